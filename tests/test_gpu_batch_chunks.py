"""Batches with smaller chunks (64 and 128 points: workgroups of one and two
wavefronts), set before the first run and between runs, with points that leave
their boxes, per-grain strengths and a re-sort in between: against the CPU oracle."""
import ctypes

import numpy as np
import pytest

import oracle
from icempm_amd import SimParams
from icempm_amd._lib import BATCH_F32, BATCH_F64
from icempm_amd.batch import Batch, batch_cases, ingest_cases

pytestmark = pytest.mark.gpu


def run_oracle(p0, soa0, nsub):
    p = SimParams()
    ctypes.memmove(ctypes.byref(p), ctypes.byref(p0), ctypes.sizeof(SimParams))
    pts = soa0.copy()
    hist, err = oracle.run(p, pts, oracle.new_grid(p), np.zeros(2 * p.n_indenter_subdivisions), nsub)
    assert err == 0
    return hist, pts


# The oracle's own sensitivity over 20 substeps: a relative 1e-15 of the positions
# and velocities grows to 6e-14 of a row's largest value, 1e-7 of the velocities
# to 1e-5.  FP64 storage rounds at ~1e-15 a substep (1e-11 with a margin), FP32
# storage at 6e-8 (1e-4).
@pytest.mark.parametrize("precision,tol", [(BATCH_F64, 1e-11), (BATCH_F32, 1e-4)], ids=["f64", "f32"])
@pytest.mark.parametrize("vx,vy", [(0.3, 0.0), (0.05, 0.25)], ids=["right", "up"])
@pytest.mark.parametrize("sizes", [(64, 64, 64), (128, 128, 128), (256, 64, 128), (64, 256, 64)],
                         ids=["64", "128", "256-64-128", "64-256-64"])
def test_chunk_sizes(gpu_available, precision, tol, vx, vy, sizes):
    print("chunks", precision, vx, vy, sizes, flush=True)
    cases = batch_cases(3, 700, 3000, seed=21)
    states = []
    for p, soa in ingest_cases(cases):
        unit = p.cellsize / p.InitialTimeStep
        soa[6, :p.nPts], soa[7, :p.nPts] = vx * unit, vy * unit
        soa[0].view(np.uint8)[p.nPtsPitch:p.nPtsPitch + 2 * p.nPts].view(np.int16)[:] = np.arange(p.nPts) % 700
        p.GrainVariability = 0.5
        states.append((p, soa))
    b = Batch(precision)
    for c, s in zip(cases, states):
        b.add_state(c, *s)
    b.set_tuning(chunk=sizes[0])
    b.finalize()
    b.run(3)
    b.set_tuning(chunk=sizes[1])
    b.run(10)
    b.resort()
    b.set_tuning(chunk=sizes[2])
    b.run(7)
    assert b.error_flag() == 0
    for c, (p, soa) in enumerate(states):
        _, ref = run_oracle(p, soa, 20)
        got, n = b.points(c), p.nPts
        assert np.array_equal(got[0].view(np.uint8)[:n], ref[0].view(np.uint8)[:n])
        for r in (4, 5, 6, 7, 8, 9, 10, 11):
            scale = np.abs(ref[r, :n]).max()
            assert np.abs(got[r, :n] - ref[r, :n]).max() <= tol * scale, (c, r)
    b.close()
