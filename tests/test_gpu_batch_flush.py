"""The two ways an FP32 batch's windows reach the grid: batches of fewer than 8192
chunks add the four of a workgroup up first, larger ones take each by itself.
The same cases in a small batch and in one of more than 8192 chunks, every value
against the CPU oracle: points at rest, and a block whose points leave their
boxes."""
import ctypes

import numpy as np
import pytest

import oracle
from icempm_amd import SimParams
from icempm_amd._lib import BATCH_F32
from icempm_amd.batch import Batch, batch_cases, ingest_cases

pytestmark = pytest.mark.gpu

JOINT_CHUNKS = 8192


def run_oracle(p0, soa0, nsub):
    p = SimParams()
    ctypes.memmove(ctypes.byref(p), ctypes.byref(p0), ctypes.sizeof(SimParams))
    pts = soa0.copy()
    hist, err = oracle.run(p, pts, oracle.new_grid(p), np.zeros(2 * p.n_indenter_subdivisions), nsub)
    assert err == 0
    return pts


# The oracle's sensitivity over 20 substeps to perturbations of 1e-7 of
# the velocities is 1e-5 of a row's largest value; FP32 storage rounds at 6e-8 a
# substep.
TOL = 1e-4


@pytest.mark.parametrize("vx,vy", [(0.0, 0.0), (0.3, 0.0), (0.05, 0.25)], ids=["rest", "right", "up"])
@pytest.mark.parametrize("large", [False, True], ids=["joint", "each"])
def test_both_flushes(gpu_available, vx, vy, large):
    print("flush", vx, vy, large, flush=True)
    cases = batch_cases(3, 700, 3000, seed=21)
    states = []
    for p, soa in ingest_cases(cases):
        unit = p.cellsize / p.InitialTimeStep
        soa[6, :p.nPts], soa[7, :p.nPts] = vx * unit, vy * unit
        states.append((p, soa))
    # every pair of rows of cells is a chunk or more
    bands = sum(c.ncy // 2 for c in cases)
    copies = -(-JOINT_CHUNKS // bands) if large else 1
    b = Batch(BATCH_F32)
    for _ in range(copies):
        for c, s in zip(cases, states):
            b.add_state(c, *s)
    b.finalize()
    b.run(3)
    b.run(17)
    assert b.error_flag() == 0
    for c, (p, soa) in enumerate(states):
        ref, n = run_oracle(p, soa, 20), p.nPts
        for k in {0, copies // 2, copies - 1}:
            got = b.points(k * len(cases) + c)
            assert np.array_equal(got[0].view(np.uint8)[:n], ref[0].view(np.uint8)[:n])
            for r in (4, 5, 6, 7, 8, 9, 10, 11):
                scale = np.abs(ref[r, :n]).max()
                assert np.abs(got[r, :n] - ref[r, :n]).max() <= TOL * scale, (c, k, r)
    b.close()
