"""Batches stepped by runs of one to five substeps, whose chunks' boxes are renewed by
some of the runs only, with points that leave their boxes in between: against the CPU
oracle's one run."""
import ctypes

import numpy as np
import pytest

import oracle
from icempm_amd import SimParams
from icempm_amd._lib import BATCH_F32, BATCH_F64
from icempm_amd.batch import Batch, batch_cases, ingest_cases

pytestmark = pytest.mark.gpu


# The tolerances of test_gpu_batch_chunks: the oracle's own sensitivity over 20
# substeps to the storage's rounding; ten times that for the forces, which are made of
# differences of velocities.
@pytest.mark.parametrize("precision,tol", [(BATCH_F64, 1e-11), (BATCH_F32, 1e-4)], ids=["f64", "f32"])
@pytest.mark.parametrize("vx,vy", [(0.3, 0.0), (0.05, 0.25)], ids=["right", "up"])
@pytest.mark.parametrize("lens", [(1,) * 20, (2,) * 10, (3, 4, 1, 4, 3, 5), (1, 8, 1, 2, 2, 5, 1)],
                         ids=["ones", "twos", "threes", "mixed"])
@pytest.mark.parametrize("prepared", [False, True], ids=["captured", "prepared"])
def test_short_runs(gpu_available, precision, tol, vx, vy, lens, prepared):
    print("short runs", precision, vx, vy, lens, prepared, flush=True)
    states, cases = [], batch_cases(3, 700, 3000, seed=21)
    for p, soa in ingest_cases(cases):
        unit = p.cellsize / p.InitialTimeStep
        soa[6, :p.nPts], soa[7, :p.nPts] = vx * unit, vy * unit
        states.append((p, soa))
    b = Batch(precision)
    for c, s in zip(cases, states):
        b.add_state(c, *s)
    b.finalize()
    assert sum(lens) == 20
    last = []
    for i, n in enumerate(lens):
        if prepared:
            b.prepare(n)
        b.run(n, use_graph=prepared or i % 3 != 1)
        last.append([b.force_history(c, n) for c in range(3)])
    assert b.error_flag() == 0
    for c, (p0, soa) in enumerate(states):
        p = SimParams()
        ctypes.memmove(ctypes.byref(p), ctypes.byref(p0), ctypes.sizeof(SimParams))
        ref = soa.copy()
        hist, err = oracle.run(p, ref, oracle.new_grid(p), np.zeros(2 * p.n_indenter_subdivisions), 20)
        assert err == 0
        force = np.concatenate([h[c] for h in last])
        assert np.abs(force - np.asarray(hist).reshape(force.shape)).max() <= 10 * tol * max(1.0, np.abs(hist).max())
        got, n = b.points(c), p.nPts
        assert np.array_equal(got[0].view(np.uint8)[:n], ref[0].view(np.uint8)[:n])
        for r in (4, 5, 6, 7, 8, 9, 10, 11):
            scale = np.abs(ref[r, :n]).max()
            assert np.abs(got[r, :n] - ref[r, :n]).max() <= tol * scale, (c, r)
    b.close()
