"""The learned map's points far from their chunk.  Crushed points whose
projection the map kernel does are not scattered by the substep kernel, but the
nodes they touch have to be cleared, and their contact counted, all the same:
three such points of one chunk fly apart, until no box holds them, far outside
what the other chunks touch, one through where another has been.  With a tolerance
that no proposal passes, the learned map is the exact one: against the CPU
oracle."""
import ctypes

import numpy as np
import pytest

import oracle
from icempm_amd import SimParams
from icempm_amd._lib import BATCH_F32, BATCH_F64
from icempm_amd.batch import Batch, batch_cases, ingest_cases
from icempm_amd.learned import init_params

pytestmark = pytest.mark.gpu


def with_flyers(state):
    """Three of the block's points put six cells above it, crushed and past the
    tension branch's limit (Jp_inv < 1, so they project in every substep): one
    going up, one right, one crossing the first one's path later."""
    p, soa = state[0].copy(), state[1].copy()
    n, h = p.nPts, p.cellsize
    unit = h / p.InitialTimeStep
    row, col = np.floor(soa[5, :n].max() / h) + 6, np.floor(soa[4, :n].mean() / h)
    for k, (dx, vx, vy) in enumerate([(0, 0.0, 0.3), (20, 0.22, 0.0), (-8, 0.1, 0.28)]):
        i = n - 1 - 40 * k
        soa[4, i], soa[5, i] = (col + dx + 0.3) * h, (row + 0.4) * h
        soa[6, i], soa[7, i] = vx * unit, vy * unit
        soa[3, i] = 0.98
        soa[0].view(np.uint8)[i] = 1
    return p, soa


def run_oracle(p0, soa0, nsub):
    p = SimParams()
    ctypes.memmove(ctypes.byref(p), ctypes.byref(p0), ctypes.sizeof(SimParams))
    pts = soa0.copy()
    hist, err = oracle.run(p, pts, oracle.new_grid(p), np.zeros(2 * p.n_indenter_subdivisions), nsub)
    assert err == 0
    return pts


# The oracle's own sensitivity over these 90 substeps, from perturbed inputs: a
# relative 1e-15 of velocity and Fe grows to at most 5e-14 of a row's largest
# value, 6e-8 to 1.5e-6.  Rounding of those sizes (FP64, FP32 storage) enters in
# each of the 90 substeps: a hundred times as much, and for FP64, where a
# substep rounds many times, twenty times that.
@pytest.mark.parametrize("precision,tol", [(BATCH_F64, 1e-10), (BATCH_F32, 1.5e-4)], ids=["f64", "f32"])
def test_deferred_points_far_from_their_chunk(gpu_available, precision, tol):
    print("deferred points", precision, flush=True)
    cases = batch_cases(2, 1500, 2500, seed=33)
    states = [with_flyers(s) for s in ingest_cases(cases)]
    b = Batch(precision)
    for c, s in zip(cases, states):
        b.add_state(c, *s)
    b.finalize()
    norm = np.array([0, 0, 0, 0, 0.5, 3e-5, 3e-5, 5e-3, 1, 0.5, 0, 0, 0, 3e-5, 3e-5, 5e-5], np.float32)
    b.set_learned(init_params(7), norm, tol=-1.0)
    for n in (3, 87):
        b.run(n)
    assert b.error_flag() == 0
    accepted, fell_back, _ = b.map_stats()
    assert accepted == 0 and fell_back >= 2 * 3 * 90
    for c, (p, soa) in enumerate(states):
        ref, got, n = run_oracle(p, soa, 90), b.points(c), p.nPts
        assert np.array_equal(got[0].view(np.uint8)[:n], ref[0].view(np.uint8)[:n])
        for r in (4, 5, 6, 7, 8, 9, 10, 11):
            scale = np.abs(ref[r, :n]).max()
            assert np.abs(got[r, :n] - ref[r, :n]).max() <= tol * scale, (c, r)
    b.close()
