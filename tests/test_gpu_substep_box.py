"""The batched substep's boxes: a workgroup keeps its points' box of nodes for
several substeps, so fast points leave it in between.  The points that gather
and scatter outside it (up to seven a wavefront through its patch, more node
by node), the chunks of every length and the grids' clearing behind a moving
block, against the CPU oracle."""
import ctypes

import numpy as np
import pytest

import oracle
from icempm_amd import SimParams
from icempm_amd._lib import BATCH_F32, BATCH_F64
from icempm_amd.batch import Batch, batch_cases, ingest_cases

pytestmark = pytest.mark.gpu


def with_velocity(state, vx, vy, shear):
    """The state with every point moving at (vx, vy) cells a substep, sheared
    by `shear` cells a substep over a cell's height (its Bp says so too)."""
    p, soa = state[0].copy(), state[1].copy()
    n, unit = p.nPts, p.cellsize / p.InitialTimeStep
    soa[6, :n] = unit * vx + (soa[5, :n] - soa[5, :n].mean()) / p.cellsize * shear * unit
    soa[7, :n] = unit * vy
    soa[13, :n] = shear / p.InitialTimeStep
    return p, soa


def run_oracle(p0, soa0, nsub):
    p = SimParams()
    ctypes.memmove(ctypes.byref(p), ctypes.byref(p0), ctypes.sizeof(SimParams))
    pts = soa0.copy()
    hist, err = oracle.run(p, pts, oracle.new_grid(p), np.zeros(2 * p.n_indenter_subdivisions), nsub)
    assert err == 0
    return hist, pts


# The oracle's own sensitivity over these 20 substeps, from perturbed inputs: a
# relative 1e-15 of the positions and velocities grows to 6e-14 of a row's
# largest value, 1e-7 of the velocities to 1e-5.  FP64 storage rounds at ~1e-15
# a substep (1e-11 with a margin), FP32 storage at 6e-8 (1e-4).
# The sheared body is FP64 only: its points are crushed, and the return map
# carries the FP32 rounding of Bp past that estimate.
@pytest.mark.parametrize("precision,tol,vx,vy,shear", [
    (BATCH_F64, 1e-11, 0.3, 0.0, 0.0), (BATCH_F64, 1e-11, 0.05, 0.25, 0.0), (BATCH_F64, 1e-11, -0.02, 0.06, 0.004),
    (BATCH_F32, 1e-4, 0.3, 0.0, 0.0), (BATCH_F32, 1e-4, 0.05, 0.25, 0.0),
], ids=["f64-right", "f64-up", "f64-shear", "f32-right", "f32-up"])
def test_points_that_leave_their_box(gpu_available, precision, tol, vx, vy, shear):
    print("box", precision, vx, vy, shear, flush=True)
    cases = batch_cases(3, 700, 3000, seed=21)
    states = [with_velocity(s, vx, vy, shear) for s in ingest_cases(cases)]
    b = Batch(precision)
    for c, s in zip(cases, states):
        b.add_state(c, *s)
    b.finalize()
    for n in (3, 17):
        b.run(n)
    assert b.error_flag() == 0
    for c, (p, soa) in enumerate(states):
        _, ref = run_oracle(p, soa, 20)
        got, n = b.points(c), p.nPts
        assert np.array_equal(got[0].view(np.uint8)[:n], ref[0].view(np.uint8)[:n])
        for r in (4, 5, 6, 7, 8, 9, 10, 11):
            scale = np.abs(ref[r, :n]).max()
            assert np.abs(got[r, :n] - ref[r, :n]).max() <= tol * scale, (c, r)
    b.close()
