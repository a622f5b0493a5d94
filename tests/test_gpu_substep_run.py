"""Runs of the single case through the substep kernel (FAST, default pass kind,
long enough) against the same runs through the grid update and the particle
pass: the copy in band order and back, the rotation of three grids, the
recording substep in the middle of a run, ragged chunks, strengths per grain,
points that leave their box."""
from dataclasses import replace

import numpy as np
import pytest

from icempm_amd import INDENT_60K, INDENT_TINY, MODE_FAST, Model, configure_params, lattice_points
from icempm_amd._lib import check_ctx

pytestmark = pytest.mark.gpu


def run(case, kind, moving, runs):
    m = Model(MODE_FAST)
    m.set_pass_kind(kind)
    configure_params(m.prms, case)
    m.prms.UpdateEveryNthStep = 50
    xy, _ = lattice_points(case)
    rng = np.random.default_rng(5)
    m.load_raw_points(xy, rng.integers(-40, 1000, xy.shape[0]).astype(np.int16), case.volume)
    n = m.prms.nPts
    pts = m.points()
    unit = m.prms.cellsize / m.prms.InitialTimeStep
    if moving:   # up to a tenth of a cell a substep, sheared
        pts[6, :n] = 0.02 * unit
        pts[7, :n] = 0.04 * unit * (pts[5, :n] - pts[5, :n].min()) / np.ptp(pts[5, :n])
        pts[6, : n // 97] = 0.1 * unit
    else:
        pts[6:8, :n] = 1e-3 * unit * rng.standard_normal((2, n))
    m.host_points()[:] = pts
    check_ctx(m._H.icempm_transfer_points_to_device(m.ctx), m.ctx)
    hist = [m.run(k) for k in runs]
    out = m.points()
    crushed = out[0].view(np.uint8)[:n]
    force = np.concatenate(hist)
    assert m.error_flag() == 0
    return n, out[:, :n], crushed, force


# Both add each node's terms in an order of their own, so they differ by
# rounding, which the scheme carries on.  Oracle runs of these inputs, positions
# and velocities perturbed by a relative 1e-15 at the start, end within 1e-10 of
# the largest value of their row (P, Q), 2e-11 (Bp), 4e-12 (the others) and
# 1.5e-12 of the force; rounding enters in each of the 75 substeps: a hundred
# times as much.
@pytest.mark.parametrize("case,moving", [
    (INDENT_TINY, False),
    (replace(INDENT_TINY, grain_variability=0.5), True),
    (replace(INDENT_60K, grain_variability=0.5), False),
    (INDENT_60K, True),
], ids=["tiny", "tiny-grains-moving", "60k-grains", "60k-moving"])
def test_run_matches_the_particle_pass(gpu_available, case, moving):
    print("substep run", case.name, moving, flush=True)
    runs = (60, 15)
    n, a, ca, fa = run(case, 2, moving, runs)
    _, b, cb, fb = run(case, 1, moving, runs)
    assert np.array_equal(ca, cb)
    for r in range(1, 16):
        tol = 1e-8 if r in (1, 2) else 2e-9 if r >= 12 else 4e-10
        assert np.abs(a[r] - b[r]).max() <= tol * np.abs(b[r]).max(), r
    assert np.abs(fa - fb).max() <= 1.5e-10 * np.abs(fb).max()
