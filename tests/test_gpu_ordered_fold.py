"""ORDERED P2G at every density, bit for bit against the CPU oracle: points in
cell order and shuffled, cells of four points (whole tiles), of a dozen (quarters
of tiles) and of dozens (past a cell's bucket), blocks that end inside a tile."""
import numpy as np
import pytest

import oracle
from icempm_amd import INDENT_TINY, MODE_ORDERED, Model, SimParams, configure_params, lattice_points
from icempm_amd._lib import check_ctx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("squeeze", [1.0, 1.08, 1.75, 3.5], ids=["4", "5", "12", "49"])
@pytest.mark.parametrize("shuffled", [False, True], ids=["sorted", "shuffled"])
def test_fold_matches_the_oracle(gpu_available, squeeze, shuffled):
    print("fold", squeeze, shuffled, flush=True)
    m = Model(MODE_ORDERED)
    configure_params(m.prms, INDENT_TINY)
    xy, _ = lattice_points(INDENT_TINY)
    grains = np.zeros(xy.shape[0], np.int16)
    m.load_raw_points(xy, grains, INDENT_TINY.volume)
    n, pitch = m.prms.nPts, m.prms.nPtsPitch
    p = SimParams()
    configure_params(p, INDENT_TINY)
    pts = oracle.ingest(p, xy, grains, INDENT_TINY.volume, pitch=pitch)
    p.nGridPitch = m.prms.nGridPitch
    rng = np.random.default_rng(11)
    for r in (4, 5):   # denser by squeeze^2, the block's corner in place
        pts[r, :n] = pts[r, :n].min() + (pts[r, :n] - pts[r, :n].min()) / squeeze
    pts[6:8, :n] = 1e-3 * p.cellsize / p.InitialTimeStep * rng.standard_normal((2, n))
    if shuffled:
        pts[3:, :n] = pts[3:, rng.permutation(n)]
    m.host_points()[:] = pts
    check_ctx(m._H.icempm_transfer_points_to_device(m.ctx), m.ctx)
    bins = np.zeros(2 * p.n_indenter_subdivisions)
    want, err = oracle.run(p, pts, oracle.new_grid(p), bins, 5)
    got = m.run(5)
    assert err == m.error_flag() == 0
    assert np.array_equal(m.points()[:, :n], pts[:, :n], equal_nan=True)
    assert np.array_equal(got, want)


def test_forces_of_one_run_and_of_single_substeps(gpu_available):
    """A run folds a substep's forces with the next one's P2G; the last one's, and
    those before the bins are cleared at a cycle's start, by themselves."""
    out = []
    for runs in ((11,), (1,) * 11, (4, 7)):
        m = Model(MODE_ORDERED)
        configure_params(m.prms, INDENT_TINY)
        m.prms.UpdateEveryNthStep = 4
        xy, _ = lattice_points(INDENT_TINY)
        m.load_raw_points(xy, np.zeros(xy.shape[0], np.int16), INDENT_TINY.volume)
        m.prms.indenter_x_initial += 0.02   # into the block's side
        m.prms.indenter_y -= 0.03
        hist = np.concatenate([m.run(n) for n in runs])
        out.append((hist, m.bins(), m.points()))
    assert np.abs(out[0][0]).max() > 0 and np.abs(out[0][1]).max() > 0
    for other in out[1:]:
        for a, b in zip(out[0], other):
            assert np.array_equal(a.view(np.uint64), b.view(np.uint64))
