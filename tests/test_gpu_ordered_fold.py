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
