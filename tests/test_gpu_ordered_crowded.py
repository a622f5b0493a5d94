"""ORDERED P2G of cells with hundreds and thousands of points, whose fold goes by
batches of ascending indices: indices that follow each other (a histogram's first
bucket holds more than a batch) and indices from everywhere, next to cells of the
usual four.  Bit for bit against the CPU oracle."""
import numpy as np
import pytest

import oracle
from icempm_amd import INDENT_60K, MODE_ORDERED, Model, SimParams, configure_params, lattice_points
from icempm_amd._lib import check_ctx

pytestmark = pytest.mark.gpu


# points with indices in a row in one cell (256 is a batch), points from everywhere in another
@pytest.mark.parametrize("row,spread", [(256, 0), (257, 300), (3000, 0), (2000, 2500)])
def test_crowded_cells(gpu_available, row, spread):
    print("crowded", row, spread, flush=True)
    m = Model(MODE_ORDERED)
    configure_params(m.prms, INDENT_60K)
    xy, _ = lattice_points(INDENT_60K)
    grains = np.zeros(xy.shape[0], np.int16)
    m.load_raw_points(xy, grains, INDENT_60K.volume)
    n, pitch = m.prms.nPts, m.prms.nPtsPitch
    p = SimParams()
    configure_params(p, INDENT_60K)
    pts = oracle.ingest(p, xy, grains, INDENT_60K.volume, pitch=pitch)
    p.nGridPitch = m.prms.nGridPitch
    rng = np.random.default_rng(17)
    col, line = np.floor(pts[4, :n].mean() / p.cellsize), np.floor(pts[5, :n].mean() / p.cellsize)
    for k, who in enumerate((np.arange(20000, 20000 + row), rng.choice(n, spread, replace=False))):
        pts[4, who] = (col + 3 * k + rng.uniform(0.6, 1.4, who.size)) * p.cellsize
        pts[5, who] = (line + 3 * k + rng.uniform(0.6, 1.4, who.size)) * p.cellsize
    pts[6:8, :n] = 1e-3 * p.cellsize / p.InitialTimeStep * rng.standard_normal((2, n))
    m.host_points()[:] = pts
    check_ctx(m._H.icempm_transfer_points_to_device(m.ctx), m.ctx)
    want, err = oracle.run(p, pts, oracle.new_grid(p), np.zeros(2 * p.n_indenter_subdivisions), 3)
    got = m.run(3)
    assert err == m.error_flag() == 0
    assert np.array_equal(m.points()[:, :n], pts[:, :n], equal_nan=True)
    assert np.array_equal(got, want)
