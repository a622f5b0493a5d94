"""The contact forces of ORDERED mode where cellsize_inv is not 1 / cellsize: the
points' cells follow the one, the nodes' places and the disc the other.  Bit for
bit against the CPU oracle."""
import numpy as np
import pytest

import oracle
from icempm_amd import INDENT_TINY, MODE_ORDERED, Model, SimParams, configure_params, lattice_points
from icempm_amd._lib import check_ctx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [1.0, 0.5, 0.3])
def test_forces_follow_the_nodes(gpu_available, scale):
    print("ordered force", scale, flush=True)
    m = Model(MODE_ORDERED)
    configure_params(m.prms, INDENT_TINY)
    xy, _ = lattice_points(INDENT_TINY)
    grains = np.zeros(xy.shape[0], np.int16)
    m.load_raw_points(xy, grains, INDENT_TINY.volume)
    n = m.prms.nPts
    p = SimParams()
    configure_params(p, INDENT_TINY)
    pts = oracle.ingest(p, xy, grains, INDENT_TINY.volume, pitch=m.prms.nPtsPitch)
    p.nGridPitch = m.prms.nGridPitch
    for q in (p, m.prms):   # the disc on the middle of the nodes that the points reach
        q.cellsize_inv = scale / q.cellsize
        q.indenter_x = q.indenter_x_initial = scale * float(pts[4, :n].mean())
        q.indenter_y = q.indenter_y_initial = scale * float(pts[5, :n].mean())
        q.IndVelocity = 2.0
    m.prepare()
    m.host_points()[:] = pts
    check_ctx(m._H.icempm_transfer_points_to_device(m.ctx), m.ctx)
    bins = np.zeros(2 * p.n_indenter_subdivisions)
    want, err = oracle.run(p, pts, oracle.new_grid(p), bins, 3)
    got = m.run(3)
    assert err == m.error_flag() == 0
    assert np.abs(want).max() > 0
    assert np.array_equal(got, want)
    assert np.array_equal(m.bins(), bins)
    assert np.array_equal(m.points()[:, :n], pts[:, :n], equal_nan=True)
