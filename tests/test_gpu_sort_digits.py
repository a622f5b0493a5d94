"""The radix sort's ranks within wavefronts, tiles and 8-bit digits: the order
must be the oracle's stable order at the edges of a wavefront's 64 and 512 keys
and of a tile's 2048, with equal keys, few and all four digits, and both signs."""
import numpy as np
import pytest

import oracle
from icempm_amd import MODE_FAST, Model

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model(gpu_available):
    m = Model(MODE_FAST)
    yield m
    m.close()


@pytest.mark.parametrize("lo,hi,gx", [(3, 4, 8), (1, 15, 16), (0, 300, 256), (0, 1000, 1 << 14), (-1000, 1000, 1 << 20)])
def test_order_at_the_edges(model, lo, hi, gx):
    for n in (2, 63, 64, 65, 511, 513, 2047, 2049, 33000):
        print("sort", lo, hi, gx, n, flush=True)
        rng = np.random.default_rng(n)
        xy = (rng.integers(lo, hi, size=(n, 2)) + 0.75).astype(np.float32)
        g = np.arange(n).astype(np.int16)
        sx, sg = model.sort_raw_points(xy, g, 1.0, gx)
        order = oracle.stable_order(oracle.cell_keys_f32(xy, 1.0, gx))
        assert np.array_equal(sx, xy[order])
        assert np.array_equal(sg, g[order])
