"""Readback of a case of more points than the scratch holds (2^16): part by part,
every point at its own index, the padding zero."""
import numpy as np
import pytest

from icempm_amd import SimParams
from icempm_amd._lib import BATCH_F32, BATCH_F64
from icempm_amd.batch import Batch, batch_cases, ingest_cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,n", [(BATCH_F64, (1 << 20) + 1), (BATCH_F32, (1 << 21) + 70), (BATCH_F64, 1 << 16),
                                         (BATCH_F32, (1 << 16) + 1)], ids=["f64", "f32", "f64-one", "f32-two"])
def test_points_come_back_in_parts(gpu_available, precision, n):
    print("read parts", precision, n, flush=True)
    cases = batch_cases(2, 700, 3000, seed=3)
    small, big = ingest_cases(cases)
    p = SimParams.from_buffer_copy(big[0])
    pitch = (n + 63) // 64 * 64 + 64
    rng = np.random.default_rng(7)
    soa = np.full((16, pitch), 7.0)
    soa[1:, :n] = big[1][1:, rng.integers(0, big[0].nPts, n)]
    soa[6:16, :n] += 1e-3 * rng.standard_normal((10, n))
    u8 = soa[0].view(np.uint8)
    u8[:n] = rng.integers(0, 2, n)
    u8[pitch:pitch + 2 * n].view(np.int16)[:] = rng.integers(-40, 1000, n)
    p.nPts, p.nPtsPitch, p.GrainVariability = n, pitch, 0.5
    b = Batch(precision)
    b.add_state(cases[0], *small)
    b.add_state(cases[1], p, soa)
    b.finalize()
    got = b.points(1)
    g8 = got[0].view(np.uint8)
    assert np.array_equal(g8[:n], u8[:n]) and np.array_equal(g8[pitch:pitch + 2 * n], u8[pitch:pitch + 2 * n])
    assert not g8[n:pitch].any() and not g8[pitch + 2 * n:].any()
    assert not got[1:3].any() and not got[3:, n:].any()
    for r in range(3, 16):
        a, c = got[r, :n], soa[r, :n]
        if precision == BATCH_F32 and r in (4, 5):
            # 48-bit fixed point: at most half of 2^-48 of 32768 cells, and two roundings
            assert np.abs(a - c).max() <= p.cellsize * 2.0 ** -33
            continue
        if precision == BATCH_F32:
            c = (c - 1).astype(np.float32).astype(np.float64) + 1.0 if r in (3, 8, 11) else c.astype(np.float32)
        assert np.array_equal(a, c), r
    assert np.array_equal(b.points(0)[3:4], small[1][3:4])
    b.close()
