"""Readback of a batch's cases: the rows a case came in with, each point at its
own index, at sizes around a wavefront and a workgroup, with a wider pitch than
the points need."""
import numpy as np
import pytest

from icempm_amd import SimParams
from icempm_amd._lib import BATCH_F32, BATCH_F64
from icempm_amd.batch import Batch, batch_cases, ingest_cases

pytestmark = pytest.mark.gpu


def cut(state, n, extra):
    """The first n points of a state, the rest of the row undefined."""
    p = SimParams.from_buffer_copy(state[0])
    soa = state[1]
    pitch = (n + 63) // 64 * 64 + extra
    out = np.full((16, pitch), 7.0)
    out[1:, :n] = soa[1:, :n]
    rng = np.random.default_rng(n)
    out[6:16, :n] += 1e-3 * rng.standard_normal((10, n))
    out[3, :n] += 1e-3 * rng.standard_normal(n)
    u8 = out[0].view(np.uint8)
    u8[:n] = rng.integers(0, 2, n)
    u8[pitch:pitch + 2 * n].view(np.int16)[:] = rng.integers(-40, 1000, n)
    p.nPts, p.nPtsPitch = n, pitch
    return p, out


@pytest.mark.parametrize("precision", [BATCH_F64, BATCH_F32], ids=["f64", "f32"])
@pytest.mark.parametrize("grains", [0.0, 0.5], ids=["uniform", "grains"])
def test_points_come_back(gpu_available, precision, grains):
    cases = batch_cases(5, 700, 3000, seed=3)
    sizes = ((1, 0), (63, 64), (64, 0), (257, 192), (640, 64))
    states = [cut(s, n, e) for s, (n, e) in zip(ingest_cases(cases), sizes)]
    b = Batch(precision)
    for c, s in zip(cases, states):
        s[0].GrainVariability = grains
        b.add_state(c, *s)
    b.finalize()
    for c, (p, soa) in enumerate(states):
        n, pitch = p.nPts, p.nPtsPitch
        print("read", precision, grains, n, pitch, flush=True)
        got, ref = b.points(c), soa.copy()
        ref[1:3] = 0        # P and Q
        ref[:, n:] = 0
        assert np.array_equal(got[0].view(np.uint8)[:n], soa[0].view(np.uint8)[:n])
        ids = soa[0].view(np.uint8)[pitch:pitch + 2 * n]
        # a batch without per-grain strengths keeps ids in its FP32 records only
        if grains or precision == BATCH_F32:
            assert np.array_equal(got[0].view(np.uint8)[pitch:pitch + 2 * n], ids)
        if precision == BATCH_F32:
            # 48-bit fixed point: at most half of 2^-48 of 32768 cells, and two roundings
            assert np.abs(got[4:6] - ref[4:6]).max() <= p.cellsize * 2.0 ** -33
            for r in (3, 8, 11):
                ref[r, :n] = (ref[r, :n] - 1).astype(np.float32).astype(np.float64) + 1.0
            for r in (6, 7, 9, 10, 12, 13, 14, 15):
                ref[r] = ref[r].astype(np.float32)
            ref[4:6] = got[4:6]
        assert np.array_equal(got[1:], ref[1:])
    b.close()
