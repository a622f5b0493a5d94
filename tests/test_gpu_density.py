"""Clouds of less than a point to dozens of points a cell, whose chunks are laid
out differently (one wavefront, rows, band order), through the one-kernel substep
of a single case and of batches in both storages, with points that leave their
boxes: against the CPU oracle."""
import ctypes

import numpy as np
import pytest

import oracle
from icempm_amd import MODE_FAST, Model, SimParams
from icempm_amd._lib import BATCH_F32, BATCH_F64, check_ctx
from icempm_amd.batch import Batch, batch_cases, ingest_cases

pytestmark = pytest.mark.gpu


def of_density(state, d, vx, vy):
    """The state's block (four points a cell) stretched or squeezed to d a cell, off
    the walls and the disc, moving at (vx, vy) cells a substep, with a smooth strain
    that leaves it intact and a few crushed points."""
    p, soa = state[0].copy(), state[1].copy()
    n, h, s = p.nPts, p.cellsize, (4 / d) ** 0.5
    unit = h / p.InitialTimeStep
    for r in (4, 5):
        soa[r, :n] = 6.2 * h + (soa[r, :n] - soa[r, :n].min()) * s
    x, y = ((soa[r, :n] - soa[r, :n].min()) / np.ptp(soa[r, :n]) for r in (4, 5))
    soa[6, :n] = (vx + 1e-5 * np.sin(2 * np.pi * x + 0.3)) * unit
    soa[7, :n] = (vy + 1e-5 * np.cos(2 * np.pi * y)) * unit
    soa[8, :n] += 1e-5 * np.cos(2 * np.pi * y)
    soa[0].view(np.uint8)[: n : 97] = 1
    p.indenter_x = p.indenter_x_initial = -1.0
    return p, soa


def run_oracle(p0, soa0, nsub):
    p = SimParams()
    ctypes.memmove(ctypes.byref(p), ctypes.byref(p0), ctypes.sizeof(SimParams))
    pts = soa0.copy()
    hist, err = oracle.run(p, pts, oracle.new_grid(p), np.zeros(2 * p.n_indenter_subdivisions), nsub)
    assert err == 0
    return hist, pts


def check(got, ref, n, pos, vel, fe):
    assert np.array_equal(got[0].view(np.uint8)[:n], ref[0].view(np.uint8)[:n])
    for rows, tol in (((4, 5), pos), ((6, 7), vel)):
        scale = max(np.abs(ref[r, :n]).max() for r in rows)
        for r in rows:
            assert np.abs(got[r, :n] - ref[r, :n]).max() <= tol * scale, r
    for r in (8, 9, 10, 11):
        assert np.abs(got[r, :n] - ref[r, :n]).max() <= fe, r


# The oracle's own sensitivity over 20 substeps.  At (0.25, 0.1) cells a substep a
# relative 1e-15 of positions and velocities grows to at most 5e-15 of the
# positions, 5e-14 of the velocities and 1e-14 of Fe (which strains by 2e-5); at
# (0.01, 0.004) a relative 6e-8 of the velocities, the rounding of FP32 storage, to
# 2e-10, 5e-8 and 1e-8.  Rounding enters in each of the 20 substeps: twenty times
# as much, and a margin of five to ten.
F64 = dict(pos=1e-12, vel=1e-11, fe=2e-12)
F32 = dict(pos=4e-8, vel=1e-5, fe=1e-6)
DENSITIES = [0.7, 1.0, 2.0, 5.5, 6.5, 9.0, 25.0, 60.0]


@pytest.mark.parametrize("density", DENSITIES)
@pytest.mark.parametrize("precision,v,tol", [(BATCH_F64, (0.25, 0.1), F64), (BATCH_F32, (0.01, 0.004), F32)],
                         ids=["f64", "f32"])
def test_batch(gpu_available, precision, v, tol, density):
    print("density, batch", precision, density, flush=True)
    cases = batch_cases(3, 700, 1200, seed=22)
    states = [of_density(s, density, *v) for s in ingest_cases(cases)]
    b = Batch(precision)
    for c, s in zip(cases, states):
        b.add_state(c, *s)
    b.finalize()
    b.run(3)
    b.run(9)
    b.resort()
    b.checkpoint()
    b.run(5)
    b.set_tuning(chunk=64)
    b.restore()
    b.run(8)
    assert b.error_flag() == 0
    for c, (p, soa) in enumerate(states):
        check(b.points(c), run_oracle(p, soa, 20)[1], p.nPts, **tol)
    b.close()


@pytest.mark.parametrize("density", DENSITIES)
def test_single(gpu_available, density):
    print("density, single", density, flush=True)
    case = batch_cases(1, 1200, 1200, seed=23)[0]
    (p, soa), = (of_density(s, density, 0.25, 0.1) for s in ingest_cases([case]))
    m = Model(MODE_FAST)
    m.load_case(case)
    m.prms.indenter_x = m.prms.indenter_x_initial = p.indenter_x_initial
    m.host_points()[:] = soa
    check_ctx(m._H.icempm_transfer_points_to_device(m.ctx), m.ctx)
    m.run(20)
    assert m.error_flag() == 0
    check(m.points(), run_oracle(p, soa, 20)[1], p.nPts, **F64)
