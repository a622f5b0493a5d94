"""How exact the one-kernel substep of a single case is: as exact as the particle
pass.  Runs of one kernel differ by the order of its atomic sums alone; what a
kernel rounds differently from the other in every run shows in the difference of
their means."""
import numpy as np
import pytest

from icempm_amd import INDENT_TINY, MODE_FAST, Model, configure_params, lattice_points
from icempm_amd._lib import check_ctx

pytestmark = pytest.mark.gpu

RUNS, SUBSTEPS = 48, 2500


def runs(kind):
    """RUNS runs by one kind: velocity, Fe - I and Bp of every point at the end."""
    m = Model(MODE_FAST)
    m.set_pass_kind(kind)
    configure_params(m.prms, INDENT_TINY)
    m.prms.UpdateEveryNthStep = 10 * SUBSTEPS
    xy, _ = lattice_points(INDENT_TINY)
    m.load_raw_points(xy, np.zeros(xy.shape[0], np.int16), INDENT_TINY.volume)
    n = m.prms.nPts
    start = m.points()
    x, y = ((start[r, :n] - start[r, :n].min()) / np.ptp(start[r, :n]) for r in (4, 5))
    # smooth fields of an indentation's size
    start[6, :n] = 0.02 * np.sin(np.pi * x + 0.3) * np.cos(np.pi * y)
    start[7, :n] = 0.02 * np.cos(np.pi * x) * np.sin(2 * np.pi * y + 0.5)
    start[8, :n] += 2e-5 * np.sin(np.pi * x + 2 * np.pi * y)
    start[11, :n] -= 2e-5 * np.cos(2 * np.pi * x)
    out = []
    for _ in range(RUNS):
        m.prms.SimulationStep, m.prms.SimulationTime = 0, 0.0
        m.host_points()[:] = start
        check_ctx(m._H.icempm_transfer_points_to_device(m.ctx), m.ctx)
        m.run(SUBSTEPS)
        p = m.points()[:, :n].copy()
        p[8], p[11] = p[8] - 1, p[11] - 1
        out.append([p[6:8].ravel(), p[8:12].ravel(), p[12:16].ravel()])
    assert m.error_flag() == 0
    return out


# The means of N runs each differ, squared, by (s1^2 + s2^2) / N on the average
# where only the order of sums tells the runs apart.  The spread is that of a few
# modes of the block, not of thousands of independent values, so three times the
# average is allowed for.  Rounding that is the kernel's own, of half the size of a
# run's spread, gives seven times.
def test_no_rounding_of_its_own(gpu_available):
    print("substep rounding", flush=True)
    a, b = runs(2), runs(1)
    for k, name in enumerate(("velocity", "Fe - I", "Bp")):
        u, v = np.array([r[k] for r in a]), np.array([r[k] for r in b])
        spread = sum(((w - w.mean(0)) ** 2).sum() / (RUNS - 1) for w in (u, v))
        apart = ((u.mean(0) - v.mean(0)) ** 2).sum()
        print(name, "apart", apart / (spread / RUNS), "spread", np.sqrt(spread / 2) / np.linalg.norm(v[0]), flush=True)
        assert apart <= 3 * spread / RUNS, name
