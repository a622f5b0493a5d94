"""The host code's refusals and its way out of failed allocations, without a
GPU: the library runs on a stand-in for the HIP runtime (tests/cpp/fake_hip.cpp)
that counts the launches and fails allocations on request.  What these calls
must not do is launch a kernel on arrays that are not there."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = r"""
import ctypes, sys
import numpy as np
sys.path.insert(0, ROOT)
from icempm_amd import SimParams, _lib
from icempm_amd._lib import *
F = ctypes.CDLL(None)
F.fake_hip_live_bytes.restype = F.fake_hip_launches.restype = F.fake_hip_nulls.restype = ctypes.c_long
F.fake_hip_pending_failure.restype = ctypes.c_long
H = _lib.hip()

def fail_at(k):
    F.fake_hip_fail_at(ctypes.c_long(k))

def launches(part):
    return F.fake_hip_launches(part.encode())

def params(n, gx=64, gy=32):
    p = SimParams()
    _lib.host().icempm_simparams_reset(ctypes.byref(p))
    p.GridX, p.GridY, p.GridTotal, p.nPts, p.nPtsPitch = gx, gy, gx * gy, n, (n + 63) // 64 * 64
    p.cellsize, p.InitialTimeStep = 0.01, 1e-6
    p.cellsize_inv, p.Dp_inv = 1. / p.cellsize, 4. / (p.cellsize * p.cellsize)
    p.ParticleVolume, p.ParticleMass = 1e-4 / 4, 1e-4 / 4 * 900
    return p

def soa(p):
    s = np.zeros((16, p.nPtsPitch))
    i = np.arange(p.nPts)
    s[3, :p.nPts] = s[8, :p.nPts] = s[11, :p.nPts] = 1
    s[4, :p.nPts] = (4 + 0.5 * (i % 80)) * p.cellsize
    s[5, :p.nPts] = (4 + 0.5 * (i // 80)) * p.cellsize
    return s

def load(ctx, n):
    p = params(n)
    assert H.icempm_update_constants(ctx, ctypes.byref(p), ctypes.sizeof(p)) == 0
    return p
def setup(mode):
    ctx = ctypes.c_void_p()
    assert H.icempm_create(ctypes.byref(ctx)) == 0
    assert H.icempm_set_mode(ctx, mode) == 0
    p = load(ctx, 300)
    pg, pp = ctypes.c_size_t(), ctypes.c_size_t()
    hp, hf = (ctypes.POINTER(ctypes.c_double)() for _ in range(2))
    assert H.icempm_allocate_arrays(ctx, p.GridTotal, 9000, 2 * p.n_indenter_subdivisions, ctypes.byref(pg),
                                    ctypes.byref(pp), ctypes.byref(hp), ctypes.byref(hf)) == 0
    return ctx
def run(ctx, n):
    t = ctypes.c_double(0)
    return H.icempm_run_substeps(ctx, 0, n, ctypes.byref(t), ctypes.c_double(0), ctypes.c_double(0), 1)
def batch(precision, n=700, finalize=True):
    b = ctypes.c_void_p()
    assert H.icempm_batch_create(ctypes.byref(b), precision) == 0
    p = params(n)
    a = soa(p)
    assert H.icempm_batch_add_case(b, ctypes.byref(p), ctypes.sizeof(p),
                                   a.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), p.nPtsPitch) == 0
    if finalize:
        assert H.icempm_batch_finalize(b) == 0
    return b, p
"""


@pytest.fixture(scope="module")
def fake_hip(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-o", so,
                    os.path.join(ROOT, "tests", "cpp", "fake_hip.cpp")], check=True)

    def run(body):
        preload = ":".join(x for x in (so, os.environ.get("LD_PRELOAD")) if x)
        r = subprocess.run([sys.executable, "-c", f"ROOT = {ROOT!r}\n{PRELUDE}\n{body}"], timeout=120,
                           env=dict(os.environ, LD_PRELOAD=preload), capture_output=True, text=True)
        assert r.returncode == 0 and "passed" in r.stdout, r.stdout + r.stderr
    return run


@pytest.mark.parametrize("precision", ["BATCH_F64", "BATCH_F32"])
def test_read_points_of_a_batch_that_is_not_finalized(fake_hip, precision):
    """The points of a batch before finalize, or after a finalize that failed
    at any of its allocations: refused, and nothing launched."""
    fake_hip(f"""
def refused(b, p):
    out = np.zeros((16, p.nPtsPitch))
    before = launches("")
    rc = H.icempm_batch_read_points(b, 0, out.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), p.nPtsPitch)
    assert rc == ICEMPM_E_STATE and b"not finalized" in H.icempm_batch_last_error(b), rc
    assert launches("") == before

b, p = batch({precision}, finalize=False)
refused(b, p)
H.icempm_batch_destroy(b)
for k in range(100):
    b, p = batch({precision}, finalize=False)
    fail_at(k)
    rc = H.icempm_batch_finalize(b)
    hit = F.fake_hip_pending_failure() < 0
    fail_at(-1)
    if not hit:
        break
    assert rc == ICEMPM_E_HIP
    refused(b, p)
    H.icempm_batch_destroy(b)
assert rc == 0 and k > 8
print("passed")
""")


def test_sort_after_a_failed_allocation(fake_hip):
    """A sort that fails at any of its allocations leaves none of its scratch
    taken for granted: a smaller one afterwards sorts with a workspace."""
    fake_hip("""
def sort(ctx, n):
    xy, g = np.ones((n, 2), np.float32), np.zeros(n, np.int16)
    return H.icempm_sort_raw_points(ctx, xy.ctypes.data_as(ctypes.POINTER(ctypes.c_float)),
                                    g.ctypes.data_as(ctypes.POINTER(ctypes.c_int16)), n, ctypes.c_double(100.), 64)
for k in range(20):
    ctx = ctypes.c_void_p()
    assert H.icempm_create(ctypes.byref(ctx)) == 0
    assert sort(ctx, 5000) == 0
    fail_at(k)
    rc = sort(ctx, 100000)
    hit = F.fake_hip_pending_failure() < 0
    fail_at(-1)
    if not hit:
        break
    assert rc == ICEMPM_E_HIP
    for arg in (0, 2):   # the keys, the workspace
        F.fake_hip_watch(b"k_minmax_key", arg)
        before = launches("k_minmax_key")
        assert sort(ctx, 5000) == 0
        assert launches("k_minmax_key") > before and F.fake_hip_nulls() == 0, (k, arg)
    H.icempm_destroy(ctx)
assert rc == 0 and k >= 3
print("passed")
""")


def test_run_after_a_failed_allocation(fake_hip):
    """The same for runs: after one that fails at any of its allocations, a
    shorter one on fewer points has its force history, chunk table and grids."""
    fake_hip("""
# kernels and the arguments that must be there
PRESENT = [("k_fill_f64", 0), ("k_update", 4), ("k_particles_wave", 3), ("k_batch_substep", 0), ("k_batch_substep", 11),
           ("k_chunk_boxes", 5), ("k_pack", 3), ("k_minmax_key", 2), ("k_node_fold", 2), ("k_node_fold", 3),
           ("k_node_fold", 4), ("k_node_fold", 5)]
seen = set()
for mode, short, long in ((MODE_FAST, 40, 4000), (MODE_ORDERED, 4, 4000)):
    for k in range(40):
        for name, arg in PRESENT:
            ctx = setup(mode)
            assert run(ctx, short) == 0
            load(ctx, 9000)
            fail_at(k)
            run(ctx, long)   # may also go by another path
            hit = F.fake_hip_pending_failure() < 0
            fail_at(-1)
            load(ctx, 300)
            F.fake_hip_watch(name.encode(), arg)
            before = launches(name)
            assert run(ctx, short) == 0, (mode, k)
            if launches(name) > before:
                seen.add(name)
            assert F.fake_hip_nulls() == 0, (mode, k, name, arg)
            H.icempm_destroy(ctx)
        if not hit:
            break
    assert k > 2
assert seen == {name for name, _ in PRESENT}, seen
print("passed")
""")


@pytest.mark.parametrize("precision", ["BATCH_F64", "BATCH_F32"])
def test_batch_after_a_failed_allocation(fake_hip, precision):
    """A re-sort, a finer chunk table, a checkpoint, a readback or a run that
    fails at any of its allocations can be asked for again, and the substeps in
    between have their chunk table."""
    fake_hip(f"""
def calls(b, p):
    out = np.zeros((16, p.nPtsPitch))
    return {{"resort": lambda: H.icempm_batch_resort(b),
             "chunks": lambda: H.icempm_batch_set_tuning(b, BATCH_TUNE_CHUNK, 64),
             "checkpoint": lambda: H.icempm_batch_checkpoint(b) or H.icempm_batch_restore(b),
             "points": lambda: H.icempm_batch_read_points(b, 0, out.ctypes.data_as(ctypes.POINTER(ctypes.c_double)),
                                                          p.nPtsPitch),
             "run": lambda: H.icempm_batch_run(b, 20, 0)}}
# kernels of what comes after, and the argument that must be there
PRESENT = {{"resort": [("k_minmax_key", 0), ("k_minmax_key", 2), ("k_batch_permute", 4), ("k_batch_substep", 0)],
            "chunks": [("k_batch_cells", 6), ("k_batch_substep", 0)], "checkpoint": [("k_batch_substep", 0)],
            "points": [("k_read_points", 4)], "run": [("k_batch_substep", 0), ("k_batch_substep", 11)]}}
for call, watch in PRESENT.items():
    for name, arg in watch:
        for k in range(20):
            b, p = batch({precision}, n=3000)
            fail_at(k)
            rc = calls(b, p)[call]()
            hit = F.fake_hip_pending_failure() < 0
            fail_at(-1)
            if hit:   # (a chunk table can be had without rearranging the points)
                assert rc == ICEMPM_E_HIP or call == "chunks", (call, k, rc)
            F.fake_hip_watch(name.encode(), arg)
            before = launches(name)
            assert H.icempm_batch_run(b, 8, 0) == 0
            assert calls(b, p)[call]() == 0, (call, k, H.icempm_batch_last_error(b))
            assert H.icempm_batch_run(b, 8, 0) == 0
            assert (launches(name) > before or rc == 0) and F.fake_hip_nulls() == 0, (call, k, name, arg)
            H.icempm_batch_destroy(b)
            if not hit:
                break
        assert not hit and k > 0, (call, k)
print("passed")
""")


def test_ordered_run_after_a_failed_launch(fake_hip):
    """An ORDERED run that fails between making the cells' lists and folding them
    leaves points in the lists: the next call clears them before it adds its own."""
    fake_hip("""
def fills(call, *args):
    before = launches("k_fill_i32")
    rc = call(*args)
    return rc, launches("k_fill_i32") - before
for fails in ("k_particles_wave", "k_node_fold", "k_point_records"):
    for again in (lambda c: run(c, 4), H.icempm_p2g):
        ctx = setup(MODE_ORDERED)
        assert run(ctx, 4) == 0
        rc, usual = fills(again, ctx)
        assert rc == 0
        F.fake_hip_fail_launch(fails.encode(), ctypes.c_long(0))
        assert run(ctx, 4) == ICEMPM_E_HIP
        rc, now = fills(again, ctx)
        assert rc == 0 and now == usual + 2, (fails, now, usual)
        assert fills(again, ctx) == (0, usual)
        H.icempm_destroy(ctx)
print("passed")
""")


def test_new_constants_keep_the_order_of_the_points(fake_hip):
    """The band order of a longer FAST run depends on the points and the grid
    alone: constants uploaded between runs do not have it made again, points do,
    and so do another point count and another grid."""
    fake_hip("""
def plans(ctx, change):
    before = launches("k_slots")
    assert change() == 0 and run(ctx, 40) == 0
    return launches("k_slots") - before
def constants(**kw):
    p = params(300, **{k: kw.pop(k) for k in ("gx", "gy") if k in kw})
    for name, value in kw.items():
        setattr(p, name, value)
    return lambda: H.icempm_update_constants(ctx, ctypes.byref(p), ctypes.sizeof(p))
ctx = setup(MODE_FAST)
assert plans(ctx, lambda: 0) == 1 and plans(ctx, lambda: 0) == 0
assert plans(ctx, constants()) == 0
assert plans(ctx, constants(IceTensileStrength=2e6, IndVelocity=0.3, InitialTimeStep=2e-6)) == 0
assert plans(ctx, constants(nPts=299)) == 1
assert plans(ctx, constants()) == 1
assert plans(ctx, lambda: H.icempm_transfer_points_to_device(ctx)) == 1
assert plans(ctx, constants(gx=32, gy=64)) == 1
assert plans(ctx, constants(gx=32, gy=64, cellsize=0.02, cellsize_inv=1. / 0.02, Dp_inv=4. / (0.02 * 0.02))) == 1
print("passed")
""")


def test_strengths_of_the_one_kernel_substep(fake_hip):
    """A negative shear strength puts the tension line below every q, which the
    one-kernel substep's comparison of squares does not hold for: such a run takes
    the grid update and the particle pass, others of its length the one kernel."""
    fake_hip("""
for shear, one in ((1e6, True), (0., True), (-1e6, False)):
    ctx = setup(MODE_FAST)
    p = params(300)
    p.IceCompressiveStrength, p.IceTensileStrength, p.IceShearStrength = 1e7, 1e6, shear
    assert H.icempm_update_constants(ctx, ctypes.byref(p), ctypes.sizeof(p)) == 0
    before = launches("k_batch_substep")
    assert run(ctx, 40) == 0
    assert (launches("k_batch_substep") > before) == one, shear
    H.icempm_destroy(ctx)
print("passed")
""")
