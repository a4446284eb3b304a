"""What the library's host code does where a one-GPU machine cannot show it:
other current devices, failures half way, several threads.  Runs the host code
itself on the CPU (hostlib.py); no kernel is executed."""
import ctypes
import shutil
import threading
import time

import numpy as np
import pytest

import hostlib

P = ctypes.c_void_p


def ptr(a):
    return a.ctypes.data_as(P)


@pytest.fixture(scope="module")
def libpath(tmp_path_factory):
    return hostlib.build(str(tmp_path_factory.mktemp("hostlib")))


def opened(path):
    h = hostlib.load(path)
    assert h.phf_init() == 0, h.phf_last_error()
    return h


@pytest.fixture(scope="module")
def H(libpath):
    return opened(libpath)


@pytest.fixture
def fresh(libpath, tmp_path):
    """The library with nothing allocated yet."""
    return opened(shutil.copy(libpath, tmp_path / "fresh.so"))


@pytest.fixture(autouse=True)
def _clean(H):
    yield
    H.hr_on_launch(None)
    H.hr_fail(b"", -1)
    H.hr_fail_new(-1)
    H.hr_pin_delay_us(0)
    H.hr_set_device(0)


def system(H, n, seed=0):
    """A system of n blobs and its arrays."""
    xyw = np.random.default_rng(seed).random((3, n))
    s = P()
    rc = H.phf_system_create(ptr(xyw[0]), ptr(xyw[1]), ptr(xyw[2]), ctypes.c_int64(n),
                             ctypes.byref(s))
    assert rc == 0, H.phf_last_error()
    return s, xyw


def get(H, s, n):
    out = np.zeros((3, n))
    rc = H.phf_system_get(s, ptr(out[0]), ptr(out[1]), ptr(out[2]))
    return rc, out


@pytest.mark.parametrize("n", [100, 300000])
def test_results_on_a_thread_of_another_device(H, n):
    """Results are fetched, in one packed transfer or through the pinned slots,
    whichever device the calling thread uses, and it stays that thread's."""
    s, xyw = system(H, n)
    for dev in (1, 0, 1):
        H.hr_set_device(dev)
        rc, out = get(H, s, n)
        assert rc == 0, (dev, H.phf_last_error())
        assert H.hr_device() == dev
        assert np.array_equal(out, xyw)
    assert H.phf_system_destroy(s) == 0


def on_launch(H, **kernels):
    """kernels: name -> f(args), called for launches whose mangled name holds
    it; args[i] points to the i-th argument.  Returns what must be kept."""
    def cb(name, args):
        for k, f in kernels.items():
            if k.encode() in name:
                f(args)
    c = hostlib.LAUNCH_CB(cb)
    H.hr_on_launch(c)
    return c


def arg(args, i, t):
    return ctypes.cast(args[i], ctypes.POINTER(t)).contents


def put_i32(args, i, v):
    """*(int32_t *)argument i = v"""
    ctypes.c_int32.from_address(arg(args, i, P).value).value = v


def ring(m):
    """Start and end points of m panels on a circle."""
    t = np.linspace(0.0, 2.0 * np.pi, m + 1)
    x, y = np.cos(t), np.sin(t)
    return [np.ascontiguousarray(a) for a in (x[:-1], y[:-1], x[1:], y[1:])]


def test_rebuild_completed_on_a_thread_of_another_device(H):
    """A square body whose normal matrix does not serve takes the pivoted LU
    when its rebuild is completed, whichever device that thread uses."""
    bad = [0]
    keep = on_launch(H, chol_check=lambda a: put_i32(a, 2, bad[0]),
                     lu_first=lambda a: put_i32(a, 3, 0))
    m = 40
    g = ring(m)
    body = P()
    assert H.phf_panels_create(*map(ptr, g), ctypes.c_int64(m), 0, ctypes.c_double(0.0),
                               ctypes.byref(body)) == 0, H.phf_last_error()
    assert H.hr_launches(b"lu_first") == 0
    bad[0] = m
    assert H.phf_panels_update_async(body, *map(ptr, g)) == 0, H.phf_last_error()
    H.hr_set_device(1)
    xc, yc = np.empty(m), np.empty(m)
    rc = H.phf_panels_info(body, None, ptr(xc), ptr(yc), None)
    assert rc == 0, H.phf_last_error()
    assert H.hr_device() == 1
    assert H.hr_launches(b"lu_first") == 1
    assert H.phf_panels_destroy(body) == 0
    del keep


class RmGeom(ctypes.Structure):
    """The remesh's layout as phf_remesh.hip has it on the device."""
    _fields_ = [(k, ctypes.c_int64) for k in
                ("imin", "imax", "jmin", "jmax", "bi", "bj", "nj", "nstart", "ncell", "nscan",
                 "m")] + [(k, ctypes.c_int32) for k in ("ok", "bits", "crowded", "pad")]


@pytest.mark.parametrize("fail", ["pc_choose", "pc_compact"])
def test_step_whose_population_control_fails(H, fail):
    """A coupled step whose population control cannot run ends with an error
    and leaves the system holding the remeshed blobs."""
    from phyflow_amd._native import METHOD_DIRECT, StepInfo, StepParams, VelParams
    n, m = 50, 90
    new = np.random.default_rng(1).random((3, m))

    def layout(a):
        g = RmGeom(imin=0, jmin=0, bi=7, bj=7, nj=10, nstart=50, ncell=100, nscan=101, m=m, ok=1)
        ctypes.memmove(arg(a, 3, P).value, ctypes.byref(g), ctypes.sizeof(g))

    def gather(a):
        for k in range(3):
            ctypes.memmove(arg(a, 8 + k, P).value, new[k].ctypes.data, 8 * m)

    def copy3(a):
        for k in range(3):
            ctypes.memmove(arg(a, 4 + k, P).value, arg(a, k, P).value,
                           8 * arg(a, 3, ctypes.c_int64).value)

    keep = on_launch(H, base_bounds_final=layout, gather_cells=gather, copy3_f64=copy3)
    s, _ = system(H, n)
    vp = VelParams(METHOD_DIRECT, 0, 0, 0, 0, 35, 0.1, 2.0, 1e-6, 0.0, 0.0)
    sp = StepParams(dt=0.0, remesh=1, remesh_sigma=0.1, remesh_overlap=1.0, pc_enabled=1,
                    pc_w_threshold=1e-8, pc_total_threshold=1e-8)
    H.hr_fail(fail.encode(), 0)
    rc = H.phf_system_step_rk2(s, ctypes.byref(vp), None, ctypes.byref(sp),
                               ctypes.byref(StepInfo()))
    assert rc != 0 and b"OutOfMemory" in H.phf_last_error()
    size = ctypes.c_int64()
    assert H.phf_system_size(s, ctypes.byref(size)) == 0 and size.value == m
    rc, out = get(H, s, m)
    assert rc == 0 and np.array_equal(out, new)
    assert H.phf_system_destroy(s) == 0
    del keep


def test_concurrent_results_do_not_pin_memory(fresh):
    """Several threads that fetch large results at once pin one set of slots
    between them, free none for the next fetch to pin again, and only the one
    that pins them waits for it."""
    H = fresh
    n, threads, rounds = 300000, 6, 5
    systems = [system(H, n, seed=k) for k in range(threads)]
    barrier = threading.Barrier(threads)
    pinned, freed = H.hr_calls(b"hipHostMalloc"), H.hr_calls(b"hipHostFree")
    H.hr_pin_delay_us(1000000)
    bad, waits = [], []

    def work(k):
        s, xyw = systems[k]
        for _ in range(rounds):
            barrier.wait()
            t = time.perf_counter()
            rc, out = get(H, s, n)
            waits.append(time.perf_counter() - t)
            if rc != 0 or not np.array_equal(out, xyw):
                bad.append(k)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
    assert H.hr_calls(b"hipHostMalloc") - pinned <= 1
    assert H.hr_calls(b"hipHostFree") == freed
    assert sum(t > 0.9 for t in waits) <= 1
    for s, _ in systems:
        assert H.phf_system_destroy(s) == 0


@pytest.mark.parametrize("nb,nt,prec,sort,near", [
    (10007, 10007, 0, 1, 1),     # even sides, 1e8 pairs
    (9000, 9000, 0, 0, 0),       # fewer
    (20011, 20011, 1, 0, 1),
    (19000, 19000, 1, 0, 0),
    (50, 2100000, 0, 0, 0),      # few sources: the targets' sort is the call
    (400, 275000, 0, 0, 0),
    (1600, 68750, 0, 0, 0),
    (3200, 156250, 0, 1, 1),
    (1600, 312500, 1, 0, 0),
    (3200, 312500, 1, 0, 1),
    (1100000, 100, 0, 1, 0),     # few targets: theirs is quick, the sources' is not
    (220000, 500, 0, 1, 0),
    (800000, 600, 1, 0, 0),
    (250000, 2000, 1, 0, 1),
])
def test_which_direct_sums_sort(H, nb, nt, prec, sort, near):
    """Direct sums sort their targets, and vorticity its sources too, where
    the pairs saved are more than the sorts cost."""
    n = [H.hr_launches(k) for k in (b"direct_f64_sorted", b"rs_scatter", b"vort_near")]
    assert direct(H, nb, nt, "velocity", prec) == 0, H.phf_last_error()
    assert (H.hr_launches(b"direct_f64_sorted") > n[0]) == bool(sort)
    assert (H.hr_launches(b"rs_scatter") > n[1]) == bool(sort)
    n[1] = H.hr_launches(b"rs_scatter")
    assert direct(H, nb, nt, "vorticity", prec) == 0, H.phf_last_error()
    assert (H.hr_launches(b"vort_near") > n[2]) == bool(near)
    assert (H.hr_launches(b"rs_scatter") > n[1]) == bool(near)


@pytest.mark.parametrize("sigma,apart,sort,near", [
    (0.02, 0.0, 1, 1), (0.2, 0.0, 0, 0), (1e9, 0.0, 0, 0), (0.2, 30.0, 1, 1), (1e-9, 1e300, 1, 1)])
@pytest.mark.parametrize("nb,nt", [(20011, 20011), (5133, 90007)])
def test_sums_of_wide_kernels_do_not_sort(H, nb, nt, sigma, apart, sort, near):
    """Kernels as wide as the points' extent leave the sorted passes nothing to
    skip: every pair without the sorts, for points that are not far apart."""
    for field, prec, kernel, expect in (("velocity", 0, b"direct_f64_sorted", sort),
                                        ("vorticity", 0, b"vort_near", near),
                                        ("vorticity", 1, b"vort_near", near)):
        n = H.hr_launches(kernel), H.hr_launches(b"rs_scatter")
        assert direct(H, nb, nt, field, prec, 2 * sigma ** 2, apart) == 0, H.phf_last_error()
        assert (H.hr_launches(kernel) > n[0]) == bool(expect), field
        assert (H.hr_launches(b"rs_scatter") > n[1]) == bool(expect), field


def fmm(H, n, order):
    """One fmm2d call of n blobs in the unit square at an expansion order."""
    from phyflow_amd._native import FmmOpts
    r = np.random.default_rng(n).random((3, n))
    o = np.empty((2, n))
    return H.phf_fmm2d(ptr(r[0]), ptr(r[1]), ptr(r[2]), ctypes.c_int64(n), ptr(r[0]), ptr(r[1]),
                       ctypes.c_int64(n), 35, ctypes.c_double(0.01), ctypes.c_double(0.05),
                       ctypes.c_double(1e-6), ctypes.byref(FmmOpts(order, 32, 0, 0)), ptr(o[0]),
                       ptr(o[1]))


def unit_box(a):
    """What bbox_final writes for points in the unit square."""
    box = np.array([0.0, 1.0, 0.0, 1.0])
    ctypes.memmove(arg(a, 2, P).value, box.ctypes.data, 32)


def test_more_tree_shapes_than_a_lane_keeps(H):
    """Calls that take more tree shapes in turn than a lane keeps the tables of
    neither allocate nor free, nor wait for the device more than a call whose
    tables are there."""
    keep = on_launch(H, bbox_final=unit_box)
    names = (b"hipMalloc", b"hipFree", b"hipStreamSynchronize")

    def calls(orders):
        n = [H.hr_calls(k) for k in names]
        for p in orders:
            assert fmm(H, 4000, p) == 0, H.phf_last_error()
        return [H.hr_calls(k) - a for k, a in zip(names, n)]

    shapes = [6, 17, 9, 30, 12, 21, 7, 24, 14]
    for _ in range(4):
        calls(shapes)
    kept = calls([shapes[-1]] * len(shapes))
    assert kept[:2] == [0, 0]
    assert calls(shapes) == kept
    del keep


def test_tables_without_memory_beyond_the_arena(H):
    """A new tree shape needs no more device memory than the call's workspace:
    its tables go there when they cannot have a buffer of their own."""
    keep = on_launch(H, bbox_final=unit_box)
    assert fmm(H, 4000, 35) == 0, H.phf_last_error()
    for p in range(25, 35):
        H.hr_fail(b"hipMalloc", 0)
        assert fmm(H, 4000, p) == 0, H.phf_last_error()
    H.hr_fail(b"", -1)
    assert fmm(H, 4000, 36) == 0, H.phf_last_error()
    del keep


def direct(H, nb, nt, field, prec=0, ks=1e-4, apart=0.0):
    r = np.random.default_rng(0)
    b, t, o = r.random((3, nb)), r.random((2, nt)), np.empty((2, nt))
    t[0] += apart
    args = [ptr(b[0]), ptr(b[1]), ptr(b[2]), ctypes.c_int64(nb), ptr(t[0]), ptr(t[1]),
            ctypes.c_int64(nt), ctypes.c_double(ks), ctypes.c_int32(prec)]
    if field == "velocity":
        return H.phf_vv2par_gauss(*args, ptr(o[0]), ptr(o[1]))
    return H.phf_ww2par_gauss(*args, ptr(o[0]))


@pytest.mark.parametrize("field,nt", [("velocity", 800000), ("vorticity", 2400000)])
def test_direct_sum_without_memory_for_its_sort(fresh, field, nt):
    """A sum that would sort, but finds the device's memory taken (its second
    block here), is done as it comes."""
    H = fresh
    H.hr_fail(b"hipMalloc", 1)
    assert direct(H, 2100, nt, field) == 0, H.phf_last_error()
    assert H.phf_last_error() == b""
    assert H.hr_launches(b"direct_f64_sorted") + H.hr_launches(b"vort_near") == 0
    assert H.hr_calls(b"hipMalloc") == (2 if field == "velocity" else 3)
    # with room it does sort
    assert direct(H, 2100, nt, field) == 0, H.phf_last_error()
    assert H.hr_launches(b"direct_f64_sorted") + H.hr_launches(b"vort_near") > 0


@pytest.mark.parametrize("what", ["get", "set"])
def test_no_host_memory_for_the_workers(H, what):
    """The checks and copies that share worker threads do without them, and
    without the pinned slots, when the host has no memory for their
    bookkeeping: no exception leaves the C entry, and the data are right."""
    n = 300000
    s, xyw = system(H, n)
    for k in range(100):
        # the runtime's own objects are made in calls before this one
        assert get(H, s, n)[0] == 0
        out = np.zeros((3, n))
        o = [ptr(a) for a in out]
        x = [ptr(a) for a in xyw]
        H.hr_fail_new(k)
        if what == "get":
            rc = H.phf_system_get(s, *o)
        else:
            rc = H.phf_system_set(s, *x, ctypes.c_int64(n))
        left = H.hr_fail_new(-1)
        assert rc == 0, H.phf_last_error()
        assert np.array_equal(get(H, s, n)[1] if what == "set" else out, xyw)
        if left:
            break
    assert left and k > 1  # each of the call's allocations has failed once
    assert H.phf_system_destroy(s) == 0


def test_no_memory_to_pin(fresh):
    """Small arrays go without the pinned staging when it cannot be had."""
    H = fresh
    n = 100
    r, o = np.random.default_rng(0).random((3, n)), np.empty((2, n))
    H.hr_fail(b"hipHostMalloc", 0)
    args = [ptr(r[0]), ptr(r[1]), ptr(r[2]), ctypes.c_int64(n), ptr(r[0]), ptr(r[1]),
            ctypes.c_int64(n), ctypes.c_double(1e-4), 0, ptr(o[0]), ptr(o[1])]
    assert H.phf_vv2par_gauss(*args) == 0, H.phf_last_error()
    s, xyw = system(H, n)
    H.hr_fail(b"hipHostMalloc", 0)
    rc, out = get(H, s, n)
    assert rc == 0 and H.phf_last_error() == b"" and np.array_equal(out, xyw)
    assert H.phf_system_destroy(s) == 0


@pytest.mark.parametrize("n", [1, 512, 1024, 2048, 3072, 4096, 5120])
def test_small_results_of_touching_allocations(H, n):
    """Arrays of whole pages can be neighbours in memory and allocations of
    their own all the same."""
    s, xyw = system(H, n)
    rc, out = get(H, s, n)
    assert rc == 0, H.phf_last_error()
    assert np.array_equal(out, xyw)
    assert H.phf_system_destroy(s) == 0
