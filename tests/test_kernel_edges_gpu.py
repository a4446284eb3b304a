"""Kernels at the sizes where their tiles and dispatch rules have edges,
against the CPU oracle or a float64 direct sum."""
import numpy as np
import pytest

from phyflow_amd import workloads as W
from phyflow_amd.cpp.blobs.kernels import gauss

pytestmark = pytest.mark.gpu
F64, F32C = gauss.PREC_F64, gauss.PREC_F32C


@pytest.mark.parametrize("order", [2, 11, 12, 15, 16, 19, 20, 23, 24, 31, 32, 40])
def test_multipole_orders(order, O):
    """Orders on both sides of each compiled power count.  One-box separation
    (ws = 1): the expansions of two boxes of side s at distance 2 s converge as
    (r / (2 - r))^k, r = sqrt(1/2); leaves of 0 to some 150 points."""
    n = 6001
    s = W.uniform_system(n, seed=order)
    x, y, w = s["x"] ** 2, s["y"], s["w"]  # uneven leaves
    xopt, cutoff = W.oseen_params(s["sigma"] * 0.1)
    ref = O.direct_oseen(x, y, w, x, y, xopt, cutoff)
    got = gauss.fmm2d_gpu(x, y, w, x, y, 35, xopt, cutoff, 1e-6, prec=F64, order=order, leaf=32)
    r = 0.5 ** 0.5
    assert O.rel_l2(got, ref) <= (r / (2 - r)) ** (order + 1) + 1e-12
    got = gauss.fmm2d_gpu(x, y, w, x, y, 35, xopt, cutoff, 1e-6, prec=F32C, order=order, leaf=32)
    assert O.rel_l2(got, ref) <= (r / (2 - r)) ** (order + 1) + 1e-6


@pytest.mark.parametrize("order", [2, 12, 19, 31, 40])
@pytest.mark.parametrize("n", [5, 300, 9001])
def test_small_and_empty_leaves(n, order, O):
    """Leaves of few points (sixteen lanes each), most of them empty, among them
    all the last ones in Morton order; the same bounds as above."""
    rng = np.random.default_rng(n + order)
    x, y = 0.3 * rng.random((2, n)) ** 2
    x[0], y[0], x[1], y[1] = 1.0, 0.0, 0.0, 1.0  # the last quarter holds no point
    w = rng.standard_normal(n)
    xopt, cutoff = W.oseen_params(1e-3)
    ref = O.direct_oseen(x, y, w, x, y, xopt, cutoff)
    r = 0.5 ** 0.5
    for prec, eps in ((F64, 1e-12), (F32C, 1e-6)):
        got = gauss.fmm2d_gpu(x, y, w, x, y, 35, xopt, cutoff, 1e-6, prec=prec, order=order,
                              leaf=1 if n < 1000 else 8)
        assert O.rel_l2(got, ref) <= (r / (2 - r)) ** (order + 1) + eps


@pytest.mark.parametrize("n", [1, 63, 65, 255, 257, 1025, 2047, 2048, 2049, 70001])
def test_population_control_chunks(n, O):
    """Chunks of 2048 and waves of 64 blobs at their edges; few, most, all and
    none of the blobs under the thresholds; values that are not finite stay."""
    from phyflow_amd.blobs.base.regrid import PopulationControl
    rng = np.random.default_rng(n)
    x, y = rng.random(n), rng.random(n)
    for lo, hi, total in ((-12, -3, 1e-7), (-14, -9, 1e-9), (-7, -3, 1e-8), (-30, -20, 1.0)):
        w = 10.0 ** rng.uniform(lo, hi, n) * rng.choice([-1.0, 1.0], n)
        got = PopulationControl(x, y, w, 1e-8, total)
        ref = O.population_control(x, y, w, 1e-8, total)
        for a, b in zip(got, ref[:3]):
            assert np.array_equal(a, b)
    w = 10.0 ** rng.uniform(-12, -3, n)
    w[n // 2] = np.nan
    w[n // 3] = np.inf
    got = PopulationControl(x, y, w, 1e-8, 1e300)
    assert np.array_equal(got[0], x[~(np.abs(w) < 1e-8)])


def _flow_and_targets(nb, nt, seed, spread=1.0):
    s = W.uniform_system(nb, seed=seed)
    p = np.random.default_rng(seed + 1).random((nt, 2)) * spread
    return s["x"], s["y"], s["w"], p[:, 0].copy(), p[:, 1].copy(), 2.0 * s["sigma"] ** 2


@pytest.mark.parametrize("nb,nt", [(9999, 10000), (10001, 10007), (3001, 65537), (70001, 1501)])
def test_direct_sorted_targets(nb, nt, O):
    """Both sides of the pair count from which targets are sorted, and of the
    second sorting pass; targets on sources and a cutoff of 0.  float64 sums of
    nb terms in another order: nb 2^-53 relative to the terms' sizes, far less
    in practice."""
    x, y, w, xt, yt, ks = _flow_and_targets(nb, nt, nb)
    m = min(nb, nt) // 2
    xt[:m], yt[:m] = x[:m], y[:m]
    sub = np.arange(0, nt, 7)
    got = gauss.vv2parGauss_gpu(x, y, w, xt, yt, ks, 128)
    ref = O.vv2par_gauss(x, y, w, xt[sub], yt[sub], ks)
    assert O.rel_l2([g[sub] for g in got], ref) <= 1e-13
    xopt = (1.2564312086261696770 * ks) ** 0.5
    for cutoff in (5.0 * xopt, 0.0):
        got = gauss.fmm2d_gpu(x, y, w, xt, yt, 35, xopt, cutoff, 0.0)
        if cutoff == 0.0:  # the oracle divides 0 by 0 where a target is a source
            assert np.all(np.isfinite(got))
            sub = sub[sub >= m]
        ref = O.direct_oseen(x, y, w, xt[sub], yt[sub], xopt, cutoff)
        assert O.rel_l2([g[sub] for g in got], ref) <= 1e-13


@pytest.mark.parametrize("prec,tol", [(F64, 1e-14), (F32C, 1e-6)])
@pytest.mark.parametrize("nb,nt", [(1, 1), (15, 64), (16, 65), (17, 127), (33, 129), (400, 400),
                                   (1023, 2025), (2081, 3), (8193, 1), (3249, 3249),
                                   (5000, 8191), (16384, 16385)])
def test_direct_source_chunks(nb, nt, prec, tol, O):
    """Source chunks of 16 and more: remainders of chunks and target groups, one
    round of waves and the rounds after it."""
    x, y, w, xt, yt, ks = _flow_and_targets(nb, nt, nb + nt)
    got = gauss.vv2parGauss_gpu(x, y, w, xt, yt, ks, 128, prec=prec)
    ref = O.vv2par_gauss(x, y, w, xt, yt, ks)
    assert O.rel_l2(got, ref) <= tol * max(1.0, (nb / 100) ** 0.5)


def test_direct_sorted_degenerate(O):
    """All targets in one point or on a line: one cell, or one row of them."""
    x, y, w, xt, yt, ks = _flow_and_targets(10007, 10007, 5)
    for xs, ys in ((np.full(10007, 0.25), np.full(10007, 0.5)), (xt, np.full(10007, 0.5))):
        got = gauss.vv2parGauss_gpu(x, y, w, xs, ys, ks, 128)
        ref = O.vv2par_gauss(x, y, w, xs[:500], ys[:500], ks)
        assert O.rel_l2([g[:500] for g in got], ref) <= 1e-13


@pytest.mark.parametrize("prec,tol", [(F64, 1e-14), (F32C, 1e-6)])
@pytest.mark.parametrize("nb,nt,spread", [(9999, 10000, 1.0), (10001, 10007, 1.0),
                                          (20011, 20021, 1.0), (2003, 200003, 1.6),
                                          (300007, 1501, 3.0)])
def test_vorticity_near(prec, tol, nb, nt, spread, O):
    """Both sides of the pair counts; with spread > 1 many targets lie where
    every term is below 2^-100: each value is held to the value itself (down to
    where float64 runs out), float32 ones to the field's size."""
    x, y, w, xt, yt, ks = _flow_and_targets(nb, nt, nt, spread)
    sub = np.arange(0, nt, max(1, nt // 700))
    got = gauss.ww2parGauss_gpu(x, y, w, xt, yt, ks, 128, prec=prec)[sub]
    ref = O.ww2par_gauss(x, y, w, xt[sub], yt[sub], ks)
    assert O.rel_l2([got], [ref]) <= tol
    if prec == F64:
        # terms of both signs cancel: the bound is on the sum of their sizes,
        # and exp's argument carries its own rounding, 2^-53 of r2 / ks <= 750
        size = O.ww2par_gauss(x, y, np.abs(w), xt[sub], yt[sub], ks)
        assert np.all(np.abs(got - ref) <= 750 * 2.0 ** -52 * size + 1e-300)


@pytest.mark.parametrize("prec", [F64, F32C])
def test_vorticity_small_sums(prec, O):
    """Sums at both ends of the second pass: targets at distances out to where
    a term is 0 and beyond, alone in their group of 64 and in whole groups; all
    circulations 0, and circulations whose sizes add up to infinity."""
    nb, nt = 20011, 40009
    x, y, w, xt, yt, ks = _flow_and_targets(nb, nt, 11)
    d = np.sqrt(ks * np.linspace(0.0, 1500.0, 4001))  # right of the unit square
    xt[:4001], yt[:4001] = 1.0 + d, 0.5
    xt[5000:5200], yt[5000:5200] = -40.0, 0.5  # beyond every term
    sub = np.r_[0:4001:7, 5000:5200:9, 6000:nt:97]
    got = gauss.ww2parGauss_gpu(x, y, w, xt, yt, ks, 128, prec=prec)
    ref = O.ww2par_gauss(x, y, w, xt[sub], yt[sub], ks)
    size = O.ww2par_gauss(x, y, np.abs(w), xt[sub], yt[sub], ks)
    # float32: some 1e-6 of the terms, and of the exponent r2 / ks times the
    # rounding of r2, until a term leaves float32's normal numbers
    big = size if prec == F64 else np.maximum(size, 2.0 ** -126 * np.max(size) * nb)
    tol = 750 * 2.0 ** -52 if prec == F64 else 104 * 2.0 ** -21
    assert np.all(np.abs(got[sub] - ref) <= tol * big + (1e-300 if prec == F64 else 0.0))
    assert not got[5000:5200].any()
    assert not gauss.ww2parGauss_gpu(x, y, 0 * w, xt, yt, ks, 128, prec=prec).any()
    if prec == F64:
        big = np.where(np.arange(nb) % 2 == 0, 2e304, -2e304)
        got = gauss.ww2parGauss_gpu(x, y, big, xt, yt, ks, 128)[sub]
        size = O.ww2par_gauss(x, y, np.full(nb, 1.0), xt[sub], yt[sub], ks)
        ref = O.ww2par_gauss(x, y, big * 5e-305, xt[sub], yt[sub], ks)
        fits = np.abs(ref) < 8e3  # of a value in float64
        assert np.count_nonzero(fits) > 0.9 * fits.size
        assert np.all((np.abs(got * 5e-305 - ref) <= 1e-12 * size + 1e-300)[fits])


@pytest.mark.parametrize("prec", [F64, F32C])
def test_vorticity_beyond_the_flow_is_not_the_whole_sum(prec):
    """A grid that reaches beyond the blobs takes longer than one among them,
    but not as long as every pair would (some fifteen times)."""
    import time
    nb, nt = 100003, 90601
    x, y, w, xt, yt, ks = _flow_and_targets(nb, nt, 3)

    def t(sx, ox):
        a, b = xt * sx + ox, yt * sx + (1.0 - sx) / 2
        runs = []
        for _ in range(7):
            t0 = time.perf_counter()
            gauss.ww2parGauss_gpu(x, y, w, a, b, ks, 128, prec=prec)
            runs.append(time.perf_counter() - t0)
        return sorted(runs)[3]

    inside = t(1.0, 0.0)
    assert t(2.0, -0.5) <= 5.0 * inside
    assert t(1.0, 2.0) <= 2.0 * inside


def test_a_few_small_sums_are_no_long_chain():
    """Broad blobs and a grid that reaches a little beyond them: the targets in
    its corners, a hundredth of all, have small sums out of most of the blobs.
    They cost what the others cost, not as much again."""
    import time
    x, y, w, xt, yt, ks = _flow_and_targets(20011, 40401, 3)
    ks = 18.0 / x.size

    def t(sx):
        a, b = (xt - 0.5) * sx + 0.5, (yt - 0.5) * sx + 0.5
        runs = []
        for _ in range(9):
            t0 = time.perf_counter()
            gauss.ww2parGauss_gpu(x, y, w, a, b, ks, 128)
            runs.append(time.perf_counter() - t0)
        return sorted(runs)[4]

    assert t(1.5) <= 1.8 * t(1.0)


@pytest.mark.parametrize("n", [1, 5461, 5462, 87381, 87382, 131072, 131073, 800001])
def test_blobs_come_back_whole(n):
    """Results by one packed transfer, by the runtime's copies and through the
    pinned slots (24 n bytes: 128 KiB, 2 MiB, whole and odd slots, more slots
    than a ring has), from several threads at once."""
    import threading
    from phyflow_amd.system import BlobSystem
    rng = np.random.default_rng(n)
    data = [tuple(rng.random(n) for _ in range(3)) for _ in range(3)]
    systems = [BlobSystem(*d) for d in data]
    wrong = []

    def check(k):
        for _ in range(3):
            for a, b in zip(systems[k].get(), data[k]):
                if not np.array_equal(a, b):
                    wrong.append(k)

    threads = [threading.Thread(target=check, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


@pytest.mark.parametrize("n", [87381, 87382, 131072, 131073, 699050, 699051, 800001])
def test_blobs_come_back_whole_alone(n):
    """Fetches that are alone go through the pinned slots from 2 MiB (24 n
    bytes) on: one slot, whole and odd ones, and as many as there are and more."""
    from phyflow_amd.system import BlobSystem
    data = np.random.default_rng(n).random((3, n))
    with BlobSystem(*data) as s:
        for _ in range(2):
            assert np.array_equal(s.get(), data)


@pytest.mark.parametrize("n", [511, 512, 1024, 2048, 3072, 4096, 4608, 5120, 5461])
def test_systems_of_whole_pages(n, O):
    """Small systems whose arrays are whole pages, and so may touch in memory
    without being one allocation: blobs and velocities come back."""
    from phyflow_amd.system import BlobSystem, vel_params
    s = W.uniform_system(n, seed=n)
    xopt, cutoff = W.oseen_params(s["sigma"])
    q = O.direct_oseen(s["x"], s["y"], s["w"], s["x"], s["y"], xopt, cutoff)
    with BlobSystem(s["x"], s["y"], s["w"]) as b:
        assert np.array_equal(b.get(), [s["x"], s["y"], s["w"]])
        v = b.velocity(vel_params(s["sigma"]))
        assert np.array_equal(v, b.last_velocity())
        # (-qi, -qr) / 2 pi at the default tolerance 1e-6
        assert O.rel_l2(v, [-q[1] / (2 * np.pi), -q[0] / (2 * np.pi)]) <= 1e-6


@pytest.mark.parametrize("leaf", [16, 128])
@pytest.mark.parametrize("prec", [F64, F32C])
def test_replay_follows_from_the_points_alone(prec, leaf):
    """A system evaluated before on points that filled its domain otherwise
    (other lanes for P2M with 16 blobs a leaf, other parts of the near field
    with 128) gives the bits that a fresh one gives."""
    from phyflow_amd.system import BlobSystem, vel_params
    n = 16000
    s = W.uniform_system(n, seed=4)
    p = vel_params(0.2 * s["sigma"], prec=prec, order=17, leaf=leaf, leaf_side=-1.0)
    x, y, w = s["x"], s["y"], s["w"]
    x[0], x[1] = 0.0, 1.0  # the same bounding box side for both
    y[0], y[1] = 0.0, 1.0
    flat = 0.3 * y
    with BlobSystem(x, y, w) as a, BlobSystem(x, flat, w) as b:
        full = a.velocity(p)
        a.set(x, flat, w)
        assert np.array_equal(a.velocity(p), b.velocity(p))
        a.set(x, y, w)
        assert np.array_equal(a.velocity(p), full)


@pytest.mark.parametrize("prec", [F64, F32C])
def test_points_that_keep_the_domain_are_replayed(prec):
    """Points that fill the same domain otherwise are evaluated by the launches
    that were recorded: a system whose points change between two such states
    every time takes about as long as one that stays, not several times that."""
    import time
    from phyflow_amd.system import BlobSystem, vel_params
    n = 16000
    s = W.uniform_system(n, seed=4)
    p = vel_params(0.2 * s["sigma"], prec=prec, order=17, leaf=16, leaf_side=-1.0)
    x, y, w = s["x"], s["y"], s["w"]
    x[0], x[1] = 0.0, 1.0
    y[0], y[1] = 0.0, 1.0
    states = y, 0.3 * y

    def t(b, turns):
        runs = []
        for k in range(12):
            b.set(x, states[k % turns], w)
            t0 = time.perf_counter()
            b.velocity(p)
            runs.append(time.perf_counter() - t0)
        return sorted(runs)[6]

    with BlobSystem(x, y, w) as b:
        assert t(b, 2) <= 2.0 * t(b, 1)


@pytest.mark.parametrize("n", [1, 7, 65536, 65537, 300001])
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_not_finite_is_refused_anywhere(n, bad):
    from phyflow_amd._native import PhfError
    from phyflow_amd.system import BlobSystem
    x = np.zeros(n)
    x[:4] = [5e-324, 1.7976931348623157e308, -0.0, 1.0][:min(4, n)]
    BlobSystem(x, x, x).close()
    for at in {0, n // 2, n - 1, min(n - 1, 65535), min(n - 1, 65536)}:
        y = x.copy()
        y[at] = bad
        with pytest.raises(PhfError, match=r"y\[%d\] is not finite" % at):
            BlobSystem(x, y, x)


def _clumps(counts, n, seed):
    """counts[k] of n points in a clump of side 0.01 within a leaf, the rest over
    the unit square."""
    rng = np.random.default_rng(seed)
    x, y = rng.random((2, n))
    x[-2:], y[-2:] = [0.0, 1.0], [0.0, 1.0]
    j = 0
    for k, c in enumerate(counts):
        x[j:j + c] = 0.11 + 0.125 * k + 0.01 * x[j:j + c]
        y[j:j + c] = 0.3 + 0.01 * y[j:j + c]
        j += c
    assert j <= n
    return x, y, rng.random(n) + 0.5


@pytest.mark.parametrize("order", [2, 12, 19, 31, 40])
def test_crowded_leaves_among_small_ones(order, O):
    """Leaves on both sides of where four have a wave each in place of sixteen
    lanes (the clumps' leaves have some 3 points more); the bounds of
    test_multipole_orders."""
    x, y, w = _clumps([27, 28, 29, 30, 31, 32, 700], 4003, order)
    xopt, cutoff = W.oseen_params(1e-3)
    ref = O.direct_oseen(x, y, w, x, y, xopt, cutoff)
    r = 0.5 ** 0.5
    for prec, eps in ((F64, 1e-12), (F32C, 1e-6)):
        got = gauss.fmm2d_gpu(x, y, w, x, y, 35, xopt, cutoff, 1e-6, prec=prec, order=order, leaf=8)
        assert O.rel_l2(got, ref) <= (r / (2 - r)) ** (order + 1) + eps


@pytest.mark.parametrize("prec", [F64, F32C])
def test_a_crowded_leaf_is_no_longer_chain_in_a_deeper_tree(prec):
    """Expanding one leaf with most of the blobs takes about as long in a tree
    whose other leaves have few (sixteen lanes, as those have, would take four
    times as long) as in one of a level less."""
    from phyflow_amd.system import BlobSystem, vel_params
    x, y, w = _clumps([9000], 10000, 1)

    def ms(leaf):
        p = vel_params(1e-4, prec=prec, order=16, leaf=leaf, leaf_side=-1.0)
        with BlobSystem(x, y, w) as s:
            runs = []
            for _ in range(8):
                s.velocity(p, fetch=False, eager=True)
                runs.append(s.last_info["ms"]["p2m"])
            return sorted(runs)[3], s.last_info["L"]

    small, wave = ms(10), ms(40)
    assert small[1] == wave[1] + 1
    assert small[0] <= 2.0 * wave[0]


def test_tree_shapes_in_turn(O):
    """More tree shapes than a lane keeps tables for, in changing order: the
    same bits every time a shape comes back, each against the direct sum.
    Shapes differ in one thing at a time: order, precision, leaf level, box
    separation, the cutoff against the leaf, targets apart from the sources."""
    n = 4000
    s = W.uniform_system(n, seed=3)
    x, y, w = s["x"], s["y"], s["w"]
    xopt, cutoff = W.oseen_params(s["sigma"])
    t = np.random.default_rng(4).random((2, 700))
    base = dict(prec=F64, order=20, leaf=16, ws=1)
    shapes = [dict(base), dict(base, order=21), dict(base, order=12), dict(base, prec=F32C),
              dict(base, prec=F32C, order=16), dict(base, prec=F32C, order=17),
              dict(base, leaf=64), dict(base, ws=2), dict(base, cut=0.3), dict(base, cut=0.5),
              dict(base, targets=True), dict(base, leaf=4000)]

    def run(kw):
        kw = dict(kw)
        c = cutoff * kw.pop("cut", 1.0)
        xt, yt = t if kw.pop("targets", False) else (x, y)
        return np.array(gauss.fmm2d_gpu(x, y, w, xt, yt, 35, xopt, c, 1e-6, **kw)), (xt, yt, c)

    first = []
    for kw in shapes:
        got, (xt, yt, c) = run(kw)
        ref = O.direct_oseen(x, y, w, xt, yt, xopt, c)
        assert O.rel_l2(got, ref) <= (1e-4 if kw["order"] < 16 else 1e-6), kw
        first.append(got)
    rng = np.random.default_rng(5)
    for k in rng.integers(0, len(shapes), 40):
        assert np.array_equal(run(shapes[k])[0], first[k]), shapes[k]


def _ellipse(m, thin, turn=0.1):
    t = np.linspace(np.pi, -np.pi, m + 1) + turn
    return np.cos(t), thin * np.sin(t)


@pytest.mark.parametrize("problem", ["fixed", "moving"])
@pytest.mark.parametrize("m,thin", [(3, 1.0), (31, 1.0), (32, 0.5), (33, 0.9), (65, 0.3),
                                    (300, 1.0), (512, 0.7), (1024, 1.0), (1025, 1.0),
                                    (200, 0.02), (400, 0.003)])
def test_square_body_solve(m, thin, problem):
    """Square panel systems at block edges and at the size where the pivoted LU
    takes over, from round bodies to thin ones (whose condition number sends
    them there); after a move as after the creation.  numpy's float64 solve of
    the body's own matrix, to its condition number times 2^-52 sqrt(m)."""
    from phyflow_amd.lagrangian import PanelBody
    xp, yp = _ellipse(m, thin)
    body = PanelBody(xp, yp, problem)
    k = 2 * np.pi * np.arange(m) / m
    vx, vy = 1.0 + 0.2 * np.sin(3 * k), 0.3 * np.cos(2 * k)
    for move in range(3):
        if move:
            body.updateBody((0.1 * move, -0.2), 0.3 * move)
            c, s = np.cos(0.3 * move), np.sin(0.3 * move)
            x, y = c * xp - s * yp + 0.1 * move, s * xp + c * yp - 0.2
        else:
            x, y = xp, yp
        g = W.panel_geometry(x, y)
        A = body.A
        rhs = -(vx * g["cosA"] + vy * g["sinA"])
        ref = np.linalg.solve(A, rhs)
        got = body.solve(vx, vy)
        cond = np.linalg.cond(A)
        assert np.linalg.norm(got - ref) <= 4 * cond * 2.0 ** -52 * m ** 0.5 * np.linalg.norm(ref)


@pytest.mark.parametrize("n,leaf", [(70, 200), (500, 1000), (3001, 3001), (3001, 100),
                                    (20011, 300), (60013, 230)])
@pytest.mark.parametrize("prec,tol", [(F64, 1e-7), (F32C, 1e-6)])
def test_leaves_in_parts(n, leaf, prec, tol, O):
    """Few leaves of many targets, each split over one to eight workgroups; the
    targets also apart from the sources.  Order 24 leaves the near field's own
    error (and 1e-8 of the expansions')."""
    s = W.uniform_system(n, seed=n)
    x, y, w = s["x"], s["y"], s["w"]
    xopt, cutoff = W.oseen_params(s["sigma"])
    t = np.random.default_rng(n).random((2, n // 3 + 1))
    for xt, yt in ((x, y), t):
        got = gauss.fmm2d_gpu(x, y, w, xt, yt, 35, xopt, cutoff, 1e-6, prec=prec, order=24,
                              leaf=leaf)
        sub = np.arange(0, xt.size, max(1, xt.size // 2000))
        ref = O.direct_oseen(x, y, w, xt[sub], yt[sub], xopt, cutoff)
        assert O.rel_l2([g[sub] for g in got], ref) <= tol
