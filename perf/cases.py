"""The work that users of phyflow_amd have it do, as cases to be timed.

Every case goes through the package's public entry points the way a program
calls them: host arrays in and out for the drop-in functions, resident
handles (BlobSystem, PanelBody, BatchSystems) for time stepping, device
pointers for the allocation-free direct sum.

    listed()            the named cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) what a program holds before the call
    run(state)          one pass and its outputs
    exact(case, seed)   the outputs in plain 64-bit torch / numpy
    work(case)          bytes and flops that a pass cannot do without
    tolerance(case)     what two correct implementations differ by
"""
import ctypes
import math

import numpy as np
import torch

from __graft_entry__ import load_package

load_package()

from phyflow_amd import autotune, workloads  # noqa: E402
from phyflow_amd._native import PREC_F32C, PREC_F64, call  # noqa: E402
from phyflow_amd.batch import BatchSystems  # noqa: E402
from phyflow_amd.blobs.base.induced import velocity, vorticity  # noqa: E402
from phyflow_amd.blobs.base.regrid import Regrid  # noqa: E402
from phyflow_amd.lagrangian import PanelBody, step_rk2  # noqa: E402
from phyflow_amd.system import BlobSystem  # noqa: E402

PREC = {"f64": PREC_F64, "f32c": PREC_F32C}
OVERLAP = 0.8        # h = 0.8 sigma, as in every configuration of this repository
EPS = 1e-12          # of the direct Gaussian kernel
EXACT_PAIRS = 1.3e11  # pairs that the 64-bit sums below do in well under 20 s


# ------------------------------------------------------------------ cases --
def listed():
    return [
        # A small flow evaluated at its own blobs by the drop-in direct sum:
        # the smallest call, bound by its latency.
        dict(name="direct_900", kind="direct", field="velocity", n=900, nt=0, prec="f64"),
        # The Lamb-Oseen lattice with device arrays, as in a loop that must
        # not allocate.
        dict(name="direct_device_4096", kind="device", side=64, prec="f32c"),
        # The velocity of a mid-size flow at probes (float64, the default).
        dict(name="direct_probes", kind="direct", field="velocity", n=20011, nt=30017,
             prec="f64"),
        # The vorticity of the same flow on a plotting grid.
        dict(name="vorticity_probes", kind="direct", field="vorticity", n=20011, nt=40401,
             prec="f64"),
        # velocity() with all its defaults (FMM, float64, tol 1e-6) at probes.
        dict(name="fmm_probes", kind="fmm", n=100003, nt=40009, prec="f64"),
        # One evaluation of a large resident system, read back by the caller.
        dict(name="evaluate_1m", kind="evaluate", n=1048576, prec="f32c", tol=1e-6),
        # Time stepping from given blobs: convection, remesh and population
        # control every step, the blobs read at the end; the accurate class
        # and the fast class at the largest size.
        dict(name="steps_f64", kind="steps", nx=401, ny=299, steps=4, prec="f64", tol=1e-12),
        dict(name="steps_1m", kind="steps", nx=1021, ny=1027, steps=3, prec="f32c", tol=1e-6),
        # Flow past a moving cylinder: panels rebuilt and solved every step.
        dict(name="cylinder", kind="cylinder", panels=512, n=262144, steps=3, prec="f32c",
             tol=1e-6),
        # The no-slip strengths of a body that has moved.
        dict(name="body_fixed", kind="body", panels=301, problem="fixed"),
        # The drop-in remesh, with viscous diffusion (Wee's parameter).
        dict(name="regrid", kind="regrid", n=262147, c=0.1),
        # A parameter sweep: many uneven systems advanced and remeshed at once.
        dict(name="sweep_64", kind="sweep", count=64, lo=1024, hi=131072, mix=0, prec="f32c"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["direct", "device", "fmm", "evaluate", "steps", "cylinder", "body",
                       "regrid", "sweep"])
    prec = rng.choice(["f64", "f32c"])
    # the accuracy classes of the measured table
    tol = rng.choice([1e-6, 1e-12]) if prec == "f64" else 1e-6
    if kind == "direct":
        nt = rng.choice([0, 1]) * _log_int(rng, 100, 40000)
        return dict(kind=kind, field=rng.choice(["velocity", "velocity", "vorticity"]),
                    n=_log_int(rng, 500, 20000), nt=nt, prec=prec)
    if kind == "device":
        return dict(kind=kind, side=_log_int(rng, 20, 200), prec=prec)
    if kind == "fmm":
        nt = rng.choice([0, 1]) * _log_int(rng, 1000, 100000)
        return dict(kind=kind, n=_log_int(rng, 10000, 200000), nt=nt, prec=prec)
    if kind == "evaluate":
        return dict(kind=kind, n=_log_int(rng, 20000, 800000), prec=prec, tol=tol)
    if kind == "steps":
        s = _log_int(rng, 60, 600)
        return dict(kind=kind, nx=s, ny=int(s * rng.uniform(0.6, 1.4)), steps=rng.choice([2, 3]),
                    prec=prec, tol=tol)
    if kind == "cylinder":
        return dict(kind=kind, panels=_log_int(rng, 64, 512), n=_log_int(rng, 8000, 200000),
                    steps=2, prec=prec, tol=tol)
    if kind == "body":
        return dict(kind=kind, panels=_log_int(rng, 40, 700),
                    problem=rng.choice(["fixed", "prescribed"]))
    if kind == "regrid":
        return dict(kind=kind, n=_log_int(rng, 5000, 400000), c=rng.choice([0.0, 0.1, 0.25]))
    return dict(kind=kind, count=rng.randint(8, 64), lo=1024, hi=_log_int(rng, 8192, 131072),
                mix=rng.randint(1, 1 << 20), prec=prec)


# ----------------------------------------------------------------- inputs --
def _flow(n, seed):
    """n blobs anywhere in the unit square, circulations of both signs."""
    return workloads.uniform_system(n, seed)


def _probes(nt, seed):
    p = np.random.default_rng([seed, 77]).random((nt, 2))
    return p[:, 0].copy(), p[:, 1].copy()


# A remesh returns as many blobs as the lattice cells it touched.  So that the
# seed does not change that count, it shuffles and weighs blobs at positions
# that the case fixes, and where they move it also scales the whole flow
# (circulations and stream by a, time step and thresholds to match).
def _scale(seed, n):
    rng = np.random.default_rng([seed, 3])
    return rng.uniform(0.5, 2.0), 1.0 + 1e-4 * rng.standard_normal(n), rng.permutation(n)


def _moving(s, seed):
    """The flow s with its blobs in another order, scaled by a."""
    a, f, p = _scale(seed, s["x"].size)
    return dict(s, x=s["x"][p], y=s["y"][p], w=(a * f * s["w"])[p], a=a)


def _lattice_flow(nx, ny, seed):
    """Blobs on an nx x ny lattice carrying smooth vortices of both signs on a
    background: the state of a run between two remeshes."""
    rng = np.random.default_rng(nx * ny)
    h = 1.0 / max(nx, ny)
    X, Y = np.meshgrid(h * (np.arange(nx) + 0.5) - 1.5 * h, h * (np.arange(ny) + 0.5) - 1.5 * h,
                       indexing="ij")
    omega = np.full_like(X, 0.5)
    for _ in range(8):
        cx, cy, a, c = rng.random(), rng.random() * ny / nx, rng.normal(0, 2), rng.uniform(.1, .3)
        omega += a * np.exp(-((X - cx) ** 2 + (Y - cy) ** 2) / (c * c))
    a = _scale(seed, 1)[0]
    return dict(x=X.ravel().copy(), y=Y.ravel().copy(), w=a * (omega * h * h).ravel(), h=h,
                sigma=h / OVERLAP, dt=0.3 * h / a,  # a few tenths of a cell per step
                control=(1e-8 * a, 1e-8 * a))  # Blobs' default, 1e-8 each and in all


def _lamb(side, seed):
    rng = np.random.default_rng(seed)
    return workloads.lamb_oseen_lattice(side, gamma0=rng.uniform(0.5, 2.0),
                                        c=rng.uniform(0.3, 0.6))


def _cylinder(case, seed):
    xp, yp = workloads.cylinder_panels(case["panels"])
    sigma = 0.004 * math.sqrt(262144.0 / case["n"])
    b = workloads.annulus_blobs(case["n"], r0=0.52, sigma=sigma, seed=case["panels"])
    return xp, yp, _moving(b, seed)


def _body(case, seed):
    """A cylinder deformed to a smooth closed body, and the external flow at
    its collocation points."""
    rng = np.random.default_rng(seed)
    xp, yp = workloads.cylinder_panels(case["panels"])
    th, r = np.arctan2(yp, xp), np.hypot(xp, yp)
    r = r * (1.0 + 0.1 * rng.uniform(-1, 1) * np.cos(2 * th + rng.uniform(0, 6)))
    xp, yp = r * np.cos(th), r * np.sin(th)
    xp[-1], yp[-1] = xp[0], yp[0]
    m = case["panels"]
    k = 2 * np.pi * np.arange(m) / m
    vx = 1.0 + 0.2 * np.sin(3 * k + rng.uniform(0, 6))
    vy = 0.3 * np.cos(2 * k + rng.uniform(0, 6))
    return xp, yp, vx, vy


def _regrid_blobs(case, seed):
    s = _flow(case["n"], case["n"])
    rng = np.random.default_rng(seed)
    p = rng.permutation(case["n"])
    return dict(s, x=s["x"][p], y=s["y"][p], w=rng.standard_normal(case["n"]) * s["h"] ** 2)


def _sweep_systems(case, seed):
    """Sizes, systems and their common time step."""
    sizes = workloads.uneven_sizes(case["count"], case["lo"], case["hi"], case["mix"])
    a = _scale(seed, 1)[0]
    systems = [_moving(_flow(int(n), i), seed) for i, n in enumerate(sizes)]
    return sizes, systems, 1e-2 / a


_stream = None


def _user_stream():
    """The one stream that this program runs its device-array calls on."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case)
    if kind in ("direct", "fmm"):
        st.update(_flow(case["n"], seed))
        st["xe"], st["ye"] = _probes(case["nt"], seed) if case["nt"] else (None, None)
    elif kind == "device":
        s = _lamb(case["side"], seed)
        st["ks"] = 2.0 * s["sigma"] ** 2
        st["t"] = [torch.from_numpy(s[k]).cuda() for k in ("x", "y", "w")]
        st["out"] = [torch.empty_like(st["t"][0]) for _ in range(2)]
        st["stream"] = _user_stream()
        st["stream"].wait_stream(torch.cuda.current_stream())
    elif kind == "evaluate":
        s = _flow(case["n"], seed)
        st["system"] = BlobSystem(s["x"], s["y"], s["w"])
        st["params"] = autotune.tuned_params(s["sigma"], case["n"], PREC[case["prec"]],
                                             case["tol"])
    elif kind == "steps":
        st.update(_lattice_flow(case["nx"], case["ny"], seed))
        st["system"] = BlobSystem(st["x"], st["y"], st["w"])
        st["params"] = autotune.tuned_params(st["sigma"], st["x"].size, PREC[case["prec"]],
                                             case["tol"])
        st["remesh"] = dict(sigma=st["sigma"], overlap=OVERLAP, population_control=st["control"])
    elif kind == "cylinder":
        xp, yp, b = _cylinder(case, seed)
        st.update(b)
        st["system"] = BlobSystem(b["x"], b["y"], b["w"])
        st["body"] = PanelBody(xp, yp, "prescribed")
        st["params"] = autotune.tuned_params(b["sigma"], case["n"], PREC[case["prec"]],
                                             case["tol"])
        st["remesh"] = dict(sigma=b["sigma"], overlap=OVERLAP)
    elif kind == "body":
        xp, yp, st["vx"], st["vy"] = _body(case, seed)
        st["body"] = PanelBody(xp, yp, case["problem"])
    elif kind == "regrid":
        st.update(_regrid_blobs(case, seed))
    else:
        sizes, systems, dt = _sweep_systems(case, seed)
        order = max(autotune.tuned_params(s["sigma"], s["x"].size, PREC[case["prec"]], 1e-6).order
                    for s in systems)
        b = BatchSystems(sizes, [s["sigma"] for s in systems], PREC[case["prec"]], order)
        for i, s in enumerate(systems):
            b.set_system(i, s["x"], s["y"], s["w"])
        b.set_remesh(OVERLAP, dt=dt)
        st["batch"] = b
    return st


# -------------------------------------------------------------------- run --
def run(s):
    kind = s["kind"]
    if kind == "direct":
        if s["field"] == "vorticity":
            return vorticity(s["x"], s["y"], s["w"], s["sigma"], xEval=s["xe"], yEval=s["ye"],
                             hardware=1, prec=PREC[s["prec"]])
        return velocity(s["x"], s["y"], s["w"], s["sigma"], xEval=s["xe"], yEval=s["ye"],
                        hardware=1, method=1, prec=PREC[s["prec"]])
    if kind == "device":
        x, y, w = (ctypes.c_void_p(t.data_ptr()) for t in s["t"])
        u, v = (ctypes.c_void_p(t.data_ptr()) for t in s["out"])
        n = s["t"][0].numel()
        call("phf_vv2par_gauss_noalloc", x, y, w, n, x, y, n, s["ks"], PREC[s["prec"]], u, v,
             ctypes.c_void_p(s["stream"].cuda_stream))
        return s["out"]
    if kind == "fmm":
        return velocity(s["x"], s["y"], s["w"], s["sigma"], xEval=s["xe"], yEval=s["ye"],
                        hardware=1, prec=PREC[s["prec"]])
    if kind == "evaluate":
        return s["system"].velocity(s["params"])
    if kind == "steps":
        s["system"].set(s["x"], s["y"], s["w"])
        for _ in range(s["steps"]):
            step_rk2(s["system"], s["params"], s["dt"], remesh=s["remesh"])
        return s["system"].get()
    if kind == "cylinder":
        s["system"].set(s["x"], s["y"], s["w"])
        for k in range(s["steps"]):
            s["body"].updateBody((1e-3 * (k + 1), 0.0), 0.01 * (k + 1), wait=False)
            step_rk2(s["system"], s["params"], 1e-3 / s["a"], vInf=(s["a"], 0.0),
                     panels=s["body"], remesh=s["remesh"])
        return s["system"].get()
    if kind == "body":
        s["body"].updateBody((0.25, -0.125), 0.3)
        return s["body"].solve(s["vx"], s["vy"])
    if kind == "regrid":
        b = (-1.5 * s["h"], 1.0)
        return Regrid(s["x"], s["y"], s["w"], s["sigma"], OVERLAP, b, b, 0, s["c"])
    s["batch"].step()
    got = [s["batch"].get_remeshed(i) for i in range(s["count"])]
    return [np.concatenate([g[k] for g in got]) for k in range(3)]


# ------------------------------------------------------------------ exact --
def _sum_pairs(xb, yb, wb, xt, yt, weight, vector):
    """sum_j weight(r2) w_j (and its products with dx, dy), float64 on the GPU."""
    xb, yb, wb, xt, yt = (torch.as_tensor(a, dtype=torch.float64, device="cuda")
                          for a in (xb, yb, wb, xt, yt))
    rows = max(1, int(1.5e8 // xb.numel()))
    out = []
    for i in range(0, xt.numel(), rows):
        dx = xt[i:i + rows, None] - xb
        dy = yt[i:i + rows, None] - yb
        g = weight(dx * dx + dy * dy).mul_(wb)
        if vector:
            out.append(torch.stack([-dy.mul_(g).sum(1), dx.mul_(g).sum(1)]))
        else:
            out.append(g.sum(1)[None])
    return torch.cat(out, 1).cpu().numpy()


def _direct_velocity(x, y, w, xt, yt, sigma):
    ks = 2.0 * sigma * sigma

    def weight(r2):
        r2 = r2.add_(EPS)
        return torch.expm1(r2 / -ks).div_(r2).neg_()

    return _sum_pairs(x, y, w, xt, yt, weight, True) / (2.0 * math.pi)


def _oseen_velocity(x, y, w, xt, yt, sigma):
    """The smoother of the FMM: exp(-shape r2) inside the cutoff, scaled to be
    continuous there; a blob has no velocity at its own centre."""
    xopt, cutoff = workloads.oseen_params(sigma)
    shape = workloads.ALPHA_OSEEN / (xopt * xopt)
    scale = -1.0 / math.expm1(-shape * cutoff * cutoff)

    def weight(r2):
        g = torch.expm1(-shape * r2).mul_(-scale).clamp_(max=1.0)
        return g.div_(r2.clamp_(min=1e-300))

    return _sum_pairs(x, y, w, xt, yt, weight, True) / (2.0 * math.pi)


def _m4(u, c):
    a = np.abs(u)
    outer = 0.5 * (2 - a) ** 2 * (1 - a) - c * c * (2 - a) ** 2 * (1 - 2 * a)
    inner = 1 - 2.5 * a * a + 1.5 * a ** 3 - c * c * (2 - 9 * a * a + 6 * a ** 3)
    return np.where(a < 1, inner, np.where((a > 1) & (a < 2), outer, 0.0))


def _remesh(x, y, w, h, x0, y0, c=0.0):
    """Every lattice cell that a blob's 4 x 4 stencil touches, row-major."""
    i0 = np.ceil(((x - x0) - 2.0 * h + 0.5 * h) / h).astype(np.int64) - 1
    j0 = np.ceil(((y - y0) - 2.0 * h + 0.5 * h) / h).astype(np.int64) - 1
    wx = [_m4(((i0 + k + 0.5) + x0 / h) - x / h, c) for k in range(4)]
    wy = [_m4(((j0 + k + 0.5) + y0 / h) - y / h, c) for k in range(4)]
    ib, jb = i0.min(), j0.min()
    cols = int(j0.max() - jb) + 4
    cells = (int(i0.max() - ib) + 4) * cols
    total, touched = np.zeros(cells), np.zeros(cells, bool)
    for a in range(4):
        for b in range(4):
            k = (i0 - ib + a) * cols + (j0 - jb + b)
            total += np.bincount(k, wx[a] * wy[b] * w, cells)
            touched[k] = True
    k = np.flatnonzero(touched)
    return ((k // cols + ib) * h + 0.5 * h) + x0, ((k % cols + jb) * h + 0.5 * h) + y0, total[k]


def _control(x, y, w, local, whole):
    while np.abs(w[np.abs(w) < local]).sum() >= whole:
        local /= 10.0
    keep = ~(np.abs(w) < local)
    return x[keep], y[keep], w[keep]


def _turned(xp, yp, cm, theta):
    c, s = math.cos(theta), math.sin(theta)
    return c * xp - s * yp + cm[0], s * xp + c * yp + cm[1]


def _influence(g):
    dx, dy = g["xcp"][:, None] - g["xs"], g["ycp"][:, None] - g["ys"]
    ca, sa, L = g["cosA"], g["sinA"], g["L"]
    xp, yp = ca * dx + sa * dy, -sa * dx + ca * dy
    u = (np.arctan2(yp, xp - L) - np.arctan2(yp, xp)) / (2 * math.pi)
    v = -np.log((xp * xp + yp * yp) / ((xp - L) ** 2 + yp * yp)) / (4 * math.pi)
    vx, vy = ca * u - sa * v, sa * u + ca * v
    return vx * ca[:, None] + vy * sa[:, None]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("direct", "fmm"):
        s = _flow(case["n"], seed)
        xe, ye = _probes(case["nt"], seed) if case["nt"] else (s["x"], s["y"])
        if case["n"] * xe.size > EXACT_PAIRS:
            return None
        if kind == "fmm":
            return tuple(_oseen_velocity(s["x"], s["y"], s["w"], xe, ye, s["sigma"]))
        if case["field"] == "velocity":
            return tuple(_direct_velocity(s["x"], s["y"], s["w"], xe, ye, s["sigma"]))
        ks = 2.0 * s["sigma"] ** 2
        return _sum_pairs(s["x"], s["y"], s["w"], xe, ye,
                          lambda r2: torch.exp(r2.add_(EPS).div_(-ks)), False)[0] / (math.pi * ks)
    if kind == "device":
        s = _lamb(case["side"], seed)
        return list(_direct_velocity(s["x"], s["y"], s["w"], s["x"], s["y"], s["sigma"]))
    if kind == "evaluate":
        if case["n"] ** 2 > EXACT_PAIRS:
            return None
        s = _flow(case["n"], seed)
        return tuple(_oseen_velocity(s["x"], s["y"], s["w"], s["x"], s["y"], s["sigma"]))
    if kind == "steps":
        if 2.0 * case["steps"] * (case["nx"] * case["ny"]) ** 2 > EXACT_PAIRS:
            return None
        s = _lattice_flow(case["nx"], case["ny"], seed)
        x, y, w, h, sigma, dt = s["x"], s["y"], s["w"], s["h"], s["sigma"], s["dt"]
        h = sigma * OVERLAP
        for _ in range(case["steps"]):
            k1 = _oseen_velocity(x, y, w, x, y, sigma)
            x1, y1 = x + dt * k1[0], y + dt * k1[1]
            k2 = _oseen_velocity(x1, y1, w, x1, y1, sigma)
            x, y = x + 0.5 * dt * (k1[0] + k2[0]), y + 0.5 * dt * (k1[1] + k2[1])
            x, y, w = _control(*_remesh(x, y, w, h, -1.5 * h, -1.5 * h), *s["control"])
        return x, y, w
    if kind == "cylinder":
        return None  # hundreds of billions of pairs and a boundary solve in between
    if kind == "body":
        xp, yp, vx, vy = _body(case, seed)
        g = workloads.panel_geometry(*_turned(xp, yp, (0.25, -0.125), 0.3))
        A, rhs = _influence(g), -(vx * g["cosA"] + vy * g["sinA"])
        if case["problem"] == "fixed":
            return np.linalg.solve(A, rhs)
        return np.linalg.lstsq(np.vstack([A, g["L"]]), np.append(rhs, 0.0), rcond=None)[0]
    if kind == "regrid":
        s = _regrid_blobs(case, seed)
        h = s["sigma"] * OVERLAP
        return _remesh(s["x"], s["y"], s["w"], h, -1.5 * s["h"], -1.5 * s["h"], case["c"])
    sizes, systems, dt = _sweep_systems(case, seed)
    if float((sizes.astype(float) ** 2).sum()) > EXACT_PAIRS:
        return None
    got = []
    for s in systems:
        h = s["sigma"] * OVERLAP
        u, v = _oseen_velocity(s["x"], s["y"], s["w"], s["x"], s["y"], s["sigma"])
        got.append(_remesh(s["x"] + dt * u, s["y"] + dt * v, s["w"], h, -1.5 * h, -1.5 * h))
    return [np.concatenate([g[k] for g in got]) for k in range(3)]


# ------------------------------------------------------------------- work --
PAIR = 17.0  # flops of one smoothed pair


def _fmm_flops(n, nt, order=13):
    """Sources inside the cutoff of every target by pairs (pi cutoff^2 / h^2,
    h = OVERLAP sigma, cutoff = 5 xopt), the rest through one expansion in
    and one out."""
    inside = math.pi * 25.0 * 2.0 * workloads.ALPHA_OSEEN / OVERLAP ** 2
    return nt * min(n, inside) * PAIR + 8.0 * (order + 1) * (n + nt)


def work(case):
    kind = case["kind"]
    if kind in ("direct", "fmm"):
        n, nt = case["n"], case["nt"] or case["n"]
        byt = 24.0 * n + (16.0 * nt if case["nt"] else 0.0)
        if kind == "fmm":
            return {"bytes": byt + 16.0 * nt, "flops": _fmm_flops(n, nt)}
        if case["field"] == "vorticity":
            return {"bytes": byt + 8.0 * nt, "flops": 8.0 * n * nt}
        return {"bytes": byt + 16.0 * nt, "flops": PAIR * n * nt}
    if kind == "device":
        n = case["side"] ** 2
        return {"bytes": 40.0 * n, "flops": PAIR * n * n}
    if kind == "evaluate":
        return {"bytes": 40.0 * case["n"], "flops": _fmm_flops(case["n"], case["n"])}
    if kind == "steps":
        n = case["nx"] * case["ny"]
        # each step reads and writes the blobs once; they come from the host
        # and go back once
        return {"bytes": 48.0 * n * (case["steps"] + 1),
                "flops": case["steps"] * (2.0 * _fmm_flops(n, n) + 16.0 * 20.0 * n)}
    if kind == "cylinder":
        n, m = case["n"], case["panels"]
        return {"bytes": 48.0 * n * (case["steps"] + 1),
                "flops": case["steps"] * (2.0 * _fmm_flops(n, n) + 16.0 * 20.0 * n
                                          + m ** 3 / 3.0 + 30.0 * m * m)}
    if kind == "body":
        m = case["panels"]
        return {"bytes": 8.0 * 7 * m, "flops": 2.0 / 3.0 * m ** 3 + 30.0 * m * m}
    if kind == "regrid":
        return {"bytes": 48.0 * case["n"], "flops": 16.0 * 20.0 * case["n"]}
    sizes = workloads.uneven_sizes(case["count"], case["lo"], case["hi"], case["mix"])
    n = float(sizes.sum())
    return {"bytes": 48.0 * n, "flops": sum(_fmm_flops(float(k), float(k)) for k in sizes)
            + 16.0 * 20.0 * n}


def tolerance(case):
    """About four times what these paths differ by from exact(), or from the
    float64 1e-12 class where there is no exact()."""
    kind = case["kind"]
    f32 = case.get("prec") == "f32c"
    tight = case.get("tol", 1e-6) < 1e-9
    if kind in ("direct", "device"):
        # float64 pairs in another order; float32 pairs with compensated sums
        return {"rel": 5e-7, "max": 1e-5} if f32 else {"rel": 1e-14, "max": 1e-12}
    if kind == "evaluate":
        # the measured orders meet their tolerance with little to spare
        return {"rel": 2e-12, "max": 1e-10} if tight else {"rel": 1e-6, "max": 3e-5}
    if kind == "fmm":
        # the order that the reference's rule gives for 1e-6 is better than that
        return {"rel": 1e-6, "max": 2e-5} if f32 else {"rel": 5e-8, "max": 2e-6}
    if kind in ("steps", "sweep"):
        # a velocity error moves a blob by dt times it, which changes the
        # weights of its cells by that over h
        return {"rel": 1e-13, "max": 1e-11} if tight else {"rel": 2e-8, "max": 4e-7}
    if kind == "cylinder":
        return {"rel": 1e-12, "max": 1e-10} if tight else {"rel": 4e-8, "max": 6e-7}
    if kind == "body":
        return {"rel": 3e-13, "max": 3e-13}  # float64 times the condition number
    return {"rel": 2e-15, "max": 1e-13}  # regrid: some 16 blobs per cell, float64
