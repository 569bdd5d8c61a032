"""The work that programs on this framework do, as cases to be timed.

A case is one pass through the public entry points (GpuBox, Ensemble, the
C-ABI operators) over the sizes the framework is used at: from a box whose
substep is all launch latency to the 1536 x 315 x 1024 box, FP64 and mixed
precision, z lengths that are powers of two and that are not, odd numbers of
planes and rows.

* step: `steps` whole RK3 steps of one box (one hipGraph per substep), then
  its fields fetched, as a program does that writes a restart file every so
  many steps.  A mixed box's fields are stored as 4-byte reals, as the
  restart file holds them.
* ensemble: the same for several uneven boxes advanced together.
* stats: one statistics sample of the current state, then the accumulators
  and the enstrophy field of the sample.
* xlines, ylines, spectral: the operators on device buffers (x lines; y
  lines; z transforms of rows and cosine transforms of lines), each
  direction the path has.
"""
import ctypes
import math
from dataclasses import replace

import numpy as np
import torch

from opentbl_amd import config, ic
from opentbl_amd.lib import FIELDS, NSTAT, OTBL_FP64, OTBL_MIXED, PD, Ensemble, GpuBox, check, lib

FIELD_NAMES = ("u", "v", "w", "p")


def listed():
    return [
        # smallest box of the tests: launches and single-block kernels
        {"name": "step-32x40x24-fp64", "kind": "step", "nx": 32, "ny": 40, "nz": 24, "mixed": False, "steps": 10},
        # the reference method's own CPU-sized box
        {"name": "step-256x96x64-fp64", "kind": "step", "nx": 256, "ny": 96, "nz": 64, "mixed": False, "steps": 10},
        # ragged sizes: odd planes and rows, a z length of 2 * 7 * 7
        {"name": "step-387x113x98-mixed", "kind": "step", "nx": 387, "ny": 113, "nz": 98, "mixed": True, "steps": 10},
        # members of the uneven ensemble, each precision
        {"name": "step-640x144x160-mixed", "kind": "step", "nx": 640, "ny": 144, "nz": 160, "mixed": True, "steps": 10},
        {"name": "step-896x176x224-fp64", "kind": "step", "nx": 896, "ny": 176, "nz": 224, "mixed": False, "steps": 5},
        # production-like FP64 box
        {"name": "step-1024x192x512-fp64", "kind": "step", "nx": 1024, "ny": 192, "nz": 512, "mixed": False,
         "steps": 5},
        # the benchmark's box
        {"name": "step-1536x315x1024-mixed", "kind": "step", "nx": 1536, "ny": 315, "nz": 1024, "mixed": True,
         "steps": 8},
        # uneven boxes advanced in one graph per substep
        {"name": "ensemble-4-mixed", "kind": "ensemble", "boxes": "256x96x64 384x112x96 512x128x128 640x144x160",
         "mixed": True, "steps": 10},
        # a statistics sample (FP64), as a production run takes every few steps
        {"name": "stats-1024x192x256-fp64", "kind": "stats", "nx": 1024, "ny": 192, "nz": 256},
        # 98,304 x lines of 1024 points
        {"name": "xlines-98304x1024", "kind": "xlines", "nx": 1024, "ny": 192, "nz": 768},
        # y columns of 315 rows, 512 planes
        {"name": "ylines-512x315x512", "kind": "ylines", "nx": 512, "ny": 315, "nz": 512},
        # z rows of 1024 points and x lines of 1535 points
        {"name": "spectral-1024-1535", "kind": "spectral", "nx": 1536, "ny": 40, "nz": 1024, "rows": 150000},
    ]


# even z lengths of factors 2, 3, 5, 7
NZ = [n for n in range(12, 1025, 2) if any(n == 2 ** a * 3 ** b * 5 ** c * 7 ** d for a in range(1, 11)
                                           for b in range(7) for c in range(5) for d in range(4))]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_box(rng, top, mixed):
    """Proportions of the framework's configurations: ny 0.16 to 0.4 of nx, nz
    0.2 to 0.75."""
    while True:
        nx = _logint(rng, 192 if mixed else 32, 1280)
        ny = min(320, max(40, int(nx * rng.uniform(0.16, 0.4))))
        x = nx * rng.uniform(0.2, 0.75)
        nz = min(NZ, key=lambda n: (abs(n - x), n))
        if nz >= (64 if mixed else 24) and nx * ny * nz <= top:
            return nx, ny, nz


def draw(rng):
    kind = rng.choice(["step"] * 6 + ["ensemble", "stats", "xlines", "ylines", "spectral"])
    if kind == "step":
        mixed = rng.random() < 0.5
        nx, ny, nz = _draw_box(rng, 1.5e8, mixed)
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "mixed": mixed, "steps": 10 if nx * ny * nz < 4e7 else 5}
    if kind == "ensemble":
        mixed = rng.random() < 0.5
        boxes = [_draw_box(rng, 2e7, mixed) for _ in range(rng.randint(2, 5))]
        return {"kind": kind, "boxes": " ".join("%dx%dx%d" % b for b in boxes), "mixed": mixed, "steps": 10}
    if kind == "stats":
        nx, ny, nz = _draw_box(rng, 5e7, False)
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz}
    # the operators: lines and rows of any number
    while True:
        nx, ny, nz = _logint(rng, 48, 2048), _logint(rng, 40, 320), rng.choice(NZ)
        if 2e5 <= nx * ny * nz <= 1.5e8:
            break
    case = {"kind": kind, "nx": nx, "ny": ny, "nz": nz}
    if kind == "spectral":
        case["rows"] = _logint(rng, 1000, min(300000, 100_000_000 // nz))
    return case


# ---------------------------------------------------------------------------
# boxes and their initial states
# ---------------------------------------------------------------------------
def _config(nx, ny, nz, seed):
    """The spacing and heights of the framework's own production boxes (a
    coarser grid does not hold the flow for the steps of many passes)."""
    Lx = 60.0 * nx / 1024
    Lz = 8.0 if nz <= 512 else 12.0
    re_theta = 300.0 if nx < 512 else 600.0 if nx < 1280 else 1000.0
    kz = max(1, min(64, nz // 3 - 1))
    return config.BoxConfig(f"{nx}x{ny}x{nz}", nx, ny, nz, Lx, 4.0, Lz, re_theta, AMP, kz, "k53", seed, 1).check()


AMP = 0.4  # peak z-rms of the perturbation: a layer past transition


def _mean(cfg):
    """The box's mean flow alone (a Blasius layer), with few z modes."""
    return ic.make_state(replace(cfg, nz=12, kzmax=0), with_perturbation=False)


def _state(cfg):
    """The boundary layer of ic.make_state with its kz^-5/3 perturbation, the
    perturbation formed on the GPU: two streamfunctions per spanwise mode
    (y-z plane for v, w; x-z plane for u, w), each discretely divergence-free
    on the staggered grid."""
    mean = _mean(cfg)
    st = dict(mean)
    nx, ny, mz, K = cfg.nx, cfg.ny, cfg.mz, cfg.kzmax
    rng = np.random.default_rng(cfg.seed)
    cu = lambda a: torch.as_tensor(np.ascontiguousarray(a), device="cuda")  # noqa: E731
    kz = ic.kaz_values(cfg)[1:K + 1]
    ak = np.arange(1, K + 1) ** (-5.0 / 6.0)
    c1, c2 = ((rng.standard_normal(K) + 1j * rng.standard_normal(K)) * ak for _ in range(2))
    m1, m2 = rng.integers(1, 7, K), rng.integers(1, 7, K)
    ph1, ph2 = rng.uniform(0, 2 * math.pi, K), rng.uniform(0, 2 * math.pi, K)
    dx = cfg.ax * math.pi / (nx + 1)
    xs = np.arange(nx) * dx
    gx1 = np.cos(2 * math.pi * np.outer(xs, m1) / cfg.Lx + ph1)
    gx2 = np.cos(2 * math.pi * np.outer(xs, m2) / cfg.Lx + ph2)
    y = mean["y"]
    yv, yu, dy = y[1:ny + 1], 0.5 * (y[:-1] + y[1:]), np.diff(y)
    psi = (yv / 0.5) ** 2 * np.exp(-(yv / 0.5) ** 2)
    chi = (yu / 0.5) ** 2 * np.exp(-(yu / 0.5) ** 2)
    chi[0] = chi[ny] = 0.0
    dpsi = np.zeros(ny + 1)
    dpsi[1:ny] = np.diff(psi) / dy[1:ny]
    dg2 = np.zeros_like(gx2)
    dg2[1:] = np.diff(gx2, axis=0) / dx
    # u = i kz chi g2 c2, v = i kz psi g1 c1, w = -dpsi g1 c1 - chi dg2 c2
    parts = {"u": [(chi, gx2, 1j * kz * c2)], "v": [(psi, gx1, 1j * kz * c1)],
             "w": [(dpsi, gx1, -c1), (chi, dg2, -c2)]}

    def outer(terms):
        return sum(cu(r)[None, :, None] * cu(g)[:, None, :] * cu(c)[None, None, :] for r, g, c in terms)

    peak = max(float((outer(t).abs() ** 2).sum(dim=2).max()) * 2 for t in parts.values()) ** 0.5
    for n, terms in parts.items():
        f = torch.zeros((nx, ny if n == "v" else ny + 1, mz), dtype=torch.complex128, device="cuda")
        f[:, :, 1:K + 1] = outer(terms) * (AMP / peak)
        if n != "w":
            f[:, :, 0] = cu(mean[n][:, :, 0])
        st[n] = f.cpu().numpy()
        del f
    st["p"] = np.zeros((nx, ny, mz), np.complex128)
    torch.cuda.empty_cache()
    return st


def _ptr(t):
    return ctypes.cast(t.data_ptr(), PD)


class _Run:
    """A box (or several) with what a program that steps it and stores its
    fields keeps: page-locked host memory for each field, and for a mixed box
    the 4-byte reals that it stores."""

    def __init__(self, cfg, mixed):
        self.box = GpuBox(cfg, _state(cfg), precision=OTBL_MIXED if mixed else OTBL_FP64, graphs=True)
        n = {f: lib().otbl_field_len(self.box.h, FIELDS[f]) for f in FIELD_NAMES}
        pinned = lambda k: torch.empty(k, dtype=torch.float64, pin_memory=True)  # noqa: E731
        if mixed:
            self.host = dict.fromkeys(n, pinned(max(n.values())))
            self.out = {f: torch.zeros(k, dtype=torch.float32) for f, k in n.items()}
        else:
            self.host = self.out = {f: pinned(k) for f, k in n.items()}

    def fetch(self):
        for f, o in self.out.items():
            h = self.host[f]
            check(lib().otbl_get_field(self.box.h, FIELDS[f], _ptr(h)), "get_field")
            if o is not h:
                o.copy_(h[:o.numel()])
        return self.out


def _rand(shape, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(shape, dtype=torch.float64, device="cuda", generator=g)


def _dims(case):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    return nx, ny, 2 * (nz // 3)


# the operators of a kind: output name, entry point, input names, arguments.
# Fields q.. hold ny+1 rows per plane (u-type), f.. ny rows (v-type).
def _ops(case):
    nx, ny, _ = _dims(case)
    if case["kind"] == "xlines":
        return [("iu", "interpxx", ("q1",), (ny + 1, 1)), ("iv", "interpxx", ("f1",), (ny, 0)),
                ("du", "difvisxx", ("q1", "q2"), (ny + 1, 1)), ("dv", "difvisxx", ("f1", "f2"), (ny, 0))]
    return [("i0", "interpyy", ("q1",), (0, nx)), ("i1", "interpyy", ("f1",), (1, nx)),
            ("d0", "differzy", ("q1",), (0, nx)), ("d1", "differzy", ("q2",), (1, nx)),
            ("vu", "vistyy", ("q1",), (ny + 1, nx)), ("vv", "vistyy", ("f1",), (ny, nx))]


RKK = -0.013  # implzy's implicit viscous factor


def _inputs(case, seed):
    nx, ny, nz1 = _dims(case)
    if case["kind"] == "spectral":
        fou = _rand((case["rows"], nz1), seed)
        return {"fou": fou, "phys": _rand((case["rows"], case["nz"]), seed + 1), "f1": _rand((nx, ny, nz1), seed + 2),
                "f2": _rand((nx, ny, nz1), seed + 3)}
    return {n: _rand((nx, ny + (n[0] == "q"), nz1), seed + k) for k, n in enumerate(("q1", "q2", "f1", "f2"))}


def prepare(case, seed):
    if case["kind"] in ("step", "ensemble"):
        sizes = case["boxes"].split() if case["kind"] == "ensemble" else ["%dx%dx%d" % (case["nx"], case["ny"], case["nz"])]
        runs = [_Run(_config(*map(int, s.split("x")), seed + 100 * k), case["mixed"]) for k, s in enumerate(sizes)]
        state = {"kind": case["kind"], "runs": runs, "steps": case["steps"]}
        state["stepper"] = Ensemble([r.box for r in runs]) if case["kind"] == "ensemble" else runs[0].box
        return state
    nx, ny, nz1 = _dims(case)
    if case["kind"] == "stats":
        cfg = _config(nx, ny, case["nz"], seed)
        box = GpuBox(cfg, _state(cfg), precision=OTBL_FP64, graphs=True)
        box.step(2)  # a pressure field
        box.stats_enable()
        pinned = lambda k, t: torch.empty(k, dtype=t, pin_memory=True)  # noqa: E731
        return {"kind": "stats", "box": box, "acc": pinned((NSTAT, nx, ny + 1), torch.float64),
                "ens": pinned((nx, ny, case["nz"]), torch.float32)}
    # operators: a box that holds the coefficients, buffers on the device
    cfg = _config(nx, ny, case["nz"], seed)
    state = {"kind": case["kind"], "case": case, "box": GpuBox(cfg, _state(cfg)), "in": _inputs(case, seed)}
    if case["kind"] == "spectral":
        out = {"c2r": torch.zeros_like(state["in"]["phys"]), "r2c": torch.zeros_like(state["in"]["fou"]),
               "dct2": torch.zeros_like(state["in"]["f1"]), "dct3": torch.zeros_like(state["in"]["f1"])}
    else:
        rows = {"iu": ny + 1, "du": ny + 1, "iv": ny, "dv": ny, "vv": ny}
        out = {o[0]: torch.zeros((nx, rows.get(o[0], ny + 1), nz1), dtype=torch.float64, device="cuda")
               for o in _ops(case)}
        if case["kind"] == "ylines":
            # boundary rows in, interior rows out
            out["mu"], out["mv"] = state["in"]["q2"].clone(), state["in"]["f2"].clone()
    state["out"] = out
    torch.cuda.synchronize()  # the box works on a stream of its own
    return state


def run(state):
    kind = state["kind"]
    if kind in ("step", "ensemble"):
        state["stepper"].step(state["steps"])
        outs = [r.fetch() for r in state["runs"]]
        return outs[0] if kind == "step" else outs
    box = state["box"]
    if kind == "stats":
        box.statsp()
        for q in range(NSTAT):
            check(lib().otbl_stats_get(box.h, q, _ptr(state["acc"][q])), "stats_get")
        check(lib().otbl_stats_get_ens(box.h, ctypes.cast(state["ens"].data_ptr(), ctypes.POINTER(ctypes.c_float))),
              "stats_get_ens")
        return {"acc": state["acc"], "ens": state["ens"]}
    x, out, case = state["in"], state["out"], state["case"]
    ptr = lambda t: t.data_ptr()  # noqa: E731
    if kind == "spectral":
        rows = case["rows"]
        box.op("fourxz", ptr(x["fou"]), ptr(out["c2r"]), 1, rows)
        box.op("fourxz", ptr(out["r2c"]), ptr(x["phys"]), -1, rows)
        box.op("cosftx", ptr(x["f1"]), ptr(out["dct2"]), -1)
        box.op("cosftx", ptr(x["f2"]), ptr(out["dct3"]), 1)
        return out
    for name, op, ins, args in _ops(case):
        box.op(op, *(ptr(x[i]) for i in ins), ptr(out[name]), *args)
    if kind == "ylines":
        box.op("implzy", ptr(out["mu"]), ptr(x["q1"]), case["ny"] + 1, RKK, case["nx"])
        box.op("implzy", ptr(out["mv"]), ptr(x["f1"]), case["ny"], RKK, case["nx"])
    return out


def work(case):
    if case["kind"] == "ensemble":
        parts = [work(dict(case, kind="step", nx=a, ny=b, nz=c)) for a, b, c in
                 (map(int, s.split("x")) for s in case["boxes"].split())]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    nx, ny, nz1 = _dims(case)
    nz, f = case["nz"], nx * ny * nz1  # values of a field
    row = lambda n: 2.5 * n * math.log2(n)  # noqa: E731  flops of a real transform
    if case["kind"] == "step":
        s = 4 if case["mixed"] else 8
        # a substep reads and writes u, v, w, p and the three right-hand sides;
        # the fields go out once at the end of the pass
        sub = 14 * s * f
        # 18 z transforms per (x, y) row, two x transforms per (y, z) line,
        # 13 compact solves with their explicit parts
        flops = 18 * nx * ny * row(nz) + 2 * ny * nz1 * row(nx) + 13 * 10 * f
        return {"bytes": 3 * case["steps"] * sub + 4 * s * f, "flops": 3 * case["steps"] * flops}
    if case["kind"] == "stats":
        acc = NSTAT * nx * (ny + 1) * 8
        return {"bytes": 4 * 8 * f + 2 * acc + 4 * nx * ny * nz, "flops": 6 * nx * ny * row(nz) + 12 * 10 * f + 100 * f}
    if case["kind"] == "spectral":
        return {"bytes": 8 * (2 * case["rows"] * (nz + nz1) + 4 * f),
                "flops": 2 * case["rows"] * row(nz) + 2 * ny * nz1 * row(nx)}
    arrays = 10 if case["kind"] == "xlines" else 18
    return {"bytes": 8 * arrays * f, "flops": (60 if case["kind"] == "xlines" else 80) * f}


# ---------------------------------------------------------------------------
# the operators in 64 bits
# ---------------------------------------------------------------------------
def _weights(lhs, rhs, deriv):
    """Weights (a, c) of the scheme g(0) + sum a_l g(lhs_l) = sum c_q f(rhs_q),
    g the deriv-th derivative of f, of the highest order the points allow.
    lhs, rhs: arrays (rows, points) of offsets."""
    n, nl = lhs.shape[1] + rhs.shape[1], lhs.shape[1]
    h = np.abs(rhs).max(axis=1, keepdims=True)
    l, r = lhs / h, rhs / h
    m, b = np.zeros((len(h), n, n)), np.zeros((len(h), n, 1))
    for k in range(n):
        falling = math.prod(range(k - deriv + 1, k + 1)) if k >= deriv else 0
        m[:, k, nl:] = r ** k
        if k >= deriv:
            m[:, k, :nl] = -falling * l ** (k - deriv)
            b[:, k, 0] = falling * (k == deriv)
    w = np.linalg.solve(m, b)[:, :, 0]
    return w[:, :nl], w[:, nl:] / h ** deriv


def _end(offsets, deriv):
    return _weights(np.zeros((1, 0)), np.array([offsets]), deriv)[1][0]


def _second_end(a, b, c):
    """f''(0) + w f''(a) = sum c_q f(0, a, a + b, a + b + c)."""
    w, e = _weights(np.array([[a]]), np.array([[0.0, a, a + b, a + b + c]]), 2)
    return w[0, 0], e[0]


def _solve(lo, up, r, diag=None):
    """The tridiagonal systems lo x(j-1) + diag x(j) + up x(j+1) = r along the
    first dimension of r, in place."""
    n = r.shape[0]
    diag = np.ones(n) if diag is None else diag
    q = np.zeros(n)
    for j in range(n):
        piv = diag[j] - (lo[j] * q[j - 1] if j else 0.0)
        q[j] = up[j] / piv
        if j:
            r[j] -= float(lo[j]) * r[j - 1]
        r[j] /= float(piv)
    for j in range(n - 2, -1, -1):
        r[j] -= float(q[j]) * r[j + 1]
    return r


def _compact(points, g, grid, deriv, first, last, rows=None):
    """A compact scheme on the rows of `points` from values g on `grid` (rows
    along the first dimension): interior rows from the row's neighbours and
    the grid points around it (their weights `rows`, or those of the highest
    order), first and last rows given."""
    n = len(points)
    x, i = points, np.arange(1, n - 1)
    nq = 3 if deriv == 2 else 2
    # nearest nq grid points of each interior row
    q0 = np.array([np.argsort(np.abs(grid - p))[:nq].min() for p in x[1:-1]])
    a, c = rows or _weights(np.stack([x[i - 1] - x[i], x[i + 1] - x[i]], 1),
                            np.stack([grid[q0 + k] - x[i] for k in range(nq)], 1), deriv)
    r = torch.empty((n,) + tuple(g.shape[1:]), dtype=g.dtype, device=g.device)
    c = torch.as_tensor(c, device=g.device)[:, :, None]
    flat, gf = r.reshape(n, -1), g.reshape(g.shape[0], -1)
    flat[1:-1] = sum(c[:, k] * gf[q0[0] + k:q0[0] + k + n - 2] for k in range(nq))
    lo, up = np.zeros(n), np.zeros(n)
    lo[1:-1], up[1:-1] = a[:, 0], a[:, 1]
    for j, (off, w, at) in ((0, first), (n - 1, last)):
        flat[j] = sum(float(v) * gf[k] for v, k in zip(w, at))
        lo[j], up[j] = (off, 0.0) if j else (0.0, off)
    return _solve(lo, up, flat).reshape(r.shape)


def _exact_x(case, x):
    nx = case["nx"]
    cfg = _config(nx, case["ny"], case["nz"], 0)
    h = cfg.ax * math.pi / (nx + 1)
    # interpolation to the point half a spacing up (u), or half a spacing
    # down with the points below and above it (v)
    p, out = np.arange(nx) * h, {}
    re = _mean(cfg)["re"]
    up, back = range(4), range(nx - 1, nx - 5, -1)
    for t, f, q in (("u", x["q1"], x["q2"]), ("v", x["f1"], x["f2"])):
        out["i" + t] = _compact(p + 0.5 * h, f, p, 0, (0.0, _end([-0.5 * h, 0.5 * h, 1.5 * h, 2.5 * h], 0), up),
                                (0.0, _end([-0.5 * h, -1.5 * h, -2.5 * h], 0), back))
        d = _compact(p - 0.5 * h, f, p, 1, (0.0, _end([0.5 * h, 1.5 * h, 2.5 * h, 3.5 * h], 1), up),
                     (0.0, _end([0.5 * h, -0.5 * h, -1.5 * h, -2.5 * h], 1), back))
        w, e = _second_end(h, h, h)
        d -= _compact(p, q, p, 2, (w, e, up), (w, e, back)) / re
        d[-1] = (q[-1] - q[-2]) / h
        out["d" + t] = d
    return out


def _y_rows(a, b, c, kind):
    """The interior weights that the method itself has on a stretched grid
    (coeft.f90:514-1168) where they are not those of the highest order: a, b
    spacings, c the one between (interpolation: the cell's)."""
    if kind == "interp":  # u rows from v rows: a above, b the cell, c below
        return (np.stack([c * b * b / ((2 * a + b) * (2 * a - b) * (c + a)), -a * b * b / ((b - 2 * c) * (b + 2 * c) * (c + a))], 1),
                np.stack([2 * c * a / (-b * b + 2 * a * b - 2 * c * b + 4 * c * a),
                          -2 * c * a / (2 * a * b + b * b - 4 * c * a - 2 * c * b)], 1))
    if kind == "first":  # u rows from v rows
        den = -c * c * a - c * c * b + 12 * b * b * a + 12 * b * a * a
        v = 12 * a * b / ((12 * a * b - c * c) * c)
        return np.stack([b * c * c / den, c * c * a / den], 1), np.stack([-v, v], 1)
    den = b ** 3 + a ** 3 + 4 * a * a * b + 4 * a * b * b
    return (np.stack([b * (a * a + a * b - b * b) / den, -a * (a * a - a * b - b * b) / den], 1),
            np.stack([12 * a / den, -12 / (a * a + 3 * a * b + b * b), 12 * b / den], 1))


def _exact_y(case, x):
    nx, ny, _ = _dims(case)
    y = ic.ygrid(_config(nx, ny, case["nz"], 0))
    dy = np.diff(y)  # dy[j] = y[j+1] - y[j]
    dyi = np.zeros(ny + 1)
    dyi[1:] = 0.5 * (dy[1:] + dy[:-1])
    yv, yu = y[1:ny + 1], 0.5 * (y[:-1] + y[1:])
    first = lambda f: f.transpose(0, 1).contiguous()  # noqa: E731
    back = lambda r: r.transpose(0, 1).contiguous()  # noqa: E731
    q1, q2, f1, f2 = (first(x[n]) for n in ("q1", "q2", "f1", "f2"))
    up, uend, vend = range(4), range(ny, ny - 4, -1), range(ny - 1, ny - 5, -1)
    chain = lambda *s: np.cumsum(s)  # noqa: E731  offsets of points one after another
    full = lambda r: torch.cat([r, torch.zeros_like(r[:1])])  # noqa: E731  row ny+1 is not written
    out = {}
    out["i0"] = full(_compact(yv, q1, yu, 0, (0.0, [0.0], [0]),
                              (0.0, _end([-0.5 * dy[ny], *chain(0.5 * dy[ny - 1], dyi[ny - 1], dyi[ny - 2])], 0),
                               uend)))
    out["i1"] = full(_compact(yu[:ny], f1, yv, 0, (0.0, _end(chain(0.5 * dy[0], dy[1], dy[2]), 0), up),
                              (0.0, _end([0.5 * dy[ny - 1], *-chain(0.5 * dy[ny - 1], dy[ny - 2], dy[ny - 3])], 0),
                               vend), _y_rows(dyi[2:ny], dy[1:ny - 1], dyi[1:ny - 1], "interp")))
    out["d0"] = _compact(yu, q1[:ny], yv, 1, (0.0, _end(chain(0.5 * dy[0], dy[1], dy[2], dy[3]), 1), up),
                         (0.0, _end(-chain(0.5 * dy[ny], dy[ny - 1], dy[ny - 2], dy[ny - 3]), 1), vend),
                         _y_rows(dyi[2:ny + 1], dyi[1:ny], dy[1:ny], "first"))
    out["d1"] = full(_compact(yv, q2, yu, 1,
                              (0.0, _end([-0.5 * dy[0], *chain(0.5 * dy[1], dyi[2], dyi[3])], 1), up),
                              (0.0, _end(-chain(0.5 * dy[ny - 1], dyi[ny - 1], dyi[ny - 2], dyi[ny - 3]), 1), vend)))
    for t, g, p, s in (("u", q1, yu, dyi[1:]), ("v", f1, yv, dy[1:ny])):
        lo_end, hi_end = _second_end(*s[:3]), _second_end(*s[:-4:-1])
        n = len(p)
        i = np.arange(1, n - 1)
        rows2 = _y_rows(p[i + 1] - p[i], p[i] - p[i - 1], 0, "second")
        out["v" + t] = _compact(p, g, p, 2, (*lo_end, up), (*hi_end, range(n - 1, n - 5, -1)), rows2)
        # implicit: (A + rkk B) u = A g on the interior rows, A, B the
        # second derivative's two sides; boundary rows kept
        a, c = rows2
        u = (q2 if t == "u" else f2).clone()
        at = torch.as_tensor(a, device=u.device)
        flat = lambda z: z.reshape(n, -1)  # noqa: E731
        G, U = flat(g), flat(u)
        r = at[:, :1] * G[:-2] + G[1:-1] + at[:, 1:] * G[2:]
        lo, di, hi = a[:, 0] + RKK * c[:, 0], 1 + RKK * c[:, 1], a[:, 1] + RKK * c[:, 2]
        r[0] -= float(lo[0]) * U[0]
        r[-1] -= float(hi[-1]) * U[-1]
        U[1:-1] = _solve(lo, hi, r, di)
        out["m" + t] = u
    return {k: back(v) for k, v in out.items()}


def _exact_spectral(case, x):
    nx, ny, nz1 = _dims(case)
    nz, mz, N = case["nz"], nz1 // 2, nx - 1
    fou = torch.view_as_complex(x["fou"].reshape(-1, mz, 2)).clone()
    fou[:, 0] = fou[:, 0].real.to(fou.dtype)
    out = {"c2r": torch.fft.irfft(fou, n=nz) * nz}
    out["r2c"] = torch.view_as_real(torch.fft.rfft(x["phys"])[:, :mz] / nz).reshape(-1, nz1)
    j = torch.arange(N, device="cuda", dtype=torch.float64)
    for name, f, iopt in (("dct2", x["f1"], -1), ("dct3", x["f2"], 1)):
        o = torch.zeros_like(f)
        a = f[1:, :ny - 1]
        if iopt < 0:  # DCT-II: 2 sum a_j cos(pi (j + 1/2) k / N), over N
            z = torch.fft.fft(torch.cat([a, a.flip(0)]), dim=0)[:N]
            o[1:, :ny - 1] = (z * torch.exp(-1j * math.pi * j / (2 * N))[:, None, None]).real / N
        else:  # DCT-III: a_0 + 2 sum a_j cos(pi j (k + 1/2) / N), halved
            z = a * torch.exp(1j * math.pi * j / (2 * N))[:, None, None]
            z[0] *= 0.5
            o[1:, :ny - 1] = torch.fft.ifft(torch.cat([z, torch.zeros_like(z)]), dim=0)[:N].real * 2 * N
        out[name] = o
    return out


def exact(case, seed):
    """The operators' results; none for whole RK3 steps and statistics, whose
    values only another flow solver would give."""
    f = {"xlines": _exact_x, "ylines": _exact_y, "spectral": _exact_spectral}.get(case["kind"])
    return f(case, _inputs(case, seed)) if f else None
