"""Workloads of trans_bl_amd, timed through its public entry points.

Each case is a call that a DNS program makes, on synthetic inputs of the kinds the tests and the benchmark use:
wavepackets on the wall-stretched grid (uniform dx, geometric y), an analytic boundary-layer base flow, modes kz = k beta.

  derivs   Context.derivs_dev: d/dx, d2/dx2, d/dy, d2/dy2 of one field
  solve    Context.solve_rhs_dev: the v-Poisson solve of every mode from zero to a residual
  rhs      Context.drv_gv_dev: the vorticity right-hand side, linear (kphys 0) or with the nonlinear terms (kphys z points)
  step     Context.rk4_step_dev: one RK4 time step (four right-hand sides, updates and `loop` calls), plain FP64
  net      guess.Net: the U-Net of the learned start, forward and forward + backward

Returned are the fields that a call writes.  Cycle counts and residuals are the stopping test's diagnostics and are not
returned: a mode whose residual lies at the tolerance may take a cycle more or less by the last bit.
"""
import functools
import json
import math
import os
from fractions import Fraction

import numpy as np
import torch

import trans_bl_amd as tb
from trans_bl_amd import autotune, guess

RE, DT, TOL = 33124.00001004055, 1e-4, 1e-9
FIELDS = ("ux", "uy", "uz", "wx", "wy", "wz")
BASE = ("uxb", "uyb", "wzb", "varg", "dvargdx")


def _grid(name, kind, nx, ny, modes, dx, dy0, stf, beta, levels=4, **more):
    return dict(name=name, kind=kind, nx=nx, ny=ny, modes=modes, levels=levels, dx=dx, dy0=dy0, stf=stf, beta=beta, **more)


SMALL = dict(dx=0.02, dy0=5e-4, stf=1.02, beta=0.2)
BATCH = dict(dx=0.02, dy0=2e-4, stf=1.015, beta=0.1)
LARGE = dict(dx=0.02, dy0=2e-4, stf=1.012, beta=0.05)


def listed():
    return [
        # a coarse trial grid: launch latency
        _grid("derivs small", "derivs", 129, 33, 4, 0.03, 1e-3, 1.03, 0.6),
        # an odd mid-size grid, no line a multiple of the wavefront
        _grid("derivs odd", "derivs", 777, 145, 20, **SMALL),
        # the production grid of the benchmark
        _grid("derivs batch", "derivs", 1025, 193, 64, **BATCH),
        # lines of the largest grid (longer than one wavefront's on-chip line)
        _grid("derivs long lines", "derivs", 2049, 257, 32, **LARGE),
        # a single small problem in the reference's arithmetic, as the shipped defaults run it
        _grid("solve small fp64", "solve", 385, 97, 8, **SMALL, precision=0, fmg=0, nu1=0, ncoarse=0, tuned=False),
        # the batched solve in the reference's arithmetic, line shapes from the committed tuning table as the benchmark sets them
        _grid("solve batch fp64", "solve", 1025, 193, 64, **BATCH, precision=0, fmg=0, nu1=0, ncoarse=0, tuned=True),
        # the batched solve in the benchmark's mixed form
        _grid("solve batch mixed", "solve", 1025, 193, 64, **BATCH, precision=1, fmg=1, nu1=3, ncoarse=3, tuned=True),
        # the largest grid, mixed form of the stage benchmark
        _grid("solve large mixed", "solve", 2049, 257, 128, **LARGE, precision=1, fmg=1, nu1=3, ncoarse=0, tuned=True),
        # the right-hand side with the nonlinear terms on the production grid
        _grid("rhs nonlinear", "rhs", 1025, 193, 64, **BATCH, kphys=128),
        # a whole time step on the production grid (linear terms, as the reference's drv_gv)
        _grid("rk4 step", "step", 1025, 193, 64, **BATCH, kphys=0, tuned=True),
        # the learned start's prediction for 64 modes on the 129x25 coarsest level
        dict(name="net forward", kind="net", H=32, W=136, N=64, backward=False),
        # one training batch: loss, parameter and input gradients
        dict(name="net gradients", kind="net", H=32, W=136, N=32, backward=True),
    ]


def draw(rng):
    def log(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    kind = rng.choice(["derivs", "derivs", "solve", "solve", "rhs", "step", "net"])
    if kind == "net":
        while True:
            H, W, N = 8 * rng.randint(2, 5), 8 * int(round(log(3, 33))), int(round(log(1, 64)))
            if H * W * N <= 32 * 136 * 64:
                return dict(kind="net", H=H, W=W, N=N, backward=bool(N <= 32 and rng.random() < 0.5))
    most = {"derivs": 2049 * 257 * 32, "solve": 2049 * 257 * 64, "rhs": 1025 * 193 * 64, "step": 1025 * 193 * 64}[kind]
    while True:
        nx, ny, modes = 8 * int(round(log(10, 256))) + 1, 8 * rng.randint(4, 32) + 1, int(round(log(1, 128)))
        if nx * ny * modes <= most and not (kind in ("rhs", "step") and modes > 64):
            break
    stf = 1.03 if ny <= 65 else 1.02 if ny <= 129 else 1.015 if ny <= 193 else 1.012
    c = dict(kind=kind, nx=nx, ny=ny, modes=modes, levels=4, dx=rng.choice([0.02, 0.03]), dy0=rng.choice([2e-4, 5e-4]),
             stf=stf, beta=rng.choice([0.05, 0.1, 0.2]))
    if kind == "solve":
        p = rng.randint(0, 1)
        f = p and rng.randint(0, 1)
        c.update(precision=p, fmg=f, nu1=3 if f else 0, ncoarse=0, tuned=bool(rng.randint(0, 1)))
    if kind == "step":
        c.update(tuned=bool(rng.randint(0, 1)))
    if kind in ("rhs", "step"):
        c["kphys"] = rng.choice([0, max(4, 1 << math.ceil(math.log2(2 * modes)))]) if kind == "rhs" else 0
    return c


# ---- inputs ---------------------------------------------------------------------------------------------------------
def _xy(c):
    x = c["dx"] * torch.arange(c["nx"], dtype=torch.float64, device="cuda")
    j = torch.arange(c["ny"], dtype=torch.float64, device="cuda")
    return x, c["dy0"] * (c["stf"] ** j - 1.0) / (c["stf"] - 1.0)


def _packets(c, seed, field=0, scale=1.0):
    """Complex (modes, ny, nx): six Gaussian wavepackets per mode and part."""
    x, y = _xy(c)
    rng = np.random.default_rng([int(seed) & 0x7FFFFFFF, field])
    lx, ytop, shape = float(x[-1]), float(y[-1]), (c["modes"], 2, 6)
    amp, sig, alp, xc, yc = (torch.as_tensor(a, device="cuda") for a in (
        rng.normal(size=shape) * scale, rng.uniform(0.05, 0.3, shape), rng.uniform(10.0, 30.0, shape),
        rng.uniform(0.1 * lx, 0.9 * lx, shape), rng.uniform(0.0, 0.5 * ytop, shape)))
    out = torch.zeros((c["modes"], c["ny"], c["nx"]), dtype=torch.complex128, device="cuda")
    for k in range(c["modes"]):
        parts = []
        for q in range(2):
            a, s, w, u, v = (t[k, q, :, None] for t in (amp, sig, alp, xc, yc))
            gx = torch.exp(-(x - u) ** 2 / (2 * s * s)) * torch.cos(w * x)
            gy = a * torch.exp(-(y - v) ** 2 / (2 * s * s))
            parts.append(gy.T @ gx)
        torch.complex(*parts, out=out[k])
    return out


def _base(c):
    x, y = _xy(c)
    X, Y = torch.meshgrid(x, y, indexing="xy")
    d = 0.002 * torch.sqrt(X + 1)
    b = dict(uxb=torch.tanh(Y / d), uyb=0.01 * (1 - torch.exp(-Y / d)), wzb=-(1 - torch.tanh(Y / d) ** 2) / d,
             varg=0.05 + 0.01 * X, dvargdx=0.01 + 0 * X)
    return {k: v.contiguous() for k, v in b.items()}


def _fields(c, seed):
    return {k: _packets(c, seed, q, 0.1 if k[0] == "w" else 1.0) for q, k in enumerate(FIELDS)}


LAYERS = [  # name, cin, cout, kernel size, level
    ("E0A", 4, 32, 3, 0), ("E0B", 32, 32, 3, 0), ("E1A", 32, 64, 3, 1), ("E1B", 64, 64, 3, 1), ("E2A", 64, 128, 3, 2),
    ("E2B", 128, 128, 3, 2), ("E3A", 128, 256, 3, 3), ("E3B", 256, 256, 3, 3), ("D2A", 384, 128, 3, 2),
    ("D2B", 128, 128, 3, 2), ("D1A", 192, 64, 3, 1), ("D1B", 64, 64, 3, 1), ("D0A", 96, 32, 3, 0), ("D0B", 32, 32, 3, 0),
    ("OUT", 32, 2, 1, 0)]


def _net_inputs(c, seed):
    """He-normal weights, images of scaled wavepackets with the kz and y channels, targets of the same kind."""
    g = torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)
    theta = []
    for name, cin, cout, ks, _ in LAYERS:
        sd = math.sqrt(2.0 / (ks * ks * cin)) * (0.1 if name == "OUT" else 1.0)
        theta.append(sd * torch.randn(ks * ks * cin * cout, generator=g, device="cuda"))
        theta.append(0.01 * torch.randn(cout, generator=g, device="cuda"))
    N, H, W = c["N"], c["H"], c["W"]
    u = lambda lo, hi: lo + (hi - lo) * torch.rand((N, 4, 6, 1, 1), generator=g, device="cuda")  # noqa: E731
    y, x = torch.arange(H, device="cuda")[:, None] / H, torch.arange(W, device="cuda")[None, :] / W
    p = (u(-1, 1) * torch.exp(-((x - u(0.1, 0.9)) ** 2 + (y - u(0, 0.5)) ** 2) / (2 * u(0.02, 0.1) ** 2))
         * torch.cos(u(20, 120) * x)).sum(2)
    p = p / p.abs().amax((2, 3), keepdim=True)
    kz = torch.linspace(0, 1, N, device="cuda")[:, None, None].expand(N, H, W)
    img = torch.stack([p[:, 0], p[:, 1], kz, y.expand(N, H, W)], dim=-1)
    return torch.cat(theta), img.float().contiguous(), p[:, 2:].permute(0, 2, 3, 1).float().contiguous()


# ---- the program's state and one pass -------------------------------------------------------------------------------
def _context(c):
    ctx = tb.Context(tb.Grid(c["nx"], c["ny"], c["modes"], c["levels"], c["dx"], c["dy0"], c["stf"], 0.0, c["beta"]))
    if c.get("tuned"):
        with open(os.path.join(os.path.dirname(tb.__file__), "weights", "linetune.json")) as f:
            autotune.apply(ctx, json.load(f))
    return ctx


def prepare(case, seed):
    c = case
    s = {"case": c}
    if c["kind"] == "net":
        theta, s["x"], s["t"] = _net_inputs(c, seed)
        s["net"] = guess.Net(c["H"], c["W"], c["N"])
        s["net"].set_params(theta.cpu().numpy())
        s["y"] = torch.zeros_like(s["t"])
        s["gx"] = torch.zeros_like(s["x"])
    else:
        s["ctx"] = _context(c)
        if c["kind"] in ("derivs", "solve"):
            s["f"] = _packets(c, seed)
            s["out"] = [torch.zeros_like(s["f"]) for _ in range(4 if c["kind"] == "derivs" else 1)]
        else:
            s["start"], s["base"] = _fields(c, seed), _base(c)
            s["fields"] = {k: v.clone() for k, v in s["start"].items()}
            if c["kind"] == "rhs":
                s["out"] = [torch.zeros_like(v) for _, v in zip(range(3), s["start"].values())]
            else:
                bd = tb.bdfc_generate(c["nx"], 10, int(c["nx"] * 0.785), int(c["nx"] * 0.88))
                s["bdfc"] = torch.from_numpy(bd).to("cuda")
                s["d2"] = torch.zeros((c["modes"], c["nx"]), dtype=torch.complex128, device="cuda")
    torch.cuda.synchronize()
    return s


def run(s):
    c = s["case"]
    if c["kind"] == "net":
        if not c["backward"]:
            s["net"].forward(s["x"].data_ptr(), s["y"].data_ptr(), c["N"])
            return s["y"]
        loss, g = s["net"].gradients(s["x"].data_ptr(), s["t"].data_ptr(), c["N"], s["gx"].data_ptr())
        return {"loss": np.float32(loss), "params": g, "input": s["gx"]}
    ctx = s["ctx"]
    if c["kind"] == "derivs":
        ctx.derivs_dev(s["f"].data_ptr(), *[o.data_ptr() for o in s["out"]])
        return s["out"]
    if c["kind"] == "solve":
        ctx.solve_rhs_dev(s["f"].data_ptr(), s["out"][0].data_ptr(), TOL, precision=c["precision"], max_cycles=20, nu1=c["nu1"],
                          ncoarse=c["ncoarse"], use_graph=1, guess=1, fmg=c["fmg"])
        return s["out"]
    base = {k: v.data_ptr() for k, v in s["base"].items()}
    if c["kind"] == "rhs":
        ctx.drv_gv_dev(RE, c["kphys"], base, *[s["fields"][k].data_ptr() for k in FIELDS], *[o.data_ptr() for o in s["out"]])
        return s["out"]
    # the step updates its fields in place: every pass starts from the same ones
    for k in FIELDS:
        s["fields"][k].copy_(s["start"][k])
    ctx.rk4_step_dev(RE, DT, c["kphys"], base, s["bdfc"].data_ptr(), s["d2"].data_ptr(),
                     {k: s["fields"][k].data_ptr() for k in FIELDS}, precision=0, use_graph=1)
    return s["fields"]


def work(case):
    c = case
    if c["kind"] == "net":
        px = c["N"] * c["H"] * c["W"]
        flops = sum(2.0 * ks * ks * cin * cout * px / 4 ** lvl for _, cin, cout, ks, lvl in LAYERS)
        nparam = sum((ks * ks * cin + 1) * cout for _, cin, cout, ks, _ in LAYERS)
        return dict(bytes=4.0 * (px * 6 + nparam), flops=flops) if not c["backward"] else \
            dict(bytes=4.0 * (px * 10 + 2 * nparam), flops=3 * flops)
    n = c["nx"] * c["ny"] * c["modes"]
    if c["kind"] == "derivs":
        return dict(bytes=16.0 * 5 * n, flops=100.0 * n)
    if c["kind"] == "solve":
        # the source read and the solution written once; a handful of stencil applications and line solves
        return dict(bytes=32.0 * n, flops=1000.0 * n)
    if c["kind"] == "rhs":
        fft = 10 * 2.5 * c["kphys"] * math.log2(c["kphys"]) / c["modes"] if c["kphys"] else 0.0
        return dict(bytes=16.0 * 9 * n, flops=(500.0 + fft) * n)
    return dict(bytes=16.0 * 12 * n, flops=8000.0 * n)


# ---- the same in 64 bits, by plain torch ----------------------------------------------------------------------------
def _moments(lhs, rhs, fixed, degree):
    """Weights of sum_u lhs f^(q_u)(h_u) = sum_u rhs f(h_u), exact on polynomials up to `degree` with the weights `fixed`
    given: rational elimination, rounded once."""
    cols = [(1, q, h) for q, h in lhs] + [(-1, q, h) for q, h in rhs]
    m = []
    for p in range(degree + 1):
        m.append([s * h ** (p - q) / math.factorial(p - q) if p >= q else Fraction(0) for s, q, h in cols] + [Fraction(0)])
    for i, v in fixed.items():
        m.append([Fraction(int(i == k)) for k in range(len(cols))] + [Fraction(v)])
    n = len(cols)
    for a in range(n):
        b = next(r for r in range(a, n) if m[r][a] != 0)
        m[a], m[b] = m[b], m[a]
        m[a] = [v / m[a][a] for v in m[a]]
        for r in range(n):
            if r != a and m[r][a] != 0:
                m[r] = [v - m[r][a] * w for v, w in zip(m[r], m[a])]
    return [float(row[n]) for row in m]


def _heights(steps, sign=1):
    out, at = [], Fraction(0)
    for s in steps:
        at += s
        out.append(sign * at)
    return out


def _y_schemes(stf, order):
    """Rows (first, second, centre, last but one, last) of the compact y scheme of f' (order 1) or f'' (order 2): weights
    on the derivatives and on the values, each with the offset of its row's first value."""
    s, d = Fraction(stf), order
    up = _heights([s ** k for k in range(4 if d == 1 else 5)])
    down = _heights([s ** k for k in reversed(range(4 if d == 1 else 5))], -1)
    zero, one = Fraction(0), Fraction(1)
    F = lambda hs: [(0, h) for h in hs]  # noqa: E731
    if d == 1:
        first = [12.0] + _moments([(1, zero)], F([zero] + up), {0: 12}, 4)[1:]
    else:
        first = _moments([(2, zero), (2, up[0])], F([zero] + up), {0: 1}, 6)
    above = _heights([s ** k for k in range(1, 5 if d == 1 else 6)])
    key = {0: 1, 4: Fraction(-5, 2)} if d == 1 else {0: 1, 5: Fraction(21, 4)}
    second = _moments([(d, -one), (d, zero), (d, above[0])], F([-one, zero] + above), key, 6 if d == 1 else 7)
    pts = [-(1 + s), -s, zero, s * s, s * s + s ** 3]
    centre = _moments([(d, pts[1]), (d, zero), (d, pts[3])], F(pts), {1: 1}, 6)
    top = s ** (4 if d == 1 else 5)
    key = {0: 1, 4: Fraction(5, 2)} if d == 1 else {0: 1, 5: Fraction(21, 4)}
    lastbut = _moments([(d, top), (d, zero), (d, down[0])], F([top, zero] + down), key, 6 if d == 1 else 7)
    last = _moments([(d, zero), (d, down[0])], F([zero] + down), {0: 1}, 5 if d == 1 else 6)
    return first, second, centre, lastbut, last


@functools.lru_cache(maxsize=2)
def _dy(ny, dy0, stf, order):
    """The dense y derivative."""
    first, second, centre, lastbut, last = _y_schemes(stf, order)
    q = [1.0 / (dy0 * stf ** j) ** order for j in range(ny - 1)]
    A, B = np.zeros((ny, ny)), np.zeros((ny, ny))
    n, w = ny - 1, 5 if order == 1 else 6
    if order == 1:
        A[0, 0], B[0, :5] = first[0], np.array(first[1:]) * q[0]
    else:
        A[0, :2], B[0, :6] = first[:2], np.array(first[2:]) * q[0]
    A[1, :3], B[1, :w + 1] = second[:3], np.array(second[3:]) * q[0]
    for j in range(2, n - 1):
        A[j, j - 1:j + 2], B[j, j - 2:j + 3] = centre[:3], np.array(centre[3:]) * q[j - 2]
    A[n - 1, n - 2:n + 1] = [lastbut[2], lastbut[1], lastbut[0]]
    B[n - 1, n - w:n + 1] = np.array(lastbut[3:])[::-1] * q[n - w]
    A[n, n - 1:n + 1] = [last[1], last[0]]
    B[n, n - w + 1:n + 1] = np.array(last[2:])[::-1] * q[n - w + 1]
    return torch.as_tensor(np.linalg.solve(A, B), device="cuda")


@functools.lru_cache(maxsize=2)
def _dx(nx, dx, order):
    """The dense x derivative."""
    A, B = np.zeros((nx, nx)), np.zeros((nx, nx))
    for i in range(2, nx - 2):
        A[i, i - 1:i + 2] = (1, 3, 1) if order == 1 else (2, 11, 2)
        B[i, i - 2:i + 3] = np.array((-1, -28, 0, 28, 1)) / 12 if order == 1 else np.array((3, 48, -102, 48, 3)) / 4
    if order == 1:
        A[0, 0], A[1, :3] = 1, (1, 6, 2)
        B[0, :5], B[1, :6] = np.array((-25, 48, -36, 16, -3)) / 12, np.array((-406, -300, 760, -80, 30, -4)) / 120
        A[-1, -2:], A[-2, -3:] = (4, 1), (2, 6, 1)
        B[-1, -5:], B[-2, -6:] = np.array((2, -16, 72, 16, -74)) / -24, np.array((-4, 30, -80, 760, -300, -406)) / -120
    else:
        A[0, :2], A[1, :3] = (13, 137), (1, 12, 3)
        B[0, :6] = np.array((9775, -20285, 11170, -550, -145, 35)) / 60
        B[1, :7] = np.array((4834, -8424, 1890, 2320, -810, 216, -26)) / 360
        A[-1, -2:], A[-2, -3:] = (137, 13), (3, 12, 1)
        B[-1, -6:], B[-2, -7:] = B[0, 5::-1], B[1, 6::-1]
    return torch.as_tensor(np.linalg.solve(A, B) / dx ** order, device="cuda")


def _along(D, f, axis):
    """D applied along y (axis 1) or x (axis 2) of a complex (modes, ny, nx) field, a mode at a time."""
    out = torch.empty_like(f)
    for k in range(f.shape[0]):
        re, im = f[k].real, f[k].imag
        out[k] = torch.complex(D @ re, D @ im) if axis == 1 else torch.complex(re @ D.T, im @ D.T)
    return out


def _four(c, f, which="x xx y yy"):
    D = {"x": (_dx, (c["nx"], c["dx"], 1), 2), "xx": (_dx, (c["nx"], c["dx"], 2), 2),
         "y": (_dy, (c["ny"], c["dy0"], c["stf"], 1), 1), "yy": (_dy, (c["ny"], c["dy0"], c["stf"], 2), 1)}
    return [_along(D[w][0](*D[w][1]), f, D[w][2]) for w in which.split()]


def _solution(c, f):
    """The discrete v-Poisson problem by diagonalising its x part: Bw v X' + C_k v = S on the columns 2..nx-1."""
    nx, ny, s = c["nx"] - 2, c["ny"], Fraction(c["stf"])
    zero, one = Fraction(0), Fraction(1)
    F = lambda hs: [(0, h) for h in hs]  # noqa: E731
    sp = _moments([(1, -one), (2, zero), (2, s)], F([-one, zero, s, s + s * s]), {1: Fraction(4, 5)}, 5)
    pts = [-(1 + s), -s, zero, s * s, s * s + s ** 3]
    cp = _moments([(2, -s), (2, zero), (2, s * s)], F(pts), {1: Fraction(11, 15)}, 6)
    pp = _moments([(2, zero)], F([-one, zero, s]), {0: 1}, 2)
    lp = _moments([(2, zero)], [(1, zero)] + F([zero, -s, -(s + 1)]), {0: 1}, 3)
    q2 = [1.0 / (c["dy0"] * c["stf"] ** j) ** 2 for j in range(ny - 1)]
    Bw, C = np.zeros((ny, ny)), np.zeros((ny, ny))
    Bw[1, 1:3], C[1, 0:4] = sp[1:3], np.array(sp[3:7]) * q2[0]
    for j in range(2, ny - 2):
        Bw[j, j - 1:j + 2], C[j, j - 2:j + 3] = cp[:3], np.array(cp[3:8]) * q2[j - 2]
    Bw[ny - 2, ny - 2], C[ny - 2, ny - 3:ny] = 1.0, np.array(pp[1:4]) * q2[ny - 3]
    Bw[ny - 1, ny - 1], C[ny - 1, ny - 3:ny] = 1.0, np.array((lp[4], lp[3], lp[2])) * q2[ny - 3]
    X = np.zeros((nx, nx))
    for i in range(nx):
        for o, w in zip(range(-2, 3), (-1, 16, -30, 16, -1)):
            if 0 <= i + o < nx:
                X[i, i + o] = w
    X[0, :5], X[-1, -5:] = (-15, -4, 14, -6, 1), (1, -6, 14, -4, -15)
    lam, P = torch.linalg.eig(torch.as_tensor(X / (12 * c["dx"] ** 2)))
    lam, P, Pi = lam.cuda(), P.cuda(), torch.linalg.inv(P).cuda()
    Bw, C = (torch.as_tensor(a[1:, 1:], dtype=torch.complex128, device="cuda") for a in (Bw, C))
    S = Bw.clone()
    S[-1] = 0
    out = torch.zeros_like(f)
    for k in range(c["modes"]):
        kz = k * c["beta"]
        Ck = C - kz * kz * Bw
        Ck[-1, -1] -= lp[1] * math.sqrt(q2[ny - 3]) * kz
        w = (S @ f[k, 1:, 1:-1]) @ Pi.T
        A = lam[:, None, None] * Bw + Ck
        out[k, 1:, 1:-1] = torch.linalg.solve(A, w.T[:, :, None])[:, :, 0].T @ P.T
    return out


def _rhs(c, seed):
    f, b = _fields(c, seed), _base(c)
    ux, uy, uz, wx, wy, wz = (f[k] for k in FIELDS)
    t = [b["uyb"] * wx - wy * b["uxb"], b["uxb"] * wz + ux * b["wzb"], -b["uyb"] * wz - uy * b["wzb"], 2 * b["uxb"] * ux]
    if c["kphys"]:
        K, N = c["modes"], c["kphys"]
        for j in range(c["ny"]):
            def physical(a):
                spec = torch.zeros((N // 2 + 1, c["nx"]), dtype=torch.complex128, device="cuda")
                spec[0], spec[N // 2] = N * a[0, j].real, 0.5 * N * a[0, j].imag
                spec[1:K] = 0.5 * N * a[1:, j].conj()
                return torch.fft.irfft(spec, n=N, dim=0)
            u, v, w, p, q, r = (physical(a) for a in (ux, uy, uz, wx, wy, wz))
            for a, z in zip(t, (v * p - u * q, u * r - w * p, w * q - v * r, u * u)):
                m = torch.fft.rfft(z, dim=0)[:K].conj() * (2.0 / N)
                m[0] = 0.5 * m[0].real
                parts = [torch.where(x.abs() < 1e-14, torch.zeros_like(x), x) for x in (m.real, m.imag)]
                a[:, j] += torch.complex(*parts)
    k = torch.arange(c["modes"], dtype=torch.float64, device="cuda")[:, None, None] * c["beta"]
    a, bb, cc, d = t
    one = lambda g, w: _four(c, g, w)[0]  # noqa: E731
    lap = lambda g: (one(g, "xx") + one(g, "yy") - k * k * g) / RE  # noqa: E731
    out = [-one(a, "y") - 1j * k * bb + b["varg"] * 1j * k * d + lap(wx), 1j * k * cc + one(a, "x") + lap(wy),
           -one(bb, "x") + one(cc, "y") + b["varg"] * one(d, "x") + b["dvargdx"] * d + lap(wz)]
    for o in out:
        o[:, 0] = 0
    return out


def _unet(theta, x):
    p, at = {}, 0
    for name, cin, cout, ks, _ in LAYERS:
        n = ks * ks * cin * cout
        p[name] = (theta[at:at + n].reshape(ks * ks, cin, cout).permute(2, 1, 0).reshape(cout, -1), theta[at + n:at + n + cout])
        at += n + cout

    def conv(name, a):
        N, _, H, W = a.shape
        col = torch.nn.functional.unfold(a, 3, padding=1) if name != "OUT" else a.reshape(N, -1, H * W)
        w, b = p[name]
        z = torch.stack([w @ m for m in col]) + b[:, None]
        z = z.reshape(N, -1, H, W)
        return torch.relu(z) if name != "OUT" else z

    def two(a, n):
        return conv(n + "B", conv(n + "A", a))

    def half(a):
        return 0.25 * (a[:, :, ::2, ::2] + a[:, :, 1::2, ::2] + a[:, :, ::2, 1::2] + a[:, :, 1::2, 1::2])

    def join(a, skip):
        return torch.cat([a.repeat_interleave(2, 2).repeat_interleave(2, 3), skip], 1)

    a0 = two(x.permute(0, 3, 1, 2), "E0")
    a1 = two(half(a0), "E1")
    a2 = two(half(a1), "E2")
    b = two(join(two(half(a2), "E3"), a2), "D2")
    b = two(join(two(join(b, a1), "D1"), a0), "D0")
    return conv("OUT", b).permute(0, 2, 3, 1)


def exact(case, seed):
    c = case
    if c["kind"] == "net":
        theta, x, t = _net_inputs(c, seed)
        theta, x, t = (a.double() for a in (theta, x, t))
        if not c["backward"]:
            with torch.no_grad():
                return _unet(theta, x)
        theta.requires_grad_(True)
        # image by image: the loss is their mean
        loss = 0.0
        for n in range(c["N"]):
            part = ((_unet(theta, x[n:n + 1]) - t[n:n + 1]) ** 2).sum() / t.numel()
            part.backward()
            loss += float(part)
        # the input's gradient crosses every layer's rectifier, whose bf16 side differs: no 64-bit value to hold it to
        return {"loss": np.float64(loss), "params": theta.grad.cpu().numpy(), "input": None}
    if c["kind"] == "derivs":
        return _four(c, _packets(c, seed))
    if c["kind"] == "rhs":
        return _rhs(c, seed)
    # a direct solve takes too long on the larger grids; a time step has no closed form in this file
    if c["kind"] == "solve" and c["nx"] <= 520 and c["nx"] * c["ny"] * c["modes"] <= 2e6:
        return [_solution(c, _packets(c, seed))]
    return None
