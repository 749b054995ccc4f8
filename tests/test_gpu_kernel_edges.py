"""Kernels at the sizes where they can go wrong: remainders, smallest and
largest of a form's range."""
import numpy as np
import pytest

import oracle
from trans_bl_amd import workload as wl

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_mod(gpu_ready):
    import torch
    return torch


def context(g):
    import trans_bl_amd as tb
    return tb.Context(g)


def rel(a, b):
    return np.max(np.abs(a - b)) / np.max(np.abs(b))


@pytest.mark.parametrize("g", [
    wl.Grid(65, 33, 3, 4, 0.05, 2e-3, 1.03, 0.0, 0.9),      # coarsest 9x5, the smallest
    wl.Grid(89, 41, 2, 4, 0.05, 1e-3, 1.03, 0.1, 0.7),      # 12x6
    wl.Grid(145, 145, 2, 4, 0.03, 3e-4, 1.015, 0.0, 0.3),   # 19x19: 18 rows, two row blocks
    wl.Grid(401, 185, 1, 4, 0.02, 2e-4, 1.015, 0.0, 0.3),   # 51x24: 17 lines, one past a tile
    wl.Grid(257, 65, 2, 2, 0.02, 5e-4, 1.02, 0.0, 0.3),     # 129x33: all 32 rows
    wl.Grid(1025, 33, 2, 2, 0.02, 1e-3, 1.03, 0.0, 0.3)],   # 513x17: 12 wavefronts
    ids=lambda g: f"{g.nx}x{g.ny}x{g.nmodes}l{g.levels}")
@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32"])
def test_coarsest_inverse_form_matches_scan(torch_mod, g, precision):
    """The coarsest level through inverse line matrices (shape 1) against the
    lane scan (shape 16): the iterates after two cycles agree to rounding,
    with wall and boundary-column data (FP64 1e-12 as the other forms of the
    same sweep; FP32 1e-5, single-precision corrections)."""
    f = wl.wavepacket_rhs(g, tag="inverse")
    u = 0.01 * wl.wavepacket_rhs(g, tag="start")
    out = []
    with context(g) as ctx:
        for shape in (1, 16):
            ctx.set_line_shape(precision, g.levels, shape)
            out.append(ctx.poi_uy(None, -f, u, 0.0, precision=precision, max_cycles=2)[0])
    assert rel(out[0], out[1]) < (1e-12 if precision == 0 else 1e-5), rel(out[0], out[1])


# x: every shape (R, W) at or next to its ends; y: every (G, R) likewise
DERIV_GRIDS = [(17, 9), (65, 49), (129, 81), (193, 113), (257, 129), (321, 145), (449, 161), (577, 177), (641, 225),
               (769, 257), (897, 289), (1025, 321), (1153, 33), (1345, 65), (1521, 97), (1729, 33), (1793, 33), (2049, 17),
               (2105, 17), (33, 449), (33, 577)]


@pytest.mark.parametrize("nx, ny", DERIV_GRIDS)
def test_derivatives_at_every_shape(torch_mod, nx, ny):
    """All five derivatives against the oracle (1e-12 of the largest value, as
    the parity tests), on random values: every point of the line counts, and
    the rows past its end must not reach it."""
    torch = torch_mod
    import trans_bl_amd as tb
    g = wl.Grid(nx, ny, 2, 2, 0.02, 1e-3, 1.004, 0.0, 0.3)
    rng = np.random.default_rng(nx + ny)
    f = rng.normal(size=(2, ny, nx)) + 1j * rng.normal(size=(2, ny, nx))
    p = oracle.make_params(g.nx, g.ny, g.nmodes, g.levels, g.dx, g.dy0, g.stf, g.alpha, g.beta)
    with context(g) as ctx:
        fd = torch.from_numpy(f).to("cuda")
        out = [torch.zeros_like(fd) for _ in range(4)]
        ctx.derivs_dev(fd.data_ptr(), *[o.data_ptr() for o in out])
        fv = torch.zeros_like(fd)
        ctx.deriv_dev(tb.DERIV_KINDS["yfv"], fd.data_ptr(), fv.data_ptr())
        ctx.synchronize()
        got = dict(zip(("x", "xx", "y", "yy"), (o.cpu().numpy() for o in out)), yfv=fv.cpu().numpy())
    for kind, v in got.items():
        assert rel(v, oracle.deriv(p, kind, f)) < 1e-12, kind


@pytest.mark.parametrize("nx, ny, nmodes", [(17, 9, 1), (129, 33, 4), (193, 65, 3), (321, 97, 5), (449, 113, 2), (577, 143, 1)],
                         ids=lambda v: str(v))
def test_derivatives_of_small_grids_in_one_launch(torch_mod, nx, ny, nmodes):
    """All four derivatives in one launch against a launch per direction: the
    same arithmetic, equal to the bit."""
    torch = torch_mod
    g = wl.Grid(nx, ny, nmodes, 2, 0.02, 1e-3, 1.004, 0.0, 0.3)
    rng = np.random.default_rng(nx * ny)
    f = rng.normal(size=(nmodes, ny, nx)) + 1j * rng.normal(size=(nmodes, ny, nx))
    with context(g) as ctx:
        fd = torch.from_numpy(f).to("cuda")
        one, two = ([torch.zeros_like(fd) for _ in range(4)] for _ in range(2))
        p = [o.data_ptr() for o in two]
        ctx.derivs_dev(fd.data_ptr(), *[o.data_ptr() for o in one])
        ctx.derivs_dev(fd.data_ptr(), p[0], p[1], 0, 0)
        ctx.derivs_dev(fd.data_ptr(), 0, 0, p[2], p[3])
        ctx.synchronize()
        for a, b in zip(one, two):
            assert torch.equal(a, b) and torch.any(a != 0)


@pytest.mark.parametrize("n, H, W", [(2, 8, 8), (3, 8, 40), (1, 40, 56), (2, 32, 136), (1, 16, 264), (1, 8, 1024)],
                         ids=lambda v: str(v))
def test_network_gradients_at_image_shapes(torch_mod, n, H, W):
    """Parameter and input gradients against the numpy network: one-column
    coarsest images, rows that do not fill a group, several images in a group,
    and a width whose finest levels take the im2col form.  Every output
    channel copies one (tap, channel) and inputs are small integers, so every value before a bf16 rounding is exact in both and rounds
    alike; what is left are the fp32 sums over up to 2^13 pixels (1e-5)."""
    torch = torch_mod
    from oracle import unet_ref as U
    from trans_bl_amd import guess
    rng = np.random.default_rng(H * W + n)
    x = rng.integers(0, 5, size=(n, H, W, 4)).astype(np.float32)
    t = rng.integers(-4, 5, size=(n, H, W, 2)).astype(np.float32)
    theta = []
    for name, cin, cout, ks, lvl, relu in U.layers():
        w = np.zeros((ks * ks, cin, cout))
        o = np.arange(cout)
        tap = np.where(o % 2 > 0, ks * ks // 2, rng.integers(0, ks * ks, cout))
        w[tap, 3 * o % cin, o] = 1.0
        if name == "OUT":
            w[:] = 1.0                            # the gradient reaches every layer
        theta += [w.ravel(), rng.integers(0, 2, cout)]
    theta = np.concatenate(theta)
    net = guess.Net(H, W, n + 1, seed=7)          # a batch below the capacity
    net.set_params(theta.astype(np.float32))
    xd, td = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
    gx = torch.zeros_like(xd)
    torch.cuda.synchronize()
    loss, g = net.gradients(xd.data_ptr(), td.data_ptr(), n, gx.data_ptr())
    again = net.gradients(xd.data_ptr(), td.data_ptr(), n, gx.data_ptr())[1]
    ref = U.UNet(theta, bf16=True)
    rloss, dout = U.mse_loss_and_grad(ref.forward(x), t)
    rg, rdx = ref.backward(dout)
    assert abs(loss - rloss) / rloss < 1e-5
    off, errs = 0, {}
    for name, cin, cout, ks, lvl, relu in U.layers():
        m = ks * ks * cin * cout + cout
        assert np.any(rg[off:off + m])
        errs[name] = np.linalg.norm(g[off:off + m] - rg[off:off + m]) / np.linalg.norm(rg[off:off + m])
        off += m
    assert max(errs.values()) < 1e-5, errs
    assert np.linalg.norm(gx.cpu().numpy() - rdx) <= 1e-5 * np.linalg.norm(rdx)
    if W < 500:
        assert np.array_equal(g, again)           # no atomics in the direct forms


@pytest.mark.parametrize("n, H, W", [(1, 8, 8), (37, 24, 152), (3, 40, 152), (1, 8, 160)], ids=lambda v: str(v))
def test_network_forward_at_image_shapes(torch_mod, n, H, W):
    """Outputs against the numpy network: a tile that one image does not fill,
    two tiles per wavefront with a rest, the widest image of the staged form
    and one past it.  Weights and inputs as in the gradients' test: every value
    before a bf16 rounding is exact in both, so the outputs agree to the fp32
    sum over 32 channels (1e-6)."""
    torch = torch_mod
    from oracle import unet_ref as U
    from trans_bl_amd import guess
    rng = np.random.default_rng(H * W + n)
    x = rng.integers(0, 5, size=(n, H, W, 4)).astype(np.float32)
    theta = []
    for name, cin, cout, ks, lvl, relu in U.layers():
        w = np.zeros((ks * ks, cin, cout))
        o = np.arange(cout)
        tap = np.where(o % 2 > 0, ks * ks // 2, rng.integers(0, ks * ks, cout))
        w[tap, 3 * o % cin, o] = 1.0
        if name == "OUT":
            w[:] = 1.0                            # the gradient reaches every layer
        theta += [w.ravel(), rng.integers(0, 2, cout)]
    theta = np.concatenate(theta)
    net = guess.Net(H, W, n, seed=7)
    net.set_params(theta.astype(np.float32))
    xd, yd = torch.from_numpy(x).cuda(), torch.zeros((n, H, W, 2), device="cuda")
    torch.cuda.synchronize()
    net.forward(xd.data_ptr(), yd.data_ptr(), n)
    out = U.UNet(theta, bf16=True).forward(x)
    assert np.any(out) and np.max(np.abs(yd.cpu().numpy() - out)) <= 1e-6 * np.max(np.abs(out))


@pytest.mark.parametrize("nmodes, kphys", [(1, 4), (2, 4), (3, 8), (4, 8), (5, 16), (16, 32), (20, 64), (33, 128),
                                           (64, 128), (65, 256), (100, 256), (40, 512), (30, 1024)])
def test_nonlinear_terms_at_every_size(torch_mod, nmodes, kphys):
    """Both forms of the nonlinear terms against the oracle (1e-13, as the
    tests of their usual sizes), the mode counts at and below kphys / 2, a plane
    that is no multiple of a group of points; fields of scales 1 to 1e-6."""
    torch = torch_mod
    g = wl.Grid(33, 17, nmodes, 2, 0.02, 1e-3, 1.02, 0.0, 0.3)
    rng = np.random.default_rng(nmodes)
    names = ("ux", "uy", "uz", "wx", "wy", "wz")
    scale = dict(zip(names, (1.0, 1e-3, 0.1, 1e-2, 10.0, 1e-6)))
    F = {k: scale[k] * (rng.normal(size=(nmodes, 17, 33)) + 1j * rng.normal(size=(nmodes, 17, 33))) for k in names}
    base = {k: rng.normal(size=(17, 33)) for k in ("uxb", "uyb", "wzb", "varg", "dvargdx")}
    p = oracle.make_params(g.nx, g.ny, g.nmodes, g.levels, g.dx, g.dy0, g.stf, g.alpha, g.beta)
    zero = {k: np.zeros((17, 33)) for k in base}
    with context(g) as ctx:
        d = {k: torch.from_numpy(F[k]).to("cuda") for k in names}
        for b in (base, zero):
            db = {k: torch.from_numpy(b[k]).to("cuda") for k in b}
            out = [torch.zeros_like(d["ux"]) for _ in range(4)]
            ctx.terms_dev(kphys, {k: v.data_ptr() for k, v in db.items()}, *[d[k].data_ptr() for k in names],
                          *[o.data_ptr() for o in out])
            ctx.synchronize()
            for o, ref in zip(out, oracle.terms(p, kphys, b, F)):
                assert rel(o.cpu().numpy(), ref) < 1e-13
        out = [torch.zeros_like(d["ux"]) for _ in range(3)]
        ctx.terms_fi_dev(kphys, None, *[d[k].data_ptr() for k in names], *[o.data_ptr() for o in out])
        ctx.synchronize()
    for o, ref in zip(out, oracle.terms_fi(p, kphys, None, F)):
        assert rel(o.cpu().numpy(), ref) < 1e-13


RHS_GRIDS = [g for g in DERIV_GRIDS if g[0] >= 65 or g[1] > 400]


@pytest.mark.parametrize("form", ["linear", "nonlinear", "flat plate", "in place"])
@pytest.mark.parametrize("nx, ny", RHS_GRIDS)
def test_right_hand_side_at_every_shape(torch_mod, nx, ny, form):
    """The right-hand side against the oracle on random values (1e-12 of the
    largest value, as the parity tests); in place: dvx over wx, dvz over wz,
    which the kernels that need their inputs twice must not take.  Row 1 keeps
    the caller's values."""
    torch = torch_mod
    g = wl.Grid(nx, ny, 3, 2, 0.02, 1e-3, 1.004, 0.0, 0.3)
    rng = np.random.default_rng(nx + ny)
    names = ("ux", "uy", "uz", "wx", "wy", "wz")
    F = {k: rng.normal(size=(3, ny, nx)) + 1j * rng.normal(size=(3, ny, nx)) for k in names}
    base = {k: rng.normal(size=(ny, nx)) for k in ("uxb", "uyb", "wzb", "varg", "dvargdx")}
    kphys = 8 if form == "nonlinear" else 0
    Re = 1e4
    p = oracle.make_params(g.nx, g.ny, g.nmodes, g.levels, g.dx, g.dy0, g.stf, g.alpha, g.beta)
    ref = oracle.drv_fi(p, Re, 0, base, F) if form == "flat plate" else oracle.drv_gv(p, Re, kphys, base, F)
    with context(g) as ctx:
        d = {k: torch.from_numpy(F[k]).to("cuda") for k in names}
        keep = {k: torch.from_numpy(base[k]).to("cuda") for k in base}
        db = {k: keep[k].data_ptr() for k in base}
        out = [torch.full_like(d["ux"], 7.0) for _ in range(3)]
        first = [7.0] * 3
        if form == "in place":
            out[0], out[2] = d["wx"], d["wz"]
            first = [F["wx"][:, 0], 7.0, F["wz"][:, 0]]
        call = ctx.drv_fi_dev if form == "flat plate" else ctx.drv_gv_dev
        call(Re, kphys, db, *[d[k].data_ptr() for k in names], *[o.data_ptr() for o in out])
        ctx.synchronize()
        got = [o.cpu().numpy() for o in out]
    for q in range(3):
        assert np.all(got[q][:, 0] == first[q])
        assert rel(got[q][:, 1:], ref[q][:, 1:]) < 1e-12, "xyz"[q]


@pytest.mark.parametrize("g", [
    wl.Grid(65, 33, 3, 4, 0.05, 2e-3, 1.03, 0.0, 0.9),      # strips of 2 columns, one row chunk
    wl.Grid(89, 41, 2, 4, 0.05, 1e-3, 1.03, 0.1, 0.7),
    wl.Grid(145, 117, 2, 3, 0.03, 3e-4, 1.015, 0.0, 0.3),   # 116 rows: two full chunks
    wl.Grid(145, 121, 2, 3, 0.03, 3e-4, 1.015, 0.0, 0.3),   # two rows in the third
    wl.Grid(609, 65, 40, 3, 0.02, 5e-4, 1.02, 0.0, 0.3)],   # strips of 32 and a rest
    ids=lambda g: f"{g.nx}x{g.ny}x{g.nmodes}l{g.levels}")
def test_fas_cycles_match_oracle(torch_mod, g):
    """Two FP64 cycles, wall and boundary columns non-zero (they are injected
    too), against the oracle in the same line order: iterates to 1e-10 (last-bit
    differences of some 600 line solves, each of condition up to 1e4), the checks'
    largest defects to 1e-5 (differences of values up to 1e6 times as large)."""
    p = oracle.make_params(g.nx, g.ny, g.nmodes, g.levels, g.dx, g.dy0, g.stf, g.alpha, g.beta)
    f = wl.wavepacket_rhs(g, tag="fas")
    u = 0.01 * wl.wavepacket_rhs(g, tag="fas-start")
    u[:, 0, :] = 0.003
    u[:, :, 0] = 0.002
    u[:, :, -1] = -0.001
    with context(g) as ctx:
        got, _, res = ctx.poi_uy(None, -f, u, 0.0, max_cycles=2)[:3]
    ref, _, rres = oracle.poi_uy(p, np.zeros_like(f), -f, u, 0.0, max_cycles=2, order=1)
    assert rel(got, ref) < 1e-10, rel(got, ref)
    assert rel(res, rres) < 1e-5, rel(res, rres)


@pytest.mark.parametrize("g, lanes", [
    (wl.Grid(65, 33, 3, 3, 0.05, 2e-3, 1.03, 0.0, 0.9), 16),       # one strip holds all columns
    (wl.Grid(129, 65, 8, 3, 0.05, 1e-3, 1.03, 0.0, 0.9), 16),
    (wl.Grid(161, 97, 6, 3, 0.03, 5e-4, 1.02, 0.0, 0.5), 32),
    (wl.Grid(89, 193, 4, 3, 0.03, 2e-4, 1.015, 0.0, 0.3), 64),     # strips of 6 columns
    (wl.Grid(545, 65, 70, 3, 0.02, 5e-4, 1.02, 0.0, 0.3), 32)],    # two rounds of lines a colour
    ids=lambda v: f"{v.nx}x{v.ny}x{v.nmodes}" if hasattr(v, "nx") else str(v))
@pytest.mark.parametrize("nu1, nu2", [(3, 1), (2, 1), (2, 2)])
def test_one_launch_sweeps_match_colour_phases(torch_mod, g, lanes, nu1, nu2):
    """FP64 solves with every level's sweeps in one launch each (direct shapes)
    against the staged colour phases, modes stopping after different cycles and
    either buffer holding the result: the same cycle counts, v to 1e-12 (the
    same operations), boundary data kept."""
    f = wl.wavepacket_rhs(g, tag="one-launch") * 10.0 ** -np.arange(g.nmodes)[:, None, None]
    u = np.zeros_like(f)
    u[:, 0, :], u[:, :, 0], u[:, :, -1] = 0.003, 0.002, -0.001
    out = []
    with context(g) as ctx:
        for sign in (1, -1):
            for lvl in range(1, g.levels):
                ctx.set_line_shape(0, lvl, sign * lanes)
            out.append(ctx.poi_uy(None, -f, u, 1e-7, nu1=nu1, nu2=nu2)[:2])
    assert np.array_equal(out[0][1], out[1][1]), (out[0][1], out[1][1])
    assert rel(out[0][0], out[1][0]) < 1e-12, rel(out[0][0], out[1][0])
    assert np.array_equal(out[0][0][:, 0], u[:, 0])
