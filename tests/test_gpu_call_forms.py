"""Forms of a call whose route through the library depends on the grid: the
result must not."""
import numpy as np
import pytest

import oracle
from trans_bl_amd import workload as wl

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_mod(gpu_ready):
    import torch
    return torch


def random_field(torch, g):
    rng = np.random.default_rng(g.nx * g.ny)
    return torch.from_numpy(rng.normal(size=(g.nmodes, g.ny, g.nx)) + 1j * rng.normal(size=(g.nmodes, g.ny, g.nx))).to("cuda")


# the first three take all four derivatives in one launch where that may be, the last does not
@pytest.mark.parametrize("nx, ny, nmodes", [(17, 9, 1), (129, 33, 4), (577, 143, 1), (641, 65, 2)], ids=lambda v: str(v))
def test_derivatives_into_overlapping_outputs(torch_mod, nx, ny, nmodes):
    """Outputs of the two directions in the same memory, whole or in part: the
    y-derivatives, written last, stand; what they do not cover holds the
    x-derivatives.  An output in the input's place is refused."""
    torch = torch_mod
    import trans_bl_amd as tb
    g = wl.Grid(nx, ny, nmodes, 2, 0.02, 1e-3, 1.004, 0.0, 0.3)
    f = random_field(torch, g)
    n = f.numel()
    with tb.Context(g) as ctx:
        ref = [torch.zeros_like(f) for _ in range(4)]
        p = [o.data_ptr() for o in ref]
        ctx.derivs_dev(f.data_ptr(), p[0], p[1], 0, 0)
        ctx.derivs_dev(f.data_ptr(), 0, 0, p[2], p[3])
        ctx.synchronize()
        a, b = torch.zeros_like(f), torch.zeros_like(f)
        torch.cuda.synchronize()
        ctx.derivs_dev(f.data_ptr(), a.data_ptr(), b.data_ptr(), a.data_ptr(), b.data_ptr())
        ctx.synchronize()
        assert torch.equal(a, ref[2]) and torch.equal(b, ref[3])
        # d/dy starts half way into d/dx's memory
        m = n // 2
        buf, c = torch.zeros(n + m, dtype=f.dtype, device="cuda"), torch.zeros_like(f)
        torch.cuda.synchronize()
        ctx.derivs_dev(f.data_ptr(), buf.data_ptr(), b.data_ptr(), buf.data_ptr() + 16 * m, c.data_ptr())
        ctx.synchronize()
        assert torch.equal(buf[:m], ref[0].flatten()[:m]) and torch.equal(buf[m:], ref[2].flatten())
        assert torch.equal(b, ref[1]) and torch.equal(c, ref[3])
        for q in range(4):
            out = [o.data_ptr() for o in (a, b, c, ref[3])]
            out[q] = f.data_ptr()
            with pytest.raises(tb.TblError):
                ctx.derivs_dev(f.data_ptr(), *out)


def test_creating_a_context_of_many_modes(torch_mod):
    """A mode costs a context its line factors, on the host, and their upload;
    their other layouts are the device's work.  128 modes of a narrow tall grid
    take 4 to 5 times as long as one mode with the factors alone, 16 to 20 times
    with the layouts formed on the host: at most 8 (the quickest of seven each)."""
    import time

    import trans_bl_amd as tb

    def create(nmodes):
        g = wl.Grid(65, 257, nmodes, 3, 0.02, 2e-4, 1.012, 0.0, 0.1)
        best = np.inf
        for _ in range(7):
            t = time.perf_counter()
            ctx = tb.Context(g)
            best = min(best, time.perf_counter() - t)
            ctx.close()
        return best

    one, many = create(1), create(128)
    print(f"creation: {1e3 * one:.2f} ms with 1 mode, {1e3 * many:.2f} with 128", flush=True)
    assert many < 8 * one


@pytest.mark.parametrize("nmodes, kphys", [(256, 512), (43, 1024), (300, 1024), (512, 1024)])
def test_nonlinear_terms_of_many_modes(torch_mod, nmodes, kphys):
    """Every mode count up to kphys / 2 at the largest kphys, against the oracle
    (1e-13 as at the other sizes; the oracle lies 8e-15 from numpy's FFT here)."""
    torch = torch_mod
    import trans_bl_amd as tb
    g = wl.Grid(33, 17, nmodes, 2, 0.02, 1e-3, 1.02, 0.0, 0.3)
    rng = np.random.default_rng(nmodes)
    names = ("ux", "uy", "uz", "wx", "wy", "wz")
    scale = dict(zip(names, (1.0, 1e-3, 0.1, 1e-2, 10.0, 1e-6)))
    F = {k: scale[k] * (rng.normal(size=(nmodes, 17, 33)) + 1j * rng.normal(size=(nmodes, 17, 33))) for k in names}
    base = {k: rng.normal(size=(17, 33)) for k in ("uxb", "uyb", "wzb", "varg", "dvargdx")}
    p = oracle.make_params(g.nx, g.ny, g.nmodes, g.levels, g.dx, g.dy0, g.stf, g.alpha, g.beta)
    with tb.Context(g) as ctx:
        d = {k: torch.from_numpy(F[k]).to("cuda") for k in names}
        db = {k: torch.from_numpy(base[k]).to("cuda") for k in base}
        out = [torch.zeros_like(d["ux"]) for _ in range(4)]
        ctx.terms_dev(kphys, {k: v.data_ptr() for k, v in db.items()}, *[d[k].data_ptr() for k in names],
                      *[o.data_ptr() for o in out])
        fi = [torch.zeros_like(d["ux"]) for _ in range(3)]
        ctx.terms_fi_dev(kphys, None, *[d[k].data_ptr() for k in names], *[o.data_ptr() for o in fi])
        ctx.synchronize()
        for bad in (kphys + 2, kphys // 2 if 2 * nmodes > kphys // 2 else kphys + 2, 2048):
            with pytest.raises(tb.TblError):
                ctx.terms_dev(bad, {k: v.data_ptr() for k, v in db.items()}, *[d[k].data_ptr() for k in names],
                              *[o.data_ptr() for o in out])
    for o, ref in zip(out + fi, oracle.terms(p, kphys, base, F) + oracle.terms_fi(p, kphys, None, F)):
        o = o.cpu().numpy()
        assert np.max(np.abs(o - ref)) < 1e-13 * np.max(np.abs(ref))


@pytest.mark.parametrize("nx, ny, nmodes", [(17, 9, 3), (33, 59, 1), (35, 59, 2), (65, 61, 5), (129, 121, 7), (1025, 193, 2)],
                         ids=lambda v: str(v))
def test_residual_maxima(torch_mod, nx, ny, nmodes):
    """Each mode's largest residual is that of the field written (2 units in the
    last place: a square root of a sum of squares against numpy's hypot), with
    one to four wavefronts in a mode's last workgroup; the largest may lie in any
    of them."""
    torch = torch_mod
    import trans_bl_amd as tb
    g = wl.Grid(nx, ny, nmodes, 2 if ny % 2 else 1, 0.02, 1e-3, 1.004, 0.0, 0.3)
    f = random_field(torch, g)
    rng = np.random.default_rng(ny)
    with tb.Context(g) as ctx:
        v, out = torch.zeros_like(f), torch.zeros_like(f)
        for _ in range(6):
            k, j, i = rng.integers(nmodes), rng.integers(1, ny), rng.integers(1, nx - 1)
            f[k, j, i] = 1e3 * (1 + 1j)
            torch.cuda.synchronize()
            res = ctx.residual_dev(0, f.data_ptr(), v.data_ptr(), out.data_ptr())
            ref = np.abs(out.cpu().numpy()).max(axis=(1, 2))
            assert ref[k] > 100 and np.all(np.abs(res - ref) <= 4.5e-16 * ref)


@pytest.mark.parametrize("shape", [0, 64], ids=["default", "direct"])
def test_line_factors_past_4_gigabytes(torch_mod, shape):
    """58400 modes of 545 rows: the FP64 factors of 64 lanes take 4.3 GB, past what
    one buffer resource reaches.  Two cycles of the last modes, staged (the
    default) and direct, against a context of two modes with the same kz (1e-12, as
    other forms of one sweep)."""
    torch = torch_mod
    import trans_bl_amd as tb
    if torch.cuda.mem_get_info()[0] < 140 << 30:
        pytest.skip("needs 140 GiB of device memory")
    nx, ny, K, beta = 15, 545, 58400, 1e-4
    rng = np.random.default_rng(5)
    one = torch.from_numpy(rng.normal(size=(1, ny, nx)) + 1j * rng.normal(size=(1, ny, nx))).to("cuda")

    def solve(nmodes, b, want):
        with tb.Context(wl.Grid(nx, ny, nmodes, 2, 0.02, 1e-3, 1.002, 0.0, b)) as ctx:
            if shape:
                ctx.set_line_shape(0, 1, shape)
            f = one.expand(nmodes, ny, nx).contiguous()
            v = torch.zeros_like(f)
            torch.cuda.synchronize()
            ctx.solve_rhs_dev(f.data_ptr(), v.data_ptr(), 0.0, precision=0, max_cycles=2, guess=1)
            return [v[k].cpu().numpy() for k in want]

    modes = (1, K // 2, K - 2, K - 1)
    for k, got in zip(modes, solve(K, beta, modes)):
        ref = solve(2, k * beta, (1,))[0]
        assert np.max(np.abs(got - ref)) < 1e-12 * np.max(np.abs(ref)), k
    torch.cuda.empty_cache()


@pytest.mark.parametrize("shape,precision,nx,ny,K", [
    (-64, 0, 15, 17, 1300000), (-64, 1, 15, 17, 1300000), (2064, 0, 15, 17, 1300000),
    (1064, 0, 15, 17, 1300000), (1064, 1, 15, 17, 1300000)])
def test_line_factors_of_a_million_modes(torch_mod, shape, precision, nx, ny, K):
    """Lines of 64 lanes whose factors, 8 kB a mode in FP64 and 3.6 to 4 in FP32, take
    two or three ranges of modes a sweep: staged and strips.  Two cycles
    of modes in and next to the ranges against a context of two modes with the
    same kz (1e-12; FP32 corrections 1e-5)."""
    torch = torch_mod
    import trans_bl_amd as tb
    if torch.cuda.mem_get_info()[0] < 200 << 30:
        pytest.skip("needs 200 GiB of device memory")
    beta = 1e-5
    rng = np.random.default_rng(7)
    one = torch.from_numpy(rng.normal(size=(1, ny, nx)) + 1j * rng.normal(size=(1, ny, nx))).to("cuda")

    def solve(nmodes, b, want):
        with tb.Context(wl.Grid(nx, ny, nmodes, 2, 0.02, 1e-2, 1.02, 0.0, b)) as ctx:
            ctx.set_line_shape(precision, 1, shape)
            f = one.expand(nmodes, ny, nx).contiguous()
            v = torch.zeros_like(f)
            torch.cuda.synchronize()
            ctx.solve_rhs_dev(f.data_ptr(), v.data_ptr(), 0.0, precision=precision, max_cycles=2, guess=1)
            return [v[k].cpu().numpy() for k in want]

    each = 4096 if precision and shape > 1000 else 3584 if precision else 8192   # bytes a mode
    most = (2 ** 32 - 1) // each
    modes = (1, most - 1, most, most + 1, K // 2 + 1, K - 2, K - 1)
    for k, got in zip(modes, solve(K, beta, modes)):
        ref = solve(2, k * beta, (1,))[0]
        assert np.max(np.abs(got - ref)) < (1e-12 if precision == 0 else 1e-5) * np.max(np.abs(ref)), k
    torch.cuda.empty_cache()


def test_x_derivatives_of_many_lines(torch_mod):
    """35 million x-lines, whose threads are past 2^32: every mode of a field of
    equal modes has the first one's derivatives."""
    torch = torch_mod
    import trans_bl_amd as tb
    if torch.cuda.mem_get_info()[0] < 140 << 30:
        pytest.skip("needs 140 GiB of device memory")
    nx, ny, K = 15, 545, 64000
    rng = np.random.default_rng(6)
    one = torch.from_numpy(rng.normal(size=(1, ny, nx)) + 1j * rng.normal(size=(1, ny, nx))).to("cuda")
    f = one.expand(K, ny, nx).contiguous()
    a, b = torch.zeros_like(f), torch.zeros_like(f)
    with tb.Context(wl.Grid(nx, ny, K, 2, 0.02, 1e-3, 1.002, 0.0, 1e-4)) as ctx:
        torch.cuda.synchronize()
        ctx.derivs_dev(f.data_ptr(), a.data_ptr(), b.data_ptr(), 0, 0)
        ctx.synchronize()
        for o in (a, b):
            assert torch.any(o[0] != 0) and all(torch.equal(o[k], o[0]) for k in range(0, K, 777))
        a.zero_()
        torch.cuda.synchronize()
        ctx.deriv_dev(tb.DERIV_KINDS["x"], f.data_ptr(), a.data_ptr())
        ctx.synchronize()
        assert torch.any(a[0] != 0) and all(torch.equal(a[k], a[0]) for k in range(0, K, 777))
    del f, a, b
    torch.cuda.empty_cache()


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32"])
def test_colour_phases_of_a_large_coarsest_level(torch_mod, precision):
    """A coarsest level past the LDS takes a launch per colour phase: direct with
    16, 32 and 64 lanes (a wavefront's lines of two modes and kinds) and staged, the
    iterates after two cycles to rounding (1e-12; FP32 corrections 1e-5)."""
    import trans_bl_amd as tb
    g = wl.Grid(257, 161, 3, 2, 0.02, 5e-4, 1.01, 0.0, 0.3)        # coarsest 129x81
    f = wl.wavepacket_rhs(g, tag="phases")
    u = 0.01 * wl.wavepacket_rhs(g, tag="start")
    out = []
    with tb.Context(g) as ctx:
        for shape in (16, 32, 64, -16, 2032):
            ctx.set_line_shape(precision, 2, shape)
            out.append(ctx.poi_uy(None, -f, u, 0.0, precision=precision, max_cycles=2)[0])
    for o in out[1:]:
        assert np.max(np.abs(o - out[0])) < (1e-12 if precision == 0 else 1e-5) * np.max(np.abs(out[0]))
