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

