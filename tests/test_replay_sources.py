"""The shape tables that the kernels' host replays restate, against the sources."""
import os
import re

import numpy as np
import pytest
import test_deriv_replay as deriv
import test_nlterms_replay as nl

import trans_bl_amd as tb


def source(name):
    with open(os.path.join(os.path.dirname(tb.__file__), "csrc", name)) as f:
        return f.read()


def table(text, macro):
    body = re.search(rf"#define {macro}\(X\)((?:.*\\\n)*.*)", text).group(1)
    rows = [tuple(int(v) for v in m.split(",")) for m in re.findall(r"X\(([\d, ]+)\)", body)]
    return [r[0] if len(r) == 1 else r for r in rows]


def constant(text, name):
    return int(re.search(rf"\b{name} = (\d+)", text).group(1))


def test_derivative_shapes():
    h, k = source("tbl_deriv.h"), source("tbl_kernels.h")
    assert table(h, "TBL_X_SHAPES") == deriv.X_SHAPES and table(h, "TBL_Y_SHAPES") == deriv.Y_SHAPES
    assert constant(h, "kDerivYCols") == 8 and constant(h, "kDerivMaxNx") == 2112
    assert constant(k, "kTriRows") == 67 and "kXTab = 6 * kTriRows + 64" in k
    assert f"kBufOff = 0x{deriv.K_BUF_OFF:x}u" in source("tbl_buf.h")


def test_nonlinear_term_sizes():
    s = source("tbl_rhs.hip")
    assert table(s, "TBL_NL_SIZES") == [4, 8, 16, 32, 64, 128, 256, 512, 1024]
    radix = re.search(r"constexpr int nl_radix\(int L\) \{ return (.*); \}", s).group(1)
    assert radix == "L % 64 == 32 || L >= 128 ? 8 : L == 8 ? 2 : 4"
    for L in (8, 16, 32, 64, 128, 256, 512):
        assert nl.radix(L) == (8 if L % 64 == 32 or L >= 128 else 2 if L == 8 else 4)
    assert "nl_slot(int n) { return n + (n >> 3); }" in s


@pytest.mark.parametrize("nx", [15, 129, 1026])
@pytest.mark.parametrize("ny", [289, 320, 321, 353, 448, 449, 545, 576])
def test_y_tiles_of_four_columns(nx, ny):
    """deriv_y_tile's forms of 64 lanes a column: test_deriv_replay.py's checks
    with their tile of 4 columns."""
    h = source("tbl_deriv_kernels.hip")
    assert "constexpr int y_cols(int G) { return G == 64 ? 4 : kDerivYCols; }" in h
    G, R = next((g, r) for g, r in deriv.Y_SHAPES if g * r >= ny)
    TX, NT, N, M = 4, 8 * G, (R + 1) // 2, G * R
    LP = M + 32 // TX
    assert G == 64
    t = np.arange(NT)
    tx, tj = t % TX, t // TX
    lds = np.zeros(2 * TX * LP, int)
    got = np.zeros((TX, ny), int)
    columns = min(TX, nx - (nx - 1) // TX * TX)                     # of the last tile
    x0 = nx - columns
    for q in range(N):
        use = ((q + 1) * 2 * G <= M) | (tj + 2 * G * q < M)
        at = (tx * LP + 2 + tj + 2 * G * q)[use]
        np.add.at(lds, at, 1)
        np.add.at(lds, at + TX * LP, 1)
        j = tj + 2 * G * q
        np.add.at(got, (tx[use & (j < ny)], j[use & (j < ny)]), 1)
        off = np.where(tx < columns, (tj * nx + x0 + tx) * 16, deriv.K_BUF_OFF) + 2 * G * nx * 16 * q
        assert off.max() < 2 ** 32
        assert np.all((off < nx * ny * 16) == ((tx < columns) & (j < ny)))
        # half a wavefront's accesses on different banks
        assert all(len(set(at[w:w + 32] % 32)) == 32 for w in range(0, len(at) - 31, 32))
    e = np.arange(8 * TX)
    np.add.at(lds, e // 4 * LP + np.where(e % 4 < 2, e % 4, M + e % 4), 1)
    used = lds.reshape(2 * TX, LP)
    assert np.all(used[:, :M + 4] == 1) and np.all(used[:, M + 4:] == 0) and np.all(got == 1)
    assert NT // G == 2 * TX
    win = np.arange(G)[:, None] * R + np.arange(R + 4)
    assert win.min() == 0 and win.max() == M + 3
    tiles = -(-nx // TX) * 3
    grid, per = -(-tiles // 8) * 8, -(-tiles // 8)
    m = np.arange(grid) % 8 * per + np.arange(grid) // 8
    assert np.array_equal(np.sort(m[m < tiles]), np.arange(tiles))
    assert (2 * TX * LP + 6 * M + 64) * 8 <= 80 * 1024              # two workgroups a CU
