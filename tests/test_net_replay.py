"""Host replay of the network kernels' dispatch and indexing (tbl_unet.hip): every
LDS and global access in bounds, every operand from the right pixel, every
output written once.  Forms and constants are read from the source."""
import os
import re

import numpy as np
import pytest

import trans_bl_amd as tb
from oracle import unet_ref as U

with open(os.path.join(os.path.dirname(tb.__file__), "csrc", "tbl_unet.hip")) as f:
    SRC = f.read()

LDS, OFF = 160 * 1024, 0x80000000
WG_ROW = int(re.search(r"constexpr int kWgRow = (\d+);", SRC).group(1))


def forms(macro):
    """The argument lists of an X-macro table."""
    text = re.search(rf"#define {macro}\(X\)((?:.*\\\n)*.*)", SRC).group(1)
    return [tuple(int(v) for v in m.split(",")) for m in re.findall(r"X\(([\d, ]+)\)", text)]


CONVS = [(cin, cout, lvl) for _, cin, cout, ks, lvl, _ in U.layers() if ks == 3]
# images of a layer: height, width, number
IMAGES = [(1, 1, 2), (2, 3, 5), (4, 17, 3), (5, 34, 2), (2, 64, 1), (3, 68, 1), (4, 136, 1), (2, 159, 1)]


def neighbours(NP, H, W):
    """Per flattened pixel and tap: the pixel the tap reads, -1 outside."""
    p = np.arange(NP)
    h, w = p // W % H, p % W
    out = np.full((NP, 9), -1)
    for t in range(9):
        hh, ww = h + t // 3 - 1, w + t % 3 - 1
        ok = (hh >= 0) & (hh < H) & (ww >= 0) & (ww < W)
        out[ok, t] = (p + (t // 3 - 1) * W + t % 3 - 1)[ok]
    return out


def slot(r, p):
    return r * 64 + ((p ^ (r >> 2 & 3)) << 4)


@pytest.mark.parametrize("H, W, n", IMAGES)
@pytest.mark.parametrize("MT, NI", forms("TBL_CONV_FORMS"))
@pytest.mark.parametrize("cin", [4, 32, 96])
def test_staged_convolution(H, W, n, MT, NI, cin):
    NP, PX, cin4 = n * H * W, 128 * MT, cin == 4
    NQ = PX + 2 * W + 2
    assert NQ <= 64 * NI                       # conv3x3s_fits
    lds = 64 * (9 * 32 + 128 * MT + 2 * W + 3)  # conv3x3s_lds
    want = neighbours(NP, H, W)
    tid = np.arange(256)
    stored = np.zeros(NP, int)
    for p0 in range(0, NP, PX):
        q0 = p0 - W - 1
        qb = max(q0, 0)
        rng = min(NP - qb, NQ) * cin * 2
        held = np.full(NQ + 1, -2)             # the pixel a staged row holds, -1 zeros
        for s in range(NI):
            e = tid + 256 * s
            q, g = (e, 0 * e) if cin4 else (e // 4, e % 4)
            xo = ((q0 - qb) * cin * 2 + (tid * cin * 2 if cin4 else (tid // 4 * cin + 8 * (tid % 4)) * 2)
                  + s * (256 if cin4 else 64) * cin * 2) % 2 ** 32
            use = (q < NQ) & (g == 0)
            inside = xo[use] < rng
            assert np.array_equal(inside, (q0 + q[use] >= 0) & (q0 + q[use] < NP))
            pix = qb + xo[use] // (cin * 2)
            assert np.all(held[q[use]] == -2)
            held[q[use]] = np.where(inside, pix, -1)
            assert np.all(pix[inside] == (q0 + q[use])[inside])
            assert np.all(9 * 32 * 64 + slot(q[q < NQ], g[q < NQ]) + 16 <= lds - 64)
        held[NQ] = -1
        assert np.all(held > -2) and 9 * 32 * 64 + NQ * 64 + 64 <= lds
        lp = np.arange(PX)
        pa = p0 + lp
        wa, ha = pa % W, pa // W % H
        for t in range(9):
            hh, ww = ha + t // 3 - 1, wa + t % 3 - 1
            ok = (hh >= 0) & (hh < H) & (ww >= 0) & (ww < W)
            r = np.where(ok, lp + W + 1 + (t // 3 - 1) * W + t % 3 - 1, NQ)
            assert r.min() >= 0 and r.max() <= NQ
            live = pa < NP
            assert np.array_equal(held[r][live], want[pa[live], t])
            # the second half of the channels: pieces half + 2, in the same row
            for half in (0, 1):
                a = slot(r, half)
                assert np.array_equal(np.where(r == NQ, NQ * 64 + 16 * half, a) // 64, r)
                assert np.array_equal((a ^ 32)[r < NQ], slot(r, half + 2)[r < NQ])
        stored[pa[pa < NP]] += 1
    assert np.all(stored == 1)
    # weights: rows [tap][32 outputs] of four pieces, later taps past the range
    e = (tid[:, None] + 256 * np.arange(5)).ravel()
    tap, o = e // 4 // 32, e // 4 % 32
    cinp, cout = (cin + 31) // 32 * 32, 64
    off = ((tid[:, None] // 4 // 32 * cout + tid[:, None] // 4 % 32) * cinp + 8 * (tid[:, None] % 4)) * 2 \
        + np.arange(5) * (64 // 32 * cout * cinp * 2)
    assert np.array_equal(off.ravel(), ((tap * cout + o) * cinp + 8 * (e % 4)) * 2)
    assert np.array_equal(np.unique(slot(e[e < 1152] // 4, e[e < 1152] % 4)), np.arange(0, 9 * 32 * 64, 16))


def test_input_gradient_forms_are_the_ones_layers_take():
    """conv3x3_dx: every layer has its form, and every compiled form a layer."""
    taken = set()
    for cin, cout, _ in CONVS:
        nt = 2 if cin % 64 == 0 and cout != 32 else 1
        taken.add((3 - nt, nt, cout))
    assert taken == set(forms("TBL_DX_SHAPES"))


@pytest.mark.parametrize("H, W, n", IMAGES)
@pytest.mark.parametrize("MT, NT, cout", forms("TBL_DX_SHAPES"))
@pytest.mark.parametrize("cin", [4, 32, 96, 192])
def test_input_gradient(H, W, n, MT, NT, cout, cin):
    NP, CT, PX, ROW, G = n * H * W, 32 * NT, 128 * MT, cout + 8, cout // 8
    NQ = PX + 2 * W + 2
    lds = (PX + 2 * W + 2 + CT) * ROW * 2                                  # dx_lds
    assert (CT * ROW + (NQ - 1) * ROW + cout) * 2 <= lds
    # one tap's weights: WP pieces a thread cover CT rows of G pieces
    WP = max(1, CT * G // 256)
    assert 256 * WP >= CT * G
    want = neighbours(NP, H, W)
    stored = np.zeros(NP, int)
    for p0 in range(0, NP, PX):
        lp = np.arange(PX)
        pa = p0 + lp
        wa, ha = pa % W, pa // W % H
        for t in range(9):
            hh, ww = ha - (t // 3 - 1), wa - (t % 3 - 1)
            ok = (pa < NP) & (hh >= 0) & (hh < H) & (ww >= 0) & (ww < W)
            row = (lp + W + 1 - ((t // 3 - 1) * W + t % 3 - 1))[ok]
            assert row.size == 0 or (row.min() >= 0 and row.max() < NQ)
            src = p0 - W - 1 + row
            assert np.all((src >= 0) & (src < NP))
            assert np.array_equal(want[src, t], pa[ok])                    # the pixels whose tap t reads pa
        # D layout: pixel of register i and lane
        i, lane, tile = np.meshgrid(np.arange(16), np.arange(64), np.arange(4 * MT), indexing="ij")
        p = p0 + 32 * tile + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3)
        np.add.at(stored, p[(lane & 31 == 0) & (p < NP)], 1)
    assert np.all(stored == 1)
    assert NT * 32 * -(-cin // (NT * 32)) >= cin


def dw_shape(W, nc):
    nr = max(1, ({4: 128, 2: 192}.get(nc, 256) + W // 2) // W)
    ks = -(-nr * W // 32)
    x_bytes = -(-((nr + 3) * (W + 2) * WG_ROW * 2) // 16) * 16
    return nr, ks, x_bytes, x_bytes + nc * 32 * ks * WG_ROW * 2 + 3 * 32 * ks * 2


@pytest.mark.parametrize("H, W, n", IMAGES + [(2, 264, 1), (1, 400, 2)])
@pytest.mark.parametrize("NC", [1, 2, 4])
@pytest.mark.parametrize("cin", [4, 32, 96])
def test_weight_gradient(H, W, n, NC, cin):
    rows, cout = n * H, 32 * NC
    nr, ks, x_bytes, lds = dw_shape(W, NC)
    if lds > LDS or (nr + 3) * (W + 2) * (WG_ROW // 4) >= 65536:           # conv3x3_back_fits
        assert W > 264
        return
    W2, npx, groups = W + 2, 32 * ks, -(-rows // nr)
    want = neighbours(rows * W, H, W)
    seen = np.zeros(rows * W, int)
    for grp in range(groups):
        r0 = grp * nr
        held = np.full((nr + 3) * W2, -2)
        q = np.arange((nr + 3) * W2)
        border = (q % W2 == 0) | (q % W2 == W + 1) | (q // W2 == nr + 2)
        held[border] = -1
        count = (nr + 2) * W
        if cin >= 8:
            # pieces of a pixel go to four threads; lr and col follow q by steps of 64
            for first in range(64):
                q, lr, col = first, first // W, first % W
                while q < count:
                    assert lr == q // W and col == q % W
                    off = ((r0 - 1) * W + q) * cin * 2 % 2 ** 32
                    at = q + 2 * lr + 1
                    assert held[at] == -2
                    held[at] = off // (cin * 2) if off < rows * W * cin * 2 else -1
                    q, lr, col = q + 64, lr + 64 // W, col + 64 % W
                    if col >= W:
                        lr, col = lr + 1, col - W
        else:
            q = np.arange(count)
            off = ((r0 - 1) * W + q) * cin * 2 % 2 ** 32
            at = q + 2 * (q // W) + 1
            assert np.all(held[at] == -2)
            held[at] = np.where(off < rows * W * cin * 2, off // (cin * 2), -1)
        assert np.all(held > -2) and held.size * WG_ROW * 2 <= x_bytes
        p = np.arange(npx)
        lr, col, inside = p // W, p % W, p < nr * W
        off = np.where(inside, ((r0 * W + p) * cout) * 2, OFF)
        z = np.where(off < rows * W * cout * 2, off // (cout * 2), -1)       # the pixel of dZ, -1 zeros
        h = (r0 + lr) % H
        for t in range(9):
            dh = t // 3 - 1
            row = np.where(inside & (h + dh >= 0) & (h + dh < H), lr + 1 + dh, nr + 2)
            unit = (row * W2 + np.where(inside, col, 0) + 1) * (WG_ROW // 4)
            assert unit.max() < 65536
            x = unit // (WG_ROW // 4) + t % 3 - 1
            assert x.min() >= 0 and x.max() < held.size
            live = z >= 0
            assert np.array_equal(held[x][live], want[z[live], t])
            assert np.all(held[x][~live] == -1)        # zeros meet zeros past the last row
        seen[z[z >= 0]] += 1
    assert np.all(seen == 1)
