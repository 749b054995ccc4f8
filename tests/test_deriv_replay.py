"""Host replay of the derivative kernels' indexing (tbl_deriv_kernels.hip):
every LDS and global access in bounds, every point written once."""
import numpy as np
import pytest

X_SHAPES = [(2, 1), (3, 1), (5, 1), (7, 1), (9, 1), (5, 2), (7, 2), (9, 2), (7, 3), (9, 3), (7, 4), (9, 4)]
Y_SHAPES = [(16, 3), (16, 5), (16, 7), (16, 9), (32, 5), (32, 7), (32, 9), (64, 5), (64, 7), (64, 9)]


K_BUF_OFF = 0x80000000


@pytest.mark.parametrize("nx", [15, 64, 127, 128, 129, 193, 320, 321, 450, 577, 777, 1025, 1088, 1152, 1153, 1729,
                                2049, 2112])
def test_x_lines(nx):
    R, W = min(((r, w) for r, w in X_SHAPES if 64 * r * w >= nx), key=lambda s: (s[1], s[0]))
    NT, N, M = 128 * W, (R + 1) // 2, 64 * R * W
    LP = M + 4
    t = np.arange(NT)
    plane = np.zeros(LP, int)                                       # writes per plane value
    glob = []
    for q in range(N):
        use = ((q + 1) * NT <= M) | (t // 64 < W)
        e = (t + NT * q)[use]
        assert e.max() < M
        np.add.at(plane, 2 + e, 1)
        glob.append(e[e < nx])                                      # the rest is past the buffer's range
    assert np.array_equal(np.sort(np.concatenate(glob)), np.arange(nx))
    np.add.at(plane, [e % 4 if e % 4 < 2 else LP - 4 + e % 4 for e in range(4)], 1)
    assert np.all(plane == 1)                                       # every value of the plane set, once
    i0 = np.arange(64 * W) * R
    rows = (i0[:, None] + np.arange(R)).ravel()
    win = i0[:, None] + np.arange(R + 4) - 2 + 2
    assert win.min() == 0 and win.max() == LP - 1
    # closures: rows 0, 1 in the first lane; the lanes of the last two points
    # take the end's weights, their wavefronts form them
    assert R >= 2
    for i in (nx - 2, nx - 1):
        lane = i // R
        assert lane * R >= nx // 2
        w = lane // 64
        assert w == 0 or (w + 1) * 64 * R > nx - 2
    table = np.where(rows < nx - 2, np.minimum(rows, 63), np.minimum(64 + rows - (nx - 2), 66))
    assert table.max() <= 66 and np.array_equal(table[rows == nx - 1], [65]) and np.all(table[rows >= nx] == 66)
    assert 8 * W + 4 * W + 4 * (W - 1) + 3 < 16 * W                 # part 1, backward, last wavefront's map
    assert (2 * LP + 16 * W + 6 * 67 + 64) * 8 <= 64 * 1024         # static LDS


@pytest.mark.parametrize("nx", [15, 129, 1025])
@pytest.mark.parametrize("ny", [9, 33, 48, 49, 63, 64, 65, 97, 112, 129, 144, 145, 161, 193, 225, 257, 288, 289, 321, 449, 545, 576])
def test_y_tiles(nx, ny):
    G, R = next((g, r) for g, r in Y_SHAPES if g * r >= ny)
    TX, NT, N, M = 8, 16 * G, (R + 1) // 2, G * R
    LP = M + 4
    t = np.arange(NT)
    tx, tj = t % TX, t // TX
    lds = np.zeros(2 * TX * LP, int)
    got = np.zeros((TX, ny), int)
    for q in range(N):
        use = ((q + 1) * 2 * G <= M) | (tj + 2 * G * q < M)
        at = (tx * LP + 2 + tj + 2 * G * q)[use]
        np.add.at(lds, at, 1)
        np.add.at(lds, at + TX * LP, 1)
        j = tj + 2 * G * q
        np.add.at(got, (tx[use & (j < ny)], j[use & (j < ny)]), 1)
        # a thread past the last column, or a row past the mode: past the range
        off = np.where(tx < 3, (tj * nx + nx - 3 + tx) * 16, K_BUF_OFF) + 2 * G * nx * 16 * q
        assert off.max() < 2 ** 32
        assert np.all((off < nx * ny * 16) == ((tx < 3) & (j < ny)))
    e = np.arange(64)
    np.add.at(lds, e // 4 * LP + np.where(e % 4 < 2, e % 4, M + e % 4), 1)
    assert np.all(lds == 1) and np.all(got == 1)
    assert NT // G == 2 * TX                                        # columns x parts
    j0 = np.arange(G) * R
    win = j0[:, None] + np.arange(R + 4)
    assert win.min() == 0 and win.max() == LP - 1
    for j in (ny - 2, ny - 1):
        assert (j // R) * R >= ny // 2
    tiles = -(-nx // TX) * 3
    grid, per = -(-tiles // 8) * 8, -(-tiles // 8)
    m = np.arange(grid) % 8 * per + np.arange(grid) // 8
    assert np.array_equal(np.sort(m[m < tiles]), np.arange(tiles))
    assert (2 * TX * LP + 6 * M + 64) * 8 <= 160 * 1024
