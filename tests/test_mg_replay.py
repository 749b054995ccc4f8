"""Host replay of the restricting defect (defect_march_kernel with RS,
tbl_mg_kernels.hip) over every strip width its rule can give, and of the rule;
the constants are read from the source."""
import os
import re

import numpy as np
import pytest

import trans_bl_amd as tb

with open(os.path.join(os.path.dirname(tb.__file__), "csrc", "tbl_mg_kernels.hip")) as f:
    SRC = f.read()


def constant(name):
    return int(re.search(rf"constexpr int {name} = (\d+);", SRC).group(1))


ROWS, WAVES, HALO = constant("kDefRowsRs"), constant("kDefWaves"), 3
GRIDS = [(1025, 193), (513, 97), (257, 49), (129, 25), (385, 97), (193, 49), (2049, 257), (65, 17), (17, 9), (15, 9),
         (89, 41), (1025, 33), (129, 145)]


def strip_rule(nx, waves, start):
    """defect_strip: `start` columns, halved down to 4 until there are kDefWaves
    wavefronts, 2 where 4 columns leave less than a quarter of them."""
    def wavefronts(w):
        return waves * -(-(nx - 2) // w)

    strip = start
    while strip > 4 and wavefronts(strip) < WAVES:
        strip //= 2
    return 2 if strip == 4 and wavefronts(4) < WAVES / 4 else strip


def test_strip_rule_as_written():
    """The lines of defect_strip that the replay's rule restates."""
    body = re.search(r"static int defect_strip\(int nx, int waves\)\n\{\n(.*?)\n\}", SRC, re.S).group(1)
    assert [line.strip() for line in body.split("\n")] == [
        "int strip = sizeof(T) == 8 && sizeof(TO) == 4 && nx >= 1024 ? 64 : nx >= 512 ? 32 : 16;",
        "auto all = [&](int w) { return static_cast<long>(waves) * ((nx - 2 + w - 1) / w); };",
        "while (strip > 4 && all(strip) < kDefWaves) strip /= 2;",
        "return strip == 4 && all(4) < kDefWaves / 4 ? 2 : strip;"]
    for nx, ny in GRIDS:
        for modes in (1, 2, 8, 64, 128, 1000):
            waves = -(-(ny - 1) // ROWS) * modes
            strip = strip_rule(nx, waves, 32 if nx >= 512 else 16)
            assert strip in (2, 4, 8, 16, 32)


@pytest.mark.parametrize("strip", [2, 4, 8, 16, 32])
@pytest.mark.parametrize("nx, ny", GRIDS)
def test_restricting_defect(nx, ny, strip):
    """A wavefront takes rows 1 + 58 c - 3 + lane and columns ia .. ia + strip - 1,
    and one more where the grid has it.  Every interior coarse source point is
    written once, from defects its wavefront formed; every coarse v point, wall
    row and boundary columns included, is injected once (the last column twice,
    with the same values, where a strip ends next to it), from its own fine point;
    loads stay in the field (others are masked) and columns are even in
    number, so that a strip starts on an odd one."""
    cnx, cny = (nx - 1) // 2 + 1, (ny - 1) // 2 + 1
    lane = np.arange(64)
    source, injected = np.zeros((cnx, cny), int), np.zeros((cnx, cny), int)
    maxima = np.zeros((nx, ny), int)
    for sc in range(-(-(nx - 2) // strip)):
        ia = 1 + sc * strip
        ib0 = min(ia + strip, nx - 1)
        ib = ib0 + 1 if ib0 < nx - 1 else ib0
        assert ia % 2 == 1 and ib <= nx - 1
        for jc in range(-(-(ny - 1) // ROWS)):
            j = 1 + jc * ROWS - HALO + lane
            own = (lane >= HALO) & (lane < HALO + ROWS) & (j >= 1) & (j < ny)
            calc = (lane >= HALO - 1) & (lane <= HALO + ROWS) & (j >= 1) & (j < ny)
            inj = (own | (j == 0)) & (j % 2 == 0)

            def inject(i):
                assert i % 2 == 0 and 0 <= i < nx
                np.add.at(injected, (i >> 1, j[inj] >> 1), 1)

            if ia == 1:
                inject(0)
            for i in range(ia, ib):
                maxima[i, j[calc]] += 1
                if i % 2 == 0 and i < ib0:
                    inject(i)
                if i == nx - 2:
                    inject(nx - 1)
                if i % 2 and i >= ia + 2 and 1 <= (i - 1) >> 1 <= cnx - 2:
                    for l in np.nonzero(own & (j % 2 == 0))[0]:
                        if not 1 <= j[l] >> 1 <= cny - 1:
                            continue
                        used = [l] if j[l] == ny - 1 else [l - 1, l, l + 1]
                        assert all(0 <= u < 64 and calc[u] for u in used)
                        source[(i - 1) >> 1, j[l] >> 1] += 1
    expect = np.zeros_like(source)
    expect[1:cnx - 1, 1:cny] = 1
    assert np.array_equal(source, expect)
    assert np.all(injected[:-1] == 1) and np.all((injected[-1] >= 1) & (injected[-1] <= 2))
    # the largest defect sees every interior point
    assert np.all(maxima[1:nx - 1, 1:ny] >= 1)
