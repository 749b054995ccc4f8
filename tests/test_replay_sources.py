"""The shape tables that the kernels' host replays restate, against the sources."""
import os
import re

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
