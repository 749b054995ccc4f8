"""Host replay of the network kernels' dispatch and indexing (tbl_unet.hip), with
the forms read from the source."""
import os
import re

import pytest

import trans_bl_amd as tb
from oracle import unet_ref as U

with open(os.path.join(os.path.dirname(tb.__file__), "csrc", "tbl_unet.hip")) as f:
    SRC = f.read()


def forms(macro):
    """The argument lists of an X-macro table."""
    text = re.search(rf"#define {macro}\(X\)((?:.*\\\n)*.*)", SRC).group(1)
    return [tuple(int(v) for v in m.split(",")) for m in re.findall(r"X\(([\d, ]+)\)", text)]


CONVS = [(cin, cout, lvl) for _, cin, cout, ks, lvl, _ in U.layers() if ks == 3]


def test_input_gradient_forms_are_the_ones_layers_take():
    """conv3x3_dx: every layer has its form, and every compiled form a layer."""
    taken = set()
    for cin, cout, _ in CONVS:
        nt = 2 if cin % 64 == 0 and cout != 32 else 1
        taken.add((3 - nt, nt, cout))
    assert taken == set(forms("TBL_DX_SHAPES"))
