"""The committed table of line shapes against the kernels it chooses from."""
import json
import os

import pytest

import trans_bl_amd as tb

with open(os.path.join(os.path.dirname(tb.__file__), "weights", "linetune.json")) as f:
    TABLE = json.load(f)


@pytest.mark.parametrize("key", sorted(TABLE))
def test_chosen_shapes_are_the_fastest_measured(key):
    e = TABLE[key]
    for prec in ("fp64", "fp32"):
        us = {int(k.split(":")[1]): v for k, v in e["us_per_sweep"].items() if k.startswith(prec)}
        assert us[e[prec]] == min(us.values()), (prec, us)


@pytest.mark.parametrize("key", sorted(k for k in TABLE if k.endswith("c") and int(k[:-1].split("x")[1]) <= 33))
def test_coarsest_classes_take_the_inverse_matrices(key):
    """Coarsest levels of up to 33 rows: the inverse line matrices (shape 1) take
    a half to a tenth of the lane scan's time at every class, so an entry with
    another shape was timed against other code."""
    e = TABLE[key]
    assert e["fp64"] == e["fp32"] == 1
    for prec in ("fp64", "fp32"):
        assert e["us_per_sweep"][f"{prec}:1"] < 0.7 * e["us_per_sweep"][f"{prec}:16"]
