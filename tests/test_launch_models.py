"""The launch models' Python forms are the library's, and the measured launches in profiles/ are what the models are said to
be off by."""
import ctypes
import os
import random

import pytest

from tuna_amd import _lib, launch_models as lm

DATA = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "profiles", "launch_model_times.csv")


@pytest.mark.parametrize("kind", list(lm.MODELS))
def test_the_python_form_is_the_librarys(kind):
    model, coefficients = lm.MODELS[kind]
    rng = random.Random(6)
    for _ in range(150):
        for r in lm.launches(kind, rng, 4):
            us = _lib.bench_lib().tuna_predicted_us(r["m"], r["n"], r["k"], r["block"], ctypes.byref(lm.config_of(r)))
            assert us == pytest.approx(model(r, coefficients), rel=1e-9), r


# (per cent, as stated beside the models in csrc/api.cpp)
@pytest.mark.parametrize("kind,launches,off", [("flow", 440, 9.7), ("narrow", 440, 10.5), ("narrow blocks", 440, 7.1), ("wide", 323, 9.6)])
def test_the_stated_errors_are_those_of_the_kept_launches(kind, launches, off):
    model, coefficients = lm.MODELS[kind]
    rows = [r for r in lm.read(DATA) if r["kind"] == kind]
    assert len(rows) == launches
    assert 100 * lm.errors(rows, model, coefficients)[0] == pytest.approx(off, abs=0.06)


@pytest.mark.parametrize("m,n,k,shares", [(229376, 40, 4096, 512), (120064, 30, 3968, 469), (24576, 20, 3072, 192)])
def test_long_decode_batches_put_two_workgroups_on_a_compute_unit(m, n, k, shares):
    """From 14 units of 32 KB per compute unit on; whole tiles where their number is below 512 and near it.  (The last one is
    short, and what it takes is not a matter of this rule.)"""
    import re

    from tuna_amd import ops

    got = re.search(r"gemm_flow_kernel<NT=\d> (\d+) shares", ops.describe_launch(m, n, k))
    if m * k // 2 >= 14 * 256 * 32768:
        assert got and int(got.group(1)) == shares
    else:
        assert got is None or int(got.group(1)) <= 256
