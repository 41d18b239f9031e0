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
@pytest.mark.parametrize("kind,launches,off", [("flow", 440, 9.7), ("narrow", 440, 10.5), ("narrow blocks", 440, 7.1), ("wide", 323, 14.4)])
def test_the_stated_errors_are_those_of_the_kept_launches(kind, launches, off):
    model, coefficients = lm.MODELS[kind]
    rows = [r for r in lm.read(DATA) if r["kind"] == kind]
    assert len(rows) == launches
    assert 100 * lm.errors(rows, model, coefficients)[0] == pytest.approx(off, abs=0.06)
