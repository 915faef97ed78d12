"""pow15 (csrc/fw_math.hpp), the x^1.5 of the FP64 Courtemanche update, against
exact integer arithmetic: within 0.5001 ulp over the range its argument
kmnai / nai can take and far beyond, and its special values."""
from __future__ import annotations

import ctypes
import math
import subprocess
from fractions import Fraction
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def pow15(tmp_path_factory):
    so = tmp_path_factory.mktemp("pow15") / "libpow15.so"
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-shared", "-fPIC", "-I",
                    str(ROOT / "finitewave_amd" / "csrc"), "-o", str(so),
                    str(ROOT / "tests" / "native" / "fw_pow_check.cpp")], check=True)
    fn = ctypes.CDLL(str(so)).fw_pow15
    fn.argtypes = [ctypes.c_void_p, ctypes.c_int64, ctypes.c_void_p]

    def call(x):
        x = np.ascontiguousarray(x, dtype=np.float64)
        out = np.empty_like(x)
        fn(x.ctypes.data, len(x), out.ctypes.data)
        return out
    return call


@pytest.mark.parametrize("lo, hi", [(0.1, 10.0), (1e-9, 1e9), (1e-150, 1e150)])
def test_pow15_is_within_half_an_ulp(pow15, lo, hi):
    rng = np.random.default_rng(3)
    x = np.exp(rng.uniform(math.log(lo), math.log(hi), 3000))
    for a, y in zip(x, pow15(x)):
        cube = Fraction(float(a)) ** 3
        y = float(y)
        ulp = Fraction(math.ulp(y))
        d = Fraction(5001, 10000) * ulp
        assert (Fraction(y) - d) ** 2 <= cube <= (Fraction(y) + d) ** 2


def test_pow15_special_values(pow15):
    y = pow15([0.0, 1.0, 4.0, math.inf, math.nan, 1e300])
    assert list(y[:4]) == [0.0, 1.0, 8.0, math.inf]
    assert math.isnan(y[4]) and y[5] == math.inf
