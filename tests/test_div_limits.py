"""div_recip (csrc/fw_math.hpp) at divisors without a finite reciprocal pair: a
parameter set to infinity or to zero divides as the machine does."""
from __future__ import annotations

import ctypes
import subprocess
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def quotients(tmp_path_factory):
    so = tmp_path_factory.mktemp("div") / "libdivv.so"
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-shared", "-fPIC", "-I",
                    str(ROOT / "finitewave_amd" / "csrc"), "-o", str(so),
                    str(ROOT / "tests" / "native" / "fw_div_values.cpp")], check=True)
    fn = ctypes.CDLL(str(so)).fw_div_values
    fn.argtypes = [ctypes.c_void_p, ctypes.c_int64, ctypes.c_double, ctypes.c_void_p]

    def run(a, b):
        out = np.empty(len(a))
        fn(a.ctypes.data, len(a), b, out.ctypes.data)
        return out
    return run


@pytest.mark.parametrize("b", [np.inf, -np.inf, 0.0, -0.0, np.nan], ids=repr)
def test_divisors_without_a_pair(quotients, b):
    a = np.array([0.3, -0.3, 1.0, -1e300, 1e-300, 0.0, -0.0, np.inf, -np.inf, np.nan])
    with np.errstate(all="ignore"):
        want = a / b
    got = quotients(a, b)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    assert got[ok].tobytes() == want[ok].tobytes()
