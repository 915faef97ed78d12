"""div_recip (csrc/fw_math.hpp), the FP64 division by a reciprocal pair: equal to
the machine's division for every literal divisor of the models and for random
ones, on random numerators and on those whose quotients lie nearest a rounding
boundary."""
from __future__ import annotations

import ctypes
import re
import subprocess
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parent.parent
CSRC = ROOT / "finitewave_amd" / "csrc"


def literal_divisors():
    """The divisors b of every divc(a, R(b)) of the models."""
    src = (CSRC / "fw_models.hpp").read_text()
    found = {3.0}
    for call in re.finditer(r"\bdivc\(", src):
        depth, end = 1, call.end()
        while depth:
            depth += {"(": 1, ")": -1}.get(src[end], 0)
            end += 1
        last = re.search(r",\s*R\((-?[0-9.e-]+)\)\)$", src[call.start():end])
        if last:
            found.add(float(last.group(1)))
    return sorted(found)


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    so = tmp_path_factory.mktemp("div") / "libdiv.so"
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-shared", "-fPIC", "-I", str(CSRC), "-o",
                    str(so), str(ROOT / "tests" / "native" / "fw_div_check.cpp")], check=True)
    fn = ctypes.CDLL(str(so)).fw_div_check
    fn.argtypes = [ctypes.c_void_p, ctypes.c_int64, ctypes.c_double]
    fn.restype = ctypes.c_int64
    return lambda a, b: fn(np.ascontiguousarray(a).ctypes.data, len(a), b)


def numerators(b, rng):
    a = np.concatenate([rng.uniform(-200, 200, 100_000),
                        np.exp(rng.uniform(-200, 200, 50_000)) * rng.choice([-1, 1], 50_000),
                        [0.0, 1.0, b, 3 * b]])
    # b times a 54-bit odd integer, rounded: quotients beside a rounding boundary
    m = rng.integers(2 ** 52, 2 ** 53, 50_000) * 2 + 1
    near = np.array([float(int(x)) for x in m[:2000]]) * b
    hard = np.concatenate([near, np.nextafter(near, np.inf), np.nextafter(near, -np.inf)])
    return np.concatenate([a, hard])


def test_every_literal_divisor(check):
    divisors = literal_divisors()
    assert len(divisors) > 40
    rng = np.random.default_rng(5)
    for b in divisors:
        assert check(numerators(b, rng), b) == 0, b


def test_random_divisors(check):
    rng = np.random.default_rng(6)
    for b in np.exp(rng.uniform(-40, 40, 60)):
        assert check(numerators(float(b), rng), float(b)) == 0, b
