"""The six-operation FP64 division of the ionic updates (csrc/fw_models.hpp, dv) equals
the machine's.  Aliev-Panfilov's v += (-dt (eap + mu_1 v / (mu_2 + u))) (v + k u (u - a -
1)) with eap = k = mu_2 = 0, v = 1 and dt = -1 is 1 + mu_1 / u, and the quotient itself
where that is 2^60 or more."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 1 << 20


@pytest.mark.parametrize("low, high", [(-3, 3), (-40, 40), (-200, 200)], ids=str)
def test_quotients(gpu, low, high):
    from finitewave_amd import _native
    rng = np.random.default_rng(high)
    idx = gpu.arange(N, dtype=gpu.int64, device="cuda")
    for k in range(12):
        b = np.exp2(rng.uniform(low, high, N)) * rng.choice([-1.0, 1.0], N)
        b[:4] = [1.0, 3.0, -7.0, 2.0 ** low]
        a = rng.uniform(1, 2) * 2.0 ** (62 + max(abs(low), abs(high)))
        u = gpu.from_numpy(b).cuda()
        un, v = gpu.zeros_like(u), gpu.ones_like(u)
        state = (ctypes.c_void_p * 1)(v.data_ptr())
        par = (ctypes.c_double * 5)(0.1, 0.0, 0.0, a, 0.0)
        _native.check(_native.lib().fw_ionic(0, 0, un.data_ptr(), u.data_ptr(), state, 1,
                                             idx.data_ptr(), N, -1.0, par, 5, None))
        got = v.cpu().numpy()
        assert np.array_equal(got, a / b), f"{np.sum(got != a / b)} quotients of {a!r} differ"
