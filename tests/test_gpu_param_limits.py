"""FP64 parameters at infinity, the plain way to switch a current or a relaxation
off: every step equals the oracle's wherever the oracle's is a number."""
from __future__ import annotations

import numpy as np
import pytest

from tests.scenarios import make_pair

pytestmark = pytest.mark.gpu


def _steps(name, params, steps=12):
    from finitewave_amd.engine import Engine
    model, sim = make_pair(name, 2, (14, 12), fibrosis=0.1)
    for p, value in params.items():
        setattr(model, p, value)
        sim.params[p] = value
    eng = Engine(model)
    eng.upload()
    compared = 0
    for s in range(steps):
        with np.errstate(all="ignore"):
            sim.one_step()
        sim.u, sim.u_new = sim.u_new, sim.u
        arrays = [sim.u] + [sim.state[n] for n in eng.state_names]
        if not all(np.isfinite(a).all() for a in arrays):
            break
        eng.run_steps(s, 1, use_graph=False)
        got = [eng.u_dev().cpu().numpy()] + [a for _, a in eng.state_values()]
        for q, (a, b) in enumerate(zip(got, arrays)):
            err = np.max(np.abs(a - b) / np.maximum(1.0, np.abs(b)))
            assert err <= 1e-12, f"step {s}, array {q}: {err}"
        compared += 1
    eng.close()
    return compared


FK = ["tau_d", "tau_o", "tau_r", "tau_si", "tau_v_m", "tau_v_p", "tau_w_m", "tau_w_p"]


@pytest.mark.parametrize("param", FK)
def test_fenton_karma_time_constants(gpu, param):
    assert _steps("fenton_karma", {param: np.inf}) == 12


@pytest.mark.parametrize("param", ["caupmax", "Vj"])
def test_courtemanche_uniform_divisors(gpu, param):
    assert _steps("courtemanche", {param: np.inf}) == 12
