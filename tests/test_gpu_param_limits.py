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


# the parameters that divide, in the node's own terms
DIVISORS = [("aliev_panfilov", ["mu_2"]), ("luo_rudy91", ["F"]),
            ("courtemanche", ["kup", "kmnai", "kmko", "kmnancx", "kmcancx", "ksatncx", "trpnmax",
                              "cmdnmax", "csqnmax", "kq10"])]


@pytest.mark.parametrize("name, param", [(n, p) for n, ps in DIVISORS for p in ps])
def test_divisors_with_a_parameter(gpu, name, param):
    assert _steps(name, {param: np.inf}) == 12


def test_a_stopped_temperature_factor(gpu):
    # kq10 = 0 freezes four gates: their time constants are infinite
    assert _steps("courtemanche", {"kq10": 0.0}) == 12


@pytest.mark.parametrize("name", ["luo_rudy91", "courtemanche"])
def test_potentials_whose_rates_overflow(gpu, name):
    # single nodes far outside the physiological range, and one ulp above 3.3328,
    # where e^x - 1 rounds to zero: one step where the oracle's is a number
    from finitewave_amd.engine import Engine
    volts = [200.0, -200.0, 1000.0, -1000.0, 3000.0, -3000.0, 3650.0, 3700.0, 4000.0, 5000.0,
             7000.0, 10000.0, 20000.0, -5000.0, 3.3328000000000007, -80.0]
    shape = (3, 2 * len(volts) + 1)
    model, sim = make_pair(name, 2, shape)
    mesh = np.full(shape, 2, dtype=np.int8)
    mesh[1, 1::2] = 1
    mesh[0], mesh[-1], mesh[:, 0], mesh[:, -1] = 0, 0, 0, 0
    model.cardiac_tissue.mesh = mesh.copy()
    model.compute_weights()
    sim.mesh = mesh.copy()
    sim.compute_weights()
    model.u[:] = sim.init_u
    sim.u[:] = sim.init_u
    model.u[1, 1::2] = volts
    sim.u[1, 1::2] = volts
    eng = Engine(model)
    eng.upload()
    eng.run_steps(0, 1, use_graph=False)
    with np.errstate(all="ignore"):
        sim.one_step()
    got = [eng.u_dev().cpu().numpy()] + [a for _, a in eng.state_values()]
    want = [sim.u_new] + [sim.state[n] for n in eng.state_names]
    numbers = 0
    for k, volt in enumerate(volts):
        pairs = [(float(a[1, 1 + 2 * k]), float(b[1, 1 + 2 * k])) for a, b in zip(got, want)]
        if not np.isfinite([b for _, b in pairs]).all():
            continue
        numbers += 1
        for q, (a, b) in enumerate(pairs):
            assert abs(a - b) <= 1e-12 * max(1.0, abs(b)), f"u = {volt}, array {q}: {a} {b}"
    eng.close()
    assert numbers >= 12
