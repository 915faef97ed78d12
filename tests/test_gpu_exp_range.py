"""FP64 updates with exps left unchecked (csrc/fw_models.hpp, SPLIT): potentials on
both sides of the range that allows it, within one wavefront and alone."""
from __future__ import annotations

import numpy as np
import pytest

from tests.scenarios import make_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("far", ["none", "one", "some", "all"])
@pytest.mark.parametrize("name", ["luo_rudy91", "tp06", "courtemanche"])
def test_potentials_beyond_the_range_follow_the_oracle(name, far):
    from finitewave_amd.engine import Engine
    shape = (9, 131)
    model, sim = make_pair(name, 2, shape, dt=0.001)
    rng = np.random.RandomState(4)
    u0 = rng.uniform(-100, 60, size=shape)
    if far == "one":
        u0[4, 60] = 160.0000001
    elif far == "some":
        hit = rng.random_sample(shape) < 0.02
        u0[hit] = rng.choice([-240.0, -161.0, -160.0, 160.0, 165.0, 230.0], size=int(hit.sum()))
    elif far == "all":
        u0 = rng.uniform(165, 240, size=shape)
    inside = model.cardiac_tissue.mesh == 1
    u0[~inside] = model.u[~inside]
    model.u[...] = u0
    sim.u[...] = u0
    eng = Engine(model)
    eng.upload()
    eng.run_steps(0, 1, use_graph=False)
    u_gpu = eng.u_dev().cpu().numpy()
    sim.one_step()
    sim.u, sim.u_new = sim.u_new, sim.u
    assert np.array_equal(np.isfinite(u_gpu), np.isfinite(sim.u))
    ok = np.isfinite(sim.u)
    assert float(np.max(np.abs(u_gpu - sim.u)[ok] / np.maximum(1.0, np.abs(sim.u[ok])))) <= 1e-11
    eng.close()
