"""The exact FP64 diffusion weights of the anisotropic steps: packed conduct
bits at the edges of a grid, heavy fibrosis, and the division by dr**2."""
from __future__ import annotations

import numpy as np
import pytest

from tests.scenarios import layered_fibers, make_pair, random_fibers

pytestmark = pytest.mark.gpu


def run_equal(shape, fibers, fibrosis, dr, steps=3):
    from finitewave_amd.engine import Engine
    model, sim = make_pair("aliev_panfilov", len(shape), shape, stencil="aniso", fibrosis=fibrosis,
                           fibers=fibers, dr=dr)
    u0 = np.random.RandomState(sum(shape)).uniform(0, 1, size=shape)
    u0[model.cardiac_tissue.mesh != 1] = 0.0
    model.u[...] = u0
    sim.u[...] = u0
    eng = Engine(model)
    eng.upload()
    eng.run_steps(0, steps, use_graph=False)
    u_gpu = eng.u_dev().cpu().numpy()
    for _ in range(steps):
        sim.one_step()
        sim.u, sim.u_new = sim.u_new, sim.u
    assert np.array_equal(u_gpu, sim.u)
    eng.close()


@pytest.mark.parametrize("dr", [0.25, 0.3])
@pytest.mark.parametrize("fibrosis", [0.0, 0.5])
@pytest.mark.parametrize("shape", [(3, 3, 3), (3, 4, 62), (5, 3, 5), (18, 7, 31), (3, 3),
                                   (4, 67), (33, 21)], ids=str)
def test_steps_equal_oracle(shape, fibrosis, dr):
    """Three steps from random potentials, bit for bit, dr**2 a power of two
    and not."""
    run_equal(shape, layered_fibers(shape) if len(shape) == 3 else
              random_fibers(shape), fibrosis, dr)
