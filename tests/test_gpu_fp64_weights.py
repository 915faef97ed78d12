"""The exact FP64 diffusion weights of the anisotropic steps: packed conduct
bits at the edges of a grid, heavy fibrosis, the division by dr**2, and per-node
fields."""
from __future__ import annotations

import ctypes

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


def inplane_fibers(shape):
    """Per-node angles in the plane of the first two axes: the fields with the
    third axis are uniform, the others full arrays."""
    ang = np.random.RandomState(2).uniform(-1.5, 1.5, size=shape)
    f = np.zeros((*shape, 3))
    f[..., 0], f[..., 1] = np.cos(ang), np.sin(ang)
    return f


@pytest.mark.parametrize("kind", ["any", "inplane"])
@pytest.mark.parametrize("shape", [(3, 3, 3), (3, 4, 62), (18, 7, 31), (33, 21)], ids=str)
def test_per_node_fibres_equal_oracle(shape, kind):
    """Full-array fields, and full ones beside uniform ones."""
    run_equal(shape, inplane_fibers(shape) if kind == "inplane" and len(shape) == 3 else
              random_fibers(shape), 0.3, 0.25)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_mixed_fields_same_with_and_without_a_plan(precision):
    """Full and uniform fields together: a plan's steps, a replayed graph's and
    the allocation-free call's are the same bits."""
    import torch
    from finitewave_amd import _native
    from finitewave_amd.engine import Engine
    shape = (9, 14, 35)
    out = []
    for mode in ("plan", "graph", "noalloc"):
        model, _ = make_pair("aliev_panfilov", 3, shape, stencil="aniso", fibrosis=0.2,
                             fibers=inplane_fibers(shape), precision=precision)
        model.u[1:4] = 1.0 * (model.cardiac_tissue.mesh[1:4] == 1)
        eng = Engine(model)
        eng.upload()
        if mode == "noalloc":
            rc = _native.lib().fw_run_noalloc(
                ctypes.byref(eng.plan.desc), eng.A.data_ptr(), eng.B.data_ptr(),
                eng._state_ptrs, 0, 20, None, None)
            _native.check(rc, "fw_run_noalloc")
            torch.cuda.synchronize()
            out.append(eng.A.cpu().numpy())
        else:
            eng.run_steps(0, 20, use_graph=mode == "graph")
            out.append(eng.u_dev().cpu().numpy())
        eng.close()
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])
