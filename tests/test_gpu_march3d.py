"""The FP32 19-point march (csrc/fw_march3d.hpp) at the edges of its tiles: rows
in twos, columns in sixty-twos, planes in chunks."""
from __future__ import annotations

import numpy as np
import pytest

import finitewave_amd as fw
from tests.scenarios import boxed_mesh, layered_fibers, make_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(3, 3, 3), (3, 4, 62), (4, 5, 63), (7, 6, 64), (18, 7, 31),
                                   (90, 130, 129)], ids=str)
@pytest.mark.parametrize("name", ["aliev_panfilov", "bueno_orovio"])
def test_one_step_matches_fp64_oracle(name, shape):
    """One step from random potentials on a 30 % fibrotic mesh within 1e-5 of
    the oracle's FP64 step; (90, 130, 129) marches several planes per block."""
    from finitewave_amd.engine import Engine
    rng = np.random.RandomState(sum(shape))
    model, sim = make_pair(name, 3, shape, stencil="aniso", fibrosis=0.3,
                           fibers=layered_fibers(shape, -70.0, 50.0), precision="fp32")
    u0 = rng.uniform(0, 1, size=shape)
    u0[model.cardiac_tissue.mesh != 1] = 0.0
    model.u[...] = u0
    sim.u[...] = u0
    eng = Engine(model)
    eng.upload()
    eng.run_steps(0, 1, use_graph=False)
    u_gpu = eng.u_dev().cpu().numpy().astype(np.float64)
    sim.one_step()
    sim.u, sim.u_new = sim.u_new, sim.u
    act = model.cardiac_tissue.mesh == 1
    if act.any():
        assert float(np.max(np.abs(u_gpu[act] - sim.u[act]))) <= 1e-5
    assert np.all(u_gpu[~act] == 0.0)
    eng.close()


def test_frozen_nodes_stimuli_probes_and_map_follow_fp64():
    """40 steps with frozen nodes, a stimulus over them inside the run, probes
    and an activation map: within float rounding of the FP64 path."""
    shape = (21, 13, 66)
    out = {}
    for precision in ("fp64", "fp32"):
        tissue = fw.CardiacTissue3D(list(shape))
        tissue.mesh = boxed_mesh(shape, 0.2, seed=5)
        tissue.fibers = layered_fibers(shape)
        tissue.special_boundaries = (np.random.RandomState(9).random_sample(shape) < 0.05
                                     ).astype(np.int8)
        m = fw.AlievPanfilov3D()
        m.dt, m.dr, m.t_max, m.prog_bar = 0.01, 0.25, 0.4, False
        m.precision = precision
        m.cardiac_tissue = tissue
        m.stim_sequence = fw.StimSequence()
        m.stim_sequence.add_stim(fw.StimVoltageCoord3D(0, 1.0, 0, 4, 0, 13, 0, 66))
        m.stim_sequence.add_stim(fw.StimCurrentCoord3D(0.1, 3.0, 0.1, 8, 20, 2, 11, 30, 64))
        act = fw.ActivationTime3DTracker()
        act.threshold = 0.25
        pot = fw.ActionPotential3DTracker()
        pot.cell_ind = [[2, 5, 40], [12, 6, 50]]
        m.tracker_sequence = fw.TrackerSequence()
        m.tracker_sequence.add_tracker(act)
        m.tracker_sequence.add_tracker(pot)
        m.run()
        out[precision] = (m.u, m.u_new, m.v, np.asarray(pot.output), np.asarray(act.output))
    for a, b in zip(out["fp64"][:4], out["fp32"][:4]):
        assert np.max(np.abs(a - b)) <= 1e-5
    a, b = out["fp64"][4], out["fp32"][4]
    assert np.array_equal(a >= 0, b >= 0) and np.count_nonzero(a >= 0) > 1000
    assert np.max(np.abs(a - b)) <= 0.01 + 1e-9
