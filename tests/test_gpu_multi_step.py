"""Multi-step launches of light 2D plans (csrc/fw_multi2d.hpp): n steps in one
call equal n one-step calls bit for bit -- both buffers, state, activation map
and probe trace -- at sizes around the regions' edges."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(3, 3), (5, 37), (20, 16), (21, 33), (66, 131), (300, 261)]


def _model(name, shape, precision, aniso, stims=(), frozen=True, seed=0):
    import finitewave_amd as fw
    rng = np.random.RandomState(seed)
    tissue = fw.CardiacTissue2D(list(shape))
    tissue.mesh = (1 + (rng.random_sample(shape) <= 0.15)).astype(np.int8)
    if aniso:
        tissue.fibers = np.stack([np.full(shape, 0.8), np.full(shape, 0.6)], axis=-1)
    if frozen:
        tissue.special_boundaries = (rng.random_sample(shape) <= 0.05).astype(np.int8)
    m = getattr(fw, name)()
    m.dt, m.dr, m.t_max, m.prog_bar = 0.01, 0.25, 1e9, False
    m.precision = precision
    m.cardiac_tissue = tissue
    m.stim_sequence = fw.StimSequence()
    for s in stims:
        m.stim_sequence.add_stim(s)
    m.initialize()
    m.u = rng.random_sample(shape) * (tissue.mesh > 0)
    m.u_new = m.u + 0.01 * rng.random_sample(shape)  # frozen nodes differ by parity
    return m


class _Act:
    threshold = 0.55


def _run(m, n, whole, probes=False, use_graph=True, stream=None):
    """(u, u_new, state.., act, probe rows) after n steps from step 3."""
    import torch
    from finitewave_amd.engine import Engine, Probes
    eng = Engine(m)
    eng.upload()
    eng.act[_Act] = torch.full(m.u.shape, -1, dtype=torch.int32, device=eng.dev)
    m.step = 0
    m._schedule_stims(eng, list(m.stim_sequence.sequence), n + 3)
    p = None
    if probes:
        cells = [int(c) for c in np.flatnonzero(m.cardiac_tissue.mesh == 1)[:3]] or [0]
        eng.set_probe_bits(cells)
        p = Probes(eng, [(c, v) for c in cells for v in (-1, 0)], n)
    torch.cuda.synchronize()
    with torch.cuda.stream(stream or torch.cuda.current_stream()):
        s = 3
        while s < n + 3:
            k = n if whole else 1
            rows = np.arange(s - 3, s - 3 + k, dtype=np.int32)
            eng.run_steps(s, k, _Act, np.ones(k, np.uint8), p, rows if p else None,
                          use_graph=use_graph, stim_first=s == 3)
            if not whole and s + 1 < n + 3:
                # one-step calls: the kernel hands no stimulus on past its call
                eng.apply_stims_at(s + 1)
            s += k
        torch.cuda.synchronize()
    out = [eng.u_dev(), eng.u_new_dev(), *eng.state, eng.act[_Act]] + ([p.buf] if p else [])
    out = [t.cpu().numpy() for t in out]
    eng.close()
    return out


def _same(a, b):
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert x.tobytes() == y.tobytes()


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("name", ["AlievPanfilov2D", "BuenoOrovio2D", "MitchellSchaeffer2D"])
def test_many_steps_equal_single_steps(name, precision, shape):
    for aniso in (False, True):
        for n in (5, 22, 39):
            m = _model(name, shape, precision, aniso)
            _same(_run(m, n, True), _run(m, n, False))


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("name", ["FentonKarma2D", "Barkley2D"])
def test_probe_rows_equal_single_steps(name, precision):
    m = _model(name, (37, 66), precision, True)
    _same(_run(m, 45, True, probes=True), _run(m, 45, False, probes=True))


@pytest.mark.parametrize("t0, duration", [(0.0, 0.0), (0.04, 0.0), (0.18, 0.03), (0.30, 0.9)])
def test_stimuli_inside_the_run(t0, duration):
    import finitewave_amd as fw
    st = (fw.StimVoltageCoord2D(t0, 0.9, 0, 40, 3, 9) if duration == 0 else
          fw.StimCurrentCoord2D(t0, 3.0, duration, 0, 40, 3, 9))
    m = _model("AlievPanfilov2D", (40, 50), "fp64", False, [st], frozen=False)
    whole = _run(m, 130, True)
    for s in m.stim_sequence.sequence:
        s.passed = False
    m.t = 0
    _same(whole, _run(m, 130, False))


def test_other_streams_keep_the_results():
    """The second state set belongs to one stream: a plan driven from another
    stream, or under capture, steps one at a time with the same results."""
    import torch
    from finitewave_amd.engine import Engine
    m = _model("AlievPanfilov2D", (70, 90), "fp64", True)
    want = _run(m, 41, True)
    eng = Engine(m)
    side = torch.cuda.Stream()
    for stream in (torch.cuda.current_stream(), side):
        eng.upload()
        eng.act[_Act] = torch.full(m.u.shape, -1, dtype=torch.int32, device=eng.dev)
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            eng.run_steps(3, 41, _Act, np.ones(41, np.uint8))
        torch.cuda.synchronize()
        _same(want, [t.cpu().numpy() for t in (eng.u_dev(), eng.u_new_dev(), *eng.state,
                                               eng.act[_Act])])
    eng.upload()
    eng.act[_Act] = torch.full(m.u.shape, -1, dtype=torch.int32, device=eng.dev)
    keep = [t.clone() for t in (eng.A, eng.B, *eng.state)]
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        eng.run_steps(3, 41, _Act, np.ones(41, np.uint8), use_graph=False)
    for _ in range(3):
        for t, k in zip((eng.A, eng.B, *eng.state), keep):
            t.copy_(k)
        eng.act[_Act].fill_(-1)
        g.replay()
        torch.cuda.synchronize()
        _same(want, [t.cpu().numpy() for t in (eng.u_dev(), eng.u_new_dev(), *eng.state,
                                               eng.act[_Act])])
    eng.close()
