"""The run loop's look-ahead over event-free steps: the same trackers, times and
state as taking every step by itself, with gates, stimuli, commands and host
events falling anywhere."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(look_after, case, monkeypatch):
    import finitewave_amd as fw
    from finitewave_amd import model as M
    monkeypatch.setattr(M, "_LOOK_AFTER", look_after)
    monkeypatch.setattr(M, "_CHUNK", 256)
    monkeypatch.setattr(M, "_LOOK_AHEAD", 64)
    tissue = fw.CardiacTissue2D([40, 34])
    m = fw.AlievPanfilov2D()
    m.dt, m.dr, m.t_max, m.prog_bar = 0.01, 0.25, case.get("t_max", 6.0), False
    m.cardiac_tissue = tissue
    m.stim_sequence = fw.StimSequence()
    m.stim_sequence.add_stim(fw.StimVoltageCoord2D(0, 1.0, 0, 40, 0, 5))
    for t in case.get("stims", ()):
        m.stim_sequence.add_stim(fw.StimCurrentCoord2D(t, 4.0, 0.05, 0, 40, 20, 25))
    seq = fw.TrackerSequence()
    act = fw.ActivationTime2DTracker()
    act.threshold, act.start_time, act.end_time = 0.5, case.get("start", 0), case.get("end", 99)
    pots = []
    for step in case.get("probes", (1,)):
        p = fw.ActionPotential2DTracker()
        p.cell_ind, p.step = [[5, 7], [20, 9]], step
        pots.append(p)
    mv = fw.MultiVariable2DTracker()
    mv.var_list, mv.cell_ind, mv.step, mv.start_time = ["u", "v"], [6, 6], 3, 1.0
    for t in [act, *pots, mv]:
        seq.add_tracker(t)
    if "ecg" in case:
        e = fw.ECG2DTracker()
        e.measure_coords, e.step = np.array([[20, 17, 5.0]]), case["ecg"]
        seq.add_tracker(e)
    m.tracker_sequence = seq
    fired = []
    if "commands" in case:
        class Mark(fw.Command):
            def execute(self, model):
                fired.append((model.step, model.t))
                model.u[30, 30] = 0.7
        m.command_sequence = fw.CommandSequence()
        for t in case["commands"]:
            m.command_sequence.add_command(Mark(t))
    m.run()
    out = [m.u, m.u_new, m.v, act.output, np.array([m.t, m.step]), np.array(m._t_hist, float),
           np.array(fired, float)]
    out += [np.array(p.act_pot) for p in pots] + [np.array(mv.vars[v]) for v in ("u", "v")]
    if "ecg" in case:
        out.append(np.asarray(seq.sequence[-1].output))
    return out


@pytest.mark.parametrize("case", [
    dict(), dict(t_max=0.35), dict(t_max=2.56, probes=()), dict(start=0.7, end=2.31, probes=(7,)),
    dict(stims=(0.333, 2.0)), dict(commands=(0.5, 0.51, 3.0), probes=(1, 4)),
    dict(ecg=50, probes=(2, 5)), dict(ecg=3), dict(stims=(1.1,), commands=(1.12,), ecg=70),
], ids=str)
def test_look_ahead_equals_step_by_step(case, monkeypatch):
    want = _run(10 ** 9, case, monkeypatch)
    for after in (1, 5, 32):
        got = _run(after, case, monkeypatch)
        assert len(got) == len(want)
        for a, b in zip(got, want):
            if "ecg" in case and a is got[-1]:  # atomics: the sum's order varies
                np.testing.assert_allclose(a, b, rtol=1e-9, atol=1e-12)
            else:
                assert a.shape == b.shape and a.tobytes() == b.tobytes()
