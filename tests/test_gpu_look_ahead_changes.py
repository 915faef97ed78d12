"""The run loop's look-ahead after a command that changes what it rests on: the
same run as taking every step by itself."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _halve_dt(model):
    model.dt = model.dt / 2


def _shorten(model):
    model.t_max = 1.9


def _retime(model):
    for tr in model.tracker_sequence.sequence:
        tr.step, tr.start_time = 7, 2.0


def _save(model):
    import finitewave_amd as fw

    class Saver(fw.StateSaver):
        def due(self, model):
            return round(model.t / model.dt) % 50 == 0

        def save(self):
            self.model.saves.append((self.model.step, self.model.t))
    model.state_saver = Saver()
    model.state_saver.initialize(model)


def _run(look_after, change, monkeypatch):
    import finitewave_amd as fw
    from finitewave_amd import model as M
    monkeypatch.setattr(M, "_LOOK_AFTER", look_after)
    tissue = fw.CardiacTissue2D([24, 20])
    m = fw.AlievPanfilov2D()
    m.dt, m.dr, m.t_max, m.prog_bar = 0.01, 0.25, 3.0, False
    m.cardiac_tissue = tissue
    m.saves = []
    m.stim_sequence = fw.StimSequence()
    m.stim_sequence.add_stim(fw.StimVoltageCoord2D(0, 1.0, 0, 24, 0, 5))
    seq = fw.TrackerSequence()
    act = fw.ActivationTime2DTracker()
    act.threshold = 0.5
    pot = fw.ActionPotential2DTracker()
    pot.cell_ind, pot.step = [[5, 7], [20, 9]], 2
    for t in (act, pot):
        seq.add_tracker(t)
    m.tracker_sequence = seq

    class Change(fw.Command):
        def execute(self, model):
            change(model)
    m.command_sequence = fw.CommandSequence()
    m.command_sequence.add_command(Change(1.0))
    m.run()
    return [m.u, m.u_new, m.v, act.output, np.array([m.t, m.step]), np.array(m._t_hist, float),
            np.array(pot.act_pot), np.array(m.saves, float)]


@pytest.mark.parametrize("change", [_halve_dt, _shorten, _retime, _save],
                         ids=lambda f: f.__name__)
def test_look_ahead_after_a_change(change, monkeypatch):
    want = _run(10 ** 9, change, monkeypatch)
    for after in (3, 32):
        for a, b in zip(_run(after, change, monkeypatch), want):
            assert a.shape == b.shape and a.tobytes() == b.tobytes()


@pytest.mark.parametrize("ecg, stim", [(100, 0.0), (50, 0.0), (33, 0.0), (0, 4.5)], ids=str)
def test_looks_end_at_the_next_event(ecg, stim, monkeypatch):
    # every step looked at is one taken, or all but: an ECG every few steps, a
    # stimulus that lasts
    import finitewave_amd as fw
    m = fw.AlievPanfilov2D()
    m.dt, m.dr, m.t_max, m.prog_bar = 0.01, 0.25, 6.0, False
    m.cardiac_tissue = fw.CardiacTissue2D([24, 20])
    m.stim_sequence = fw.StimSequence()
    m.stim_sequence.add_stim(fw.StimVoltageCoord2D(0, 1.0, 0, 24, 0, 5))
    if stim:
        m.stim_sequence.add_stim(fw.StimCurrentCoord2D(1.0, 0.01, stim, 0, 24, 10, 15))
    m.tracker_sequence = fw.TrackerSequence()
    if ecg:
        e = fw.ECG2DTracker()
        e.measure_coords, e.step = np.array([[12, 10, 5.0]]), ecg
        m.tracker_sequence.add_tracker(e)
    looks = []
    whole = type(m)._look_ahead

    def look(self, n, *args):
        out = whole(self, n, *args)
        looks.append((n, len(out[0])))
        return out
    monkeypatch.setattr(type(m), "_look_ahead", look)
    m.run()
    assert bool(looks) == (ecg != 33)
    assert sum(n for n, _ in looks) <= sum(k for _, k in looks) + 2 * len(looks)
