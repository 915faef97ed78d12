"""fw_run_graph_prepare: the first graph-replayed run after it captures nothing.  A
capture takes milliseconds and a replay's launches tens of microseconds, so the
two are told apart by the host time of the call, on fresh plans."""
from __future__ import annotations

import time

import numpy as np
import pytest

from tests.test_gpu_multi_step import _model, _same

pytestmark = pytest.mark.gpu


def _first_call(torch, name, shape, steps, stim, prepare):
    """(host seconds of the first run, its results)."""
    import finitewave_amd as fw
    from finitewave_amd.engine import Engine
    stims = [fw.StimCurrentCoord2D(0.1, 0.5, stim, 0, shape[0], 3, 9)] if stim else []
    m = _model(name, shape, "fp64", False, stims, frozen=False)
    eng = Engine(m)
    eng.upload()
    m.step = 0
    m._schedule_stims(eng, list(m.stim_sequence.sequence), steps)
    if prepare:
        eng.prepare_graphs(steps)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    eng.run_steps(0, steps)
    took = time.perf_counter() - t0
    torch.cuda.synchronize()
    out = [t.cpu().numpy() for t in (eng.u_dev(), eng.u_new_dev(), *eng.state)]
    eng.close()
    return took, out


# a plan without multi-step launches, a run too short for them, a stimulus across
# which single steps are replayed
@pytest.mark.parametrize("name, shape, steps, stim", [
    ("BuenoOrovio2D", (514, 514), 254, 0.0),
    ("AlievPanfilov2D", (102, 102), 4, 0.0),
    ("AlievPanfilov2D", (102, 102), 300, 1.25),
], ids=["single", "short", "stimulus"])
def test_a_prepared_run_captures_nothing(gpu, name, shape, steps, stim):
    _first_call(gpu, name, shape, steps, stim, False)  # the kernels' first load
    cold = min(_first_call(gpu, name, shape, steps, stim, False)[0] for _ in range(4))
    runs = [_first_call(gpu, name, shape, steps, stim, True) for _ in range(4)]
    assert min(t for t, _ in runs) < 0.5 * cold
    _same(runs[0][1], _first_call(gpu, name, shape, steps, stim, False)[1])
