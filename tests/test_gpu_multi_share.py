"""One plan, several buffer sets: runs that two host threads enqueue on one stream
or on two, and runs that move from stream to stream, equal the same runs taken one
after the other (the plan's second state set serves one run at a time)."""
from __future__ import annotations

import threading

import numpy as np
import pytest

from tests.test_gpu_multi_step import _model, _same

pytestmark = pytest.mark.gpu

RUNS, STEPS = 25, 41


def _engines(torch, n):
    """n engines on one plan, each with its own state."""
    from finitewave_amd.engine import Engine
    engines = []
    for q in range(n):
        m = _model("FentonKarma2D", (61, 75), "fp64", True, seed=3)
        m.u = m.u * (0.5 + 0.25 * q)  # the same tissue, another state
        e = Engine(m)
        if q:
            e.plan.close()
            e.plan = engines[0].plan
        e.upload()
        engines.append(e)
    torch.cuda.synchronize()
    return engines


def _drive(eng, runs):
    for r in range(runs):
        eng.run_steps(r * STEPS, STEPS, use_graph=False)


def _values(eng):
    return [t.cpu().numpy() for t in (eng.u_dev(), eng.u_new_dev(), *eng.state)]


def _close(engines):
    for e in engines[1:]:
        e.plan = None
    engines[0].close()


@pytest.fixture(scope="module")
def serial(gpu):
    engines = _engines(gpu, 2)
    for e in engines:
        _drive(e, RUNS)
        gpu.cuda.synchronize()
    want = [_values(e) for e in engines]
    _close(engines)
    return want


@pytest.mark.parametrize("streams", ["one", "two"])
def test_two_threads_on_one_plan(gpu, serial, streams):
    engines = _engines(gpu, 2)
    side = [gpu.cuda.current_stream(), gpu.cuda.Stream()] if streams == "two" else \
        [gpu.cuda.current_stream()] * 2
    gate = threading.Barrier(2)
    failed = []

    def work(q):
        try:
            gpu.cuda.set_device(0)
            gate.wait(30)
            with gpu.cuda.stream(side[q]):
                _drive(engines[q], RUNS)
        except Exception as e:  # pragma: no cover
            failed.append(e)

    threads = [threading.Thread(target=work, args=(q,)) for q in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    gpu.cuda.synchronize()
    assert not failed
    for e, want in zip(engines, serial):
        _same(_values(e), want)
    _close(engines)


def test_runs_that_move_between_streams(gpu, serial):
    # two tissues of one plan, a run of each in turn: on a stream of its own, on the
    # other's, on a new one after its stream is gone, without waiting in between
    engines = _engines(gpu, 2)
    streams, done = [gpu.cuda.Stream(), gpu.cuda.Stream()], [None, None]
    for r in range(RUNS):
        if r % 8 == 7:
            gpu.cuda.synchronize()
        if r % 5 == 4:
            streams[1] = gpu.cuda.Stream()
        for q, e in enumerate(engines):
            s = streams[(q + r // 3) % 2]
            if done[q] is not None:
                s.wait_event(done[q])
            with gpu.cuda.stream(s):
                e.run_steps(r * STEPS, STEPS, use_graph=False)
            done[q] = s.record_event()
    gpu.cuda.synchronize()
    for e, want in zip(engines, serial):
        _same(_values(e), want)
    _close(engines)
