"""The batch tuner chooses a launch shape for the stencils a batch holds: one timed on
5-point tissues is not taken for 9-point tissues of the same size."""
from __future__ import annotations

import pytest

import finitewave_amd as fw
from finitewave_amd.batch import TissueBatch
from tests.test_gpu_batch import _sims

pytestmark = pytest.mark.gpu


def _tuned(kinds, n=3):
    b = TissueBatch(fw.MitchellSchaeffer2D, precision="fp32", max_tissues=8, tune_steps=4)
    for k, kind in enumerate(kinds):
        for s in _sims(kind, n=n, seed=12 + k, t_max=3.0):
            b.admit(s)
    b.run_all()
    out = b.tuning, b._tuned_key
    b.close()
    return out


def test_each_stencil_is_timed(gpu, tmp_path, monkeypatch):
    from finitewave_amd import batch as B
    monkeypatch.setenv("FW_AUTOTUNE_CACHE", str(tmp_path / "tune.json"))
    monkeypatch.setattr(B, "_TUNE_CACHE", {})
    first = _tuned(["iso"])
    assert first[0] is not None
    other = _tuned(["aniso"])
    assert other[0] is not None and other[1] != first[1]
    assert _tuned(["iso"]) == (None, first[1])  # from the cache
