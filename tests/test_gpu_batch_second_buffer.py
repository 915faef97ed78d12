"""A batch tissue whose second potential buffer and second state set hold no numbers
when it is admitted: the multi-step shapes, which write every node of a tissue, step
it as one whose buffers are filled."""
from __future__ import annotations

import numpy as np
import pytest

import finitewave_amd as fw
from finitewave_amd.batch import TissueBatch
from tests.test_gpu_batch import _check_same
from tests.test_gpu_batch_edges import edge_sims

pytestmark = pytest.mark.gpu


def _run(model, prec, variant, fill):
    sims = edge_sims(3)
    b = TissueBatch(getattr(fw, model), precision=prec, max_tissues=6, autotune=False,
                    chunk_cap=23)
    b.set_variant(variant)
    for s in sims:
        buf = b.buffers[b.admit(s)]
        if fill:
            for t in (buf["un"], *buf["state_alt"]):
                t.fill_(float("nan"))
    b.run_all()
    b.close()
    return [s.result for s in sims]


@pytest.mark.parametrize("model,prec", [("MitchellSchaeffer2D", "fp32"),
                                        ("AlievPanfilov2D", "fp64")])
def test_unfilled_second_buffers(gpu, model, prec):
    b = TissueBatch(getattr(fw, model), precision=prec, max_tissues=2)
    variants = [v for v in b.variants() if v & 8]
    b.close()
    for v in variants:
        for a, r in zip(_run(model, prec, v, True), _run(model, prec, v, False)):
            assert np.isfinite(a["u"]).all()
            _check_same(a, r)
