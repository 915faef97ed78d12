"""The multi-step batch shapes on tissues whose outer columns get no lanes
(csrc/fw_batch_tb.hpp): activation times and the probe of the outer layer."""
from __future__ import annotations

import numpy as np
import pytest

import finitewave_amd as fw
from finitewave_amd.batch import BatchSim, TissueBatch
from tests.test_gpu_batch import _check_same

pytestmark = pytest.mark.gpu


def edge_sims(seed):
    """Widths of 64, 120 and 124 inner columns (one strip fewer without the
    outer ones) and their neighbours; a threshold below rest records every
    node, and the probes lie on the outer columns."""
    rng = np.random.default_rng(seed)
    out = []
    for k, (ni, nj) in enumerate([(70, 66), (270, 126), (9, 122), (3, 65), (40, 123), (33, 67)]):
        t = fw.CardiacTissue2D([ni, nj])
        mesh = (1 + (rng.random((ni, nj)) <= 0.2)).astype(np.int8)
        mesh[0], mesh[-1], mesh[:, 0], mesh[:, -1] = 0, 0, 0, 0
        t.mesh = mesh
        out.append(BatchSim(tissue=t, t_max=0.6 + 0.05 * k,
                            stims=[fw.StimVoltageCoord2D(0, 1.0, 0, ni, 0, 5)],
                            probe=(ni // 2, 0 if k % 2 else nj - 1), act_threshold=-0.5,
                            act_start=0.03 * k, apd_threshold=0.5))
    return out


@pytest.mark.parametrize("model,prec", [("MitchellSchaeffer2D", "fp32"),
                                        ("AlievPanfilov2D", "fp64")])
def test_outer_columns_equal_the_single_step_shape(model, prec):
    results = {}
    b = TissueBatch(getattr(fw, model), precision=prec, max_tissues=2)
    variants = [v for v in b.variants() if v & 8]
    b.close()
    for v in [0] + variants:
        sims = edge_sims(3)
        b = TissueBatch(getattr(fw, model), precision=prec, max_tissues=6, autotune=False,
                        chunk_cap=23)
        b.set_variant(v)
        for s in sims:
            b.admit(s)
        b.run_all()
        b.close()
        results[v] = [s.result for s in sims]
    for r in results[0]:
        assert np.all(r["act_t"][:, [0, -1]] >= 0)
    for v in variants:
        for a, r in zip(results[v], results[0]):
            _check_same(a, r)
