"""Device memory of a plan: a second state set only where launches of several
steps use it."""
from __future__ import annotations

import pytest

from tests.test_gpu_multi_step import _model

pytestmark = pytest.mark.gpu

SIDE = 1026


@pytest.mark.parametrize("name, precision, aniso, state_bytes", [
    ("BuenoOrovio2D", "fp64", False, 0), ("FentonKarma2D", "fp64", True, 0),
    ("BuenoOrovio2D", "fp32", False, 0), ("FentonKarma2D", "fp32", True, 0),
    ("AlievPanfilov2D", "fp64", False, 8), ("FentonKarma2D", "fp32", False, 8),
])
def test_second_state_set(gpu, name, precision, aniso, state_bytes):
    from finitewave_amd.engine import Engine
    eng = Engine(_model(name, (SIDE, SIDE), precision, aniso, frozen=False))
    gpu.cuda.synchronize()
    with_plan = gpu.cuda.mem_get_info()[0]
    eng.plan.close()
    gpu.cuda.synchronize()
    held = gpu.cuda.mem_get_info()[0] - with_plan
    eng.plan = None
    # the allocator's granularity is 2 MiB
    assert abs(held - state_bytes * SIDE * SIDE) <= 4 << 20, held
