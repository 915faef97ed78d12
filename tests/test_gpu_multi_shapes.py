"""Every launch shape of the light 2D plans' multi-step launches -- 20, 24 and 32
region rows at 8 steps per launch, 16 and 32 at 4, the shorter launches of short
runs -- for each model, precision and stencil: bit for bit single steps, and the
shape is the one the sheet's size is meant to get."""
from __future__ import annotations

from ctypes import byref, c_int32

import pytest

from tests.test_gpu_multi_step import _model, _run, _same

pytestmark = pytest.mark.gpu

MODELS = ["AlievPanfilov2D", "Barkley2D", "MitchellSchaeffer2D", "FentonKarma2D",
          "BuenoOrovio2D"]
TANH = ("FentonKarma2D", "BuenoOrovio2D")
SHAPES = [(61, 75), (129, 161), (200, 205), (301, 262)]


def _shape(eng, n):
    from finitewave_amd import _native
    k, rows = c_int32(), c_int32()
    _native.check(_native.lib().fw_plan_launch_shape(eng.plan.handle, n, byref(k), byref(rows)))
    return k.value, rows.value


def _expected(name, shape, precision, aniso):
    f64 = precision == "fp64"
    if name in TANH and f64:
        return {61: (8, 20), 129: (4, 16), 200: (4, 16), 301: (1, 0)}[shape[0]]
    if shape[0] < 301:
        return {61: (8, 20), 129: (8, 24), 200: (8, 32)}[shape[0]]
    if name in TANH:
        return (4, 16) if aniso or name == "BuenoOrovio2D" else (4, 32)
    return (4, 16) if aniso and f64 else (4, 32)


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("name", MODELS)
def test_every_launch_shape(gpu, name, precision, shape):
    from finitewave_amd.engine import Engine
    for aniso in (False, True):
        m = _model(name, shape, precision, aniso, seed=shape[0])
        eng = Engine(m)
        want = _expected(name, shape, precision, aniso)
        assert _shape(eng, 40) == want
        if want != (1, 0):
            # FP64 Bueno-Orovio takes no two-step launches
            two = (1, 0) if (name, precision) == ("BuenoOrovio2D", "fp64") else (2, want[1])
            assert _shape(eng, 5) == two and _shape(eng, 9) == (4, want[1])
        assert _shape(eng, 4) == (1, 0)
        eng.close()
        for n in (5, 9, 27):
            _same(_run(m, n, True), _run(m, n, False))


# (model, precision, aniso, side) on either side of the sizes up to which several
# steps per launch, and two steps for a short run, are the faster
@pytest.mark.parametrize("name, precision, aniso, side, many, few", [
    ("AlievPanfilov2D", "fp64", True, 724, 4, 1), ("AlievPanfilov2D", "fp64", True, 725, 1, 1),
    ("MitchellSchaeffer2D", "fp64", True, 627, 4, 2),
    ("MitchellSchaeffer2D", "fp64", True, 628, 1, 1),
    ("MitchellSchaeffer2D", "fp64", False, 1619, 4, 1),
    ("MitchellSchaeffer2D", "fp64", False, 1620, 1, 1),
    ("Barkley2D", "fp64", False, 2048, 4, 1), ("Barkley2D", "fp64", False, 2049, 1, 1),
    ("AlievPanfilov2D", "fp32", False, 1254, 4, 1), ("AlievPanfilov2D", "fp32", False, 1255, 1, 1),
    ("AlievPanfilov2D", "fp32", True, 627, 4, 2), ("AlievPanfilov2D", "fp32", True, 628, 4, 1),
    ("FentonKarma2D", "fp32", True, 512, 4, 2), ("FentonKarma2D", "fp32", True, 513, 1, 1),
])
def test_where_the_lines_lie(gpu, name, precision, aniso, side, many, few):
    from finitewave_amd.engine import Engine
    eng = Engine(_model(name, (side, side), precision, aniso, frozen=False))
    assert _shape(eng, 40)[0] == many and _shape(eng, 5)[0] == few
    eng.close()
