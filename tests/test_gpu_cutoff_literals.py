"""Specialised kernels whose one cutoff configuration is compiled in, with and
without an inner radius, and those of a model with several, against the
generic kernels (the bounds of test_gpu_specialized.py: both evaluate the same
expressions, FP64 to rounding, FP32 to the mixed path's bounds)."""
import os

import pytest

from n2p2_amd import engine
from n2p2_amd import workloads as W
from tests import cases
from tests.test_gpu_specialized import _compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [engine.PRECISION_FP64,
                                  engine.PRECISION_MIXED])
@pytest.mark.parametrize("two", [False, True])
@pytest.mark.parametrize("cut", ["1", "1 0.4", "2", "3 0.2", "4 0.3", "6",
                                 "6 0.5", "8 0.1"])
def test_cutoff_literals(tmp_path, cut, two, prec):
    text = W.water_settings().replace("cutoff_type 1", "cutoff_type " + cut)
    if two:
        text = text.replace("symfunction_short H 2 O 1.0000000000e-03 0.0 "
                            "6.3500", "symfunction_short H 2 O "
                            "1.0000000000e-03 0.0 5.1000")
        assert "5.1000" in text
    d = os.path.join(str(tmp_path), "m")
    W.write_model(d, text, W.WATER_ELEMENTS, (1, 8), (25, 25), seed=7)
    r, elem, box = W.water(64, 12.42, 1234)
    cases.scale_from_oracle(d, r, elem, box)
    ctx = engine.Context(engine.Model.load_dir(d))
    ctx.set_structure(r, elem, box)
    _compare(ctx, prec)
