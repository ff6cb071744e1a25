"""The energy sum over one block (up to 8,192 atoms) and over several whose
last one adds the parts: against the atomic energies, bitwise the same on
every call, alone and together with forces."""
import math

import numpy as np
import pytest

from n2p2_amd import engine
from tests import cases

pytestmark = pytest.mark.gpu


# 8,193 atoms: three blocks; 1,048,600 would be the 256-block limit's first
# size, so 66,000 and its 17 blocks stand for the many-block form.
@pytest.mark.parametrize("n", [1, 1023, 1025, 8192, 8193, 66000])
def test_energy_sum(tmp_path, n):
    ctx = engine.Context(engine.Model.load_dir(
        cases.mixed_case(tmp_path)[0]))
    rng = np.random.default_rng(n)
    box = np.eye(3) * (n / 0.02) ** (1.0 / 3.0)
    ctx.set_structure(rng.uniform(0, box[0, 0], (n, 3)),
                      rng.integers(0, 3, n), box)
    e = ctx.evaluate(engine.FORCES_CONSISTENT)
    ea = ctx.atomic_energies()
    want = math.fsum(ea)
    # Trees of at most 1024 and 256 leaves over strided runs.
    tol = (n / 1024 + 30) * np.finfo(float).eps * np.abs(ea).sum()
    print("[gpu-energy]", n, e - want, tol, flush=True)
    assert abs(e - want) <= tol
    for _ in range(3):
        assert ctx.calculate_energy() == e
        assert ctx.evaluate(engine.FORCES_CONSISTENT) == e
        assert ctx.evaluate(-1) == e
