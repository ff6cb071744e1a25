"""Forces with the partner map beside the force kernel (an evaluation) and
beside the symmetry functions (calls one by one), after evaluations that left
the map out or ended in an error: bitwise those of a context that did nothing
else."""
import numpy as np
import pytest

from n2p2_amd import engine
from n2p2_amd import workloads as W
from tests import cases

pytestmark = pytest.mark.gpu


def _stepwise(ctx, rc):
    ctx.calculate_neighbor_list(rc)
    ctx.calculate_symmetry_function_groups()
    ctx.calculate_atomic_neural_networks()
    ctx.calculate_energy()
    ctx.calculate_forces(engine.FORCES_CONSISTENT)
    return ctx.forces()


@pytest.mark.parametrize("n", [300, 3000])
def test_partner_order(tmp_path, n):
    m = engine.Model.load_dir(cases.mixed_case(tmp_path)[0])
    rng = np.random.default_rng(n)
    box = np.eye(3) * (n / 0.05) ** (1.0 / 3.0)
    elem = rng.integers(0, 3, n)
    sets = [rng.uniform(0, box[0, 0], (n, 3)) for _ in range(3)]
    want = []
    for r in sets:
        ctx = engine.Context(m)
        ctx.set_structure(r, elem, box)
        want.append(_stepwise(ctx, m.max_cutoff))
        ctx.close()
    ctx = engine.Context(m)
    for r, f in zip(sets, want):
        ctx.set_structure(r, elem, box)
        ctx.evaluate(engine.FORCES_CONSISTENT)
        assert np.array_equal(ctx.forces(), f)
        ctx.calculate_forces(engine.FORCES_CONSISTENT)
        assert np.array_equal(ctx.forces(), f)
    for r, f in zip(sets, want):
        ctx.set_structure(r, elem, box)
        ctx.evaluate(-1)
        ctx.calculate_atomic_neural_networks()
        ctx.calculate_forces(engine.FORCES_CONSISTENT)
        assert np.array_equal(ctx.forces(), f)
        assert np.array_equal(_stepwise(ctx, m.max_cutoff), f)
    for r, f in zip(sets, want):
        ctx.set_structure(r, elem, box)
        with pytest.raises(RuntimeError, match="force mode"):
            ctx.evaluate(7)
        ctx.calculate_forces(engine.FORCES_CONSISTENT)
        assert np.array_equal(ctx.forces(), f)
    for r, f in reversed(list(zip(sets, want))):
        ctx.set_positions(r)
        ctx.evaluate(engine.FORCES_CONSISTENT)
        assert np.array_equal(ctx.forces(), f)
