"""Neighbour lists that are refused: by a check before anything changed the list
before stays in use, in its own processing order."""
import numpy as np
import pytest

from n2p2_amd import engine
from n2p2_amd import workloads as W
from tests import cases

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    d = cases.mixed_case(tmp_path_factory.mktemp("refused"))[0]
    return engine.Model.load_dir(d)


@pytest.mark.parametrize("n", [300, 2400])
def test_refusal_keeps_the_list(model, n):
    """3,000 atoms leave their cell order behind; the structure after them is
    gathered in its own order (300 atoms) or another one (2,400)."""
    ctx = engine.Context(model)
    ctx.set_structure(*W.random_structure(3000, seed=1))
    ctx.evaluate(engine.FORCES_CONSISTENT)
    r, elem, box = W.random_structure(n, seed=2)
    ctx.set_structure(r, elem, box)
    ctx.evaluate(engine.FORCES_CONSISTENT)
    f = ctx.forces()
    print("[gpu-refused]", n, flush=True)
    with pytest.raises(RuntimeError, match="60 periodic images"):
        ctx.calculate_neighbor_list(70.0 * box[0, 0])
    ctx.calculate_forces(engine.FORCES_CONSISTENT)
    assert np.array_equal(ctx.forces(), f)
