"""Neighbour lists that are refused: by a check before anything changed the list
before stays in use, in its own processing order; once the build has changed the
device's list nothing is left to evaluate on, also in an MD run."""
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


@pytest.mark.parametrize("n", [1, 2200])
def test_failure_leaves_no_list(model, n):
    """More than 8,192 neighbours, found by the count: without cells (one atom)
    and by the per-atom kernels behind the cells."""
    if n == 1:
        r, elem, box = np.array([[0.3, 0.2, 0.1]]), np.array([1]), np.eye(3) * 2
    else:
        r, elem, box = W.random_structure(n, seed=3)
    ctx = engine.Context(model)
    ctx.set_structure(r, elem, box)
    e = ctx.evaluate(engine.FORCES_CONSISTENT)
    f = ctx.forces()
    # 8,192 neighbours fill a sphere of this radius; 10% beyond it.
    rc = 1.1 * (8192 * np.linalg.det(box) / n / (4 / 3 * np.pi)) ** (1 / 3)
    print("[gpu-refused]", n, rc, flush=True)
    with pytest.raises(RuntimeError, match="8192"):
        ctx.calculate_neighbor_list(rc)
    for call in (ctx.calculate_symmetry_function_groups, ctx.neighbors):
        with pytest.raises(RuntimeError, match="not calculated"):
            call()
    for call in (ctx.calculate_forces, ctx.calculate_energy,
                 ctx.calculate_atomic_neural_networks):
        with pytest.raises(RuntimeError):
            call()
    assert ctx.evaluate(engine.FORCES_CONSISTENT) == e
    assert np.array_equal(ctx.forces(), f)


def test_failed_md_start(model):
    """A skin that makes the first list too large."""
    r, elem, box = W.random_structure(300, seed=4)
    ctx = engine.Context(model)
    ctx.set_structure(r, elem, box)
    with pytest.raises(RuntimeError, match="8192"):
        ctx.md_init([10.8, 12.0, 14.0], 0.1, skin=30.0)
    with pytest.raises(RuntimeError, match="no neighbour list"):
        ctx.md_run(1)
    ctx.md_init([10.8, 12.0, 14.0], 0.1, skin=1.0)
    ctx.md_run(2)


@pytest.mark.parametrize("end", ["refused list", "tuning"])
@pytest.mark.parametrize("n", [300, 2400])
def test_end_of_md_leaves_an_ordinary_list(model, n, end):
    """The list of the last step, with its images and partners, after a call that
    ends the run and builds no other one."""
    r, elem, box = W.random_structure(n, seed=5)
    ctx = engine.Context(model)
    ctx.set_structure(r, elem, box)
    ctx.md_init([10.8, 12.0, 14.0], 0.2, skin=1.0)
    ctx.md_run(5)
    x, _ = ctx.md_state()
    if end == "tuning":
        ctx.set_tuning(8)
    else:
        with pytest.raises(RuntimeError, match="60 periodic images"):
            ctx.calculate_neighbor_list(70.0 * box[0, 0])
    with pytest.raises(RuntimeError, match="No MD run"):
        ctx.md_run(1)
    ctx.calculate_symmetry_function_groups()
    ctx.calculate_atomic_neural_networks()
    e = ctx.calculate_energy()
    ctx.calculate_forces(engine.FORCES_CONSISTENT)
    got = (*ctx.neighbors(), ctx.forces())
    ctx.set_structure(x, elem, box)
    assert ctx.evaluate(engine.FORCES_CONSISTENT) == e
    print("[gpu-refused]", n, end, e, flush=True)
    for a, b in zip(got, (*ctx.neighbors(), ctx.forces())):
        assert np.array_equal(a, b)


def test_unstable_md_leaves_no_list(model):
    """The step in which a coordinate runs away filtered a list that was not
    rebuilt."""
    r, elem, box = W.random_structure(300, seed=6)
    v = np.zeros_like(r)
    v[3] = 1e8
    ctx = engine.Context(model)
    ctx.set_structure(r, elem, box)
    ctx.md_init([10.8, 12.0, 14.0], 0.2, skin=1.0, v=v)
    with pytest.raises(RuntimeError, match="unstable"):
        ctx.md_run(2)
    for call in (ctx.calculate_symmetry_function_groups, ctx.neighbors):
        with pytest.raises(RuntimeError, match="not calculated"):
            call()
