"""Neighbour lists of single structures around the size up to which they are
built without cells (2,048 atoms), bitwise against the oracle's: remainders
of a wave, few and many images, sheared and open cells, atoms on the faces of
their cell, a cutoff that outgrows the slots of the build before, and the limit of
8,192 neighbours."""
import numpy as np
import pytest

from n2p2_amd import engine
from n2p2_amd import workloads as W
from tests import cases
from tests.oracle_lib import OModel, OStruct

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    d = cases.mixed_case(tmp_path_factory.mktemp("lists"))[0]
    return engine.Model.load_dir(d), OModel.from_dir(d)


def _check(ctx, om, r, elem, box, rc):
    ctx.calculate_neighbor_list(rc)
    off, idx, _, d, dr = ctx.neighbors()
    s = OStruct(om, r, elem, box)
    s.neighbor_list(rc, cells=len(r) > 1000)
    ooff, oidx, od, odr = s.neighbors()
    assert np.array_equal(off, ooff)
    assert np.array_equal(idx, oidx)
    assert np.array_equal(d, od)
    assert np.array_equal(dr, odr)
    return off


@pytest.mark.parametrize("kind", ["ortho", "sheared", "faces", "open"])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1000, 2047, 2048, 2049])
def test_small_lists(model, n, kind):
    em, om = model
    r, elem, box = W.random_structure(n, seed=n)
    if kind == "sheared":
        r, box = W.sheared(r, box, [[1, 0.2, 0], [0, 1, 0.1], [0.3, 0, 1]])
    elif kind == "faces":
        k = np.random.default_rng(n).random((n, 3))
        r = np.where(k < 0.1, 0.0, np.where(
            k > 0.9, np.nextafter(box[0, 0], 0.0), r))
    elif kind == "open":
        box = None
    ctx = engine.Context(em)
    ctx.set_structure(r, elem, box)
    _check(ctx, om, r, elem, box, 4.0)
    off = _check(ctx, om, r, elem, box, 6.0)       # outgrows the slots
    print("[gpu-lists]", n, kind, int(off[-1]), flush=True)
    _check(ctx, om, r, elem, box, 5.0)


@pytest.mark.parametrize("rc", [24.0, 26.0])
def test_neighbor_limit(model, rc):
    em, om = model
    r, elem, box = np.array([[0.3, 0.2, 0.1]]), np.array([1]), np.eye(3) * 2.0
    ctx = engine.Context(em)
    ctx.set_structure(r, elem, box)
    if rc > 25.0:
        with pytest.raises(RuntimeError, match="8192"):
            ctx.calculate_neighbor_list(rc)
        # The refused list's counts are on the device: nothing may run on them.
        for call in (ctx.calculate_symmetry_function_groups, ctx.neighbors):
            with pytest.raises(RuntimeError, match="not calculated"):
                call()
        _check(ctx, om, r, elem, box, 12.0)
        ctx.set_structure(r, elem, box)
        _check(ctx, om, r, elem, box, 12.0)
        return
    _check(ctx, om, r, elem, box, rc)
