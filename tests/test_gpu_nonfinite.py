"""Lists of structures with atoms at non-finite coordinates: those have no
neighbours, and the others' lists are what they are without them, bit for bit.
Small structures, batches and cells, whose non-finite atoms share a cell with
others (in a periodic cell all of them the first one) and are most of it, so
that whichever atom the cell's kernel starts from is one of them in nearly every
run."""
import numpy as np
import pytest

from n2p2_amd import engine
from n2p2_amd import workloads as W
from tests import cases

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    d = cases.mixed_case(tmp_path_factory.mktemp("nonfinite"))[0]
    return engine.Model.load_dir(d)


def _list(ctx, load, rc):
    load(ctx)
    ctx.calculate_neighbor_list(rc)
    off, idx, _, d, dr = ctx.neighbors()
    centre = np.repeat(np.arange(len(off) - 1), np.diff(off))
    return centre, idx, d, dr


@pytest.mark.parametrize("kind", ["periodic", "open", "batch"])
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("n,nbad", [(300, 3), (3000, 200)])
def test_lists_without_them(model, n, nbad, value, kind):
    r, elem, box = W.random_structure(n, seed=n)
    rng = np.random.default_rng(1)
    bad = np.zeros(n, bool)
    bad[rng.permutation(n)[:nbad]] = True
    q = r.copy()
    q[bad, 0] = value
    box = None if kind == "open" else box

    def load(x):
        if kind == "batch":
            return lambda c: c.set_structures([(x, elem, box), (r, elem, box)])
        return lambda c: c.set_structure(x, elem, box)

    ctx = engine.Context(model)
    want = _list(ctx, load(r), 5.0)
    got = _list(ctx, load(q), 5.0)
    out = np.concatenate([bad, np.zeros(n, bool)])
    keep = ~out[want[0]] & ~out[want[1]]
    print("[gpu-nonfinite]", n, nbad, value, kind, len(want[0]),
          int(keep.sum()), len(got[0]), flush=True)
    for w, g in zip(want, got):
        assert np.array_equal(w[keep], g)
