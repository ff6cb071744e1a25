"""The table of contributions per caller atom of a caller-given list against
the reference's loop, bit for bit: targets with as many contributions as fill
a wave, the device's sort or more (counted on the host), centres that share a
target, centres without entries, lists without entries, and refused indices
and elements."""
import numpy as np
import pytest

from n2p2_amd import engine
from tests import cases
from tests.lammps_like import full_lists, ghost_domain

pytestmark = pytest.mark.gpu


def _loop(nout, off, idx, ctr, sf, pf):
    f = np.zeros((nout, 3))
    for i in range(len(off) - 1):
        f[ctr[i]] -= -sf[i]
        for q in range(off[i], off[i + 1]):
            f[idx[q]] -= -pf[q]
    return f


@pytest.fixture(scope="module")
def setup(tmp_path_factory):
    d, r, e, box = cases.water_case(tmp_path_factory.mktemp("targets"))
    m = engine.Model.load_dir(d)
    x, el, _, nl = ghost_domain(r, e, box, m.max_cutoff)
    off, idx, dr = full_lists(x, nl, m.max_cutoff)
    ctx = engine.Context(m)
    return ctx, el[:nl], np.asarray(off), el[idx], dr


@pytest.mark.parametrize("k", [0, 1, 63, 64, 65, 511, 512, 513, 5000, None])
@pytest.mark.parametrize("ctr", ["own", "shared"])
def test_table(setup, k, ctr):
    ctx, el, off, ne, dr = setup
    rng = np.random.default_rng(3)
    n, M, nout = len(el), len(ne), 600
    # Target 0: k entries spread over the list (None: all of them).
    idx = rng.integers(1, nout, M).astype(np.int32)
    idx[rng.permutation(M)[:M if k is None else k]] = 0
    ci = np.arange(1, n + 1) if ctr == "own" else rng.integers(1, 4, n)
    # Every third centre without entries.
    keep = np.ones(M, bool)
    for i in range(0, n, 3):
        keep[off[i]:off[i + 1]] = False
        if k is not None and k <= 513:
            # keep target 0's count as asked for
            keep[off[i]:off[i + 1]] |= idx[off[i]:off[i + 1]] == 0
    o2 = np.concatenate([[0], np.cumsum([keep[off[i]:off[i + 1]].sum()
                                         for i in range(n)])])
    ctx.set_neighbor_list(el, o2, idx[keep], ne[keep], dr[keep], ci)
    ctx.evaluate(engine.FORCES_CONSISTENT)
    sf, pf = ctx.pair_forces()
    got = ctx.scattered_forces(nout)
    assert np.array_equal(got, _loop(nout, o2, idx[keep], ci, sf, pf))
    assert np.array_equal(got, ctx.scattered_forces_noalloc(nout))


def test_no_entries_and_refused(setup):
    ctx, el, off, ne, dr = setup
    n, M = len(el), len(ne)
    ctx.set_neighbor_list(el, np.zeros(n + 1, int), [], [], np.zeros((0, 3)))
    ctx.evaluate(engine.FORCES_CONSISTENT)
    sf, _ = ctx.pair_forces()
    assert np.array_equal(ctx.scattered_forces(n), 0.0 - (-sf))
    idx = np.zeros(M, np.int32)
    for q in (0, M // 2, M - 1):
        bad = idx.copy()
        bad[q] = -1
        with pytest.raises(RuntimeError, match="Neighbour index"):
            ctx.set_neighbor_list(el, off, bad, ne, dr)
        assert ctx.num_atoms() == 0
        for e in (-1, 2):
            bade = ne.copy()
            bade[q] = e
            with pytest.raises(RuntimeError, match="Element index"):
                ctx.set_neighbor_list(el, off, idx, bade, dr)
    ctx.set_neighbor_list(el, off, idx, ne, dr)
    ctx.evaluate(engine.FORCES_CONSISTENT)
