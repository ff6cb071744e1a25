"""The pair search of the angular groups (blocks of four neighbours on the
matrix cores, hits queued) at its edges: element blocks of 0 to 9 neighbours
and around a step of 16 blocks, one and several elements, group cutoffs below
the list's, the wide type with all and with some neighbours inside, a
structure whose pairs lie at rjk = rc to rounding, and lists of several
hundred neighbours, against the FP64 oracle.

G and forces in FP64 within 1e-11 of their largest value (sums of up to 1e5
terms of one sign pattern or another, 64 sqrt(n) eps), mixed 2e-5 and 2e-4
(the bounds the mixed path meets everywhere else).
"""
import os

import numpy as np
import pytest

from n2p2_amd import engine
from n2p2_amd import workloads as W
from tests import cases
from tests.oracle_lib import OModel, OStruct

pytestmark = pytest.mark.gpu

TOL = {engine.PRECISION_FP64: (1e-11, 1e-11),
       engine.PRECISION_MIXED: (2e-5, 2e-4)}


def _settings(types, rc_ang, cut):
    el = ("B", "C", "N")
    out = ["number_of_elements 3", "elements B C N", "cutoff_type " + cut,
           "global_hidden_layers_short 1", "global_nodes_short 6",
           "global_activation_short l l"]
    for e in el:
        for e1 in el:
            out.append("symfunction_short %s 2 %s 0.05 0.0 6.0" % (e, e1))
        for t in types:
            for i in range(3):
                for k in range(i, 3):
                    for lam, zeta in ((1, 1), (-1, 2), (1, 16)):
                        out.append("symfunction_short %s %d %s %s 0.01 %d %d "
                                   "%.2f" % (e, t, el[i], el[k], lam, zeta,
                                             rc_ang))
    return "\n".join(out) + "\n"


def _check(tmp, r, elem, box, types=(3,), rc=6.0, cut="1"):
    d = os.path.join(str(tmp), "m")
    if not os.path.exists(d):
        W.write_model(d, _settings(types, rc, cut), W.MIXED_ELEMENTS,
                      (5, 6, 7), (6,), seed=3)
    m = engine.Model.load_dir(d, scaling=False)
    s = OStruct(OModel.from_dir(d, scaling=False), r, elem, box)
    s.evaluate(cells=False, force_mode=1)
    ns = s.G().shape[1]
    for spec in (True, False):
        for prec in (engine.PRECISION_FP64, engine.PRECISION_MIXED):
            ctx = engine.Context(m)
            ctx.set_precision(prec)
            ctx.set_specialized(spec)
            ctx.set_structure(r, elem, box)
            ctx.evaluate(engine.FORCES_CONSISTENT)
            g = np.abs(ctx.G()[:, :ns] - s.G()).max() / np.abs(s.G()).max()
            fs = np.abs(s.forces()).max()
            f = np.abs(ctx.forces() - s.forces()).max() / fs
            print("[gpu-pairs]", len(r), types, rc, cut, spec, prec,
                  "%.1e %.1e" % (g, f), flush=True)
            assert g <= TOL[prec][0] and f <= TOL[prec][1]


@pytest.mark.parametrize("counts", [
    (0, 2, 0), (1, 1, 1), (3, 4, 5), (4, 8, 9), (17, 1, 0), (64, 5, 2),
    (65, 31, 16), (7, 90, 33)])
def test_block_sizes(tmp_path, counts):
    """A cluster small enough that all atoms see each other, so an atom's
    element blocks have the counts given (one less for its own)."""
    rng = np.random.default_rng(sum(counts))
    n = 1 + sum(counts)
    elem = np.concatenate([[0]] + [np.full(c, k) for k, c
                                   in enumerate(counts)])
    r = []
    while len(r) < n:
        p = rng.uniform(-2.9, 2.9, 3)
        if p @ p < 2.95 ** 2 and all(np.sum((p - q) ** 2) > 0.4 for q in r):
            r.append(p)
    _check(tmp_path, np.array(r), elem.astype(np.int32), None)


@pytest.mark.parametrize("types,rc,cut", [
    ((3,), 6.0, "0"), ((3,), 4.1, "1"), ((9,), 6.0, "2"), ((9,), 4.0, "6"),
    ((3, 9), 5.0, "6 0.3"), ((3, 9), 6.0, "4")])
def test_types_and_cutoffs(tmp_path, types, rc, cut):
    r, elem, box = W.random_structure(90, seed=5)
    _check(tmp_path, r, elem, box, types, rc, cut)


@pytest.mark.parametrize("cut,scale", [
    ("1", 1.0), ("6", 1.0), ("0", 1.0 - 1e-6), ("0", 1.0 + 2e-6)])
def test_pairs_at_the_cutoff(tmp_path, cut, scale):
    """A lattice with spacing rc / 3, moved off exactness by a few ulp: many
    pairs at rjk = rc (1 +- 1e-15), which the search lets through and the
    evaluation has to cut off.  The hard cutoff jumps at rc, so there the pairs
    lie 1e-6 rc inside, where all count, and 2e-6 rc outside: far above the
    rounding of FP32 (1e-7), and within the 4e-6 rc that the search lets
    through, so that the evaluation alone keeps them out."""
    g = np.stack(np.meshgrid(*[np.arange(5) * 2.0] * 3, indexing="ij"),
                 -1).reshape(-1, 3)
    rng = np.random.default_rng(1)
    r = g * (1.0 + rng.uniform(-1, 1, g.shape) * 4e-16) * scale
    elem = rng.integers(0, 3, len(r)).astype(np.int32)
    _check(tmp_path, r, elem, None, cut=cut)


def test_long_list(tmp_path):
    """About 640 neighbours: past the record's 256, FP64 staging beyond
    64 KiB."""
    r, elem, box = W.random_structure(60, density=0.7, dmin=0.7, seed=9)
    _check(tmp_path, r, elem, box)
