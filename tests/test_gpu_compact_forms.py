"""The compact pass (k_compact) over the forms its launch takes, against the
oracle: groups longer than the member sums held in registers, more angle
functions than a chunk's columns, cr(r_jk) carried over from members with
another core, neighbour counts around the batch of 64 pairs, and lists long
enough for two waves, one wave and partial radial tables.

FP64 tolerances of the compact parity tests: energy 1e-10 relative, G 1e-11 of
its scale, forces 1e-9 of the largest (sums over up to 50,000 pairs, 60
functions each).
"""
import os

import numpy as np
import pytest

from n2p2_amd import engine
from n2p2_amd import workloads as W
from tests import cases
from tests.oracle_lib import OModel, OStruct

pytestmark = pytest.mark.gpu


def _head():
    return ["number_of_elements 2", "elements C N", "cutoff_type 6 0.0",
            "scale_symmetry_functions", "scale_min_short 0.0",
            "scale_max_short 1.0", "global_hidden_layers_short 1",
            "global_nodes_short 8", "global_activation_short t l"]


def _lines(kind):
    out = []
    for e in "CN":
        for e1 in "CN":
            out.append("%s 20 %s -6.0 6.0 p2" % (e, e1))
            out.append("%s 20 %s 1.0 5.5 e" % (e, e1))
        out.append("%s 23 0.5 6.0 p3a" % e)
        if kind == "many":          # 60 members, 3 angle functions
            for t in (21, 22):
                for k in range(20):
                    for al, ar in ((0, 120), (60, 180), (49.1, 169.1)):
                        out.append("%s %d C N %.2f %.2f %.1f %.1f p2a"
                                   % (e, t, -6.0 + 0.3 * k, 6.0 - 0.1 * k,
                                      al, ar))
        elif kind == "angles":      # one radial function, 40 angle functions
            for t in (21, 22):
                for k in range(40):
                    out.append("%s %d C N 0.0 6.0 %.1f %.1f p3"
                               % (e, t, 2.0 * k, 100.0 + 2.0 * k))
                out.append("%s %d N N 0.5 6.0 0.0 180.0 e" % (e, t))
            out.append("%s 24 0.0 6.0 30.0 150.0 p1" % e)
            out.append("%s 25 0.0 6.0 30.0 150.0 p4a" % e)
        else:                       # equal (rl, rc) at the change of core
            for core in ("p1", "p1a", "p2", "p2a", "p3", "p4", "e"):
                out.append("%s 21 C N 1.0 6.0 0.0 110.0 %s" % (e, core))
                out.append("%s 21 C N 1.0 6.0 70.0 180.0 %s" % (e, core))
                out.append("%s 24 0.5 5.0 20.0 120.0 %s" % (e, core))
    return ["symfunction_short " + x for x in out]


def _cluster(n, step, seed):
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"),
                 -1).reshape(-1, 3)[:n] * step
    return (g + rng.uniform(-0.15 * step, 0.15 * step, (n, 3)),
            rng.integers(0, 2, n).astype(np.int32), None)


@pytest.mark.parametrize("kind,n,step", [
    ("many", 1, 1.6), ("many", 2, 1.6), ("many", 3, 1.6), ("many", 23, 1.6),
    ("many", 120, 1.6), ("angles", 40, 1.6), ("angles", 130, 1.2),
    ("carry", 24, 1.6), ("carry", 90, 1.5), ("many", 330, 0.9),
    ("angles", 300, 0.9), ("carry", 500, 0.75)])
def test_compact_forms(tmp_path, kind, n, step):
    d = os.path.join(str(tmp_path), "m")
    W.write_model(d, "\n".join(_head() + _lines(kind)) + "\n", ("C", "N"),
                  (6, 7), (8,), seed=5)
    r, elem, box = _cluster(60, 1.6, 3)
    cases.scale_from_oracle(d, r, elem, box)
    r, elem, box = _cluster(n, step, 4)
    ctx = engine.Context(engine.Model.load_dir(d))
    ctx.set_structure(r, elem, box)
    e = ctx.evaluate(0)
    s = OStruct(OModel.from_dir(d), r, elem, box)
    oe = s.evaluate(cells=True, force_mode=0)
    G, oG = ctx.G(), s.G()
    scale = np.maximum(np.abs(oG).max(0), 1e-300)
    f, of = ctx.forces(), s.forces()
    eg = np.max(np.abs(G - oG) / scale)
    ef = np.abs(f - of).max() / max(np.abs(of).max(), 1e-300)
    print("[gpu-compact-forms] %s %d: neighbours %d, E %.2e G %.2e F %.2e"
          % (kind, n, ctx.num_neighbor_entries() // n,
             abs(e - oe) / abs(oe), eg, ef), flush=True)
    assert abs(e - oe) <= 1e-10 * abs(oe)
    assert eg <= 1e-11
    assert ef <= 1e-9
    # Repeated evaluations are bitwise equal.
    assert ctx.evaluate(0) == e and np.array_equal(ctx.forces(), f)
