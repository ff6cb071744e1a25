"""Two atoms at one place.  Their own symmetry functions have no value (the
angle at r = 0), so the specialised kernels must give NaN there and for the
energy, as the formula and the oracle do; every other atom sees two neighbours
at distance 0 from each other, which is no special case: G and energies are the
oracle's (bounds of test_gpu_pair_search.py)."""
import os

import numpy as np
import pytest

from n2p2_amd import engine
from n2p2_amd import workloads as W
from tests.oracle_lib import OModel, OStruct
from tests.test_gpu_pair_search import TOL, _settings

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cut", ["1", "1 0.3", "6"])
@pytest.mark.parametrize("types", [(3,), (9,), (3, 9)])
def test_coincident_atoms(tmp_path, types, cut):
    r, elem, box = W.random_structure(90, seed=5)
    r[41] = r[7]
    d = os.path.join(str(tmp_path), "m")
    W.write_model(d, _settings(types, 6.0, cut), W.MIXED_ELEMENTS, (5, 6, 7),
                  (6,), seed=3)
    m = engine.Model.load_dir(d, scaling=False)
    s = OStruct(OModel.from_dir(d, scaling=False), r, elem, box)
    assert np.isnan(s.evaluate(cells=False, force_mode=1))
    two = np.isin(np.arange(len(r)), (7, 41))
    og = s.G()[~two]
    assert np.array_equal(np.isnan(s.G()).any(1), two)
    for prec in (engine.PRECISION_FP64, engine.PRECISION_MIXED):
        for spec in (True, False):
            ctx = engine.Context(m)
            ctx.set_precision(prec)
            ctx.set_specialized(spec)
            ctx.set_structure(r, elem, box)
            e = ctx.evaluate(engine.FORCES_CONSISTENT)
            g, ea, f = ctx.G(), ctx.atomic_energies(), ctx.forces()
            bad = np.isnan(g).any(1)
            print("[gpu-coincident]", types, cut, prec, spec, e,
                  np.flatnonzero(bad), flush=True)
            if spec:
                assert np.isnan(e)
                assert np.array_equal(bad, two)
                assert np.isnan(f[two]).all()
            assert not bad[~two].any()
            err = np.abs(g[~two][:, :og.shape[1]] - og).max()
            assert err <= TOL[prec][0] * np.abs(og).max()
            oa = s.atomic_energies()[~two]
            assert np.abs(ea[~two] - oa).max() <= 1e-4 * np.abs(oa).max()
