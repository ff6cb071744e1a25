"""The training tangent kernel (k_train_u) over the forms its dispatch takes:
cutoff types with and without their own code, chunks of 8 and 16 members,
narrow, wide and weighted functions, integer and non-integer zeta, shifted
Gaussians, and neighbour counts at the edges of its 64-pair batches, up to
lists whose LDS exceeds 64 KiB.

The gradient of w_f / (3N) sum |F - Fref|^2 at Fref = F - d is
(2 w_f / 3N) sum d . dF/dw.  Its product with a random weight direction is
compared with the central difference of the engine's own forces (checked
against the oracle elsewhere) along that direction, over five points
(truncation h^4): with h = 2e-3 and forces good to 1e-13 of their scale the
quotient is good to a few 1e-10; 2e-8 of the sum's scale is allowed, and
1e-3 on the mixed path (forces to 1e-6 of their scale over h).
"""
import os

import numpy as np
import pytest

from n2p2_amd import engine
from n2p2_amd import workloads as W
from tests import cases

pytestmark = pytest.mark.gpu


def _model(tmp, text, el, z, hidden, r, elem, box):
    d = os.path.join(str(tmp), "m")
    W.write_model(d, text, el, z, hidden, seed=5)
    cases.scale_from_oracle(d, r, elem, box)
    return engine.Model.load_dir(d)


def _cluster(n, nel, seed):
    """n atoms of nel elements, open, at least 1.1 A apart."""
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"),
                 -1).reshape(-1, 3)[:n] * 1.6
    return (g + rng.uniform(-0.25, 0.25, (n, 3)),
            rng.integers(0, nel, n).astype(np.int32), None)


def _check(ctx, r, elem, box, tol, h=2e-3):
    rng = np.random.default_rng(9)
    n = len(elem)
    w0 = ctx.get_weights()
    w0 = w0 + rng.normal(scale=0.02, size=w0.size)
    delta = rng.normal(size=w0.size)
    delta /= np.linalg.norm(delta)
    d = rng.normal(size=(n, 3))

    def forces(x):
        ctx.set_weights(w0 + x * delta)
        ctx.set_structure(r, elem, box)
        ctx.evaluate(engine.FORCES_CONSISTENT)
        return ctx.forces()

    dF = (8.0 * (forces(h) - forces(-h))
          - (forces(2 * h) - forces(-2 * h))) / (12.0 * h)
    F = forces(0.0)
    want = 2.0 / (3 * n) * np.sum(d * dF)
    scale = 2.0 / (3 * n) * np.sum(np.abs(d * dF))
    ctx.set_structure(r, elem, box)
    g, _ = ctx.train_gradient(F - d, 0.0, 0.0, 1.0)
    got = float(g @ delta)
    print("[gpu-train-u] n %d want %.12e got %.12e scale %.3e"
          % (n, want, got, scale), flush=True)
    assert np.all(np.isfinite(g))
    if n > 1:
        assert scale > 0.0
    assert abs(got - want) <= tol * max(scale, 1e-12)


@pytest.mark.parametrize("cutoff", [1, 2, 5, 6])
def test_cutoff_types_narrow(tmp_path, cutoff):
    r, elem, box = W.water(64, 12.42, 3)
    m = _model(tmp_path, W.water_settings(cutoff_type=cutoff),
               W.WATER_ELEMENTS, (1, 8), (25, 25), r, elem, box)
    _check(engine.Context(m), r, elem, box, 2e-8)


@pytest.mark.parametrize("n", [1, 2, 3, 12, 13, 66, 140])
def test_wide_members_of_16(tmp_path, n):
    """12 members per chunk; n - 1 neighbours: no pair, one, and 64 pairs
    and one more of the whole list among the sizes."""
    r, elem, box = _cluster(140, 3, 1)
    m = _model(tmp_path, W.mixed_settings(), W.MIXED_ELEMENTS, (5, 6, 7),
               (30, 30), r, elem, box)
    _check(engine.Context(m), r[:n], elem[:n], box, 2e-8)


@pytest.mark.parametrize("n", [12, 66])
def test_weighted_shifted_noninteger(tmp_path, n):
    r, elem, box = _cluster(66, 3, 2)
    m = _model(tmp_path, W.weighted_settings(), W.MIXED_ELEMENTS, (5, 6, 7),
               (20, 20), r, elem, box)
    _check(engine.Context(m), r[:n], elem[:n], box, 2e-8)


@pytest.mark.parametrize("n,prec,tol", [(700, engine.PRECISION_FP64, 2e-8),
                                        (1000, engine.PRECISION_MIXED, 1e-3)])
def test_long_lists(tmp_path, n, prec, tol):
    """The longest lists the evaluation takes in FP64 (88 bytes of LDS per
    neighbour) and on the mixed path (56 bytes there, 88 here: past
    64 KiB).  Linear layers: the sums over hundreds of thousands of triplets
    would saturate others, and the forces are then of second order in the
    weights, for which the five-point difference has no truncation."""
    rng = np.random.default_rng(4)
    m = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"),
                 -1).reshape(-1, 3)[:n] * 0.62
    r = g + rng.uniform(-0.1, 0.1, (n, 3))
    elem = np.zeros(n, dtype=np.int32)
    elem[::7] = 1
    text = "\n".join([
        "number_of_elements 2", "elements H O", "cutoff_type 1",
        "global_hidden_layers_short 1", "global_nodes_short 6",
        "global_activation_short l l"]
        + ["symfunction_short %s %s" % (e, x) for e in "HO" for x in
           ("2 H 0.02 0.0 6.35", "2 O 0.3 2.0 6.35",
            "3 H O 0.03 1.0 2.0 6.35", "3 O O 0.02 -1.0 1.0 6.35")]) + "\n"
    d = os.path.join(str(tmp_path), "m")
    W.write_model(d, text, W.WATER_ELEMENTS, (1, 8), (6,), seed=5)
    ctx = engine.Context(engine.Model.load_dir(d, scaling=False))
    ctx.set_precision(prec)
    w = ctx.get_weights()
    ctx.set_structure(r, elem, None)
    ctx.calculate_neighbor_list(6.35)
    off = ctx.neighbors()[0]
    most = int(np.diff(off).max())
    print("[gpu-train-u] most neighbours", most, flush=True)
    assert (738 < most <= 1161) if prec else (600 < most <= 738)
    rng = np.random.default_rng(9)
    nat = len(elem)
    dvec = rng.normal(size=(nat, 3))
    delta = rng.normal(size=w.size)
    delta /= np.linalg.norm(delta)

    def forces(x):
        ctx.set_weights(w + x * delta)
        ctx.evaluate(engine.FORCES_CONSISTENT)
        return ctx.forces()

    h = 0.1
    dF = (8.0 * (forces(h) - forces(-h))
          - (forces(2 * h) - forces(-2 * h))) / (12.0 * h)
    F = forces(0.0)
    want = 2.0 / (3 * nat) * np.sum(dvec * dF)
    scale = 2.0 / (3 * nat) * np.sum(np.abs(dvec * dF))
    gr, _ = ctx.train_gradient(F - dvec, 0.0, 0.0, 1.0)
    print("[gpu-train-u] want %.10e got %.10e scale %.3e"
          % (want, gr @ delta, scale), flush=True)
    assert abs(float(gr @ delta) - want) <= tol * scale
