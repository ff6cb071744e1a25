"""Atomic networks in one launch over the elements, against numpy from the
engine's descriptors: layers at the edges of the 16-column tiles that a
workgroup's waves share, networks too wide for the tile kernel, elements with
no atoms, and atom counts at which a workgroup has one, two or four waves.

FP64: sums of at most a few hundred products, 64 n eps of the largest value
gives 1e-12.  FP32 tiles: the same with FP32's eps, n the widest sum: 102
products and two layers behind it, 4 n eps = 1e-4 at worst and 2e-5 allowed
here, since the errors of the products are independent.
"""
import os

import numpy as np
import pytest

from n2p2_amd import engine
from n2p2_amd import workloads as W
from tests import cases

pytestmark = pytest.mark.gpu

ACT = {"t": (np.tanh, lambda z: 1.0 - np.tanh(z) ** 2),
       "p": (lambda z: np.logaddexp(0.0, z), lambda z: 1 / (1 + np.exp(-z))),
       "l": (lambda z: z, lambda z: np.ones_like(z))}


def _numpy(G, elem, w, sizes, acts):
    e_at, dedg = np.zeros(len(G)), np.zeros_like(G)
    p = 0
    for e in range(3):
        sel = elem == e
        x, Ws, ders = G[sel], [], []
        for (a, b), f in zip(zip(sizes[:-1], sizes[1:]), acts):
            Wl = w[p:p + a * b].reshape(b, a)
            z = x @ Wl.T + w[p + a * b:p + a * b + b]
            p += a * b + b
            Ws.append(Wl)
            x = ACT[f][0](z)
            ders.append(ACT[f][1](z))
        e_at[sel] = x[:, 0]
        g = ders[-1]
        for l in range(len(Ws) - 1, -1, -1):
            g = g @ Ws[l]
            if l:
                g = g * ders[l - 1]
        dedg[sel] = g
    return e_at, dedg


def _run(tmp, hidden, act, n, only, precision):
    r, elem, box = W.random_structure(100, seed=6)
    text = W.mixed_settings().replace(
        "global_hidden_layers_short 2", "global_hidden_layers_short %d"
        % len(hidden)).replace(
        "global_nodes_short 30 30", "global_nodes_short "
        + " ".join(str(h) for h in hidden)).replace(
        "global_activation_short p p l", "global_activation_short " + act)
    d = os.path.join(str(tmp), "m")
    W.write_model(d, text, W.MIXED_ELEMENTS, (5, 6, 7), hidden, seed=8)
    cases.scale_from_oracle(d, r, elem, box)
    ctx = engine.Context(engine.Model.load_dir(d))
    w = ctx.get_weights()
    w = w + np.random.default_rng(2).normal(scale=0.1, size=w.size)
    ctx.set_weights(w)
    ctx.set_precision(precision)
    rng = np.random.default_rng(7)
    box = np.eye(3) * (n / 0.02) ** (1.0 / 3.0)
    r, elem = rng.uniform(0, box[0, 0], (n, 3)), rng.integers(0, 3, n)
    if only is not None:
        elem = np.full(n, only)
    ctx.set_structure(r, elem, box)
    ctx.evaluate(engine.FORCES_CONSISTENT)
    want_e, want_g = _numpy(ctx.G()[:, :102], elem, w,
                            [102] + list(hidden) + [1], act.split())
    ge = np.abs(ctx.atomic_energies() - want_e).max() / np.abs(want_e).max()
    gg = np.abs(ctx.dEdG()[:, :102] - want_g).max() / np.abs(want_g).max()
    print("[gpu-networks]", hidden, n, only, precision, "%.1e %.1e"
          % (ge, gg), flush=True)
    return max(ge, gg)


@pytest.mark.parametrize("hidden,act", [
    ((1,), "t l"), ((15, 16), "t p l"), ((17, 33, 2), "p t t l"),
    ((64, 65), "t t l"), ((700,), "p l")])
@pytest.mark.parametrize("n,only", [(1, None), (17, 2), (50, None)])
def test_widths(tmp_path, hidden, act, n, only):
    assert _run(tmp_path, hidden, act, n, only, engine.PRECISION_FP64) <= 1e-12
    assert _run(tmp_path, hidden, act, n, only, engine.PRECISION_MIXED) <= 2e-5


# One to 512 workgroups: the widest layer's tiles, at most four waves; more:
# two; small networks (a tile of at most 10 KiB) from 4,096 workgroups: one.
@pytest.mark.parametrize("hidden,n", [((30, 30), 8160), ((30, 30), 8260),
                                      ((5,), 66000)])
def test_wave_counts(tmp_path, hidden, n):
    act = "t " * len(hidden) + "l"
    for precision, tol in ((engine.PRECISION_FP64, 1e-12),
                           (engine.PRECISION_MIXED, 2e-5)):
        assert _run(tmp_path, hidden, act, n, None, precision) <= tol
