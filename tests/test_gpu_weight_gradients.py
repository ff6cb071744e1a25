"""Weight gradients of the energies (k_energy_wgrad) and of the energy loss
(k_train_grad with w_f = 0) against numpy backpropagation from the engine's
scaled descriptors, for networks that fill a block's 32 atom records, that
leave room for fewer (wide layers) and that have one layer, and for atom
counts around the block size.

Both sides are FP64 sums of at most a few hundred products of the same
factors; 1e-12 of the largest component is allowed (64 n eps with n a few
hundred terms).
"""
import os

import numpy as np
import pytest

from n2p2_amd import engine
from n2p2_amd import workloads as W
from tests import cases

pytestmark = pytest.mark.gpu


def _setup(tmp, hidden, act, natoms):
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
    r, elem, box = W.random_structure(natoms, seed=7)
    ctx.set_structure(r, elem, box)
    return ctx, w, elem


def _act(a, z):
    if a == "t":
        t = np.tanh(z)
        return t, 1.0 - t * t
    if a == "p":
        return np.log1p(np.exp(z)), 1.0 / (1.0 + np.exp(-z))
    return z, np.ones_like(z)


def _numpy_gradient(G, elem, w, sizes, acts):
    """Sum over the atoms of dE_i/dw, flat weight order."""
    out, p = [], 0
    for e in range(3):
        x = G[elem == e]
        layers, vals, ders = [], [x], []
        for (a, b), f in zip(zip(sizes[:-1], sizes[1:]), acts):
            Wl = w[p:p + a * b].reshape(b, a)
            p += a * b
            bl = w[p:p + b]
            p += b
            v, d = _act(f, vals[-1] @ Wl.T + bl)
            layers.append(Wl)
            vals.append(v)
            ders.append(d)
        delta = ders[-1]
        grads = []
        for l in range(len(layers) - 1, -1, -1):
            grads.append((delta.T @ vals[l], delta.sum(0)))
            if l:
                delta = (delta @ layers[l]) * ders[l - 1]
        for gw, gb in reversed(grads):
            out += [gw.reshape(-1), gb]
    return np.concatenate(out)


@pytest.mark.parametrize("hidden,act,natoms", [
    ((30, 30), "p p l", 1), ((30, 30), "p p l", 79),
    ((25, 7, 3), "t p t l", 80), ((1,), "t l", 81), ((130, 60), "t t l", 33),
    ((700,), "p l", 40)])
def test_weight_gradients(tmp_path, hidden, act, natoms):
    ctx, w, elem = _setup(tmp_path, hidden, act, natoms)
    e = ctx.evaluate(engine.FORCES_CONSISTENT)
    want = _numpy_gradient(ctx.G()[:, :102], elem, w, [102] + list(hidden)
                           + [1], act.split())
    scale = np.abs(want).max()
    eref = e - 3.0
    g, _ = ctx.train_gradient(np.zeros((natoms, 3)), eref, 1.0, 0.0)
    kappa = 2.0 * (e - eref) / natoms ** 2
    err = np.abs(g / kappa - want).max() / scale
    print("[gpu-wgrad]", hidden, natoms, "loss gradient %.2e" % err,
          flush=True)
    assert err <= 1e-12
    wide = max(hidden) + 102 + 2 * sum(hidden) + 1 > 256
    ctx.calculate_neighbor_list(6.0)
    if wide:
        with pytest.raises(RuntimeError, match="too wide"):
            ctx.energy_weight_jacobian(file_order=False)
        return
    J = ctx.energy_weight_jacobian(file_order=False)[0]
    err = np.abs(J - want).max() / scale
    print("[gpu-wgrad] jacobian %.2e" % err, flush=True)
    assert err <= 1e-12
