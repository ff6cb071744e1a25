"""Performance cases: what programs do with this framework, through the Python
API over its C ABI (n2p2_amd.engine).

Kinds of work
  predict   one structure per call from host arrays, energy and forces back on
            the host (nnp-predict, a Monte Carlo move, an external driver).
  eval      one structure with positions and forces resident on the GPU (a
            simulation code on the same device), neighbour list rebuilt.
  batch     a set of independent uneven periodic structures per call, on the
            device (ensembles, replica runs).
  dataset   the same from host arrays, loaded anew on every call (nnp-dataset).
  md        velocity-Verlet steps with the device integrator, then the state
            is read for a trajectory frame.
  adam      one nnp-train step with gradient descent: a structure is loaded,
            the gradient of the energy + force loss formed, Adam applied.
  kalman    one energy and two force-component updates of nnp-train's Kalman
            filter on one structure.
  lammps    the pair_style path: a neighbour list with ghost atoms handed over
            from the host, forces on owned and ghost atoms back.

Models
  water     H/O, 8 G2 per neighbour element and 8 narrow G3 per element pair,
            rc 6.35 A, network 40-25-25-1 (tanh); cutoff type 1 (cosine), or
            2 (tanh^3) and 6 (polynomial) in drawn cases.
  bcn       B/C/N, 10 G2 per element and 12 wide G9 per element pair, rc 6 A,
            polynomial cutoff, network 102-30-30-1 (softplus).
  compact   B/C/N with the compact families in the form of the SCAN molecule
            models: asymmetric radial windows (type 20) and 18 wide angular
            functions (type 22) per element pair, network 126-30-20-1.

Sizes: water boxes of 64 to 65,536 molecules at the density of the 192-,
24,576- and 196,608-atom boxes of the tests and the benchmark; B/C/N
structures of 16 to 512 atoms at 0.08 atoms/A^3, up to 512 of them.
"""
import functools
import math
import os
import tempfile

import numpy as np
import torch

from n2p2_amd import engine, workloads as W

PREC = {"fp64": engine.PRECISION_FP64, "mixed": engine.PRECISION_MIXED,
        "mixed16": engine.PRECISION_MIXED16,
        "mixed_bf16": engine.PRECISION_MIXED_BF16}

WATER_EDGE = 12.42 / 4.0          # A per molecule^(1/3) (64 molecules: 12.42)
BCN_DENSITY = 0.08                # atoms / A^3
MD_STEPS = 10
MD_DT = 0.25                      # fs


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # A single-point prediction of the smallest box of the tests: launches
        # and synchronisations count.
        {"name": "predict_192_fp64", "kind": "predict", "model": "water",
         "cut": 1, "size": 64, "prec": "fp64"},
        # An external driver (geometry optimiser, Monte Carlo) with host
        # arrays and an ordinary box.
        {"name": "predict_1536_mixed", "kind": "predict", "model": "water",
         "cut": 1, "size": 512, "prec": "mixed"},
        # A simulation code on the same device, odd size, FP16 networks.
        {"name": "eval_24573_mixed16", "kind": "eval", "model": "water",
         "cut": 1, "size": 8191, "prec": "mixed16"},
        # The large box, plain FP64 and mixed precision.
        {"name": "eval_196608_fp64", "kind": "eval", "model": "water",
         "cut": 1, "size": 65536, "prec": "fp64"},
        {"name": "eval_196608_mixed", "kind": "eval", "model": "water",
         "cut": 1, "size": 65536, "prec": "mixed"},
        # 512 uneven structures in one call, wide angular functions.
        {"name": "batch_512_mixed", "kind": "batch", "model": "bcn",
         "size": 512, "lo": 16, "hi": 512, "prec": "mixed"},
        # A data-set evaluation: small uneven structures from the host.
        {"name": "dataset_24_fp64", "kind": "dataset", "model": "bcn",
         "size": 24, "lo": 16, "hi": 200, "prec": "fp64"},
        # Molecular dynamics of a mid-size box, one frame written per pass.
        {"name": "md_24576_mixed", "kind": "md", "model": "water", "cut": 1,
         "size": 8192, "prec": "mixed"},
        # Training on energies and forces with Adam.
        {"name": "adam_1536", "kind": "adam", "model": "water", "cut": 1,
         "size": 512, "prec": "fp64"},
        # Training with the Kalman filter on small structures.
        {"name": "kalman_192", "kind": "kalman", "model": "water", "cut": 1,
         "size": 64, "prec": "fp64"},
        # A LAMMPS domain: caller-given list with ghosts.
        {"name": "lammps_3072_mixed", "kind": "lammps", "model": "water",
         "cut": 1, "size": 1024, "prec": "mixed"},
        # A model of compact functions on a bulk structure.
        {"name": "compact_1000_fp64", "kind": "eval", "model": "compact",
         "size": 1000, "prec": "fp64"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["predict", "predict", "eval", "eval", "eval", "batch",
                       "dataset", "md", "adam", "kalman", "lammps",
                       "compact"])
    prec = rng.choice(["fp64", "mixed", "mixed", "mixed16", "mixed_bf16"])
    water = {"model": "water", "cut": rng.choice([1, 1, 2, 6]), "prec": prec}
    if kind == "predict":
        return {"kind": kind, "size": _log_int(rng, 40, 4000), **water}
    if kind == "eval":
        return {"kind": kind, "size": _log_int(rng, 64, 60000), **water}
    if kind in ("batch", "dataset"):
        lo = _log_int(rng, 16, 64)
        return {"kind": kind, "model": "bcn", "prec": prec, "lo": lo,
                "size": _log_int(rng, 4, 500 if kind == "batch" else 64),
                "hi": _log_int(rng, lo + 1, 512)}
    if kind == "md":
        return {"kind": kind, "size": _log_int(rng, 64, 4000), **water}
    if kind == "adam":
        return {"kind": kind, "size": _log_int(rng, 40, 1024),
                **water, "prec": "fp64"}
    if kind == "kalman":
        return {"kind": kind, "size": _log_int(rng, 40, 256),
                **water, "prec": "fp64"}
    if kind == "lammps":
        return {"kind": kind, "size": _log_int(rng, 64, 2048), **water}
    return {"kind": "eval", "model": "compact",
            "size": _log_int(rng, 64, 2000), "prec": prec}


# --------------------------------------------------------- models and inputs

def _compact_settings():
    """Asymmetric windows and angle intervals of the SCAN molecule models,
    scaled to rc 6 A."""
    el = W.MIXED_ELEMENTS
    windows = ((-6.0, 6.0), (-5.0, 5.0), (-4.0, 4.0), (0.0, 6.0), (1.0, 5.0),
               (2.0, 6.0))
    angles = ((0.0, 120.0), (60.0, 180.0), (90.0, 270.0))
    out = ["number_of_elements 3", "elements B C N", "cutoff_type 6 0.0",
           "scale_symmetry_functions", "scale_min_short 0.0",
           "scale_max_short 1.0", "global_hidden_layers_short 2",
           "global_nodes_short 30 20", "global_activation_short p p l"]
    for e in el:
        for e1 in el:
            for rl, rc in windows:
                out.append("symfunction_short %s 20 %s %.2f %.2f p2a"
                           % (e, e1, rl, rc))
        for i1 in range(3):
            for i2 in range(i1, 3):
                for rl, rc in windows:
                    for al, ar in angles:
                        out.append("symfunction_short %s 22 %s %s %.2f %.2f "
                                   "%.1f %.1f p2a" % (e, el[i1], el[i2], rl,
                                                      rc, al, ar))
    return "\n".join(out) + "\n"


def _settings(model, cut):
    """(settings text, element symbols, atomic numbers, hidden layers)."""
    if model == "water":
        return (W.water_settings(cutoff_type=cut), W.WATER_ELEMENTS, (1, 8),
                (25, 25))
    if model == "bcn":
        return W.mixed_settings(), W.MIXED_ELEMENTS, (5, 6, 7), (30, 30)
    return _compact_settings(), W.MIXED_ELEMENTS, (5, 6, 7), (30, 20)


def _bcn(n, seed):
    """B/C/N at 0.4/0.4/0.2 on a jittered lattice at 0.08 atoms/A^3 (least
    distance about 1.8 A)."""
    rng = np.random.default_rng(seed)
    L = (n / BCN_DENSITY) ** (1.0 / 3.0)
    m = int(math.ceil(round(n ** (1.0 / 3.0), 9)))
    g = (np.arange(m) + 0.5) * (L / m)
    sites = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    sites = sites[np.sort(rng.permutation(len(sites))[:n])]
    room = max(0.5 * (L / m - 1.5), 0.05)
    r = sites + rng.uniform(-room, room, (n, 3))
    elem = rng.permutation(np.arange(n) % 5)
    elem = np.array([0, 0, 1, 1, 2], dtype=np.int32)[elem]
    box = np.diag([L, L, L])
    return W.remap(r, box), elem, box


def _structures(case, seed):
    """[(r, elem, box), ...] of a case."""
    n = case["size"]
    if case["model"] == "water":
        return [W.water(n, WATER_EDGE * n ** (1.0 / 3.0), seed)]
    if case["kind"] in ("batch", "dataset"):
        # The sizes belong to the case, the atoms to the seed.
        rng = np.random.default_rng([n, case["lo"], case["hi"]])
        sizes = rng.integers(case["lo"], case["hi"] + 1, n)
        return [_bcn(int(k), seed * 1000 + q) for q, k in enumerate(sizes)]
    return [_bcn(n, seed)]


@functools.lru_cache(maxsize=None)
def _scaling(model, cut):
    """Rows (min, max, mean, sigma) per element and function, from one small
    structure in 64 bits on the CPU: what nnp-scaling writes."""
    ref = _Reference(model, cut, "cpu")
    case = {"model": model, "size": 64 if model == "water" else 96,
            "kind": "eval"}
    nb = _neighbours(_structures(case, 4711), ref.rc, "cpu")
    G = ref.descriptors(nb, slice(0, nb["n"]), nb["dr"])
    out = []
    for e in range(len(ref.sf)):
        g = G[nb["elem"] == e][:, :len(ref.sf[e])].numpy()
        mn, mx = g.min(0), g.max(0)
        mx = np.where(mx > mn, mx, mn + 1.0)
        sd = g.std(0, ddof=1)
        out.append(np.stack([mn, mx, g.mean(0), np.where(sd > 0, sd, 1.0)], 1))
    return out


def _load_model(case):
    """The model of a case, from the files a user has."""
    cut = case.get("cut", 6)
    text, symbols, z, hidden = _settings(case["model"], cut)
    with tempfile.TemporaryDirectory() as d:
        W.write_model(d, text, symbols, z, hidden)
        W.write_scaling(os.path.join(d, "scaling.data"),
                        _scaling(case["model"], cut))
        return engine.Model.load_dir(d)


def _context(case, model):
    ctx = engine.Context(model)
    ctx.set_precision(PREC[case["prec"]])
    return ctx


def _training_data(case, r, seed):
    """Reference energy and forces of a training structure (forces of a
    liquid: 0.5 eV/A)."""
    rng = np.random.default_rng(seed + 77)
    return float(0.02 * len(r) * rng.normal()), rng.normal(0.0, 0.5, r.shape)


class _DeviceArray:
    """The engine's force buffer as an array on the device (keeps the context
    alive as long as the array is used)."""

    def __init__(self, ctx):
        self.ctx = ctx
        self.__cuda_array_interface__ = {
            "shape": (ctx.n, 3), "typestr": "<f8", "version": 3,
            "data": (ctx.forces_device_ptr(), False)}


def prepare(case, seed):
    kind = case["kind"]
    model = _load_model(case)
    sts = _structures(case, seed)
    r, elem, box = sts[0]
    ctx = _context(case, model)
    s = {"kind": kind, "model": model, "ctx": ctx}
    if kind in ("predict", "eval"):
        ctx.set_structure(r, elem, box)
        s["r"] = r if kind == "predict" else torch.from_numpy(r).cuda()
    elif kind == "batch":
        ctx.set_structures(sts)
        s["r"] = torch.from_numpy(np.concatenate([t[0] for t in sts])).cuda()
    elif kind == "dataset":
        s["structures"] = sts
    elif kind == "md":
        ctx.set_structure(r, elem, box)
        masses = np.array(W.WATER_MASSES)
        v = W.maxwell_boltzmann(masses[elem], 300.0, seed)
        ctx.md_init(masses, MD_DT, skin=1.0, v=v)
    elif kind in ("adam", "kalman"):
        s["structure"] = (r, elem, box)
        s["e_ref"], s["f_ref"] = _training_data(case, r, seed)
        if kind == "kalman":
            ctx.kalman_init()
            s["components"] = _components(case, r, seed)
    else:
        s.update(_domain(r, elem, box, model.max_cutoff))
    torch.cuda.synchronize()
    return s


def _components(case, r, seed):
    rng = np.random.default_rng(seed + 78)
    return [(int(rng.integers(len(r))), int(rng.integers(3)))
            for _ in range(2)]


def _domain(r, elem, box, rc):
    """What LAMMPS hands over: per owned atom its neighbours within rc, those
    in periodic images as ghost atoms behind the owned ones, and force rows
    for all of them with LAMMPS' headroom."""
    dev = "cuda"
    nb = _neighbours([(r, elem, box)], rc, dev)
    mask = nb["mask"]
    i, k = torch.nonzero(mask, as_tuple=True)
    j, dr = nb["idx"][i, k], nb["dr"][i, k]
    R = torch.from_numpy(r).to(dev)
    inv = torch.from_numpy(np.linalg.inv(box)).to(dev)
    b = torch.round((dr - (R[i] - R[j])) @ inv).to(torch.int64)
    code = ((b[:, 0] + 8) * 17 + b[:, 1] + 8) * 17 + b[:, 2] + 8
    home = (8 * 17 + 8) * 17 + 8
    n = len(r)
    ghost = code != home
    _, inverse = torch.unique((j * 4913 + code)[ghost], return_inverse=True)
    index = j.clone()
    index[ghost] = n + inverse
    off = np.zeros(n + 1, dtype=np.int64)
    np.cumsum(mask.sum(1).cpu().numpy(), out=off[1:])
    return {"centre_elem": elem, "offsets": off,
            "nbr_index": index.to(torch.int32).cpu().numpy(),
            "nbr_elem": np.ascontiguousarray(elem[j.cpu().numpy()]),
            "dr": dr.cpu().numpy(), "nout": _rows(n, np.diag(box), rc)}


def _rows(n, edges, rc):
    """Owned atoms and the ghosts of a shell of width rc, and a quarter."""
    return int(1.25 * n * float(np.prod(1.0 + 2.0 * rc / edges))) + 64


def run(s):
    ctx, kind = s["ctx"], s["kind"]
    if kind == "predict":
        ctx.set_positions(s["r"])
        e = ctx.evaluate(engine.FORCES_REFERENCE)
        return {"energy": e, "forces": ctx.forces()}
    if kind in ("eval", "batch"):
        ctx.set_positions_device(s["r"].data_ptr())
        e = ctx.evaluate(engine.FORCES_CONSISTENT)
        f = torch.as_tensor(_DeviceArray(ctx), device="cuda")
        if kind == "eval":
            return {"energy": e, "forces": f}
        return {"energy": e, "energies": ctx.structure_energies(), "forces": f}
    if kind == "dataset":
        ctx.set_structures(s["structures"])
        ctx.evaluate(engine.FORCES_CONSISTENT)
        return {"energies": ctx.structure_energies(), "forces": ctx.forces()}
    if kind == "md":
        epot, ekin = ctx.md_run(MD_STEPS)
        r, v = ctx.md_state()
        return {"epot": epot, "ekin": ekin, "r": r, "v": v}
    if kind == "adam":
        ctx.set_structure(*s["structure"])
        grad, loss = ctx.train_gradient(s["f_ref"], s["e_ref"], 1.0, 10.0)
        ctx.train_adam(1e-3)
        return {"grad": grad, "loss": loss, "weights": ctx.get_weights()}
    if kind == "kalman":
        # As n2p2_amd.train runs an epoch: each update loads its structure.
        n = len(s["structure"][0])
        ctx.set_structure(*s["structure"])
        ctx.calculate_neighbor_list(s["model"].max_cutoff)
        h = ctx.energy_weight_jacobian(file_order=False)[0] / n
        e = ctx.evaluate(-1)
        ctx.kalman_update(h, (s["e_ref"] - e) / n)
        jac = [h]
        for i, c in s["components"]:
            ctx.set_structure(*s["structure"])
            ctx.evaluate(engine.FORCES_CONSISTENT)
            f = ctx.forces()
            f_ref = f.copy()
            f_ref[i, c] -= 1.5 * n       # loss gradient = dF_ic / dw
            h, _ = ctx.train_gradient(f_ref, 0.0, 0.0, 1.0)
            ctx.kalman_update(h, s["f_ref"][i, c] - f[i, c])
            jac.append(h)
        return {"jacobians": jac, "weights": ctx.get_weights()}
    ctx.set_neighbor_list(s["centre_elem"], s["offsets"], s["nbr_index"],
                          s["nbr_elem"], s["dr"])
    e = ctx.evaluate(engine.FORCES_REFERENCE)
    return {"energy": e, "atomic": ctx.atomic_energies(),
            "forces": ctx.scattered_forces(s["nout"])}


# ------------------------------------------------------- work and tolerances

def _atoms(case):
    if case["model"] == "water":
        return 3 * case["size"]
    if case["kind"] in ("batch", "dataset"):
        return case["size"] * (case["lo"] + case["hi"]) / 2
    return case["size"]


# Operations per atom of one energy + force evaluation at these densities,
# every triplet taken once and its member sums contracted before the vector
# work: pair tests 8, triplet geometry and force 70 (narrow) or 50 (wide),
# member 8 with its power, radial member 14, networks 4 per weight.
#   water: 5,444 pairs, 2,488 triplets x 8 members, 107 neighbours x 8
#   bcn: 2,556 triplets x 12 members, 72 neighbours x 10
#   compact: 2,556 triplets, 3 angle windows x 20, 18 products x 8
_FLOPS = {"water": 5444 * 8 + 2488 * (70 + 8 * 8) + 107 * 8 * 14 + 4 * 1650,
          "bcn": 2556 * (50 + 12 * 8) + 72 * 10 * 14 + 4 * 3990,
          "compact": 2556 * (60 + 3 * 20 + 18 * 8) + 72 * 6 * 20 + 4 * 4400}
_NEIGHBOURS = {"water": 107, "bcn": 72, "compact": 72}


def work(case):
    n, kind, model = _atoms(case), case["kind"], case["model"]
    flops, bytes_ = n * _FLOPS[model], n * (24 + 4 + 24)
    if kind == "md":
        # positions and velocities read and written each step
        return {"flops": MD_STEPS * flops, "bytes": MD_STEPS * n * 96}
    if kind == "adam":
        # the evaluation and the forward tangent of the descriptors; value,
        # tangent and adjoints through the networks
        return {"flops": 2 * flops + n * 16 * 1650, "bytes": 2 * bytes_}
    if kind == "kalman":
        # the covariance (3,402 weights) read and written by each of 3 updates
        nw = 2 * (40 * 25 + 25 + 25 * 25 + 25 + 25 + 1)
        return {"flops": 5 * flops + 3 * 4 * nw * nw,
                "bytes": 3 * 2 * 8 * nw * nw}
    if kind == "lammps":
        # the list's entries: index, element, vector
        return {"flops": flops,
                "bytes": bytes_ + n * _NEIGHBOURS[model] * 32}
    return {"flops": flops, "bytes": bytes_}


def tolerance(case):
    kind = case["kind"]
    mixed = case["prec"] != "fp64"
    if kind == "kalman":
        # three filter updates, each from the weights of the one before
        return {"rel": 1e-10, "max": 1e-8}
    if not mixed:
        return {"rel": 1e-12, "max": 1e-10}
    # Four times the largest error against 64 bits seen over the kinds, cutoff
    # types and sizes: forces 1.4e-5 (bf16) and 4e-6.
    if case["prec"] == "mixed_bf16":
        return {"rel": 6e-5, "max": 4.5e-4}
    return {"rel": 1.6e-5, "max": 1.3e-4}


# ----------------------------------------- the same in plain torch, 64 bits

class _Reference:
    """A model in plain torch: descriptors, networks, parameters."""

    def __init__(self, model, cut, dev, scaling=False):
        text, symbols, z, hidden = _settings(model, cut)
        self.dev, self.cut = dev, cut
        self.soft = "p p l" in text
        at = {s: i for i, s in enumerate(symbols)}
        self.sf = [[] for _ in symbols]
        for line in text.splitlines():
            w = line.split()
            if w[0] != "symfunction_short":
                continue
            e, t, x = at[w[1]], int(w[2]), w[3:]
            ne = 1 if t in (2, 20) else 2
            el = tuple(at[q] for q in x[:ne])
            p = x[ne:]
            if t in (20, 22):
                par = tuple(float(q) for q in p[:-1])      # rl rc [al ar]
                # order: type, elements, rc, rl, angles
                key = (t, el, par[1], par[0]) + par[2:]
            elif t == 2:
                par = tuple(float(q) for q in p)           # eta rs rc
                key = (t, par[2], par[0], par[1], el)
            else:
                eta, lam, zeta, rc = (float(q) for q in p)
                par = (eta, lam, zeta, rc)
                # order: type, rc, eta, zeta, lambda, elements
                key = (t, rc, eta, zeta, lam, el)
            self.sf[e].append((key, t, el, par))
        for s in self.sf:
            s.sort(key=lambda q: q[0])
        self.rc = max(q[3][1] if q[1] in (20, 22) else q[3][-1]
                      for s in self.sf for q in s)
        self.nets = []
        for k in range(len(symbols)):
            sizes = [len(self.sf[k])] + list(hidden) + [1]
            w = torch.from_numpy(W.xavier_weights(sizes, 7 + 101 * k))
            layers, p = [], 0
            for a, b in zip(sizes[:-1], sizes[1:]):
                Wl = w[p:p + a * b].reshape(a, b).T.contiguous()
                p += a * b
                layers.append([Wl.to(dev), w[p:p + b].clone().to(dev)])
                p += b
            self.nets.append(layers)
        self.range = None
        if scaling:
            self.range = [torch.from_numpy(q).to(dev)
                          for q in _scaling(model, cut)]

    def fc(self, r, rc):
        x = r / rc
        if self.cut == 1:
            f = 0.5 * (torch.cos(math.pi * x) + 1.0)
        elif self.cut == 2:
            f = torch.tanh(1.0 - x) ** 3
        else:
            f = ((15.0 - 6.0 * x) * x - 10.0) * x ** 3 + 1.0
        return torch.where(r < rc, f, torch.zeros_like(f))

    @staticmethod
    def window(x, lo, hi, asym):
        """Compact function on the open interval (lo, hi), core p2."""
        y = ((x - 0.5 * (lo + hi)) / (0.5 * (hi - lo))).abs()
        inside = (x > lo) & (x < hi)
        y = torch.where(inside, y, torch.zeros_like(y))
        if asym:
            y = (2.0 - y) * y
        f = ((15.0 - 6.0 * y) * y - 10.0) * y ** 3 + 1.0
        return torch.where(inside, f, torch.zeros_like(f))

    def descriptors(self, nb, part, dr):
        """Unscaled G (atoms x functions) of a range of atoms from their
        neighbour vectors dr (atoms x K x 3).  The elements share their lists
        of parameters, so each term is formed once for all of them."""
        mask, ej = nb["mask"][part], nb["ej"][part]
        r = torch.sqrt(torch.where(mask, (dr * dr).sum(-1), 4e4))
        ne = len(self.sf)
        hot = [(mask & (ej == q)).to(dr.dtype) for q in range(ne)]
        K = dr.shape[1]
        a, b = torch.triu_indices(K, K, 1, device=dr.device)
        fc = self.fc(r, self.rc)
        geo = None
        cache = {}
        cols = []
        for key, t, el, par in self.sf[0]:
            if t == 2:
                if par not in cache:
                    eta, rs, rc = par
                    cache[par] = torch.exp(-eta * (r - rs) ** 2) * fc
                cols.append((cache[par] * hot[el[0]]).sum(1))
                continue
            if t == 20:
                if par not in cache:
                    cache[par] = self.window(r, *par, True)
                cols.append((cache[par] * hot[el[0]]).sum(1))
                continue
            if geo is None:
                dj, dk = dr[:, a], dr[:, b]
                both = mask[:, a] & mask[:, b]
                rj, rk = r[:, a], r[:, b]
                cos = (dj * dk).sum(-1) / (rj * rk)
                if t == 3:
                    d2 = torch.where(both, ((dj - dk) ** 2).sum(-1), 1.0)
                    s2 = rj * rj + rk * rk + d2
                    pf = fc[:, a] * fc[:, b] * self.fc(torch.sqrt(d2),
                                                       self.rc)
                elif t == 9:
                    s2 = rj * rj + rk * rk
                    pf = fc[:, a] * fc[:, b]
                else:
                    th = torch.acos(torch.where(both, cos, 0.5))
                types = []
                index = {}
                for q in range(ne):
                    for p in range(q, ne):
                        index[(q, p)] = len(types)
                        m = hot[q][:, a] * hot[p][:, b]
                        if p != q:
                            m = m + hot[p][:, a] * hot[q][:, b]
                        types.append(m)
                types = torch.stack(types, 2)
                geo = True
            if (t, par) not in cache:
                if t == 22:
                    rl, rc, al, ar = par
                    if ("w", rl, rc) not in cache:
                        cache[("w", rl, rc)] = self.window(r, rl, rc, True)
                    if ("a", al, ar) not in cache:
                        cache[("a", al, ar)] = self.window(
                            th, math.radians(al), math.radians(ar), False)
                    w = cache[("w", rl, rc)]
                    v = w[:, a] * w[:, b] * cache[("a", al, ar)]
                else:
                    eta, lam, zeta, rc = par
                    if ("e", eta) not in cache:
                        cache[("e", eta)] = torch.exp(-eta * s2) * pf
                    pl = (1.0 + lam * cos).clamp_min(0.0)
                    v = 2.0 ** (1.0 - zeta) * pl ** zeta * cache[("e", eta)]
                cache[(t, par)] = torch.matmul(v.unsqueeze(1), types)[:, 0]
            cols.append(cache[(t, par)][:, index[el]])
        return torch.stack(cols, 1)

    def scaled(self, G, elem):
        lo = torch.stack([q[:, 0] for q in self.range])[elem]
        hi = torch.stack([q[:, 1] for q in self.range])[elem]
        return (G - lo) / (hi - lo)

    def slope(self, elem):
        lo = torch.stack([q[:, 0] for q in self.range])[elem]
        hi = torch.stack([q[:, 1] for q in self.range])[elem]
        return 1.0 / (hi - lo)

    def networks(self, G, elem):
        E = torch.zeros(len(G), dtype=G.dtype, device=G.device)
        for e, layers in enumerate(self.nets):
            at = torch.nonzero(elem == e)[:, 0]
            x = G[at]
            for k, (w, b) in enumerate(layers):
                x = x @ w.T + b
                if k + 1 < len(layers):
                    x = (torch.nn.functional.softplus(x) if self.soft
                         else torch.tanh(x))
            E = E.index_add(0, at, x[:, 0])
        return E


def _neighbours(structures, rc, dev):
    """Padded neighbour lists of all atoms of a set of periodic structures:
    idx, mask, element of the neighbour, dr = r_i - r_j(image)."""
    rows, cols, vecs, elems, base = [], [], [], [], 0
    for r, elem, box in structures:
        n = len(r)
        R = torch.from_numpy(np.ascontiguousarray(r)).to(dev)
        L = np.diag(box)
        nc = np.floor(L / (rc * (1 + 1e-9))).astype(int)
        if n > 2500 and nc.min() >= 3:
            c = torch.from_numpy(np.minimum(np.floor(r / L * nc), nc - 1)
                                 .astype(np.int64)).to(dev)
            NC = torch.from_numpy(nc.astype(np.int64)).to(dev)
            cid = (c[:, 0] * nc[1] + c[:, 1]) * nc[2] + c[:, 2]
            order = torch.argsort(cid, stable=True)
            cnt = torch.bincount(cid, minlength=int(nc.prod()))
            start = torch.cumsum(cnt, 0) - cnt
            most = int(cnt.max())
            sh = torch.tensor([(x, y, z) for x in (-1, 0, 1)
                               for y in (-1, 0, 1) for z in (-1, 0, 1)],
                              device=dev)
            slot = torch.arange(most, device=dev)
            Lt = torch.from_numpy(L.copy()).to(dev)
            for i0 in range(0, n, 4096):
                i1 = min(n, i0 + 4096)
                cc = c[i0:i1, None] + sh
                wrap = torch.div(cc, NC, rounding_mode="floor")
                cc = cc - wrap * NC
                q = (cc[..., 0] * nc[1] + cc[..., 1]) * nc[2] + cc[..., 2]
                ok = slot < cnt[q][..., None]
                j = order[(start[q][..., None] + slot).clamp_max(n - 1)]
                img = (wrap.to(R.dtype) * Lt)[:, :, None]
                d = R[i0:i1, None, None] - R[j] - img
                d2 = (d * d).sum(-1)
                i, x, y = torch.nonzero(ok & (d2 < rc * rc) & (d2 > 1e-12),
                                        as_tuple=True)
                rows.append(base + i0 + i)
                cols.append(base + j[i, x, y])
                vecs.append(d[i, x, y])
        else:
            p = [int(math.floor(rc / x)) + 1 for x in L]
            img = torch.tensor([(x * L[0], y * L[1], z * L[2])
                                for x in range(-p[0], p[0] + 1)
                                for y in range(-p[1], p[1] + 1)
                                for z in range(-p[2], p[2] + 1)],
                               dtype=R.dtype, device=dev)
            step = max(1, int(2e7 / (n * len(img))))
            for i0 in range(0, n, step):
                d = (R[i0:i0 + step, None, None] - R[None, :, None]
                     - img[None, None])
                d2 = (d * d).sum(-1)
                i, j, k = torch.nonzero((d2 < rc * rc) & (d2 > 1e-12),
                                        as_tuple=True)
                rows.append(base + i0 + i)
                cols.append(base + j)
                vecs.append(d[i, j, k])
        elems.append(torch.from_numpy(elem.astype(np.int64)).to(dev))
        base += n
    rows, cols, vecs = torch.cat(rows), torch.cat(cols), torch.cat(vecs)
    elem = torch.cat(elems)
    count = torch.bincount(rows, minlength=base)
    K = int(count.max())
    first = torch.cumsum(count, 0) - count
    pos = torch.arange(len(rows), device=dev) - first[rows]
    idx = torch.zeros((base, K), dtype=torch.int64, device=dev)
    mask = torch.zeros((base, K), dtype=torch.bool, device=dev)
    dr = torch.zeros((base, K, 3), dtype=torch.float64, device=dev)
    dr[..., 0] = 200.0
    idx[rows, pos] = cols
    mask[rows, pos] = True
    dr[rows, pos] = vecs
    return {"n": base, "elem": elem, "idx": idx, "mask": mask, "dr": dr,
            "ej": elem[idx]}


def _chunks(nb, ref):
    K = nb["mask"].shape[1]
    types = len(ref.sf) * (len(ref.sf) + 1) // 2
    step = max(1, int(4e7 / (K * K * (types + 8))))
    return [slice(i, min(nb["n"], i + step)) for i in range(0, nb["n"], step)]


def _energy_forces(ref, nb, descriptors=False):
    """Atomic energies and forces F_m = -dE/dr_m."""
    F = torch.zeros((nb["n"], 3), dtype=torch.float64, device=nb["dr"].device)
    E, Gs = [], []
    for part in _chunks(nb, ref):
        dr = nb["dr"][part].clone().requires_grad_(True)
        G = ref.scaled(ref.descriptors(nb, part, dr), nb["elem"][part])
        e = ref.networks(G, nb["elem"][part])
        g, = torch.autograd.grad(e.sum(), dr)
        g = g * nb["mask"][part][..., None]
        F[part] -= g.sum(1)
        F.index_add_(0, nb["idx"][part].reshape(-1), g.reshape(-1, 3))
        E.append(e.detach())
        if descriptors:
            Gs.append(G.detach())
    return torch.cat(E), F, torch.cat(Gs) if descriptors else None


def _tangent(ref, nb, d):
    """t_as = sum_i d_i . dG_as/dr_i of the scaled descriptors."""
    out = []
    for part in _chunks(nb, ref):
        step = (d[part][:, None] - d[nb["idx"][part]]) \
            * nb["mask"][part][..., None]
        _, t = torch.func.jvp(lambda x: ref.descriptors(nb, part, x),
                              (nb["dr"][part],), (step,))
        out.append(t * ref.slope(nb["elem"][part]))
    return torch.cat(out)


def _flat(tensors):
    """Weights per element and layer, W[k][j] then b (the engine's order)."""
    return torch.cat([x.reshape(-1) for net in tensors for wb in net
                      for x in wb])


def _weight_gradient(ref, G, elem, kappa, t):
    """d/dw of sum_a kappa E_a + (dE_a/dG . t_a)."""
    par = [x.requires_grad_(True) for net in ref.nets for wb in net
           for x in wb]
    G = G.detach().clone().requires_grad_(True)
    E = ref.networks(G, elem)
    total = kappa * E.sum()
    if t is not None:
        dEdG, = torch.autograd.grad(E.sum(), G, create_graph=True)
        total = total + (dEdG * t).sum()
    got = torch.autograd.grad(total, par, allow_unused=True)
    out = torch.cat([(torch.zeros_like(p) if g is None else g).reshape(-1)
                     for g, p in zip(got, par)])
    for x in par:
        x.requires_grad_(False)
    return out


def _host(x):
    return x.detach().cpu().numpy()


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    kind = case["kind"]
    ref = _Reference(case["model"], case.get("cut", 6), dev, scaling=True)
    sts = _structures(case, seed)
    r, elem, box = sts[0]
    if kind == "md":
        return _exact_md(ref, r, elem, box, seed, dev)
    nb = _neighbours(sts, ref.rc, dev)
    E, F, G = _energy_forces(ref, nb, kind in ("adam", "kalman"))
    if kind in ("predict", "eval"):
        return {"energy": float(E.sum()), "forces": _host(F)}
    if kind in ("batch", "dataset"):
        parts = torch.split(E, [len(s[0]) for s in sts])
        out = {"energies": np.array([float(p.sum()) for p in parts]),
               "forces": _host(F)}
        if kind == "batch":
            out["energy"] = float(E.sum())
        return out
    if kind == "lammps":
        d = _domain(r, elem, box, ref.rc)
        # Forces on owned and ghost rows from each entry's own term.
        f = np.zeros((d["nout"], 3))
        g = _entry_gradients(ref, nb)
        i, k = torch.nonzero(nb["mask"], as_tuple=True)
        ge = _host(g[i, k])
        np.subtract.at(f, _host(i), ge)
        np.add.at(f, d["nbr_index"], ge)
        return {"energy": float(E.sum()), "atomic": _host(E), "forces": f}
    e_ref, f_ref = _training_data(case, r, seed)
    n = len(r)
    if kind == "adam":
        w0 = _flat(ref.nets)
        d = F - torch.from_numpy(f_ref).to(dev)
        t = -(2.0 * 10.0 / (3.0 * n)) * _tangent(ref, nb, d)
        de = float(E.sum()) - e_ref
        grad = _weight_gradient(ref, G, nb["elem"], 2.0 * de / n ** 2, t)
        w = w0 - 1e-3 * grad / (grad.abs() + 1e-8)
        return {"grad": _host(grad),
                "loss": (de * de / n ** 2,
                         10.0 * float((d * d).sum()) / (3.0 * n)),
                "weights": _host(w)}
    # Kalman filter from P = 100 I (epsilon 0.01), the default annealing.
    w = _flat(ref.nets)
    P = 100.0 * torch.eye(len(w), dtype=torch.float64, device=dev)
    eta, q = 0.01, 0.01
    updates = [None] + _components(case, r, seed)
    jac = []
    for u in updates:
        _set_weights(ref, w)
        dE = ref.networks(G, nb["elem"])
        if u is None:
            h = _weight_gradient(ref, G, nb["elem"], 1.0, None) / n
            xi = (e_ref - float(dE.sum())) / n
        else:
            i, c = u
            d = torch.zeros((n, 3), dtype=torch.float64, device=dev)
            d[i, c] = 1.0
            t = _tangent(ref, nb, d)
            h = -_weight_gradient(ref, G, nb["elem"], 0.0, t)
            Gv = G.detach().clone().requires_grad_(True)
            g, = torch.autograd.grad(ref.networks(Gv, nb["elem"]).sum(), Gv)
            xi = f_ref[i, c] + float((g * t).sum())
        if eta < 1.0:
            eta *= math.exp(2.302)
        X = P @ h
        den = float(h @ X) + 1.0 / eta
        P = P - torch.outer(X, X) / den
        P.diagonal().add_(q)
        w = w + X * (xi / den)
        if q > 1e-6:
            q *= math.exp(-2.302)
        jac.append(_host(h))
    return {"jacobians": jac, "weights": _host(w)}


def _set_weights(ref, w):
    p = 0
    for net in ref.nets:
        for wb in net:
            for k in range(2):
                m = wb[k].numel()
                wb[k] = w[p:p + m].reshape(wb[k].shape).clone()
                p += m


def _entry_gradients(ref, nb):
    out = []
    for part in _chunks(nb, ref):
        dr = nb["dr"][part].clone().requires_grad_(True)
        G = ref.scaled(ref.descriptors(nb, part, dr), nb["elem"][part])
        g, = torch.autograd.grad(ref.networks(G, nb["elem"][part]).sum(), dr)
        out.append(g * nb["mask"][part][..., None])
    return torch.cat(out)


def _exact_md(ref, r, elem, box, seed, dev):
    if len(r) > 30000:
        return None
    m = torch.from_numpy(np.array(W.WATER_MASSES)[elem]).to(dev)[:, None]
    v = torch.from_numpy(W.maxwell_boltzmann(_host(m)[:, 0], 300.0,
                                             seed)).to(dev)
    x = torch.from_numpy(r.copy()).to(dev)
    L = torch.from_numpy(np.diag(box).copy()).to(dev)

    def forces(x):
        inside = _host(x - torch.floor(x / L) * L)
        nb = _neighbours([(inside, elem, box)], ref.rc, dev)
        E, F, _ = _energy_forces(ref, nb)
        return float(E.sum()), F

    _, F = forces(x)
    h = 0.5 * MD_DT * W.FTOA / m
    epot, ekin = [], []
    for _ in range(MD_STEPS):
        v = v + h * F
        x = x + MD_DT * v
        e, F = forces(x)
        v = v + h * F
        epot.append(e)
        ekin.append(0.5 / W.FTOA * float((m * v * v).sum()))
    return {"epot": np.array(epot), "ekin": np.array(ekin), "r": _host(x),
            "v": _host(v)}
