"""The measured workloads of the library: what its users have it do, through
its public entry points, from the smallest call to the largest.

listed() holds the fixed cases and draw(rng) one more of the same ranges.
prepare(case, seed) makes what a program has in hand before the call (inputs
in GPU memory, output buffers, a plan or a network), run(state) is one pass,
work(case) the bytes and FP64 / bf16 operations a pass cannot do without, and
exact(case, seed) the same outputs in plain 64-bit torch.

Kinds of case:
  map        the four cross-sections over (K, q) pairs of one element, one
             process or all four, FP64 or mixed precision, into new tensors
             or into the caller's
  batch      one plan over many elements with uneven pair counts
  recoil     DEL and CEL recoil integrals over a vector of kinetic energies
  coulomb    Coulomb data and transport of each element of a mixture, then
             its hard-scattering cutoff
  soft       soft-scattering transport over a vector of kinetic energies
  pumas      a PUMAS DCS table with its envelope
  surrogate  the trained network with exact fallback over 48 elements
  train      one epoch of the network's training
"""
import math
import os
import random

import numpy as np
import torch

import noa_amd
from noa_amd import dcs, pumas
from noa_amd.batch import BatchPlan
from noa_amd.physics import AtomicElement

MUON = 0.10565839
TAU = 1.77682
ME = 0.510998910e-03
NA = 6.02214076e+23
ROCK = (11, 22.0, 0.1364e-6)
DEV = "cuda:0"
F64 = torch.float64

# Z, A (g/mol), I (GeV) of the elements that drawn single-element cases use:
# standard rock, hydrogen, oxygen, iron, lead
ELEMENTS = (ROCK, (1, 1.008, 19.2e-9), (8, 15.999, 95e-9), (26, 55.845, 286e-9), (82, 207.2, 823e-9))
PROCESSES = ("bremsstrahlung", "pair_production", "photonuclear", "ionisation")


# ---- the cases ----

def _map(process, n, precision="f64", in_place=False, element=0, mass="muon"):
    return {"kind": "map", "process": process, "n": n, "precision": precision, "in_place": in_place,
            "element": element, "mass": mass}


def listed():
    return [
        # the reference's notebook: one process over 10,000 pairs, called from an interactive session
        dict(_map("bremsstrahlung", 10000), name="map_brems_1e4"),
        # a test or a sampling step: all four processes over 2^16 standard-rock pairs
        dict(_map("all", 1 << 16), name="map_all_2e16"),
        # the headline: all four processes over 2^24 pairs, into the caller's tensors
        dict(_map("all", 1 << 24, in_place=True), name="map_all_2e24"),
        # the faster form over an uneven number of pairs, results allocated by the call
        dict(_map("all", 3000017, precision="f32mixed"), name="mixed_all_3e6"),
        # a material library: 48 elements with 2^10 to 2^20 pairs each, replayed as one plan
        {"name": "batch48_f64", "kind": "batch", "elements": 48, "log2_min": 10.0, "log2_max": 20.0,
         "precision": "f64"},
        # the energy grid of a transport table: DEL and CEL at 146 kinetic energies
        {"name": "recoil_146", "kind": "recoil", "n": 146, "min_points": 180, "element": 0, "mass": "muon"},
        # the same for a population of particles
        {"name": "recoil_2e16", "kind": "recoil", "n": 1 << 16, "min_points": 180, "element": 0, "mass": "muon"},
        # elastic scattering of particles in a three-element material
        {"name": "coulomb_mix3_2e16", "kind": "coulomb", "n": 1 << 16, "elements": 3, "mass": "muon"},
        # soft scattering of particles in one material
        {"name": "soft_2e16", "kind": "soft", "n": 1 << 16, "element": 0, "mass": "muon"},
        # a transport code's start-up: the DCS tables of 48 elements on 146 energies
        {"name": "pumas_48x146", "kind": "pumas", "elements": 48, "n": 146, "cutoff": 0.05, "mass": "muon"},
        # serving the surrogate at 3% over 48 elements
        {"name": "surrogate_2e22", "kind": "surrogate", "n": 1 << 22, "tol": 0.03},
        # training it: 16 Adam steps at the batch that it is trained with
        {"name": "train_2e17", "kind": "train", "n": 1 << 17, "batch": 8192},
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("map", "map", "map", "batch", "recoil", "coulomb", "soft", "pumas", "surrogate", "train"))
    el, mass = rng.randrange(len(ELEMENTS)), rng.choice(("muon", "muon", "muon", "tau"))
    if kind == "map":
        precision = rng.choice(("f64", "f64", "f32mixed"))
        process = "all" if precision == "f32mixed" else rng.choice(("all", "all") + PROCESSES)
        return _map(process, _size(rng, 100, 1 << 24), precision, rng.random() < 0.5, el, mass)
    if kind == "batch":
        lo = rng.uniform(5.0, 12.0)
        return {"kind": "batch", "elements": rng.randint(2, 48), "log2_min": lo,
                "log2_max": lo + rng.uniform(2.0, 8.0), "precision": rng.choice(("f64", "f64", "f32mixed"))}
    if kind == "recoil":
        return {"kind": "recoil", "n": _size(rng, 30, 1 << 16), "min_points": rng.choice((30, 60, 100, 180)),
                "element": el, "mass": mass}
    if kind == "coulomb":
        return {"kind": "coulomb", "n": _size(rng, 50, 1 << 16), "elements": rng.randint(1, 6), "mass": mass}
    if kind == "soft":
        return {"kind": "soft", "n": _size(rng, 50, 1 << 16), "element": el, "mass": mass}
    if kind == "pumas":
        return {"kind": "pumas", "elements": rng.randint(1, 40), "n": rng.randint(20, 146),
                "cutoff": rng.choice((0.05, 0.05, 0.01, 0.1)), "mass": mass}
    if kind == "surrogate":
        return {"kind": "surrogate", "n": _size(rng, 1 << 13, 1 << 22), "tol": rng.choice((0.01, 0.03, 0.1))}
    batch = rng.choice((1024, 2048, 4096, 8192))
    return {"kind": "train", "n": batch + rng.randrange(1 << 16), "batch": batch}


# ---- inputs ----

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _mass(case):
    return TAU if case.get("mass") == "tau" else MUON


def _pairs(n, seed):
    """K log-uniform in [1e-3, 1e6] GeV, nu = q / K log-uniform in [1e-6, 1)."""
    g = _gen(seed)
    K = 10.0 ** (-3.0 + 9.0 * torch.rand(n, dtype=F64, device=DEV, generator=g))
    nu = 10.0 ** (-6.0 * (1.0 - torch.rand(n, dtype=F64, device=DEV, generator=g)))
    return K, torch.minimum(nu, torch.tensor(1.0 - 2.0 ** -40, dtype=F64, device=DEV)) * K


def _energies(n, seed):
    return 10.0 ** (-3.0 + 9.0 * torch.rand(n, dtype=F64, device=DEV, generator=_gen(seed)))


def _grid(n, seed):
    """An ascending grid of n energies over [1e-3, 1e6] GeV, as a table has it."""
    u = torch.rand(n, dtype=F64, device=DEV, generator=_gen(seed))
    at = (torch.arange(n, dtype=F64, device=DEV) + 0.1 + 0.8 * u) / n
    return 10.0 ** (-3.0 + 9.0 * at)


def _batch_of(count, log2_min=10.0, log2_max=20.0):
    """Elements (Z, A, I) with Z over 1..92 and the offsets of their pair ranges."""
    r = random.Random(48)
    els, off = [], [0]
    for _ in range(count):
        Z = r.randint(1, 92)
        els.append((Z, Z * r.uniform(2.0, 2.6), 16e-9 * Z ** 0.9))
        off.append(off[-1] + int(2.0 ** r.uniform(log2_min, log2_max)))
    return els, off


def _mixture(count):
    return [ELEMENTS[(0, 2, 3, 1, 4)[i % 5]] for i in range(count)]


def _element(e):
    return AtomicElement(A=float(e[1]), I=float(e[2]), Z=int(e[0]))


def _process(name):
    return dcs.PROCESSES[PROCESSES.index(name)]


CHECKPOINT = os.path.join(os.path.dirname(os.path.abspath(noa_amd.__file__)), "surrogate_48el.npz")
LAYERS = ((3, 128), (128, 128), (128, 128), (128, 128), (128, 4))


def _train_inputs(case, seed):
    """Features over their domain, standardised smooth targets, the masks of
    closed processes, and Kaiming-uniform parameters."""
    g = _gen(seed)
    n = case["n"]
    X = (2.0 * torch.rand(n, 3, device=DEV, generator=g) - 1.0).contiguous()
    a, b, z = X[:, 0], X[:, 1], X[:, 2]
    T = torch.stack([torch.sin(3 * a + b), torch.cos(2 * b - a) * z, torch.sin(a * b * 4), 0.5 * a - torch.cos(3 * z)], 1)
    T = (1.2 * T + 0.05 * torch.randn(n, 4, device=DEV, generator=g)).contiguous()
    M = torch.stack([torch.ones_like(a), (b > -0.6 - a).float(), (b > 0.2 - a).float(), (b < 0.8).float()], 1).contiguous()
    p = []
    for k, (i, o) in enumerate(LAYERS):
        w = (2.0 * torch.rand(o * i, device=DEV, generator=g) - 1.0) * math.sqrt(6.0 / i)
        p += [0.1 * w if k == 4 else w, torch.zeros(o, device=DEV)]
    return X, T * M, M, torch.cat(p).cpu().numpy().astype(np.float32)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "map":
        K, q = _pairs(case["n"], seed)
        s = {"K": K, "q": q, "el": _element(ELEMENTS[case["element"]]), "m": _mass(case)}
        if case["in_place"]:
            t = F64 if case["precision"] == "f64" else torch.float32
            s["out"] = [torch.zeros(case["n"], dtype=t, device=DEV)
                        for _ in range(4 if case["process"] == "all" else 1)]
    elif kind == "batch":
        els, off = _batch_of(case["elements"], case["log2_min"], case["log2_max"])
        K, q = _pairs(off[-1], seed)
        s = {"plan": BatchPlan([_element(e) for e in els], off, K, q, MUON, precision=case["precision"])}
    elif kind == "recoil":
        K = _energies(case["n"], seed)
        s = {"K": K, "el": _element(ELEMENTS[case["element"]]), "m": _mass(case),
             "dels": [torch.zeros_like(K) for _ in range(4)], "cels": [torch.zeros_like(K) for _ in range(4)]}
    elif kind == "coulomb":
        n, nel = case["n"], case["elements"]
        new = lambda *shape: torch.zeros(*shape, dtype=F64, device=DEV)  # noqa: E731
        s = {"K": _energies(n, seed), "els": [_element(e) for e in _mixture(nel)], "m": _mass(case),
             "one": torch.ones(1, dtype=F64, device=DEV), "fCM": new(nel, n, 2), "screening": new(nel, n, 9),
             "fspin": new(nel, n), "invlambda": new(nel, n), "G": new(nel, n, 2), "mu0": new(n), "lb_h": new(n)}
    elif kind == "soft":
        K = _energies(case["n"], seed)
        s = {"K": K, "el": _element(ELEMENTS[case["element"]]), "m": _mass(case), "ms1": torch.zeros_like(K)}
    elif kind == "pumas":
        els, _ = _batch_of(case["elements"])
        s = {"K": _grid(case["n"], seed), "Z": [float(e[0]) for e in els], "A": [e[1] for e in els], "m": _mass(case)}
    elif kind == "surrogate":
        from noa_amd import surrogate
        sur = surrogate.Surrogate.load(CHECKPOINT)
        sur.set_tolerance(case["tol"])
        K, q = _pairs(case["n"], seed)
        s = {"sur": sur, "K": K, "q": q, "offsets": surrogate.equal_offsets(len(sur.elements), case["n"])}
    else:
        from noa_amd import surrogate
        X, T, M, p = _train_inputs(case, seed)
        net = surrogate.Network(max_rows=case["batch"])
        net.set_params(p)
        s = {"net": net, "X": X, "T": T, "M": M}
    s["case"] = case
    return s


# ---- one pass ----

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "map":
        args = (s["K"], s["q"], s["el"], s["m"])
        if case["process"] != "all":
            f = _process(case["process"])
            if not case["in_place"]:
                return dcs.map(f)(*args)
            dcs.vmap(f)(s["out"][0], *args)
            return s["out"][0]
        if case["precision"] == "f64":
            if not case["in_place"]:
                return dcs.hip.map_all(*args)
            dcs.hip.vmap_all(s["out"], *args)
            return s["out"]
        if not case["in_place"]:
            return dcs.hip.map_all_f32mixed(*args)
        dcs.eval_f32mixed(*args, *s["out"])
        return s["out"]
    if kind == "batch":
        s["plan"].launch()
        return s["plan"].outputs
    if kind == "recoil":
        dcs.recoil_integrals(s["K"], 0.05, s["el"], s["m"], case["min_points"], s["dels"], s["cels"])
        return {"del": s["dels"], "cel": s["cels"]}
    if kind == "coulomb":
        for e, el in enumerate(s["els"]):
            dcs.coulomb_data(s["fCM"][e], s["screening"][e], s["fspin"][e], s["invlambda"][e], s["K"], el, s["m"])
            dcs.coulomb_transport(s["G"][e], s["screening"][e], s["fspin"][e], s["one"])
        dcs.hard_scattering(s["mu0"], s["lb_h"], s["G"], s["fCM"], s["screening"], s["invlambda"], s["fspin"])
        return {k: s[k] for k in ("fCM", "screening", "fspin", "invlambda", "G", "mu0", "lb_h")}
    if kind == "soft":
        dcs.soft_scattering(s["ms1"], s["K"], s["el"], s["m"])
        return s["ms1"]
    if kind == "pumas":
        return pumas.dcs_table(s["Z"], s["A"], s["m"], case["cutoff"], s["K"])
    if kind == "surrogate":
        out, counters = s["sur"].evaluate(s["K"], s["q"], s["offsets"])
        # counters[0] is the launch's own work counter, the others are results
        return {"out": out, "counters": counters[1:]}
    losses = s["net"].train(s["X"], s["T"], s["M"], epochs=1, batch=case["batch"])
    return {"losses": losses, "params": s["net"].get_params()}


# ---- what a pass cannot do without ----

# FP64 operations of one pair and process where it is open in full, and on
# average over the pairs that _pairs draws (+, -, x, / and sqrt as one, log and
# exp as 19 and 20)
PAIR_FLOPS = {"bremsstrahlung": 72, "pair_production": 1201, "photonuclear": 932, "ionisation": 47}
MLP_FLOPS = 2 * sum(i * o for i, o in LAYERS)


def work(case):
    kind = case["kind"]
    n = case.get("n", 0)
    if kind in ("map", "batch"):
        if kind == "batch":
            n = _batch_of(case["elements"], case["log2_min"], case["log2_max"])[1][-1]
        names = PROCESSES if case.get("process", "all") == "all" else (case["process"],)
        out = 8 if case["precision"] == "f64" else 4
        return {"bytes": n * (16 + out * len(names)), "flops": n * sum(PAIR_FLOPS[p] for p in names)}
    if kind == "recoil":  # q above K / 20: pair production nearly always open, photonuclear on ~60%
        nodes = -(-case["min_points"] // 6) * 6
        return {"bytes": n * 72, "flops": n * nodes * 4400}
    if kind == "coulomb":  # data ~150, transport ~120; ~20 objective evaluations of ~110 per element
        nel = case["elements"]
        return {"bytes": n * (8 + nel * 8 * 15 + 16), "flops": n * nel * (150 + 120 + 20 * 110)}
    if kind == "soft":  # 102 nodes: a photonuclear integral where open, and the ratio's three logarithms
        return {"bytes": n * 16, "flops": n * 102 * 1200}
    if kind == "pumas":  # per node and element: bremsstrahlung ~200, pair ~8400, photonuclear ~3600; the
        nx = pumas.n_table_dcs(case["cutoff"])  # envelope's search ~150 interpolations of ~100 a row
        rows = case["elements"] * n
        return {"bytes": rows * 3 * (nx * 8 + 8), "flops": rows * (nx * 12200 + 3 * 150 * 100)}
    if kind == "surrogate":
        return {"bytes": n * 32, "flops": n * (MLP_FLOPS + 400)}
    steps = n // case["batch"]
    return {"bytes": steps * (case["batch"] * 44 + 50564 * 24), "flops": steps * case["batch"] * 3 * MLP_FLOPS}


# ---- the same outputs in plain 64-bit torch ----

GL6 = ((0.03376524, 0.16939531, 0.38069041, 0.61930959, 0.83060469, 0.96623476),
       (0.08566225, 0.18038079, 0.23395697, 0.23395697, 0.18038079, 0.08566225))
GL8 = ((0.01985507, 0.10166676, 0.2372338, 0.40828268, 0.59171732, 0.7627662, 0.89833324, 0.98014493),
       (0.05061427, 0.11119052, 0.15685332, 0.18134189, 0.18134189, 0.15685332, 0.11119052, 0.05061427))
GL9 = ((0.0, -0.8360311073266358, 0.8360311073266358, -0.9681602395076261, 0.9681602395076261,
        -0.3242534234038089, 0.3242534234038089, -0.6133714327005904, 0.6133714327005904),
       (0.3302393550012598, 0.1806481606948574, 0.1806481606948574, 0.0812743883615744, 0.0812743883615744,
        0.3123470770400029, 0.3123470770400029, 0.2606106964029354, 0.2606106964029354))
# 12-point rule on [0, 1]: nodes and weights of the lower half, mirrored
_G12 = ((0.0092196828766404, 0.0479413718147625, 0.1150486629028477, 0.2063410228566913, 0.3160842505009099,
         0.4373832957442655),
        (0.0235876681932559, 0.0534696629976592, 0.0800391642716731, 0.1015837133615330, 0.1167462682691774,
         0.1245735229067014))
GL12 = (_G12[0] + tuple(1.0 - x for x in reversed(_G12[0])), _G12[1] + tuple(reversed(_G12[1])))


class _El:
    """An element's values, as floats or one value per pair."""

    def __init__(self, Z, A, I):
        as_t = lambda v: v if torch.is_tensor(v) else torch.tensor(float(v), dtype=F64, device=DEV)  # noqa: E731
        self.Z, self.A, self.I = as_t(Z), as_t(A), as_t(I)
        self.H = self.Z == 1

    def pick(self, h, other):
        return torch.where(self.H, torch.as_tensor(h, dtype=F64, device=DEV), torch.as_tensor(other, dtype=F64, device=DEV))

    def at(self, i):
        sub = lambda v: v[i] if v.dim() else v  # noqa: E731
        return _El(sub(self.Z), sub(self.A), sub(self.I))


def _brems(K, q, e, m):
    BZn = e.pick(202.4, 182.7 * e.Z ** (-1. / 3.))
    BZe = e.pick(446., 1429. * e.Z ** (-2. / 3.))
    Dn = 1.54 * e.A ** 0.27
    sq = 1.648721271
    E = K + m
    nu = q / E
    delta = 0.5 * m * m / E * nu / (1. - nu)
    Pn = torch.log(BZn * (m + delta * (Dn * sq - 2.)) / (Dn * (ME + delta * sq * BZn))).clamp_min(0.)
    Pe = torch.log(BZe * m / ((1. + delta * m / (ME * ME * sq)) * (ME + delta * sq * BZe))).clamp_min(0.)
    Pe = torch.where(q < E / (1. + 0.5 * m * m / (ME * E)), Pe, torch.zeros_like(Pe))
    r = 7.297182E-07 * (5.63588E-13 * ME / m) ** 2 * e.Z * (e.Z * Pn + Pe) * (4. / 3. * (1. / nu - 1.) + nu)
    return r.clamp_min(0.) * 1E+03 * NA / e.A


def _ion(K, q, e, m):
    P2, E = K * (K + 2. * m), K + m
    Wmax = 2. * ME * P2 / (m * m + ME * (ME + 2. * E))
    on = ~((Wmax < 0.05 * K) | (q > Wmax) | (q <= 0.62 * e.I))
    cs = 1.535336E-05 * E * e.Z / e.A * (0.5 / P2 + 1. / q * (-1. / Wmax + E * E / P2 / q))
    L1 = torch.log(1. + 2. * q / ME)
    d = 1.16141E-03 * L1 * (torch.log(4. * E * (E - q) / (m * m)) - L1)
    d = torch.where(K >= 0.5 * (m - ME) ** 2 / ME, d, torch.zeros_like(d))
    return torch.where(on, cs * (1. + d), torch.zeros_like(cs))


def _pair_on(K, q, e, m):
    Z13 = e.Z ** (1. / 3.)
    gamma = 1. + K / m
    x0 = 4. * ME / q
    x1 = 6. / (gamma * (gamma - q / m))
    arg = (x0 + 2. * (1. - x0) * x1) / (1. + (1. - x1) * torch.sqrt((1. - x0).clamp_min(0.)))
    on = (q > 4. * ME) & (q < K + m * (1. - 0.75 * 1.6487212707 * Z13)) & (arg < 1.) & (arg > 0.)
    return on, arg, gamma, Z13


def _pair(K, q, e, m):
    on, arg, gamma, Z13 = _pair_on(K, q, e, m)
    nu = q / (K + m)
    beta = 0.5 * nu * nu / (1. - nu)
    r = m / ME
    xf = 0.5 * r * r * beta
    AZ = e.pick(202.4, 183.) / Z13
    cL = 2. * 1.6487212707 * ME * AZ
    cLe = 2.25 * Z13 * Z13 / (r * r)
    tmin = torch.log(arg)
    I = 0.
    for t, w in zip(*GL8):
        eps = torch.exp(t * tmin)
        rho = 1. - eps
        r2 = rho * rho
        r21 = eps * (2. - eps)
        xi = xf * r21
        Be = torch.where(xi >= 1E+03, 0.5 / xi * ((3. - r2) + 2. * beta * (1. + r2)),
                         ((2. + r2) * (1. + beta) + xi * (3. + r2)) * torch.log(1. + 1. / xi) +
                         (r21 - beta) / (1. + xi) - 3. - r2)
        Ye = (5. - r2 + 4. * beta * (1. + r2)) / (2. * (1. + 3. * beta) * torch.log(3. + 1. / xi) - r2 -
                                                  2. * beta * (2. - r2))
        xe = (1. + xi) * (1. + Ye)
        Le = torch.log(AZ * torch.sqrt(xe) * q / (q + cL / r21 * xe)) - 0.5 * torch.log(1. + cLe * xe)
        Bm = torch.where(xi <= 1E-03, 0.5 * xi * (5. - r2 + beta * (3. + r2)),
                         ((1. + r2) * (1. + 1.5 * beta) - 1. / xi * (1. + 2. * beta) * r21) * torch.log(1. + xi) +
                         xi * (r21 - beta) / (1. + xi) + (1. + 2. * beta) * r21)
        Ym = (4. + r2 + 3. * beta * (1. + r2)) / ((1. + r2) * (1.5 + 2. * beta) * torch.log(3. + xi) + 1. - 1.5 * r2)
        Lm = torch.log(r * AZ * q / (1.5 * Z13 * (q + cL / r21 * ((1. + xi) * (1. + Ym)))))
        I = I - ((Be * Le).clamp_min(0.) + (Bm * Lm).clamp_min(0.) / (r * r)) * (1. - rho) * tmin * w
    zeta = 0.073 * torch.log(gamma / (1. + e.pick(4.4E-05, 1.95E-05) * gamma * Z13 * Z13)) - 0.26
    z2 = 0.058 * torch.log(gamma / (1. + e.pick(4.8E-05, 5.30E-05) * gamma * Z13)) - 0.14
    zeta = torch.where((gamma > 35.) & (zeta > 0.), zeta / z2, torch.zeros_like(zeta))
    d = 1.794664E-34 * e.Z * (e.Z + zeta) * (K + m - q) * I / (q * (K + m))
    return torch.where(on, d.clamp_min(0.) * 1E+03 * NA * (m + K) / e.A, torch.zeros_like(d))


def _photo_on(K, q, m):
    M, mpi = 0.931494, 0.134977
    E = K + m
    y = q / E
    lo, hi = m * m * y * y / (1. - y), 2. * M * (q - mpi) - mpi * mpi
    on = (q >= 1.) & (q >= 2E-03 * K) & (q < E - m) & (q > mpi * (1. + 0.5 * mpi / M)) & (hi >= lo) & (lo >= 0)
    return on, lo, hi


def _allm(x, Q2, M2):
    W2 = Q2 * (1. / x - 1.)  # W^2 - M^2
    t = torch.log(torch.log((Q2 + 0.52544) / 0.06527) / math.log(0.52544 / 0.06527))
    xP, xR = (Q2 + 49.457) / (Q2 + 49.457 + W2), (Q2 + 0.15052) / (Q2 + 0.15052 + W2)
    cP = 0.28067 + (0.28067 - 0.22291) * (1. / (1. + t ** 2.1979) - 1.)
    aP = -0.0808 + (-0.0808 + 0.44812) * (1. / (1. + t ** 1.1709) - 1.)
    bP = 0.36292 + 1.8917 * t ** 1.8439
    cR, aR, bR = 0.80107 + 0.97307 * t ** 3.4942, 0.58400 + 0.37888 * t ** 2.6063, 0.01147 + 3.7582 * t ** 0.49338
    l1x = torch.log(1. - x)
    return Q2 / (Q2 + 0.31985) * (cP * torch.exp(aP * torch.log(xP) + bP * l1x) +
                                  cR * torch.exp(aR * torch.log(xR) + bR * l1x))


def _photo(K, q, e, m):
    on, lo, hi = _photo_on(K, q, m)
    E = K + m
    y = q / E
    l0, l1 = torch.log(lo), torch.log(hi)
    ds = 0.
    for t, w in zip(*GL9):
        Q2 = torch.exp(0.5 * (l1 + l0) + 0.5 * (l1 - l0) * t)
        x = 0.5 * Q2 / (0.931494 * q)
        F2 = _allm(x, Q2, None)
        a = torch.where(x < 0.0014, torch.exp(-0.1 * torch.log(e.A)) + 0. * x,
                        torch.where(x < 0.04, torch.exp((0.069 * torch.log10(x) + 0.097) * torch.log(e.A)),
                                    torch.ones_like(x)))
        F2 = 0.5 * e.A * a * (2. + x * (-1.85 + x * (2.45 + x * (-2.35 + x)))) * F2
        q2 = Q2.clamp_min(0.3)
        th = 1. + 12. * q2 / (1. + q2) * 0.015625 / (0.015625 + x * x)
        R = 0.635 / torch.log(q2 / 0.04) * th + 0.5747 / q2 - 0.3534 / (0.09 + q2 * q2)
        dd = (1. - y + 0.5 * (1. - 2. * m * m / Q2) * (y * y + Q2 / (E * E)) / (1. + R)) / (Q2 * Q2) - 0.25 / (E * E * Q2)
        ds = ds + 2.603096E-35 * F2 * dd / q * Q2 * w
    ds = ds.clamp_min(0.) * 0.5 * (l1 - l0) * 1E+03 * NA * (m + K) / e.A
    return torch.where(on, ds, torch.zeros_like(ds))


def _all_dcs(K, q, e, m, which=PROCESSES, chunk=1 << 21):
    """The processes of `which` over pairs, the two integrals only where open."""
    full = {"bremsstrahlung": _brems, "ionisation": _ion}
    out = []
    for name in which:
        parts = []
        for a in range(0, K.numel(), chunk):
            k, x, el = K[a:a + chunk], q[a:a + chunk], e.at(slice(a, a + chunk))
            if name in full:
                parts.append(full[name](k, x, el, m))
                continue
            i = torch.nonzero(_pair_on(k, x, el, m)[0] if name == "pair_production" else _photo_on(k, x, m)[0])[:, 0]
            r = torch.zeros_like(k)
            if i.numel():
                r[i] = (_pair if name == "pair_production" else _photo)(k[i], x[i], el.at(i), m)
            parts.append(r)
        out.append(torch.cat(parts))
    return out


def _exact_recoil(K, e, m, min_points, xlow=0.05):
    itv = -(-min_points // 6)
    E = K + m
    dels, cels = [torch.zeros_like(K) for _ in range(4)], [torch.zeros_like(K) for _ in range(4)]
    lb, ub = torch.log(K * xlow), torch.log(K)
    h = (ub - lb) / itv
    for i in range(itv):
        for x, w in zip(*GL6):
            q = torch.exp(lb + h * (i + x))
            for p, d in enumerate(_all_dcs(K, q, e, m)):
                dels[p] += d * q * h * w / E
                cels[p] += d * q * q * h * w / E
    P2 = K * (K + 2. * m)
    Wmax = 2. * ME * P2 / (m * m + ME * (ME + 2. * E))
    Wmin = torch.maximum(0.62 * e.I + 0. * K, K * xlow)
    a0, a1, a2 = 0.5 / P2, -1. / Wmax, E * E / P2
    L = torch.log(Wmax / Wmin)
    f = 1.535336E-05 * e.Z / e.A
    low = K <= 0.5 * (m - ME) ** 2 / ME
    off = (Wmax < 0.05 * K) | (Wmax <= Wmin)
    for dst, v in ((dels, a0 * (Wmax - Wmin) + a1 * L + a2 * (1. / Wmin - 1. / Wmax)),
                   (cels, 0.5 * a0 * (Wmax * Wmax - Wmin * Wmin) + a1 * (Wmax - Wmin) + a2 * L)):
        dst[3] = torch.where(low, torch.where(off, torch.zeros_like(v), f * v), dst[3])
    return {"del": dels, "cel": cels}


def _coulomb_one(K, Z, A, m):
    Ma = A * 0.931494
    si = 1. / torch.sqrt((m + Ma) ** 2 + 2. * Ma * K)
    et = K + m + Ma
    b2 = K * (K + 2. * m) / (et * et)
    fCM = torch.stack([et * si, torch.sqrt((m / Ma) ** 2 * (1. - b2) + b2)], 1)
    k0 = ((K * Ma + m * (m + Ma)) * si - m).clamp_min(1E-9)
    e = k0 + m
    p2 = k0 * (k0 + 2. * m)
    d = 5.8406E-02 / p2
    s1, s2 = d / (1.02934 * A ** (1. / 3) + 0.435) ** 2, d / 4.
    z2 = 5.3251346E-05 * (Z * e) ** 2 / p2
    f = sum(z2 / (i * (i * i + z2)) for i in range(1, 11 + Z))
    cK = torch.where(z2 > 1., torch.exp(f), torch.exp(1. - 1. / (1. + z2) + z2 * (0.2021 + z2 * (0.0083 * z2 - 0.0369))))
    r = (k0 / e) ** 2
    s0 = 5.179587126E-12 * Z ** (2. / 3.) * (r * cK + (1. - r) * (1. + 3.34 * z2)) / p2
    d01, d02, d12 = 1. / (s0 - s1), 1. / (s0 - s2), 1. / (s1 - s2)
    s6, s7, s8 = (d01 * d02) ** 2, (d01 * d12) ** 2, (d12 * d02) ** 2
    S = torch.stack([s0, s1, s2, 2. * s6 * (d01 + d02), 2. * s7 * (d12 - d01), -2. * s8 * (d12 + d02), s6, s7, s8], 1)
    dw = p2 / (Z * e)
    return fCM, S, k0 * (e + m) / (e * e), 1. / (A * 2.54910918E+08 * s0 * (1. + s0) * dw * dw)


def _transport(S, fs, mu):
    s0, s1, s2 = S[:, 0], S[:, 1], S[:, 2]
    L, r, k = torch.log(1. + mu / s0), mu / (mu + s0), s0 * (1. + s0)
    a0 = k * (r / s0 - fs * (L - r))
    a1 = 2. * k * (L - r - fs * (mu - s0 * (r - 2. * L)))
    g0 = g1 = 0.
    for i in range(3):
        s = S[:, i]
        r, L = mu / (mu + s), torch.log(1. + mu / s)
        I0, I1, I2 = r / s, L - r, mu - 2. * L * s + r * s
        J0, J1, J2 = L, mu - L * s, 0.5 * mu * mu + L * s * s - mu * s
        g0 = g0 + S[:, 3 + i] * (J0 - fs * J1) + S[:, 6 + i] * (I0 - fs * I1)
        g1 = g1 + S[:, 3 + i] * (J1 - fs * J2) + S[:, 6 + i] * (I1 - fs * I2)
    c = k * s1 * s1 * s2 * s2
    point = mu < 1E-08 * torch.minimum(s1, s2)
    return torch.stack([torch.where(point, a0, g0 * c), torch.where(point, a1, g1 * 2. * c)], 1)


def _restricted(mu, S, fs):
    s0, s1, s2 = S[:, 0], S[:, 1], S[:, 2]
    k = s0 * (1. + s0)
    L, r = torch.log((s0 + 1.) / (s0 + mu)), (1. - mu) / ((s0 + mu) * (s0 + 1.))
    a = k * (r - fs * (L - s0 * r))
    cs = 0.
    for i in range(3):
        s = S[:, i]
        L, r = torch.log((s + 1.) / (s + mu)), (1. - mu) / ((s + mu) * (s + 1.))
        cs = cs + S[:, 3 + i] * (L - fs * (mu - s * L)) + S[:, 6 + i] * (r - fs * (L - s * r))
    v = torch.where(mu < 1E-08 * torch.minimum(s1, s2), a, k * s1 * s1 * s2 * s2 * cs)
    return torch.where(mu >= 1., torch.zeros_like(v), v)


def _exact_coulomb(K, els, m):
    per = [_coulomb_one(K, Z, A, m) for Z, A, _ in els]
    one = torch.ones_like(K)
    G = [_transport(S, fs, one) for _, S, fs, _ in per]
    inv_m, inv1, sl, sh = 0., 0., 0., 0.
    for (fCM, S, fs, il), g in zip(per, G):
        inv_m, sh, sl = inv_m + il * g[:, 0], sh + S[:, 0] * il, sl + il / S[:, 0]
        inv1 = inv1 + il * g[:, 1] / (fCM[:, 0] * (1. + fCM[:, 1])) ** 2
    lb_m = 1. / inv_m
    lb = (1E-4 / inv1).clamp_max(1E+9)
    hard = lb_m < lb
    sm = torch.where(lb > 2. * lb_m, sh * lb_m, 1. / (sl * lb_m))
    mu0 = sm * (lb - lb_m) / (sm * lb + lb_m)
    obj = lambda mu: sum(il * _restricted(mu, S, fs) for _, S, fs, il in per) - 1. / lb  # noqa: E731
    top = 0.5 * (1. - math.cos(math.pi / 180.))
    hi, lo = (4. * mu0).clamp_max(1.), 0.25 * mu0
    f_hi = obj(hi)
    keep = f_hi > 0.  # the estimates stay
    f_lo = obj(lo)
    down = f_lo < 0.
    hi, lo, f_hi = torch.where(down, lo, hi), torch.where(down, 0. * lo, lo), torch.where(down, f_lo, f_hi)
    f_lo = obj(lo)
    root = lo < top
    a, b = lo, hi.clamp_max(top)
    bracket = root & ~(f_lo * f_hi > 0)
    for _ in range(90):
        c = 0.5 * (a + b)
        up = obj(c) > 0.  # the objective falls with mu
        a, b = torch.where(up, c, a), torch.where(up, b, c)
    mu = torch.where(bracket, 0.5 * (a + b), mu0).clamp_max(top)
    cs = obj(mu) + 1. / lb
    lbh = torch.where(cs <= 1E-9, torch.full_like(cs, 1E+9), 1. / cs)
    mu, lbh = torch.where(keep, mu0, mu), torch.where(keep, lb, lbh)
    return {"fCM": torch.stack([p[0] for p in per]), "screening": torch.stack([p[1] for p in per]),
            "fspin": torch.stack([p[2] for p in per]), "invlambda": torch.stack([p[3] for p in per]),
            "G": torch.stack(G), "mu0": torch.where(hard, mu, torch.zeros_like(mu)),
            "lb_h": torch.where(hard, lbh, lb_m)}


def _exact_soft(K, e, m):
    E = K + m
    p2 = K * (K + 2. * m)
    Wmax = 2. * ME * p2 / (m * m + ME * (ME + 2. * E))
    W0 = 2. * p2 / ME
    top = Wmax / W0
    mu3, mu2 = torch.minimum(K * 0.05 / W0, top), 0.62 * e.I / W0
    t = 2. * 1.535336E-05 / e.A * e.Z * (0.25 * W0 / p2 * (mu3 * mu3 - mu2 * mu2) - (mu3 - mu2) / Wmax +
                                         E * E / (W0 * p2) * torch.log(mu3 / mu2))
    t = torch.where(mu2 >= mu3, torch.zeros_like(t), t)
    h = -math.log(1E-06) / 17
    acc = 0.
    for i in range(17):
        for x, w in zip(*GL6):
            nu = 0.05 * math.exp(math.log(1E-06) + h * (i + x))
            q = nu * K
            q2, hi, lo = q * q, 1.876544 * q, q * q * m * m / (E * (E - q))
            b, c = 1. / (1. - q2 / 0.4), 1. / (1. - 0.4 / q2)
            L1, L2 = b * torch.log((q2 + hi) / (q2 + lo)), c * torch.log((0.4 + hi) / (0.4 + lo))
            I0 = torch.log(hi / lo) - L1 - L2
            I1 = L1 * q2 + L2 * 0.4
            I2 = (hi - lo) * (b * q2 + c * 0.4) - L1 * q2 * q2 - L2 * 0.16
            ratio = (I1 * hi - I2) / ((I0 * hi - I1) * K * (K + 2. * m))
            acc = acc + _all_dcs(K, q, e, m, ("photonuclear",))[0] * ratio * nu * h * w
    return t + 2. * acc


# the radiation logarithms of the PUMAS models, by Z; 182.7 elsewhere
_RL = dict(zip(list(range(1, 23)) + [26, 29, 32, 35, 42, 50, 53, 74, 82, 92],
               (202.4, 151.9, 159.9, 172.3, 177.9, 178.3, 176.6, 173.4, 170.0, 165.8, 165.8, 167.1, 169.1, 170.8, 172.2,
                173.4, 174.3, 174.8, 175.1, 175.6, 176.2, 176.8, 175.8, 173.1, 173.0, 173.5, 175.9, 177.4, 178.6, 177.6,
                178.0, 179.8)))
PM = 0.5 * (0.938272 + 0.939565)
PPI = 0.13957018
ALPHA = 7.2973525693E-03


def _li2(x):
    """The dilogarithm on (0, 1), by its series and the reflection."""
    small = x <= 0.5
    y = torch.where(small, x, 1. - x)
    s, p = torch.zeros_like(y), torch.ones_like(y)
    for k in range(1, 60):
        p = p * y
        s = s + p / (k * k)
    other = math.pi ** 2 / 6 - torch.log(x.clamp_min(1e-300)) * torch.log((1. - x).clamp_min(1e-300)) - s
    return torch.where(small, s, other)


def _pumas_dcs(p, Z, A, m, K, q):
    """The atomic DCS in m^2/kg of one process and element, zero where closed."""
    rl = _RL.get(int(Z), 182.7)
    z13, me, mm = Z ** (1. / 3.), 0.5109989461, m * 1E+03
    dn, re, sqe = 1.54 * A ** 0.27, 2.8179403227E-13, 1.648721270700128
    energy = (K + m) * 1E+03
    v = q / (K + m)
    if p == 0:
        on = q < K + m * (1. - 0.75 * sqe * z13)
        d = mm * mm * v / (2. * energy * (1. - v))
        rz, r1 = rl / z13, 446. if Z == 1 else 1429.
        e = math.exp
        phi1 = torch.log(rz * (mm / me) / (1. + rz * e(0.5) * d / me))
        phi2 = torch.log(rz * e(-1. / 6.) * (mm / me) / (1. + rz * e(1. / 3.) * d / me))
        mq = mm / (105.6583745 * e(1.) / dn)
        rho = math.sqrt(1. + 4. * mq * mq)
        lr = math.log((rho + 1.) / (rho - 1.))
        phi1 = phi1 - (math.log(mq) + 0.5 * rho * lr) * (1. - 1. / Z)
        phi2 = phi2 - (math.log(mq) + 0.25 * (3. * rho - rho ** 3) * lr + 2. * mq * mq) * (1. - 1. / Z)
        s1 = torch.log(mm / d / (mm * d / (me * me) + sqe))
        s2 = torch.log(1. + me / (d * r1 / (z13 * z13) * sqe))
        sa = (4. / 3. * (1. - v) + v * v) * (s1 - s2)
        t, lv = torch.log(1. - v), torch.log(v)
        sr = torch.where(v < 0.02, -0.00349 + 148.84 * v - 987.531 * v * v, torch.where(
            v < 0.1, 0.1642 + 132.573 * v - 585.361 * v * v + 1407.77 * v ** 3, torch.where(
                v < 0.9, -2.8922 - 19.0156 * v + 57.698 * v * v - 63.418 * v * lv + 14.1166 * t + 1.84206 * t * t,
                2134.19 + 581.823 * v - 2708.85 * v * v + 4767.05 * v * lv + 1.52918 * t + 0.361933 * t * t)))
        r = (2. - 2. * v + v * v) * phi1 - 2. / 3. * (1. - v) * phi2 + sa / Z + 0.25 * ALPHA * phi1 * sr
        out = (2 * (me / mm) * re * Z) ** 2 * (ALPHA / q) * r * 1E-04
        on = on & (r > 0)
    elif p == 1:
        gamma = 1. + K / m
        x0, x1 = 1. - 4. * ME / q, 1. - 6. / (gamma * (gamma - q / m))
        ri = 1. - torch.sqrt(x0.clamp_min(0.)) * x1
        on = (q > 4. * ME) & (q < K + m * (1. - 0.75 * 1.6487212707 * z13)) & (x0 > 0) & (x1 > 0) & (ri > 0) & (ri < 1)
        tmin = torch.log(ri)
        g1, g2 = (4.4E-05, 4.8E-05) if Z == 1 else (1.95E-05, 5.3E-05)
        ze1 = 0.073 * torch.log(energy / mm / (1. + g1 * z13 * z13 * energy / mm)) - 0.26
        ze2 = 0.058 * torch.log(energy / mm / (1. + g2 * z13 * energy / mm)) - 0.14
        zeta = torch.where((ze1 > 0) & (ze2 > 0), ze1 / ze2, torch.zeros_like(ze1))
        pref = 4. / (3. * math.pi) * Z * (ALPHA * re) ** 2 * (Z + zeta) * (1. - v) / v
        beta = v * v / (2. * (1. - v))
        out = 0.
        for x, w in zip(*GL12):
            eps = torch.exp(x * tmin)
            rho = 1. - eps
            r2 = rho * rho
            o = 1. - r2
            xi = (mm * v / (2. * me)) ** 2 * o / (1. - v)
            u = 1. + xi
            c05, c13 = (2. * me * math.exp(k) * rl / z13 * u / (energy * v * o) for k in (0.5, 1. / 3.))
            li = torch.log(1. + 1. / xi)
            Pe = (2. + r2) * (1. + beta) + xi * (3. + r2)
            Be = Pe * li + (1. - r2 - beta) / u - (3. + r2)
            C2 = (o * (1. + beta) + xi * (3. - r2)) * li + 2. * (1. - beta - r2) / u - (3. - r2)
            De = Pe * _li2(1. / u) - (2. + r2) * xi * li - (xi + r2 + beta) / u
            sx = rl / z13 * torch.sqrt(u)
            rr = De / Be

            def Le(f, c, g):
                X, Y = torch.where(rr < 100, torch.exp(-rr), 0. * rr), torch.where(rr > -100, torch.exp(rr), 0. * rr)
                k = (me / mm * dn) ** 2 * g * u
                return torch.where(rr > 0, torch.log(f * sx / (X + c)) - rr - 0.5 * torch.log(X + k),
                                   torch.log(f * sx / (1. + Y * c)) - 0.5 * rr - 0.5 * torch.log(1. + Y * k))
            de = pref * ((Be - C2) * Le(1., c05, 1.) + C2 * Le(math.exp(-1. / 6.), c13, math.exp(-1. / 3.)))
            lx, b15 = torch.log(u), 1. + 1.5 * beta
            Pm = (1. + r2) * b15 - (1. + 2. * beta) * o / xi
            Bm = Pm * lx + xi * (1. - r2 - beta) / u + (1. + 2. * beta) * o
            C2 = ((1. - beta) * o - xi * (1. + r2)) * lx / xi - 2. * (1. - beta - r2) / u + 1. - beta - (1. + beta) * r2
            Dm = Pm * _li2(xi / u) + b15 * o / xi * lx + (1. - r2 - beta / 2. * (1. + r2) + o / (2. * xi) * beta) * xi / u
            num = mm / me * rl / z13 / dn
            rm = Dm / Bm

            def Lm(c):
                X, Y = torch.where(rm < 100, torch.exp(-rm), 0. * rm), torch.where(rm > -100, torch.exp(rm), 0. * rm)
                return torch.where(rm > 0, torch.log(num / (X + c)) - rm, torch.log(num / (1. + c * Y)))
            dm = pref * (me / mm) ** 2 * ((Bm - C2) * Lm(c05) + C2 * Lm(c13))
            out = out - (de.clamp_min(0.) + dm.clamp_min(0.)) * 1E-01 / energy * eps * w * tmin
    else:
        lo, hi = m * m * (q * q - 0.5 * m * m) / ((K + m) * (K + m - q)), 2. * PM * (q - PPI) - PPI * PPI
        on = (q > PPI + 0.5 * PPI * PPI / PM) & (q < K + m - 0.5 * (PM + m * m / PM)) & (hi >= lo) & (lo >= 0)
        l0, dx = torch.log(lo), torch.log(hi) - torch.log(lo)
        E = K + m
        out = 0.
        for t, w in zip(*GL9):
            Q2 = torch.exp(l0 + dx * 0.5 * (1. + t))
            x = 0.5 * Q2 / (PM * q)
            F2 = _allm(x, Q2, None)
            if Z != 1:
                F2 = F2 * torch.where(x < 0.0014, math.exp(-0.1 * math.log(A)) + 0. * x, torch.where(
                    x < 0.04, torch.exp((0.069 * torch.log10(x) + 0.097) * math.log(A)), torch.ones_like(x)))
            F2 = F2 * (Z + (A - Z) * (1. + x * (-1.85 + x * (2.45 + x * (-2.35 + x)))))
            dd = (1. - v + 0.5 * (1. - 2. * m * m / Q2) * (v * v + Q2 / (E * E))) / (Q2 * Q2) - 0.25 / (E * E * Q2)
            f = 4 * math.pi * (ALPHA * 1.973269804E-16) ** 2 * F2 * dd / q
            out = out + f.clamp_min(0.) * 0.5 * w * dx * Q2
    out = torch.where(on, out, torch.zeros_like(out)).clamp_min(0.)
    return out * 1E+03 * NA * (m + K) / A


def _pchip(x, y):
    """Slopes of rows y [r, n] over x [n]: a linear first bin, then PCHIP."""
    h = x[1:] - x[:-1]
    s = (y[:, 1:] - y[:, :-1]) / h
    d = torch.zeros_like(y)
    n = y.shape[1]
    if n == 1:
        return d
    if n <= 3:
        d[:, 0] = s[:, 0]
        d[:, 1:] = s[:, -1:]
        return d
    d[:, 0] = s[:, 0]
    a = (h[1:-1] + 2 * h[2:]) / (3 * (h[1:-1] + h[2:]))
    p = s[:, 1:-1] * s[:, 2:]
    d[:, 2:-1] = torch.where(p > 0, p / ((1 - a) * s[:, 1:-1] + a * s[:, 2:]), torch.zeros_like(p))
    for i, (j, k) in ((1, (2, 3)), (n - 1, (n - 2, n - 3))):
        h1, h2 = x[j] - x[i], x[k] - x[i]
        D = h1 * h2 * (h2 - h1)
        c1, c2 = h2 * h2 / D, -h1 * h1 / D
        d[:, i] = -(c1 + c2) * y[:, i] + c1 * y[:, j] + c2 * y[:, k]
    return d


def _exact_pumas(K, Zs, As, m, cutoff):
    n = 20
    mm = max(int(math.log10(0.6 / cutoff) * 15), 10)
    n += mm
    xs = [math.log(cutoff) + i * math.log(0.6 / cutoff) / (mm - 1) for i in range(mm)]
    dx = math.log((0.95 - 0.6) / 1E-03) / 20
    x = torch.tensor(xs + [math.log(0.95 - 1E-03 * math.exp((n - 1 - j) * dx)) for j in range(mm, n)], dtype=F64, device=DEV)
    table = torch.zeros(3, len(Zs), K.numel(), n, 2, dtype=F64, device=DEV)
    q = K[:, None] * torch.exp(x)[None, :]
    for e, (Z, A) in enumerate(zip(Zs, As)):
        for p in range(3):
            d = _pumas_dcs(p, Z, A, m, K[:, None].expand_as(q), q)
            on = d > 0
            first = torch.where(on.any(1), on.float().argmax(1), torch.full((q.shape[0],), n, device=DEV))
            j = torch.arange(n, device=DEV)[None, :]
            ends = ((~on) & (j > first[:, None])).float()
            last = torch.where(ends.any(1), ends.argmax(1) - 1, torch.full_like(first, n - 1))
            y = torch.log(d.clamp_min(1e-300))
            for a, b in sorted(set(zip(first.tolist(), last.tolist()))):
                if a >= n:
                    continue
                r = torch.nonzero((first == a) & (last == b))[:, 0]
                table[p, e, r, a:b + 1, 0] = y[r, a:b + 1]
                table[p, e, r, a:b + 1, 1] = _pchip(x[a:b + 1], y[r, a:b + 1])
    return table, x, None


def _split_params(p):
    p = torch.as_tensor(p, device=DEV).to(F64)
    out, k = [], 0
    for i, o in LAYERS:
        out.append([p[k:k + i * o].reshape(o, i).clone(), p[k + i * o:k + i * o + o].clone()])
        k += i * o + o
    return out


def _net(layers, X):
    for w, b in layers[:-1]:
        X = torch.nn.functional.silu(X @ w.T + b)
    return X @ layers[-1][0].T + layers[-1][1]


def _mix64(z):
    with np.errstate(over="ignore"):
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return z ^ (z >> np.uint64(31))


def _exact_surrogate(case, seed):
    d = np.load(CHECKPOINT, allow_pickle=False)
    els = torch.tensor(d["elements"], dtype=F64, device=DEV)  # A, I, Z
    nel = els.shape[0]
    n = case["n"]
    counts = torch.full((nel,), n // nel, device=DEV)
    counts[:n % nel] += 1
    of = torch.repeat_interleave(torch.arange(nel, device=DEV), counts)
    K, q = _pairs(n, seed)
    e = _El(els[of, 2], els[of, 0], els[of, 1])
    true = _all_dcs(K, q, e, MUON)
    nu = q / K
    inside = (K >= 1e-3) & (K <= 1e6) & (nu >= 1e-6) & (nu < 1.)
    lk, ln = torch.log10(K), torch.log10(nu)
    a, b, z = (lk - 1.5) / 4.5, (ln + 3.) / 3., e.Z / 46. - 1.
    err = torch.tensor(d["cell_err"].astype(np.float32), device=DEV)
    bad = (err > 0.5 * case["tol"]) | (err < 0)
    bins = err.shape[-1]
    ik, iq = ((lk + 3.) / 9. * bins).long().clamp(0, bins - 1), ((ln + 6.) / 6. * bins).long().clamp(0, bins - 1)
    recheck = torch.tensor(_mix64(np.arange(n, dtype=np.uint64)) % np.uint64(1000) < 10, device=DEV)
    layers = _split_params(d["params"])
    Y = torch.cat([_net(layers, torch.stack([a, b, z], 1)[i:i + (1 << 19)]) for i in range(0, n, 1 << 19)])
    phi = torch.stack([a, b, a * a, b * b, a * b, a ** 3, b ** 3, a * a * b, a * b * b, z, z * a, z * b, z * z], 1)
    trend = torch.tensor(d["trend"], dtype=F64, device=DEV)
    out = []
    for p in range(4):
        net = torch.exp(float(d["mean"][p]) + phi @ trend[p] + float(d["std"][p]) * Y[:, p] - torch.log(e.A))
        exact_here = bad[p][of, ik, iq] | recheck | ~inside
        v = torch.where(exact_here, true[p], net)
        out.append(torch.where(true[p] > 0, v, torch.zeros_like(v)))
    return {"out": out, "counters": None}


def _order(n, epoch=0, seed=0):
    """The keyed order in which an epoch visits its rows: a 4-round Feistel
    network over the smallest even number of bits, walked back into [0, n)."""
    M = 0xFFFFFFFF

    def fmix(x):
        x = x ^ (x >> 16)
        x = (x * 0x85EBCA6B) & M
        x = x ^ (x >> 13)
        x = (x * 0xC2B2AE35) & M
        return x ^ (x >> 16)
    bits = 1
    while (1 << bits) < n:
        bits += 1
    half = (bits + 1) // 2
    mask = (1 << half) - 1
    keys = [fmix((seed & M) ^ fmix((seed >> 32) ^ fmix(epoch * 4 + i + 1))) for i in range(4)]
    y = np.arange(n, dtype=np.uint64)
    todo = np.ones(n, dtype=bool)
    while todo.any():
        L, R = y[todo] >> np.uint64(half), y[todo] & np.uint64(mask)
        for k in keys:
            x = R ^ np.uint64(k)
            x = x ^ (x >> np.uint64(16))
            x = (x * np.uint64(0x85EBCA6B)) & np.uint64(M)
            x = x ^ (x >> np.uint64(13))
            x = (x * np.uint64(0xC2B2AE35)) & np.uint64(M)
            x = x ^ (x >> np.uint64(16))
            L, R = R, L ^ (x & np.uint64(mask))
        y[todo] = (L << np.uint64(half)) | R
        todo[todo] = y[todo] >= n
    return torch.tensor(y.astype(np.int64), device=DEV)


def _exact_train(case, seed):
    X, T, M, p = _train_inputs(case, seed)
    X, T, M = X.to(F64), T.to(F64), M.to(F64)
    flat = torch.tensor(p, device=DEV).to(F64)
    m1, m2 = torch.zeros_like(flat), torch.zeros_like(flat)
    B, order = case["batch"], _order(case["n"])
    steps = case["n"] // B
    total = 0.
    for s in range(steps):
        i = order[s * B:(s + 1) * B]
        flat = flat.detach().requires_grad_(True)
        w, k = [], 0
        for a, o in LAYERS:
            w.append((flat[k:k + a * o].reshape(o, a), flat[k + a * o:k + a * o + o]))
            k += a * o + o
        loss = (((_net(w, X[i]) - T[i]) * M[i]) ** 2).sum() / (B * 4)
        g, = torch.autograd.grad(loss, flat)
        lr = 2e-5 + (2e-3 - 2e-5) * 0.5 * (1. + math.cos(math.pi * s / max(1, steps)))
        m1, m2 = 0.9 * m1 + 0.1 * g, 0.999 * m2 + 0.001 * g * g
        flat = flat.detach() - lr * (m1 / (1 - 0.9 ** (s + 1))) / (torch.sqrt(m2 / (1 - 0.999 ** (s + 1))) + 1e-8)
        total += float(loss)
    return {"losses": np.array([total / steps]), "params": flat.cpu().numpy()}


def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad() if kind != "train" else torch.enable_grad():
        if kind == "map":
            K, q = _pairs(case["n"], seed)
            which = PROCESSES if case["process"] == "all" else (case["process"],)
            r = _all_dcs(K, q, _El(*ELEMENTS[case["element"]]), _mass(case), which)
            return r if case["process"] == "all" else r[0]
        if kind == "batch":
            els, off = _batch_of(case["elements"], case["log2_min"], case["log2_max"])
            K, q = _pairs(off[-1], seed)
            t = torch.tensor(els, dtype=F64, device=DEV)
            of = torch.repeat_interleave(torch.arange(len(els), device=DEV), torch.tensor(np.diff(off), device=DEV))
            return _all_dcs(K, q, _El(t[of, 0], t[of, 1], t[of, 2]), MUON)
        if kind == "recoil":
            return _exact_recoil(_energies(case["n"], seed), _El(*ELEMENTS[case["element"]]), _mass(case),
                                 case["min_points"])
        if kind == "coulomb":
            return _exact_coulomb(_energies(case["n"], seed), _mixture(case["elements"]), _mass(case))
        if kind == "soft":
            return _exact_soft(_energies(case["n"], seed), _El(*ELEMENTS[case["element"]]), _mass(case))
        if kind == "pumas":
            els, _ = _batch_of(case["elements"])
            return _exact_pumas(_grid(case["n"], seed), [float(e[0]) for e in els], [e[1] for e in els], _mass(case),
                                case["cutoff"])
        if kind == "surrogate":
            return _exact_surrogate(case, seed)
        return _exact_train(case, seed)
