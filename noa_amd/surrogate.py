"""Learned surrogate of the four DCS processes, validated against and backed by
the exact FP64 kernel.

Pipeline (all on the GPU):
  1. dataset: seeded (K, q) pairs over an element batch, exact DCS from the
     FP64 kernel; features (log10 K, log10 nu, Z) and targets ln(A * DCS)
     standardised per process, masked where the DCS is zero;
  2. training: hand-written bf16 MFMA forward/backward and Adam
     (noa_dcs_mlp_train);
  3. validation on held-out pairs against the FP64 kernel, per element and
     per (log10 K, log10 nu) cell: cells whose worst relative error exceeds the
     tolerance are flagged, and flagged queries are evaluated exactly;
  4. inference: the fused register-resident MFMA kernel, exact FP64 fallback
     for flagged / out-of-domain / seeded-recheck queries.
"""
from __future__ import annotations

import ctypes
import os
import time

import numpy as np
import torch

from . import _lib, workload
from .batch import BatchPlan
from .physics import MUON_MASS

NPROC = 4
HERE = os.path.dirname(os.path.abspath(__file__))
CHECKPOINT = os.path.join(HERE, "surrogate_48el.npz")
MAP_BINS = 64
NO_SAMPLES = -1.0  # error-map value of a cell where the process had no non-zero validation sample
MIN_CELL_SAMPLES = 8  # fewer non-zero samples than this: the cell's worst error is unknown (+inf)


def _p(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _stream(dev):
    return ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)


class Network:
    """The MLP 3 -> 128 x4 (SiLU) -> 4 with its device state."""

    def __init__(self, seed: int = 0, max_rows: int = 8192, device=None):
        self.device = device or torch.device("cuda", torch.cuda.current_device())
        self.max_rows = max_rows
        h = ctypes.c_void_p()
        with torch.cuda.device(self.device):
            _lib.check(_lib.lib().noa_dcs_mlp_create(seed, max_rows, ctypes.byref(h)))
        self.handle = h
        self.nparam = _lib.lib().noa_dcs_mlp_num_params()

    def get_params(self) -> np.ndarray:
        out = np.zeros(self.nparam, dtype=np.float32)
        _lib.check(_lib.lib().noa_dcs_mlp_get_params(self.handle, out.ctypes.data_as(ctypes.c_void_p), self.nparam))
        return out

    def set_params(self, p: np.ndarray) -> None:
        p = np.ascontiguousarray(p, dtype=np.float32)
        _lib.check(_lib.lib().noa_dcs_mlp_set_params(self.handle, p.ctypes.data_as(ctypes.c_void_p), p.size))

    def forward(self, X: torch.Tensor) -> torch.Tensor:
        Y = torch.empty(X.shape[0], NPROC, dtype=torch.float32, device=X.device)
        _lib.check(_lib.lib().noa_dcs_mlp_forward(self.handle, _p(X), X.shape[0], _p(Y), _stream(X.device)))
        return Y

    def forward_fused(self, X: torch.Tensor) -> torch.Tensor:
        Y = torch.empty(X.shape[0], NPROC, dtype=torch.float32, device=X.device)
        _lib.check(_lib.lib().noa_dcs_mlp_infer_fused(self.handle, _p(X), X.shape[0], _p(Y), _stream(X.device)))
        return Y

    def forward_backward(self, X, T, M) -> tuple[float, np.ndarray]:
        loss = ctypes.c_double()
        g = np.zeros(self.nparam, dtype=np.float32)
        _lib.check(_lib.lib().noa_dcs_mlp_forward_backward(self.handle, _p(X), _p(T), _p(M), X.shape[0],
                                                           ctypes.byref(loss), g.ctypes.data_as(ctypes.c_void_p),
                                                           _stream(X.device)))
        return loss.value, g

    def train(self, X, T, M, epochs: int, batch: int = 8192, lr_max: float = 2e-3, lr_min: float = 2e-5,
              seed: int = 0) -> np.ndarray:
        losses = np.zeros(max(epochs, 1), dtype=np.float32)
        _lib.check(_lib.lib().noa_dcs_mlp_train(self.handle, _p(X), _p(T), _p(M), X.shape[0], batch, epochs,
                                                lr_max, lr_min, seed, losses.ctypes.data_as(ctypes.c_void_p),
                                                _stream(X.device)))
        return losses[:epochs]

    def close(self) -> None:
        if getattr(self, "handle", None) is not None:
            _lib.lib().noa_dcs_mlp_destroy(self.handle)
            self.handle = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


def features(K: torch.Tensor, q: torch.Tensor, offsets, elements) -> torch.Tensor:
    """[n x 3] FP32 features, element by element (noa_dcs_mlp_features)."""
    X = torch.empty(K.numel(), 3, dtype=torch.float32, device=K.device)
    for e, el in enumerate(elements):
        a, b = int(offsets[e]), int(offsets[e + 1])
        if b > a:
            _lib.check(_lib.lib().noa_dcs_mlp_features(_p(K[a:]), _p(q[a:]), b - a, int(el.Z), _p(X[a:]),
                                                       _stream(K.device)))
    return X


def exact_dcs(K, q, offsets, elements, mass=MUON_MASS):
    """Exact FP64 DCS of a batch (the batched kernel)."""
    plan = BatchPlan(elements, offsets, K, q, mass, precision="f64", tile=2048, waves_per_cu=4, use_graph=False)
    plan.launch()
    out = plan.outputs
    plan.close()
    return out


def equal_offsets(n_elements: int, n_total: int) -> np.ndarray:
    counts = np.full(n_elements, n_total // n_elements, dtype=np.int64)
    counts[: n_total % n_elements] += 1
    return np.concatenate([[0], np.cumsum(counts)])


def make_pairs(offsets, seed: int, device):
    n = int(offsets[-1])
    K = torch.empty(n, dtype=torch.float64, device=device)
    q = torch.empty_like(K)
    workload.fill_device_batch(K, q, offsets, seed=seed)
    return K, q


NTREND = 13


def trend_basis(X: torch.Tensor) -> torch.Tensor:
    """[n x 13] cubic basis of the features (a, b, z) = (log K, log nu, Z):
    a, b, a^2, b^2, ab, a^3, b^3, a^2 b, a b^2, z, za, zb, z^2 (the order the
    inference kernel adds them in)."""
    a, b, z = X[:, 0].double(), X[:, 1].double(), X[:, 2].double()
    return torch.stack([a, b, a * a, b * b, a * b, a * a * a, b * b * b, a * a * b, a * b * b, z, z * a, z * b,
                        z * z], 1)


def _tall_gram(A, B):
    """A^T B for a tall FP64 A [n, f] and B [n, g], as a split-K sum of batched
    products. Done as one product, the n-long reduction lands on a single
    output tile of the library GEMM (~0.45 s at n = 2^22 on MI355X)."""
    n, f = A.shape
    g = B.shape[1]
    P = 256
    m = n // P
    G = torch.zeros(f, g, dtype=A.dtype, device=A.device)
    if m > 0:
        At = A[:P * m].reshape(P, m, f).transpose(1, 2).contiguous()
        G = torch.bmm(At, B[:P * m].reshape(P, m, g).contiguous()).sum(0)
    if P * m < n:
        G = G + A[P * m:].T @ B[P * m:]
    return G


def _tall_matvec(A, c):
    """A c for a tall A [n, f] and a short c [f] (elementwise, no GEMV of
    one output column)."""
    return (A * c).sum(1)


def targets(dcs, elements, offsets, X, stats=None, exclude=None):
    """Standardised residual of ln(A * DCS) over a per-process cubic trend in
    the features, mask = DCS > 0 and not excluded. The trend (least squares over the active
    pairs, FP64) carries the bulk of the dynamic range, which the FP32 epilogue
    of the inference kernel adds back, so that the BF16 network resolves only
    the residual (std 0.1-0.7 instead of 2.5-9 in ln units)."""
    n = dcs[0].numel()
    lnA = torch.empty(n, dtype=torch.float64, device=dcs[0].device)
    for e, el in enumerate(elements):
        lnA[int(offsets[e]):int(offsets[e + 1])] = float(np.log(el.A))
    Y = torch.zeros(n, NPROC, dtype=torch.float64, device=lnA.device)
    M = torch.zeros(n, NPROC, dtype=torch.float32, device=lnA.device)
    for p in range(NPROC):
        act = dcs[p] > 0
        Y[act, p] = torch.log(dcs[p][act]) + lnA[act]
        if exclude is not None:  # [n x 4] bool: samples left out of the fit
            act = act & ~exclude[:, p]
        M[:, p] = act.float()
    Phi = trend_basis(X)
    if stats is None:
        mean, std, trend = np.zeros(NPROC), np.ones(NPROC), np.zeros((NPROC, NTREND))
        for p in range(NPROC):
            act = M[:, p] > 0
            if not bool(act.any()):
                continue
            A = torch.cat([torch.ones(int(act.sum()), 1, dtype=torch.float64, device=Y.device), Phi[act]], 1)
            G = _tall_gram(A, A).cpu().numpy()
            r = _tall_gram(A, Y[act, p].unsqueeze(1)).squeeze(1).cpu().numpy()
            c = np.linalg.solve(G + 1e-12 * np.trace(G) * np.eye(G.shape[0]), r)
            mean[p], trend[p] = c[0], c[1:]
            res = Y[act, p] - _tall_matvec(A, torch.from_numpy(c).to(Y.device))
            std[p] = max(float(res.std().item()), 1e-6)
        stats = {"mean": mean, "std": std, "trend": trend}
    dev = Y.device
    tr = torch.from_numpy(stats["trend"]).to(dev)
    base = torch.from_numpy(stats["mean"]).to(dev) + torch.stack([_tall_matvec(Phi, tr[p]) for p in range(NPROC)], 1)
    T = ((Y - base) / torch.from_numpy(stats["std"]).to(dev)) * M
    return T.float().contiguous(), M.contiguous(), stats


class Surrogate:
    """A trained network with its output statistics and validation error map."""

    def __init__(self, net: Network, elements, stats: dict, flag_map: np.ndarray | None, tol: float,
                 meta: dict | None = None, cell_err: np.ndarray | None = None):
        self.net = net
        self.elements = list(elements)
        self.stats = stats
        self.tol = tol
        self.meta = meta or {}
        self.cell_err = cell_err  # worst validation error per (element, log K, log nu) cell
        self.flag_map_host = flag_map
        self.flag_map = (torch.from_numpy(flag_map.astype(np.uint8)).to(net.device)
                         if flag_map is not None else None)

    def set_tolerance(self, tol: float) -> None:
        """Re-derive the flag map from the validation error map: process p of
        a cell is served by the network only where its worst validation error
        there is below half the tolerance (bit p of the cell's flag byte set =
        evaluate exactly). A map of the worst error over the processes
        ([elements, bins, bins]) flags all four together."""
        if self.cell_err is None:
            raise ValueError("no validation error map to derive flags from")
        self.tol = tol
        bad = (self.cell_err > 0.5 * tol) | (self.cell_err < 0)
        if bad.ndim == 3:
            flags = np.where(bad, 0xF, 0)
        else:
            flags = sum(bad[p].astype(np.int64) << p for p in range(NPROC))
        self.flag_map_host = flags.astype(np.uint8)
        self.flag_map = torch.from_numpy(self.flag_map_host).to(self.net.device)

    def served_fraction(self) -> np.ndarray:
        """Share of cells served by the network, per process, among the cells
        where the validation saw the process open (all cells without an
        error map)."""
        f = np.stack([(self.flag_map_host >> p) & 1 for p in range(NPROC)])
        res = []
        for p in range(NPROC):
            have = (self.cell_err[p] >= 0) if (self.cell_err is not None and self.cell_err.ndim == 4) else \
                np.ones(f[p].shape, bool)
            res.append(float(((f[p] == 0) & have).sum()) / max(int(have.sum()), 1))
        return np.array(res)

    def config(self, recheck_per_mille: int = 10, seed: int = 0, use_map: bool = True) -> _lib.SurrogateConfig:
        c = _lib.SurrogateConfig()
        for p in range(NPROC):
            c.out_mean[p] = float(self.stats["mean"][p])
            c.out_std[p] = float(self.stats["std"][p])
            for j in range(NTREND):
                c.trend[p][j] = float(self.stats["trend"][p][j])
        c.flag_map = _p(self.flag_map) if (use_map and self.flag_map is not None) else None
        c.bins = MAP_BINS
        c.recheck_per_mille = recheck_per_mille
        c.seed = seed
        return c

    def evaluate(self, K, q, offsets, mass=MUON_MASS, recheck_per_mille: int = 10, seed: int = 0,
                 use_map: bool = True, outputs=None, workspace=None):
        """Surrogate DCS (FP32) with exact fallback; returns (outputs, counters) (see read_counters)."""
        n = K.numel()
        dev = K.device
        if outputs is None:
            # (every query of the offsets' range is written)
            new = torch.empty if int(offsets[0]) == 0 and int(offsets[-1]) == n else torch.zeros
            outputs = tuple(new(n, dtype=torch.float32, device=dev) for _ in range(NPROC))
        counters = self.workspace(n, dev) if workspace is None else workspace
        els = (_lib.Element * len(self.elements))(*[_lib.Element(e.A, e.I, e.Z) for e in self.elements])
        offs = (ctypes.c_int64 * len(offsets))(*[int(x) for x in offsets])
        out = _lib.OutputsF32(*(_p(o) for o in outputs))
        cfg = self.config(recheck_per_mille, seed, use_map)
        with torch.cuda.device(dev):
            _lib.check(_lib.lib().noa_dcs_surrogate_eval(self.net.handle, els, offs, len(self.elements), float(mass),
                                                         _p(K), _p(q), ctypes.byref(out), ctypes.byref(cfg),
                                                         _p(counters), _stream(dev)))
        return outputs, counters

    @staticmethod
    def workspace(n: int, dev):
        """The device counters of one evaluation (see read_counters)."""
        return torch.zeros(4, dtype=torch.int32, device=dev)

    @staticmethod
    def read_counters(counters) -> tuple[int, float]:
        """(exact integral evaluations: pair production + photonuclear, largest
        relative error of the network over the recheck sample)."""
        c = counters.cpu().numpy().astype(np.uint32)
        return int(c[1]) + int(c[3]), float(np.frombuffer(c[2:3].tobytes(), dtype=np.float32)[0])

    @staticmethod
    def read_counters_full(counters) -> dict:
        c = counters.cpu().numpy().astype(np.uint32)
        return {"exact_pair": int(c[1]), "exact_photo": int(c[3]),
                "recheck_max_rel": float(np.frombuffer(c[2:3].tobytes(), dtype=np.float32)[0])}

    def save(self, path: str = CHECKPOINT) -> None:
        np.savez_compressed(path, params=self.net.get_params(), mean=self.stats["mean"], std=self.stats["std"],
                            trend=self.stats["trend"],
                            cell_err=(np.minimum(self.cell_err, 6e4).astype(np.float16) if self.cell_err is not None
                                      else np.zeros(0, np.float16)),
                            flag_map=self.flag_map_host if self.flag_map_host is not None else np.zeros(0, np.uint8),
                            elements=np.array([[e.A, e.I, e.Z] for e in self.elements]), tol=self.tol,
                            meta=np.array([repr(self.meta)]))

    @classmethod
    def load(cls, path: str = CHECKPOINT, device=None) -> "Surrogate":
        from .physics import AtomicElement
        d = np.load(path, allow_pickle=False)
        net = Network(device=device)
        net.set_params(d["params"])
        els = [AtomicElement(A=float(a), I=float(i), Z=int(z)) for a, i, z in d["elements"]]
        fm = d["flag_map"]
        ce = d["cell_err"].astype(np.float32) if "cell_err" in d.files else np.zeros(0, np.float32)
        return cls(net, els, {"mean": d["mean"], "std": d["std"], "trend": d["trend"]}, fm if fm.size else None,
                   float(d["tol"]), {"saved": str(d["meta"][0])}, ce if ce.size else None)


def error_map(sur_out, exact, K, q, offsets, bins: int = MAP_BINS) -> torch.Tensor:
    """Worst relative error per process and (element, log10 K bin, log10 nu
    bin), [4, elements, bins, bins]; a zero / non-zero mismatch counts as
    error 1. A cell where the process had no non-zero sample reads
    NO_SAMPLES (-1); one with fewer than MIN_CELL_SAMPLES reads +inf: the
    flags send both to the exact path (free for the queries where the
    process is kinematically closed, which return 0 either way)."""
    dev = K.device
    cell = cell_index(K, q, offsets, bins)
    maps = []
    for p in range(NPROC):
        s = sur_out[p].double()
        e = exact[p]
        rel = torch.where(e > 0, (s - e).abs() / e.clamp_min(1e-300), (s != 0).double())
        m = torch.zeros((len(offsets) - 1) * bins * bins, dtype=torch.float32, device=dev)
        m.scatter_reduce_(0, cell, rel.float(), reduce="amax")
        cnt = torch.zeros_like(m).scatter_add_(0, cell, (e > 0).float())
        m = torch.where(cnt == 0, torch.full_like(m, NO_SAMPLES),
                        torch.where(cnt < MIN_CELL_SAMPLES, torch.full_like(m, float("inf")), m))
        maps.append(m.reshape(len(offsets) - 1, bins, bins))
    return torch.stack(maps)


LATTICE = 32  # lattice intervals per cell side in lattice_error_map


def _lattice(bins: int, sub: int, dev):
    """The closed lattice of (bins sub + 1)^2 (K, q) points over the domain
    (log10 K in [-3, 6], log10 nu in [-6, 0]), K-major; nu = 1 is outside the
    domain (q < K), so the last line sits just below it."""
    side = bins * sub + 1
    lk = torch.linspace(-3.0, 6.0, side, dtype=torch.float64, device=dev)
    lnu = torch.linspace(-6.0, 0.0, side, dtype=torch.float64, device=dev)
    Kg = (10.0 ** lk)[:, None].expand(side, side)
    nug = (10.0 ** lnu)[None, :].expand(side, side)
    nug = torch.where(nug >= 1.0, torch.full_like(nug, 1.0 - 2.0 ** -40), nug)
    return Kg.reshape(-1).contiguous(), (Kg * nug).reshape(-1).contiguous(), side


def _cell_pool(v: torch.Tensor, sub: int) -> torch.Tensor:
    """Max of v [n, side, side] over each closed cell of the lattice."""
    return torch.nn.functional.max_pool2d(v[:, None], kernel_size=sub + 1, stride=sub)[:, 0]


def lattice_error_map(sur: "Surrogate", bins: int = MAP_BINS, sub: int = LATTICE, chunk: int = 4) -> torch.Tensor:
    """Worst relative error of the network per process and (element, log10 K
    bin, log10 nu bin) cell over a closed lattice of (sub + 1)^2 points per
    cell (the cell's edges and corners included, shared with its
    neighbours), [4, elements, bins, bins]. A cell where the exact process is
    open at some lattice points and closed at others contains a kinematic
    threshold, near which the DCS falls steeply to zero: it reads +inf (always
    exact); a cell where it is closed at every point reads NO_SAMPLES."""
    Kf, qf, side = _lattice(bins, sub, sur.net.device)
    npt = side * side
    maps = []
    for e0 in range(0, len(sur.elements), chunk):
        els = sur.elements[e0:e0 + chunk]
        off = np.arange(len(els) + 1, dtype=np.int64) * npt
        K, q = Kf.repeat(len(els)), qf.repeat(len(els))
        ex = exact_dcs(K, q, off, els)
        part = Surrogate(sur.net, els, sur.stats, None, sur.tol)
        out, _ = part.evaluate(K, q, off, recheck_per_mille=0, use_map=False)
        per = []
        for p in range(NPROC):
            e = ex[p].reshape(len(els), side, side)
            s = out[p].double().reshape(len(els), side, side)
            rel = torch.where(e > 0, (s - e).abs() / e.clamp_min(1e-300), (s != 0).double())
            worst = _cell_pool(rel, sub)
            opened, closed = _cell_pool((e > 0).double(), sub), _cell_pool((e <= 0).double(), sub)
            m = torch.where(opened == 0, torch.full_like(worst, NO_SAMPLES),
                            torch.where(closed > 0, torch.full_like(worst, float("inf")), worst))
            per.append(m.float())
        maps.append(torch.stack(per))
        del K, q, ex, out
    return torch.cat(maps, dim=1)


def threshold_cells(elements, dev, bins: int = MAP_BINS, sub: int = LATTICE, chunk: int = 4) -> torch.Tensor:
    """[4, elements, bins, bins] bool: the cells where the exact process is
    open at some lattice points and closed at others (a kinematic threshold
    crosses them). The network never serves them, so training leaves their
    samples out."""
    Kf, qf, side = _lattice(bins, sub, dev)
    npt = side * side
    maps = []
    for e0 in range(0, len(elements), chunk):
        els = elements[e0:e0 + chunk]
        off = np.arange(len(els) + 1, dtype=np.int64) * npt
        ex = exact_dcs(Kf.repeat(len(els)), qf.repeat(len(els)), off, els)
        per = []
        for p in range(NPROC):
            e = ex[p].reshape(len(els), side, side)
            per.append((_cell_pool((e > 0).double(), sub) > 0) & (_cell_pool((e <= 0).double(), sub) > 0))
        maps.append(torch.stack(per))
        del ex
    return torch.cat(maps, dim=1)


def cell_index(K: torch.Tensor, q: torch.Tensor, offsets, bins: int = MAP_BINS) -> torch.Tensor:
    """Flat (element, log10 K bin, log10 nu bin) cell of each pair."""
    dev = K.device
    el = torch.empty(K.numel(), dtype=torch.int64, device=dev)
    for e in range(len(offsets) - 1):
        el[int(offsets[e]):int(offsets[e + 1])] = e
    ik = ((torch.log10(K) + 3.0) / 9.0 * bins).long().clamp(0, bins - 1)
    inu = ((torch.log10(q / K) + 6.0) / 6.0 * bins).long().clamp(0, bins - 1)
    return (el * bins + ik) * bins + inu


def combine_maps(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """Cell-wise worst of two error maps; NO_SAMPLES only where both have none."""
    both_none = (a == NO_SAMPLES) & (b == NO_SAMPLES)
    return torch.where(both_none, torch.full_like(a, NO_SAMPLES), torch.maximum(a, b))


def max_rel_errors(out, exact) -> list[dict]:
    res = []
    for p in range(NPROC):
        s = out[p].double()
        e = exact[p]
        nz = e > 0
        rel = (s[nz] - e[nz]).abs() / e[nz]
        res.append({"max_rel": float(rel.max().item()) if rel.numel() else 0.0,
                    "p99_rel": float(torch.quantile(rel[:1 << 24].float(), 0.99).item()) if rel.numel() else 0.0,
                    "zero_mismatch": int(((s != 0) != nz).sum().item())})
    return res


def train_surrogate(elements, n_train: int = 1 << 22, n_val: int = 1 << 26, epochs: int = 200, batch: int = 8192,
                    tol: float = 1e-3, seed: int = 0, device=None, log=print, lr_max: float = 2e-3,
                    lr_min: float = 2e-5, skip_threshold_cells: bool = True) -> tuple[Surrogate, dict]:
    dev = device or torch.device("cuda", 0)
    t0 = time.time()
    off_tr = equal_offsets(len(elements), n_train)
    K, q = make_pairs(off_tr, seed=1000 + seed, device=dev)
    ex = exact_dcs(K, q, off_tr, elements)
    X = features(K, q, off_tr, elements)
    exclude = None
    if skip_threshold_cells:  # never served: the fit leaves them out
        tc = threshold_cells(elements, dev).reshape(NPROC, -1)
        cell = cell_index(K, q, off_tr)
        exclude = torch.stack([tc[p][cell] for p in range(NPROC)], 1)
        log(f"threshold cells per process {[round(float(tc[p].float().mean()), 3) for p in range(NPROC)]}")
    T, M, stats = targets(ex, elements, off_tr, X, exclude=exclude)
    del ex, exclude
    log(f"dataset {n_train} pairs in {time.time() - t0:.1f}s; active fraction per process "
        f"{[round(float(M[:, p].mean()), 3) for p in range(NPROC)]}")
    net = Network(seed=seed, max_rows=batch, device=dev)
    t1 = time.time()
    # chunks of epochs, each with its piece of one cosine schedule, so that
    # progress is reported while training runs
    chunk = max(10, epochs // 40)
    cos = lambda f: lr_min + (lr_max - lr_min) * 0.5 * (1 + np.cos(np.pi * f))  # noqa: E731
    losses = []
    for c0 in range(0, epochs, chunk):
        c1 = min(epochs, c0 + chunk)
        losses += list(net.train(X, T, M, epochs=c1 - c0, batch=batch, lr_max=cos(c0 / epochs),
                                 lr_min=cos(c1 / epochs), seed=seed + c0))
        log(f"epoch {c1}/{epochs}: loss {losses[-1]:.3e} ({time.time() - t1:.0f}s)")
    losses = np.array(losses)
    torch.cuda.synchronize()
    t_train = time.time() - t1
    log(f"trained {epochs} epochs in {t_train:.1f}s; loss {losses[0]:.3e} -> {losses[-1]:.3e}")
    del K, q, X, T, M
    sur = Surrogate(net, elements, stats, None, tol)
    report = {"n_train": n_train, "epochs": epochs, "batch": batch, "train_s": t_train,
              "skip_threshold_cells": skip_threshold_cells,
              "loss_first": float(losses[0]), "loss_last": float(losses[-1]), "lr_max": lr_max, "lr_min": lr_min}
    report.update(validate(sur, n_val=n_val, seed=seed, log=log))
    sur.meta = {**sur.meta, **report}
    return sur, report


def validate(sur: Surrogate, n_val: int = 1 << 26, seed: int = 0, log=print) -> dict:
    """Held-out validation (disjoint seed) and the lattice check: the
    per-process, per-cell worst error map the flags derive from (the worst of
    the held-out samples and of lattice_error_map; stored in sur.cell_err,
    flags set for sur.tol), and the raw error figures of the held-out
    samples."""
    dev = sur.net.device
    off_va = equal_offsets(len(sur.elements), n_val)
    Kv, qv = make_pairs(off_va, seed=2000 + seed, device=dev)
    exv = exact_dcs(Kv, qv, off_va, sur.elements)
    outv, _ = sur.evaluate(Kv, qv, off_va, recheck_per_mille=0, use_map=False)
    emap = error_map(outv, exv, Kv, qv, off_va)
    raw = max_rel_errors(outv, exv)
    del Kv, qv, exv, outv
    emap = combine_maps(emap, lattice_error_map(sur))
    sur.cell_err = emap.cpu().numpy().astype(np.float32)
    sur.set_tolerance(sur.tol)
    worst = emap.max(dim=0).values
    report = {"n_val": n_val, "tol": sur.tol, "val_raw_errors": raw,
              "served_cells_per_process": sur.served_fraction().tolist(),
              "median_cell_err_per_process": [float(emap[p][emap[p] >= 0].median().item()) for p in range(NPROC)],
              # share of the cells with samples that the network serves, per
              # process and for all four, at other tolerances
              "cells_within": {str(tl): {"per_process": [float(((emap[p] >= 0) & (emap[p] <= 0.5 * tl)).sum().item()
                                                               / max(int((emap[p] >= 0).sum().item()), 1))
                                                         for p in range(NPROC)],
                                         "all_four": float(((worst >= 0) & (worst <= 0.5 * tl)).sum().item()
                                                           / max(int((worst >= 0).sum().item()), 1))}
                               for tl in (1e-3, 3e-3, 1e-2, 3e-2, 1e-1)}}
    sur.meta = {**sur.meta, **report}
    log(f"validation raw max rel err {[round(r['max_rel'], 4) for r in raw]}, p99 "
        f"{[round(r['p99_rel'], 5) for r in raw]}; served cells per process "
        f"{[round(x, 3) for x in report['served_cells_per_process']]}")
    return report


def smoke(dev) -> str:
    """Tiny end-to-end pass: a few training steps, fused == layered forward,
    and the surrogate evaluation with everything routed exactly."""
    from .physics import STANDARD_ROCK
    els = [STANDARD_ROCK]
    off = np.array([0, 8192])
    K, q = make_pairs(off, seed=7, device=dev)
    ex = exact_dcs(K, q, off, els)
    X = features(K, q, off, els)
    T, M, stats = targets(ex, els, off, X)
    net = Network(seed=1, max_rows=1024, device=dev)
    losses = net.train(X, T, M, epochs=2, batch=1024)
    d = (net.forward(X) - net.forward_fused(X)).abs().max().item()
    assert d < 2e-2, d
    sur = Surrogate(net, els, stats, np.full((1, MAP_BINS, MAP_BINS), 0xF, np.uint8), 1e-3)
    out, cnt = sur.evaluate(K, q, off, recheck_per_mille=0)
    nfb, _ = Surrogate.read_counters(cnt)
    n_act = int((ex[1] > 0).sum().item() + (ex[2] > 0).sum().item())
    assert abs(nfb - n_act) <= 16, (nfb, n_act)
    for p in range(NPROC):
        assert torch.equal(out[p], ex[p].float()), p
    net.close()
    return f"surrogate smoke ok (loss {losses[0]:.3f} -> {losses[-1]:.3f}, fused-vs-layered {d:.1e})"


# Dense multiply-add flops of one forward pass: 2 (3 x 128 + 3 x 128 x 128 + 128 x 4).
FORWARD_FLOPS = 2 * (3 * 128 + 3 * 128 * 128 + 128 * 4)
# One training sample: the forward pass, the activation gradients and the weight gradients.
TRAIN_FLOPS = 3 * FORWARD_FLOPS
BF16_MFMA_PEAK_TFLOPS = 2500.0  # MI355X dense BF16 matrix peak


def training_entry(dev, epochs: int = 2, batch: int = 8192, n: int = 1 << 22) -> dict:
    """Training throughput at the stated workload: a fresh network on 2^22
    samples of the 48-element batch labelled by the FP64 kernel, `epochs`
    epochs at `batch` rows per step (three fused kernels per step), timed
    with HIP events on the stream; samples/s and the MFMA roofline."""
    elements, _ = workload.element_batch(48, seed=0)
    off = equal_offsets(len(elements), n)
    K, q = make_pairs(off, seed=1000, device=dev)
    ex = exact_dcs(K, q, off, elements)
    X = features(K, q, off, elements)
    T, M, _ = targets(ex, elements, off, X)
    del ex, K, q
    net = Network(seed=0, max_rows=batch, device=dev)
    net.train(X, T, M, epochs=1, batch=batch)  # warm-up
    stream = torch.cuda.current_stream(dev)
    s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda.synchronize()
    s.record(stream)
    losses = net.train(X, T, M, epochs=epochs, batch=batch, seed=1)
    e.record(stream)
    torch.cuda.synchronize()
    sec = s.elapsed_time(e) * 1e-3
    net.close()
    steps = epochs * (n // batch)
    rate = steps * batch / sec
    achieved = rate * TRAIN_FLOPS / 1e12
    return {"samples_per_s": rate, "ms_per_step": sec * 1e3 / steps, "batch": batch, "n_train": n,
            "epochs": epochs, "loss_per_epoch": [float(x) for x in losses],
            "roofline": {"bound": "mfma", "achieved": achieved, "peak": BF16_MFMA_PEAK_TFLOPS, "unit": "TFLOP/s",
                         "frac": achieved / BF16_MFMA_PEAK_TFLOPS, "flops_per_sample": TRAIN_FLOPS}}


def bench_entry(K, q, ref, steps, warmup, stream, wall_f64, tolerances=(None, 3e-2)) -> dict:
    """Config-4 style measurement: the committed checkpoint on 2^28 queries
    over its 48 elements, 1% seeded recheck, flagged cells exact; errors
    against the FP64 kernel over every query. Measured at the checkpoint's
    stated tolerance (None) and at the other tolerances given, with the flag
    map re-derived from the stored validation error map."""
    if not os.path.exists(CHECKPOINT):
        raise FileNotFoundError(CHECKPOINT)
    dev = K.device
    sur = Surrogate.load(CHECKPOINT, device=dev)
    n = 1 << 28
    off = equal_offsets(len(sur.elements), n)
    Kq, qq = make_pairs(off, seed=4, device=dev)
    outs = tuple(torch.empty(n, dtype=torch.float32, device=dev) for _ in range(NPROC))
    ws = Surrogate.workspace(n, dev)
    reps = max(1, min(steps, 5))
    # the exact FP64 kernel on the same queries, for the speedup and the errors
    plan = BatchPlan(sur.elements, off, Kq, qq, MUON_MASS, precision="f64", tile=2048, waves_per_cu=4)
    plan.launch()
    torch.cuda.synchronize()
    t = time.perf_counter()
    for _ in range(reps):
        plan.launch()
    torch.cuda.synchronize()
    dt_exact = (time.perf_counter() - t) / reps
    stated = sur.tol
    res = {"n_queries": n, "exact_f64_evals_per_s_same_queries": n / dt_exact, "stated_tolerance": stated}
    # every query through the network (no flags, no recheck): the inference
    # kernel's roofline against the dense BF16 MFMA peak
    for _ in range(max(1, warmup // 2)):
        sur.evaluate(Kq, qq, off, recheck_per_mille=0, use_map=False, outputs=outs, workspace=ws)
    torch.cuda.synchronize()
    t = time.perf_counter()
    for _ in range(reps):
        sur.evaluate(Kq, qq, off, recheck_per_mille=0, use_map=False, outputs=outs, workspace=ws)
    torch.cuda.synchronize()
    dt_net = (time.perf_counter() - t) / reps
    achieved = n * FORWARD_FLOPS / dt_net / 1e12
    res["network_only"] = {"evals_per_s": n / dt_net, "speedup_vs_f64": dt_exact / dt_net,
                           "roofline": {"bound": "mfma", "achieved": achieved, "peak": BF16_MFMA_PEAK_TFLOPS,
                                        "unit": "TFLOP/s", "frac": achieved / BF16_MFMA_PEAK_TFLOPS,
                                        "flops_per_query": FORWARD_FLOPS}}
    for tol in tolerances:
        tol = stated if tol is None else tol
        if sur.cell_err is not None:
            sur.set_tolerance(tol)
        for _ in range(max(1, warmup // 2)):
            sur.evaluate(Kq, qq, off, outputs=outs, workspace=ws)
        torch.cuda.synchronize()
        t = time.perf_counter()
        for _ in range(reps):
            sur.evaluate(Kq, qq, off, outputs=outs, workspace=ws)
        torch.cuda.synchronize()
        dt = (time.perf_counter() - t) / reps
        c = Surrogate.read_counters_full(ws)
        errs = max_rel_errors(outs, plan.outputs)
        res[f"tol_{tol:g}"] = {
            "evals_per_s": n / dt, "speedup_vs_f64": dt_exact / dt,
            "exact_pair_fraction": c["exact_pair"] / n, "exact_photo_fraction": c["exact_photo"] / n,
            "served_cells_per_process": ([round(float(x), 4) for x in sur.served_fraction()]
                                         if sur.flag_map_host is not None else [1.0] * NPROC),
            "recheck_max_rel": c["recheck_max_rel"], "max_rel_err_vs_f64": errs}
    plan.close()
    return res


def main() -> None:
    """python -m noa_amd.surrogate [--epochs E] [--out PATH]: trains on the
    48-element batch (2^22 samples), validates on 2^26 held-out pairs and
    writes the checkpoint with its error map."""
    import argparse
    import json
    ap = argparse.ArgumentParser()
    ap.add_argument("--epochs", type=int, default=200)
    ap.add_argument("--batch", type=int, default=8192)
    ap.add_argument("--n-train", type=int, default=1 << 22)
    ap.add_argument("--n-val", type=int, default=1 << 26)
    ap.add_argument("--tol", type=float, default=1e-3)
    ap.add_argument("--lr", type=float, default=2e-3, help="peak learning rate of the cosine schedule")
    ap.add_argument("--out", default=CHECKPOINT)
    ap.add_argument("--keep-threshold-cells", action="store_true",
                    help="train on the samples of cells crossed by a kinematic threshold too")
    ap.add_argument("--revalidate", metavar="CHECKPOINT",
                    help="recompute the validation error map of a trained checkpoint and write it to --out")
    a = ap.parse_args()
    if a.revalidate:
        sur = Surrogate.load(a.revalidate)
        sur.tol = a.tol
        report = validate(sur, n_val=a.n_val, log=lambda s: print(s, flush=True))
        sur.save(a.out)
        print(json.dumps(report), flush=True)
        return
    elements, _ = workload.element_batch(48, seed=0)
    sur, report = train_surrogate(elements, n_train=a.n_train, n_val=a.n_val, epochs=a.epochs, batch=a.batch,
                                  tol=a.tol, log=lambda s: print(s, flush=True), lr_max=a.lr, lr_min=a.lr / 100,
                                  skip_threshold_cells=not a.keep_threshold_cells)
    sur.save(a.out)
    print(json.dumps(report), flush=True)


if __name__ == "__main__":
    main()
