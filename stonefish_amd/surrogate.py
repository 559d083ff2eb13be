"""The learned surrogate of the hydrodynamics path (no counterpart in the reference).

A small MLP per hull shape maps 13 features of a body's state (CG-frame
relative linear and angular velocity, direction of gravity, depth of the
centre of buoyancy below the local surface, normal of the local surface) to the CG-frame
total force and torque that SolidEntity::ComputeHydrodynamicForces
(SolidEntity.cpp:1799-1850) produces after CorrectHydrodynamicForces.

  Net               libsfmlp.so (include/sfmlp.h): BF16 MFMA forward, backward
                    and Adam kernels, FP32 master weights
  Norm              feature/target normalisation and the training range that
                    decides the exact fallback (sfh_surrogate_norm)
  features / apply  the feature build, out-of-distribution mask, decode and
                    audit kernels of libsfhydro.so
  HullDataset       samples of one hull generated by the exact batch kernel
  train / evaluate  the training loop and the held-out error against the
                    exact kernel

Torch tensors carry device memory and streams only; every arithmetic step of
the feature build, the network and the optimiser runs in the HIP libraries.
"""
from __future__ import annotations

import ctypes as C
import math
import time
from dataclasses import dataclass

import numpy as np

from . import _native as N
from . import transforms as T

try:
    import torch
except ImportError:  # pragma: no cover - torch is part of the image
    torch = None

D = N.SFM_DIMS
LAYER_SHAPES = tuple((D[l + 1], D[l]) for l in range(N.SFM_LAYERS))   # padded [out, in]
REAL_DIMS = (N.SFM_IN, 256, 256, 256, 256, N.SFM_OUT)
FORWARD_FLOPS = 2 * sum(REAL_DIMS[l] * REAL_DIMS[l + 1] for l in range(N.SFM_LAYERS))   # 402,944 per sample


def _p(t) -> C.c_void_p:
    return C.c_void_p(0 if t is None else t.data_ptr())


def _stream(stream) -> C.c_void_p:
    if stream is None:
        return C.c_void_p(0)
    if isinstance(stream, int):
        return C.c_void_p(stream)
    return C.c_void_p(stream.cuda_stream)


class Net:
    """One surrogate network (sfm_net): 13 -> 4 x 256 GELU -> 6."""

    def __init__(self, max_batch: int = 65536, seed: int = 0):
        lib = N.load_mlp()
        h = C.c_void_p()
        N.check_mlp(lib.sfm_create(max_batch, seed, C.byref(h)))
        self.handle = h
        self.max_batch = max_batch

    def param_count(self) -> int:
        c = C.c_uint64()
        N.check_mlp(N.load_mlp().sfm_param_count(self.handle, C.byref(c)))
        return c.value

    def layer(self, l: int):
        """FP32 master weights [out, in] and bias [out] of layer l (padded shapes)."""
        o, i = LAYER_SHAPES[l]
        w = np.zeros((o, i), dtype=np.float32)
        b = np.zeros(o, dtype=np.float32)
        N.check_mlp(N.load_mlp().sfm_layer_io(self.handle, l, w.ctypes.data_as(N.c_float_p),
                                              b.ctypes.data_as(N.c_float_p), 0))
        return w, b

    def set_layer(self, l: int, w: np.ndarray, b: np.ndarray) -> None:
        o, i = LAYER_SHAPES[l]
        w = np.ascontiguousarray(w, dtype=np.float32).reshape(o, i)
        b = np.ascontiguousarray(b, dtype=np.float32).reshape(o)
        N.check_mlp(N.load_mlp().sfm_layer_io(self.handle, l, w.ctypes.data_as(N.c_float_p),
                                              b.ctypes.data_as(N.c_float_p), 1))

    def forward(self, x, y, stream=None) -> None:
        """x: (B, 32) bfloat16 device tensor, y: (B, 6) float32 device tensor."""
        assert x.dtype == torch.bfloat16 and x.shape[1] == N.SFM_IN_PAD and x.is_contiguous()
        assert y.dtype == torch.float32 and y.shape[0] >= x.shape[0] and y.is_contiguous()
        N.check_mlp(N.load_mlp().sfm_forward(self.handle, _p(x), x.shape[0], _p(y), _stream(stream)))

    def forward_layers(self, x, y, stream=None) -> None:
        """Same through the per-layer kernels of the training path."""
        assert x.dtype == torch.bfloat16 and x.shape[1] == N.SFM_IN_PAD and x.is_contiguous()
        assert y.dtype == torch.float32 and y.shape[0] >= x.shape[0] and y.is_contiguous()
        N.check_mlp(N.load_mlp().sfm_forward_layers(self.handle, _p(x), x.shape[0], _p(y), _stream(stream)))

    def train_step(self, x, target, loss, lr: float, beta1: float = 0.9, beta2: float = 0.999,
                   eps: float = 1e-8, stream=None) -> None:
        """One Adam step on the mean squared error of the batch; loss: 1-float device tensor."""
        assert x.dtype == torch.bfloat16 and x.is_contiguous() and target.is_contiguous()
        N.check_mlp(N.load_mlp().sfm_train_step(self.handle, _p(x), _p(target), x.shape[0], lr, beta1, beta2, eps,
                                                _p(loss), _stream(stream)))

    def gradients(self, l: int):
        o, i = LAYER_SHAPES[l]
        dw = torch.empty((o, i), dtype=torch.float32, device="cuda")
        db = torch.empty(o, dtype=torch.float32, device="cuda")
        N.check_mlp(N.load_mlp().sfm_gradients(self.handle, l, _p(dw), _p(db), C.c_void_p(0)))
        return dw, db

    def timing(self, on: bool) -> None:
        N.check_mlp(N.load_mlp().sfm_timing(self.handle, int(on)))

    def kernel_ms(self):
        ms, fl, c = C.c_double(), C.c_double(), C.c_uint32()
        N.check_mlp(N.load_mlp().sfm_kernel_ms(self.handle, C.byref(ms), C.byref(fl), C.byref(c)))
        return ms.value, fl.value, c.value

    def close(self) -> None:
        if self.handle:
            N.check_mlp(N.load_mlp().sfm_destroy(self.handle))
            self.handle = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


def forward_group(nets, counts, x, y, stream=None) -> None:
    """One launch over several networks: rows of x grouped per network (counts)."""
    assert x.dtype == torch.bfloat16 and x.is_contiguous() and y.is_contiguous()
    assert sum(counts) <= x.shape[0] and sum(counts) <= y.shape[0]
    hs = (C.c_void_p * len(nets))(*[n.handle.value for n in nets])
    cs = (C.c_uint32 * len(counts))(*counts)
    N.check_mlp(N.load_mlp().sfm_forward_group(hs, len(nets), cs, _p(x), _p(y), _stream(stream)))


def to_bf16(x, out=None, stream=None):
    """FP32 device tensor -> bfloat16 (round to nearest even) by the library kernel."""
    if out is None:
        out = torch.empty(x.shape, dtype=torch.bfloat16, device=x.device)
    N.check_mlp(N.load_mlp().sfm_to_bf16(_p(x), _p(out), x.numel(), _stream(stream)))
    return out


def probe_mfma(a, b, c) -> None:
    N.check_mlp(N.load_mlp().sfm_probe_mfma(_p(a), _p(b), _p(c), C.c_void_p(0)))


# ---- normalisation --------------------------------------------------------------

@dataclass
class Norm:
    in_shift: np.ndarray
    in_scale: np.ndarray
    in_lo: np.ndarray
    in_hi: np.ndarray
    out_shift: np.ndarray
    out_scale: np.ndarray
    gate_band: float = 0.0   # error-aware gate (fit_gate); 0: off

    @staticmethod
    def fit(raw: np.ndarray, raw_target: np.ndarray, t_weight: float = 1.0) -> "Norm":
        """Standardises features and targets; the training range is the
        features' observed [min, max].  The torque targets are scaled to a
        standard deviation of t_weight, so the squared-error loss weights
        their errors by t_weight^2 against the force's."""
        raw = np.asarray(raw, dtype=np.float64)
        tgt = np.asarray(raw_target, dtype=np.float64)
        mu, sd = raw.mean(0), raw.std(0)
        sd = np.where(sd > 1e-6, sd, 1.0)
        tmu, tsd = tgt.mean(0), tgt.std(0)
        tsd = np.where(tsd > 1e-9, tsd, 1.0)
        tsd[3:6] /= t_weight
        return Norm(mu.astype(np.float32), (1.0 / sd).astype(np.float32), raw.min(0).astype(np.float32),
                    raw.max(0).astype(np.float32), tmu.astype(np.float32), tsd.astype(np.float32))

    def c(self) -> N.sfh_surrogate_norm:
        n = N.sfh_surrogate_norm()
        n.in_shift[:] = [float(v) for v in self.in_shift]
        n.in_scale[:] = [float(v) for v in self.in_scale]
        n.in_lo[:] = [float(v) for v in self.in_lo]
        n.in_hi[:] = [float(v) for v in self.in_hi]
        n.out_shift[:] = [float(v) for v in self.out_shift]
        n.out_scale[:] = [float(v) for v in self.out_scale]
        n.gate_band = float(self.gate_band)
        return n

    def to_dict(self) -> dict:
        d = {k: np.asarray(getattr(self, k)).tolist() for k in
             ("in_shift", "in_scale", "in_lo", "in_hi", "out_shift", "out_scale")}
        d["gate_band"] = float(self.gate_band)
        return d


def features(batch, ocean, d_states, first: int, count: int, norm: Norm | None = None, rows: int | None = None,
             raw=None, x=None, ood=None, pos=None, exact=None, raw_target=None, target=None, stream=None) -> None:
    """sfh_surrogate_features over bodies first .. first+count-1 (see include/sfhydro.h)."""
    nc = norm.c() if norm is not None else None
    rows = count if rows is None else rows
    N.check(N.load().sfh_surrogate_features(batch.handle, ocean.handle, _p(d_states), first, count, rows,
                                            C.byref(nc) if nc is not None else None, _p(raw), _p(x), _p(ood),
                                            _p(pos), _p(exact), _p(raw_target), _p(target), _stream(stream)))


def apply(batch, ocean, d_states, first: int, count: int, norm: Norm, y, ft, ood=None, pos=None, exact=None,
          err=None, stream=None) -> None:
    """sfh_surrogate_apply: world-frame F/T of the bodies (exact where ood, zero out of the water), audit errors."""
    nc = norm.c()
    N.check(N.load().sfh_surrogate_apply(batch.handle, ocean.handle, _p(d_states), first, count, C.byref(nc), _p(y),
                                         _p(ood), _p(pos), _p(exact), _p(ft), _p(err), _stream(stream)))


# ---- sampling -------------------------------------------------------------------

def sample_states(rng: np.random.Generator, n: int, xy_range=(0.0, 1024.0), depth_range=(-1.0, 3.0),
                  v_max: float = 2.0, w_max: float = 1.0) -> np.ndarray:
    """(n, 22) states: position x, y uniform on the wave tile, CG depth uniform,
    uniform random orientation, v ~ U[-v_max, v_max]^3, omega ~ U[-w_max, w_max]^3."""
    pos = np.stack([rng.uniform(*xy_range, n), rng.uniform(*xy_range, n), rng.uniform(*depth_range, n)], axis=1)
    out = np.zeros((n, N.SFH_STATE_DOUBLES))
    out[:, :16] = T.quat_to_gl(T.random_unit_quaternions(rng, n), pos)
    out[:, 16:19] = rng.uniform(-v_max, v_max, (n, 3))
    out[:, 19:22] = rng.uniform(-w_max, w_max, (n, 3))
    return out


class HullDataset:
    """Samples of several hulls generated by the exact batch kernel.

    The batch holds `per_hull` bodies of each hull (body h * per_hull + i is
    hull h).  Each generation step draws new states for every body and runs
    the exact kernel; the states and exact outputs of every step stay in
    device memory, and the network inputs and targets are derived from them
    by the feature kernel."""

    def __init__(self, batch, ocean, n_hulls: int, per_hull: int, steps: int, holdout_steps: int, seed: int = 0,
                 xy_range=(0.0, 1024.0), depth_range=(-1.0, 3.0), v_max: float = 2.0, w_max: float = 1.0):
        assert per_hull % 256 == 0 and 0 < holdout_steps < steps
        self.batch, self.ocean = batch, ocean
        self.n_hulls, self.per_hull, self.steps, self.holdout = n_hulls, per_hull, steps, holdout_steps
        nb = n_hulls * per_hull
        assert batch.n == nb
        rng = np.random.default_rng(seed)
        self.states = torch.empty((steps, nb, N.SFH_STATE_DOUBLES), dtype=torch.float64, device="cuda")
        self.exact = torch.zeros((steps, nb, N.SFH_OUT_DOUBLES), dtype=torch.float64, device="cuda")
        t0 = time.perf_counter()
        for s in range(steps):
            self.states[s].copy_(torch.from_numpy(sample_states(rng, nb, xy_range, depth_range, v_max, w_max)))
            batch.compute(ocean, self.states[s].data_ptr(), self.exact[s].data_ptr())
        torch.cuda.synchronize()
        self.gen_seconds = time.perf_counter() - t0

    @property
    def train_steps(self) -> int:
        return self.steps - self.holdout

    def raw(self, hull: int, steps: range):
        """Raw features (n, 13) and raw CG-frame targets (n, 6) of one hull over steps."""
        P = self.per_hull
        raw = torch.empty((len(steps), P, N.SFH_SUR_FEATURES), dtype=torch.float32, device="cuda")
        tgt = torch.empty((len(steps), P, 6), dtype=torch.float32, device="cuda")
        for j, s in enumerate(steps):
            features(self.batch, self.ocean, self.states[s], hull * P, P, raw=raw[j], exact=self.exact[s],
                     raw_target=tgt[j])
        return raw.reshape(-1, N.SFH_SUR_FEATURES), tgt.reshape(-1, 6)

    def fit_norm(self, hull: int, t_weight: float = 1.0) -> Norm:
        raw, tgt = self.raw(hull, range(self.train_steps))
        return Norm.fit(raw.cpu().numpy(), tgt.cpu().numpy(), t_weight)

    def inputs(self, hull: int, norm: Norm, steps: range, with_pos: bool = False):
        """Network inputs (n, 32) bfloat16, normalised targets (n, 6), OOD mask
        (n,) and, with_pos, the body/fluid positions (n,)."""
        P = self.per_hull
        x = torch.empty((len(steps), P, N.SFM_IN_PAD), dtype=torch.bfloat16, device="cuda")
        t = torch.empty((len(steps), P, 6), dtype=torch.float32, device="cuda")
        ood = torch.empty((len(steps), P), dtype=torch.uint8, device="cuda")
        pos = torch.empty((len(steps), P), dtype=torch.int8, device="cuda")
        for j, s in enumerate(steps):
            features(self.batch, self.ocean, self.states[s], hull * P, P, norm=norm, rows=P, x=x[j], ood=ood[j],
                     pos=pos[j], exact=self.exact[s], target=t[j])
        out = (x.reshape(-1, N.SFM_IN_PAD), t.reshape(-1, 6), ood.reshape(-1))
        return out + (pos.reshape(-1),) if with_pos else out


@dataclass
class TrainConfig:
    steps: int = 6000
    batch: int = 4096
    lr: float = 2e-3
    lr_min: float = 2e-5
    warmup: int = 200
    beta1: float = 0.9
    beta2: float = 0.999
    eps: float = 1e-8
    seed: int = 0
    t_weight: float = 1.0   # torque outputs' weight in the loss (their standard deviation divided by it)


def lr_at(cfg: TrainConfig, step: int) -> float:
    if step < cfg.warmup:
        return cfg.lr * (step + 1) / cfg.warmup
    p = (step - cfg.warmup) / max(1, cfg.steps - cfg.warmup)
    return cfg.lr_min + 0.5 * (cfg.lr - cfg.lr_min) * (1.0 + math.cos(math.pi * min(1.0, p)))


def train(net: Net, x, t, cfg: TrainConfig, log_every: int = 0, log=None) -> dict:
    """Trains on (x, t) with mini-batches drawn from a fresh permutation each
    epoch; returns the loss history and timing."""
    n = x.shape[0]
    g = torch.Generator(device="cuda")
    g.manual_seed(cfg.seed)
    loss = torch.zeros(1, dtype=torch.float32, device="cuda")
    hist = []
    perm = torch.randperm(n, device="cuda", generator=g)
    pos = 0
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for step in range(cfg.steps):
        if pos + cfg.batch > n:
            perm = torch.randperm(n, device="cuda", generator=g)
            pos = 0
        idx = perm[pos:pos + cfg.batch]
        pos += cfg.batch
        xb = x.index_select(0, idx)
        tb = t.index_select(0, idx)
        net.train_step(xb, tb, loss, lr_at(cfg, step), cfg.beta1, cfg.beta2, cfg.eps,
                       stream=torch.cuda.current_stream())
        if log_every and (step % log_every == 0 or step == cfg.steps - 1):
            hist.append((step, float(loss.item())))
            if log:
                log(f"step {step} loss {hist[-1][1]:.3e}")
    torch.cuda.synchronize()
    return {"loss": hist, "seconds": time.perf_counter() - t0, "steps": cfg.steps, "batch": cfg.batch}


def train_many(nets, xs, ts, cfg: TrainConfig) -> dict:
    """Trains several networks at once, each on its own (x, t) and its own
    stream (default priority), step by step in turn: one network's step is a
    few dozen small launches, so networks trained side by side fill the GPU
    that one leaves mostly idle.  Same schedule and sampling as train()."""
    k = len(nets)
    assert len(xs) == len(ts) == k
    streams = [torch.cuda.Stream() for _ in range(k)]
    gens, perms, pos, losses = [], [], [0] * k, []
    torch.cuda.synchronize()
    for i in range(k):
        g = torch.Generator(device="cuda")
        g.manual_seed(cfg.seed + i)
        gens.append(g)
        with torch.cuda.stream(streams[i]):
            perms.append(torch.randperm(xs[i].shape[0], device="cuda", generator=g))
            losses.append(torch.zeros(1, dtype=torch.float32, device="cuda"))
    t0 = time.perf_counter()
    for step in range(cfg.steps):
        lr = lr_at(cfg, step)
        for i in range(k):
            with torch.cuda.stream(streams[i]):
                n = xs[i].shape[0]
                if pos[i] + cfg.batch > n:
                    perms[i] = torch.randperm(n, device="cuda", generator=gens[i])
                    pos[i] = 0
                idx = perms[i][pos[i]:pos[i] + cfg.batch]
                pos[i] += cfg.batch
                nets[i].train_step(xs[i].index_select(0, idx), ts[i].index_select(0, idx), losses[i], lr,
                                   cfg.beta1, cfg.beta2, cfg.eps, stream=streams[i])
    torch.cuda.synchronize()
    return {"seconds": time.perf_counter() - t0, "steps": cfg.steps, "batch": cfg.batch,
            "final_loss": [float(l.item()) for l in losses]}


def predict(net: Net, x, chunk: int | None = None):
    """Network outputs (n, 6) FP32 for inputs x (n, 32), n a multiple of 32."""
    n = x.shape[0]
    y = torch.empty((n, 6), dtype=torch.float32, device="cuda")
    chunk = chunk or net.max_batch
    s = torch.cuda.current_stream()
    for i in range(0, n, chunk):
        j = min(n, i + chunk)
        net.forward(x[i:j], y[i:j], stream=s)
    return y


def evaluate(ds: HullDataset, hull: int, net: Net, norm: Norm, delivered: bool = False) -> dict:
    """Held-out error of the network against the exact kernel: per sample,
    |F - F_exact| / |F_exact| and |T - T_exact| / |T_exact| on the total force
    and torque (sfh_surrogate_apply's audit), over the bodies the network
    answers; with delivered, also the error of the step's outputs, where the
    flagged bodies take the exact totals (delivered_summary)."""
    P = ds.per_hull
    steps = range(ds.train_steps, ds.steps)
    x, _, ood, pos = ds.inputs(hull, norm, steps, with_pos=True)
    y = predict(net, x)
    errs = []
    ft = torch.empty((P, 6), dtype=torch.float64, device="cuda")
    for j, s in enumerate(steps):
        err = torch.empty((P, 2), dtype=torch.float32, device="cuda")
        apply(ds.batch, ds.ocean, ds.states[s], hull * P, P, norm, y[j * P:(j + 1) * P], ft,
              pos=pos[j * P:(j + 1) * P], exact=ds.exact[s], err=err)
        errs.append(err)
    e = torch.cat(errs).cpu().numpy()
    o, p = ood.cpu().numpy().astype(bool), pos.cpu().numpy()
    r = error_summary(e, o, p)
    if delivered:
        r["delivered"] = delivered_summary(e, o, p)
    return r


def delivered_summary(e: np.ndarray, flagged: np.ndarray, pos: np.ndarray | None = None) -> dict:
    """Error of what the step delivers, over the bodies in the water: the
    flagged bodies (out of distribution or gated) get the exact kernel's
    totals, so their error is zero and they count."""
    return error_summary(np.where(flagged[:, None], 0.0, e), None, pos)


def fit_gate(depth: np.ndarray, err: np.ndarray, in_lo9: float, tau: float, bins: int = 20) -> float:
    """The error-aware gate of one hull (sfh_surrogate_norm.gate_band) from the
    network's errors on training samples of bodies crossing the surface: depth
    their depth feature (feature 9), err the larger of their F and T errors.
    The samples are binned by depth at quantiles; walking up from the
    shallowest bin, each bin whose median error exceeds tau joins the gated
    band, and the first bin at or below tau ends it.  Returns the band's upper
    edge minus in_lo9 (0: nothing gated)."""
    depth = np.asarray(depth, np.float64)
    err = np.asarray(err, np.float64)
    ok = np.isfinite(depth) & np.isfinite(err)
    depth, err = depth[ok], err[ok]
    if depth.size < 8 * bins:
        return 0.0
    q = np.quantile(depth, np.linspace(0.0, 1.0, bins + 1))
    idx = np.clip(np.searchsorted(q, depth, side="right") - 1, 0, bins - 1)
    edge = None
    for i in range(bins):
        m = idx == i
        if not m.any():
            continue
        if np.median(err[m]) > tau:
            edge = q[i + 1]
        else:
            break
    return 0.0 if edge is None else max(0.0, float(edge) - float(in_lo9))


def with_gate(norm: Norm, band: float) -> Norm:
    """A copy of norm with the error-aware gate band set."""
    return Norm(**{k: getattr(norm, k) for k in ("in_shift", "in_scale", "in_lo", "in_hi", "out_shift", "out_scale")},
                gate_band=band)


def gate_errors(ds: "HullDataset", hull: int, net: Net, norm: Norm, steps) -> tuple[np.ndarray, np.ndarray]:
    """Depth feature and larger-of-F/T network error of the bodies of one hull
    crossing the surface in the given (training) steps."""
    P = ds.per_hull
    dep, err = [], []
    for s in steps:
        raw = torch.empty((P, N.SFH_SUR_FEATURES), dtype=torch.float32, device="cuda")
        x = torch.zeros((P, N.SFM_IN_PAD), dtype=torch.bfloat16, device="cuda")
        pos = torch.empty(P, dtype=torch.int8, device="cuda")
        features(ds.batch, ds.ocean, ds.states[s], hull * P, P, norm=norm, rows=P, raw=raw, x=x, pos=pos)
        y = predict(net, x)
        e = torch.empty((P, 2), dtype=torch.float32, device="cuda")
        ft = torch.empty((P, 6), dtype=torch.float64, device="cuda")
        apply(ds.batch, ds.ocean, ds.states[s], hull * P, P, norm, y, ft, exact=ds.exact[s], err=e)
        m = (pos == 2).cpu().numpy()
        dep.append(raw.cpu().numpy()[m, 9])
        err.append(e.cpu().numpy()[m].max(1))
    return np.concatenate(dep), np.concatenate(err)


def error_summary(e: np.ndarray, ood: np.ndarray | None = None, pos: np.ndarray | None = None) -> dict:
    """Quantiles of the per-body F and T errors over the bodies in the water
    (position 1 or 2) inside the training range; bodies out of the water get
    exactly zero from both paths and are counted apart."""
    ok = np.ones(e.shape[0], bool)
    n_out = 0
    if pos is not None:
        wet = pos > 0
        n_out = int((~wet).sum())
        ok &= wet
    if ood is not None:
        ok &= ~ood
    n_inf = int((ok & ~np.isfinite(e).all(1)).sum())
    ok &= np.isfinite(e).all(1)
    F, Tq = e[ok, 0], e[ok, 1]
    q = lambda a, p: float(np.quantile(a, p)) if a.size else float("nan")   # noqa: E731
    return {"n": int(ok.sum()), "n_ood": int(0 if ood is None else ood.sum()), "n_out_of_water": n_out,
            "n_zero_exact": n_inf,
            "F_median": q(F, 0.5), "F_p90": q(F, 0.9), "F_p99": q(F, 0.99), "F_mean": float(F.mean()) if F.size else float("nan"),
            "T_median": q(Tq, 0.5), "T_p90": q(Tq, 0.9), "T_p99": q(Tq, 0.99), "T_mean": float(Tq.mean()) if Tq.size else float("nan"),
            "F_within_1pct": float((F <= 0.01).mean()) if F.size else float("nan"),
            "T_within_1pct": float((Tq <= 0.01).mean()) if Tq.size else float("nan")}


# ---- the training workload: 8 hulls of the fleet distribution -------------------

def hull_set(n_hulls: int = 8, seed: int = 17):
    """n hull shapes drawn like the fleet workload's bodies (ellipsoids or boxes,
    half-axes U[0.1, 2] m, face count log-uniform in [500, 50,000]) plus its sea
    state (1024 x 1024 grid from 64 Pierson-Moskowitz sinusoids)."""
    from . import workloads as WL
    return WL.fleet(n_hulls, seed=seed, waves=True)


def make_ocean(sea, device="cuda"):
    """Device ocean with the sea state's wave grid built on the GPU; returns
    (Ocean, grid tensor) - the grid must stay alive with the ocean."""
    from . import hydro as H
    from . import waves as W
    ocean = H.Ocean(sea.density, sea.gravity)
    grid = None
    if sea.wave_components is not None:
        n = sea.wave_n
        grid = torch.empty((n, n), dtype=torch.float32, device=device)
        W.build_grid_device(sea.wave_components, n, grid.data_ptr())
        ocean.set_waves(None, n, 1, [sea.wave_len], device_ptr=grid.data_ptr())
        torch.cuda.synchronize()
    return ocean, grid


def make_hull_batch(bodies, per_hull: int, faces_per_lane: int = 0):
    """A batch with `per_hull` consecutive bodies of each hull (shared meshes)."""
    from . import hydro as H
    descs = []
    meshes = []
    for b in bodies:
        m = H.Mesh(b.mesh)
        meshes.append(m)
        d = H.BodyDesc(mesh=m, Cd=b.Cd, Cf=b.Cf, volume=b.volume, surface=b.surface)
        descs.extend([d] * per_hull)
    return H.BodyBatch(descs, faces_per_lane=faces_per_lane), meshes


def run_training_workload(n_hulls: int = 8, per_hull: int = 8192, steps: int = 31, holdout: int = 3,
                          cfg: TrainConfig | None = None, seed: int = 17, log=None,
                          gate_tau: float | None = None) -> dict:
    """Generates n_hulls * per_hull * steps samples with the exact kernel, trains
    one network per hull and reports the held-out error against the exact
    kernel.  Returns the metrics with the trained networks and norms; with
    gate_tau, also each hull's error-aware gate fitted on four training steps
    (fit_gate), the norms carrying it ("norms_gated") and the held-out error
    with it (per hull "gated": the bodies it flags, the network's error on the
    others, the delivered error), and the training errors the gate was fitted
    on ("gate_data": per hull the crossing bodies' depth features and errors,
    for fitting other thresholds)."""
    cfg = cfg or TrainConfig()
    w = hull_set(n_hulls, seed)
    ocean, grid = make_ocean(w.sea)
    batch, meshes = make_hull_batch(w.bodies, per_hull)
    ds = HullDataset(batch, ocean, n_hulls, per_hull, steps, holdout, seed=seed + 1,
                     xy_range=(0.0, w.sea.wave_len), depth_range=(-1.0, 3.0))
    if log:
        log(f"generated {n_hulls * per_hull * steps} samples in {ds.gen_seconds:.2f}s")
    t0 = time.perf_counter()
    tables = attach_tables(batch, ocean, [(h * per_hull, per_hull) for h in range(n_hulls)])
    if log:
        log(f"hydrostatic tables in {time.perf_counter() - t0:.2f}s")
    norms = [ds.fit_norm(h, cfg.t_weight) for h in range(n_hulls)]
    xs, ts = [], []
    for h in range(n_hulls):
        x, t, _ = ds.inputs(h, norms[h], range(ds.train_steps))
        xs.append(x)
        ts.append(t)
    nets = [Net(max(cfg.batch, 65536), seed=cfg.seed + h) for h in range(n_hulls)]
    hist = train_many(nets, xs, ts, cfg)
    flops = 3.0 * FORWARD_FLOPS * cfg.batch * cfg.steps * n_hulls
    train_tflops = flops / hist["seconds"] / 1e12
    if log:
        log(f"trained {n_hulls} networks side by side, {cfg.steps} steps of {cfg.batch} each, "
            f"in {hist['seconds']:.1f}s ({train_tflops:.1f} TFLOP/s)")
    hulls = []
    for h in range(n_hulls):
        ev = evaluate(ds, h, nets[h], norms[h])
        b = w.bodies[h]
        info = {"hull": h, "faces": int(b.mesh.nf), "half_axes": [round(float(v), 3) for v in b.half_axes],
                "train_samples": int(xs[h].shape[0]), "final_loss": hist["final_loss"][h],
                "train_seconds": round(hist["seconds"], 3), "train_tflops": round(train_tflops, 2), **ev}
        if log:
            log(f"hull {h} F={b.mesh.nf}: F err median {ev['F_median']:.4f} p90 {ev['F_p90']:.4f}, "
                f"T err median {ev['T_median']:.4f}")
        hulls.append(info)
    del xs, ts
    norms_gated = None
    gate_data = None
    if gate_tau is not None:
        norms_gated, gate_data = [], []
        for h in range(n_hulls):
            d, e = gate_errors(ds, h, nets[h], norms[h], range(min(4, ds.train_steps)))
            gate_data.append((d, e))
            band = fit_gate(d, e, float(norms[h].in_lo[9]), gate_tau)
            g = with_gate(norms[h], band)
            norms_gated.append(g)
            ev = evaluate(ds, h, nets[h], g, delivered=True)
            hulls[h]["gated"] = {"tau": gate_tau, "band": band, "depth_below": float(norms[h].in_lo[9]) + band, **ev}
            if log:
                log(f"hull {h} gate tau {gate_tau}: depth < {float(norms[h].in_lo[9]) + band:.3f} m flags "
                    f"{ev['n_ood']} of {ev['n'] + ev['n_ood']}; delivered F median {ev['delivered']['F_median']:.4f} "
                    f"T median {ev['delivered']['T_median']:.4f}")
    return {"hulls": hulls, "nets": nets, "norms": norms, "norms_gated": norms_gated, "gate_data": gate_data,
            "dataset": ds, "workload": w,
            "ocean": ocean,
            "grid": grid, "batch": batch, "meshes": meshes, "tables": tables, "train_tflops": train_tflops,
            "train_seconds": hist["seconds"]}


# ---- mixed rollout: surrogate for every body, exact fallback and audits -----------

def integrate(ocean, d_states, count: int, d_ft, mass: float, inertia, dt: float, stream=None, ood=None,
              exact=None) -> None:
    """sfh_rollout_integrate: one rigid-body step of count bodies (with ood and
    exact, the flagged bodies' exact totals replace d_ft first)."""
    rg = N.sfh_rigid(float(mass), (C.c_double * 3)(*[float(v) for v in inertia]))
    N.check(N.load().sfh_rollout_integrate(ocean.handle, _p(d_states), count, _p(d_ft), _p(ood), _p(exact),
                                           C.byref(rg), float(dt), _stream(stream)))


class MixedRollout:
    """Steps n identical bodies (a BodyBatch or CompoundBatch of one hull) with
    the surrogate.  A step (captured in a HIP graph): the one-launch surrogate
    step (features, out-of-distribution flags, network, decode), the exact
    kernel restricted to the out-of-distribution bodies, and the rigid-body
    step, which first takes those bodies' exact totals.  Every
    `audit_every` steps the exact kernel runs for all bodies instead and the
    surrogate's errors against it are recorded; `audit_batch` (the same
    bodies in a batch set up for whole steps; default: `batch`) runs it."""

    def __init__(self, batch, ocean, net: Net, norm: Norm, states, mass: float, inertia, dt: float = 1e-3,
                 audit_every: int = 100, audit_batch=None):
        self.batch, self.ocean, self.net, self.norm = batch, ocean, net, norm
        self.audit_batch = batch if audit_batch is None else audit_batch
        if self.audit_batch.n != batch.n:
            raise ValueError("audit_batch must hold the same bodies as batch")
        self.n = batch.n
        self.states = states
        self.mass, self.inertia, self.dt, self.audit_every = mass, inertia, dt, audit_every
        dev = states.device
        self.plan = Plan(batch, [net], [norm], [self.n])
        self.ood = torch.zeros(self.n, dtype=torch.uint8, device=dev)
        self.pos = torch.zeros(self.n, dtype=torch.int8, device=dev)
        self.exact = torch.zeros((self.n, N.SFH_OUT_DOUBLES), dtype=torch.float64, device=dev)
        self.ft = torch.zeros((self.n, 6), dtype=torch.float64, device=dev)
        self.err = torch.zeros((self.n, 2), dtype=torch.float32, device=dev)
        self.audits = []
        self.k = 0
        self.graph = None

    def _step(self, audit: bool, stream=None) -> None:
        s = 0 if stream is None else stream.cuda_stream
        self.plan.run(self.ocean, self.states, self.ft, ood=self.ood, pos=self.pos, stream=stream)
        st = self.states.data_ptr()
        if audit:
            self.audit_batch.compute_masked(self.ocean, st, None, self.exact.data_ptr(), s)
            self.plan.merge(self.exact, self.ft, ood=self.ood, err=self.err, stream=stream)
            integrate(self.ocean, self.states, self.n, self.ft, self.mass, self.inertia, self.dt, stream=stream)
        else:
            self.batch.compute_masked(self.ocean, st, self.ood.data_ptr(), self.exact.data_ptr(), s)
            integrate(self.ocean, self.states, self.n, self.ft, self.mass, self.inertia, self.dt, stream=stream,
                      ood=self.ood, exact=self.exact)   # merge and step in one launch

    def capture(self) -> None:
        """Captures the ordinary (non-audit) step into a HIP graph."""
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        torch.cuda.synchronize()
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph, stream=s):
            self._step(False, stream=s)
        torch.cuda.synchronize()

    def step(self) -> None:
        audit = self.audit_every > 0 and self.k % self.audit_every == 0
        if audit:
            self._step(True, stream=torch.cuda.current_stream())
            self.audits.append((self.k, self.err.clone(), self.ood.clone(), self.pos.clone()))
        elif self.graph is not None:
            self.graph.replay()
        else:
            self._step(False, stream=torch.cuda.current_stream())
        self.k += 1

    def audit_summary(self) -> dict:
        if not self.audits:
            return {}
        e = torch.cat([a[1] for a in self.audits]).cpu().numpy()
        o = torch.cat([a[2] for a in self.audits]).cpu().numpy().astype(bool)
        p = torch.cat([a[3] for a in self.audits]).cpu().numpy()
        out = error_summary(e, o, p)
        out["audits"] = len(self.audits)
        out["delivered"] = delivered_summary(e, o, p)
        return out


class SurrogateStep:
    """The surrogate's evaluation of every body of a batch whose units are
    grouped by hull (counts[h] consecutive units per hull): one launch of the
    plan (features, network, decode to world-frame F/T, zero out of the
    water), capturable in a HIP graph."""

    def __init__(self, batch, ocean, nets, norms, counts, states):
        assert len(nets) == len(norms) == len(counts) and sum(counts) == batch.n
        self.batch, self.ocean = batch, ocean
        self.states = states
        n = batch.n
        dev = states.device
        self.plan = Plan(batch, nets, norms, counts)
        self.ood = torch.zeros(n, dtype=torch.uint8, device=dev)
        self.pos = torch.zeros(n, dtype=torch.int8, device=dev)
        self.ft = torch.zeros((n, 6), dtype=torch.float64, device=dev)
        self.exact = torch.zeros((n, N.SFH_OUT_DOUBLES), dtype=torch.float64, device=dev)
        self.graph = None

    def run(self, stream=None) -> None:
        self.plan.run(self.ocean, self.states, self.ft, ood=self.ood, pos=self.pos, stream=stream)

    def run_with_fallback(self, stream=None) -> None:
        """The whole step: the surrogate for every body, the exact kernel for
        the bodies it flags out of distribution, and their exact totals
        merged into ft."""
        self.run(stream)
        s = 0 if stream is None else stream.cuda_stream
        self.batch.compute_masked(self.ocean, self.states.data_ptr(), self.ood.data_ptr(), self.exact.data_ptr(), s)
        self.plan.merge(self.exact, self.ft, ood=self.ood, stream=stream)

    def capture(self, with_fallback: bool = False) -> None:
        """Captures run() (or run_with_fallback()) into a HIP graph (replay with replay())."""
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        torch.cuda.synchronize()
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph, stream=s):
            if with_fallback:
                self.run_with_fallback(stream=s)
            else:
                self.run(stream=s)
        torch.cuda.synchronize()

    def replay(self) -> None:
        self.graph.replay()


class Plan:
    """One-launch surrogate step over a batch whose units are grouped by hull
    (sfh_surrogate_plan_create / sfh_surrogate_run / sfh_surrogate_merge)."""

    def __init__(self, batch, nets, norms, counts):
        assert len(nets) == len(norms) == len(counts)
        lib, mlp = N.load(), N.load_mlp()
        ptrs = (N.sfh_net_ptrs * len(nets))()
        for g, net in enumerate(nets):
            w = (C.c_void_p * 5)()
            b = (C.c_void_p * 5)()
            N.check_mlp(mlp.sfm_weights(net.handle, w, b))
            ptrs[g].weights[:] = list(w)
            ptrs[g].bias[:] = list(b)
        ns = (N.sfh_surrogate_norm * len(norms))(*[n.c() for n in norms])
        cs = (C.c_uint32 * len(counts))(*counts)
        h = C.c_void_p()
        N.check(lib.sfh_surrogate_plan_create(batch.handle, len(nets), cs, ns, ptrs, C.byref(h)))
        self.handle = h
        self.batch, self.nets = batch, nets   # keep alive

    def run(self, ocean, d_states, ft, ood=None, pos=None, stream=None) -> None:
        N.check(N.load().sfh_surrogate_run(self.handle, ocean.handle, _p(d_states), _p(ood), _p(pos), _p(ft),
                                           _stream(stream)))

    def merge(self, exact, ft, ood=None, err=None, stream=None) -> None:
        N.check(N.load().sfh_surrogate_merge(self.handle, _p(ood), _p(exact), _p(ft), _p(err), _stream(stream)))

    def close(self) -> None:
        if self.handle:
            N.check(N.load().sfh_surrogate_plan_destroy(self.handle))
            self.handle = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


# ---- hydrostatic tables ---------------------------------------------------------

def table_grid(ns: int = 65, nth: int = 33, nph: int = 64):
    """Nodes of a hydrostatic table: immersion s in [-1, 1], polar angle in
    [0, pi], azimuth in [-pi, pi) (periodic), flattened in that order."""
    s = np.linspace(-1.0, 1.0, ns)
    th = np.linspace(0.0, np.pi, nth)
    ph = -np.pi + 2.0 * np.pi * np.arange(nph) / nph
    S_, TH, PH = np.meshgrid(s, th, ph, indexing="ij")
    return S_.ravel(), TH.ravel(), PH.ravel()


def _basis_with_row2(g):
    """Rotations R (n, 3, 3) whose third row is the unit vector g (n, 3)."""
    g = g / np.linalg.norm(g, axis=1, keepdims=True)
    a = np.where(np.abs(g[:, 0:1]) < 0.9, np.array([[1.0, 0.0, 0.0]]), np.array([[0.0, 1.0, 0.0]]))
    r0 = np.cross(a, g)
    r0 /= np.linalg.norm(r0, axis=1, keepdims=True)
    r1 = np.cross(g, r0)
    return np.stack([r0, r1, g], axis=1)


def build_hydrostatic_table(batch, ocean, first: int, count: int, aabb_min, aabb_max, P_CB, volume: float,
                            ns: int = 65, nth: int = 33, nph: int = 64):
    """Hydrostatic table of the hull shared by units first .. first+count-1 of
    the batch (sfh_surrogate_set_table layout): the exact kernel evaluates the
    hull at rest on the ocean's surface (which must be flat, gravity along +z)
    at every node, `count` nodes per pass.  Returns a (ns*nth*nph*6,) FP32
    device tensor."""
    g = np.asarray(ocean.gravity, dtype=np.float64)
    gn = float(np.linalg.norm(g))
    assert gn > 0 and abs(g[0]) + abs(g[1]) < 1e-12 * gn and g[2] > 0, "gravity along +z"
    lo, hi = np.asarray(aabb_min, np.float64), np.asarray(aabb_max, np.float64)
    c, h = 0.5 * (hi + lo), 0.5 * (hi - lo)
    Lc = float(h.max())
    P_CB = np.asarray(P_CB, np.float64)
    sv, th, ph = table_grid(ns, nth, nph)
    gb = np.stack([np.sin(th) * np.cos(ph), np.sin(th) * np.sin(ph), np.cos(th)], axis=1)
    R = _basis_with_row2(gb)
    hz = np.abs(gb) @ h
    z = sv * hz - gb @ c
    npts = sv.size
    states = np.zeros((npts, N.SFH_STATE_DOUBLES))
    Rt = np.transpose(R, (0, 2, 1))           # OpenGL column-major: columns of R
    states[:, 0:3], states[:, 4:7], states[:, 8:11] = Rt[:, 0], Rt[:, 1], Rt[:, 2]
    states[:, 14] = z
    states[:, 15] = 1.0
    n_units = batch.n
    d_states = torch.zeros((n_units, N.SFH_STATE_DOUBLES), dtype=torch.float64, device="cuda")
    d_states[:, 15] = 1.0
    d_states[:, [0, 5, 10]] = 1.0
    out = torch.zeros((n_units, N.SFH_OUT_DOUBLES), dtype=torch.float64, device="cuda")
    active = torch.zeros(n_units, dtype=torch.uint8, device="cuda")
    active[first:first + count] = 1
    rows = []
    for i0 in range(0, npts, count):
        m = min(count, npts - i0)
        d_states[first:first + m] = torch.from_numpy(states[i0:i0 + m]).cuda()
        if m < count:
            active[first + m:first + count] = 0
        out.zero_()
        batch.compute_masked(ocean, d_states.data_ptr(), active.data_ptr(), out.data_ptr())
        rows.append(out[first:first + m].cpu().numpy())
    o = np.concatenate(rows)
    wm = o[:, 20].astype(np.int64)
    Fw = np.where((wm & 1)[:, None] == 1, o[:, 0:3], 0.0)
    Tw = np.where((wm & 2)[:, None] == 1, o[:, 3:6], 0.0)
    Fb = np.einsum("nji,nj->ni", R, Fw)          # R^T F
    Tb = np.einsum("nji,nj->ni", R, Tw)
    sb = ocean.density * gn * volume
    tab = np.concatenate([Fb / sb, Tb / (sb * Lc)], axis=1).astype(np.float32)
    return torch.from_numpy(tab.reshape(-1)).cuda()


def set_table(batch, first: int, count: int, table, ns: int = 65, nth: int = 33, nph: int = 64) -> None:
    N.check(N.load().sfh_surrogate_set_table(batch.handle, first, count, _p(table), ns, nth, nph))


def unit_geometry(batch, i: int):
    """(aabb_min, aabb_max, P_CB, volume) of unit i of a BodyBatch or CompoundBatch."""
    from . import hydro as H
    d = batch.bodies[i]
    if isinstance(d, H.CompoundDesc):
        d = d.body
    if d.aabb_min is None:
        mn, mx = H.cg_frame_aabb(d.mesh.aabb_min, d.mesh.aabb_max, d.T_CG2C)
    else:
        mn, mx = d.aabb_min, d.aabb_max
    return np.asarray(mn, np.float64), np.asarray(mx, np.float64), np.asarray(d.P_CB, np.float64), float(d.volume)


def attach_tables(batch, ocean, groups, ns: int = 65, nth: int = 33, nph: int = 64, tables=None):
    """Builds (or reuses) one hydrostatic table per group (first, count) of a
    batch whose groups each hold one hull, and sets it on the group's units.
    `ocean` supplies density and gravity; the tables are evaluated on a flat
    surface.  Returns the tables (keep them alive with the batch)."""
    from . import hydro as H
    flat = H.Ocean(ocean.density, ocean.gravity)
    out = []
    for j, (first, count) in enumerate(groups):
        if tables is not None:
            t = tables[j]
        else:
            mn, mx, pcb, vol = unit_geometry(batch, first)
            t = build_hydrostatic_table(batch, flat, first, count, mn, mx, pcb, vol, ns, nth, nph)
        set_table(batch, first, count, t, ns, nth, nph)
        out.append(t)
    torch.cuda.synchronize()
    return out
