"""The plan of a Sinkhorn result without forming it: its marginals and its action on a vector.

P_ij = a_i b_j exp((f_i + g_j - C_ij) / eps) on the result's normalised coordinates (the dense form is
transport_plan, src/trnopt/sinkhorn.py:397-403). Both functions here are log-sum-exps over one side's scores,

    log (P v)_i = log a_i + (f_i - |x_i|^2) / eps + LSE_j((2 x_i . y_j + g_j - |y_j|^2) / eps + log b_j + log v_j),

which is the half-step's log-sum-exp with kappa = 1 and no offset: on the GPU each is one sk_half_step_f32 call
per side (the fused kernel, scores never stored), elsewhere a blocked PyTorch computation in the backend's
dtype. They serve what the reference computes on the host in float64 from saved potentials: the plan's row and
column sums (examples/sinkhorn_libs_compare.py:43-56, and the unbalanced masses of sinkhorn.py:381-389) and
wot's ancestor pull-back p_t0 ∝ P p_t1 (examples/singlecell_figures.py:35-47).
"""

from __future__ import annotations

import numpy as np
import torch

from .sinkhorn import SinkhornOptions, SinkhornResult, _log_weights, _use_hip

_NEG = -1.0e9          # log of a zero weight: exactly zero after exp, finite (src/trnopt/sinkhorn.py:59)


def _normalised(x, y, res: SinkhornResult):
    root = np.sqrt(res.cost_scale)
    x = (np.asarray(x, dtype=np.float64) - res.center) / root
    y = (np.asarray(y, dtype=np.float64) - res.center) / root
    if x.ndim != 2 or y.ndim != 2 or x.shape[1] != y.shape[1]:
        raise ValueError("x (n, d) and y (m, d) must share d")
    if len(res.f) != len(x) or len(res.g) != len(y):
        raise ValueError("the result's potentials do not match x and y")
    return x, y


def _log_vector(v, m: int) -> np.ndarray:
    v = np.asarray(v, dtype=np.float64)
    if v.shape != (m,) or np.any(v < 0) or not np.any(v > 0):
        raise ValueError(f"v must be {m} non-negative values, not all zero")
    with np.errstate(divide="ignore"):
        return np.where(v > 0, np.log(np.where(v > 0, v, 1.0)), _NEG)


def _lse_torch(rows, cols, h_cols, log_w_cols, eps, be, block=2048) -> np.ndarray:
    """LSE_j((2 r_i . c_j + h_j) / eps + log_w_j) for every row, blocked, in the backend's dtype."""
    dev = torch.device(be.device)
    R = torch.as_tensor(rows, dtype=be.dtype, device=dev)
    cT = torch.as_tensor(cols.T.copy(), dtype=be.dtype, device=dev)
    h = torch.as_tensor(h_cols, dtype=be.dtype, device=dev)
    lw = torch.as_tensor(log_w_cols, dtype=be.dtype, device=dev)
    out = np.empty(len(rows))
    for s in range(0, len(rows), block):
        z = (2.0 * (R[s:s + block] @ cT) + h) / eps + lw
        out[s:s + block] = torch.logsumexp(z, dim=1).to("cpu", torch.float64).numpy()
    return out


class _HipPlan:
    """Both clouds on the GPU once, for the log-sum-exps of either side on the fused kernel: each one
    sk_half_step_f32 with |x|^2 = 0, no offset, kappa = 1, so that its output is exactly -eps lse, with the scores in
    log2 units from the matrix cores (the first cloud's log2-unit copy made for this eps, by the first of them)."""

    def __init__(self, xs, log_a, ys, log_b, eps, opts):
        from . import hip_sinkhorn as hk
        dev = torch.device(opts.backend.device)
        self.dev = torch.device("cuda", torch.cuda.current_device()) if dev.index is None else dev
        self.eps, self.hk, self.baked = eps, hk, False
        with torch.cuda.device(self.dev):
            self.X = hk.HipCloud(xs, log_a, self.dev, role=0)
            self.Y = hk.HipCloud(ys, log_b, self.dev, role=1)
            self.sc = hk.scalars(eps, 1.0, self.dev)

    def lse(self, role: int, h_cols) -> torch.Tensor:
        """Enqueued: -eps lse of x's rows against y's columns (role 0) or the reverse, (n,) on the GPU."""
        R, C = (self.X, self.Y) if role == 0 else (self.Y, self.X)
        with torch.cuda.device(self.dev):
            h = np.zeros(C.npad, dtype=np.float32)
            h[:C.n] = h_cols
            R.sq = torch.zeros_like(R.sq)
            out = self.hk.half_step(R, C, torch.from_numpy(h).to(self.dev), self.sc, use_off=False, log2=not self.baked)
        self.baked = True
        return out[:R.n]

    def read(self, *outs) -> list:
        host = (outs[0] if len(outs) == 1 else torch.cat(outs)).to("cpu", torch.float64).numpy()
        return [-v / self.eps for v in np.split(host, np.cumsum([len(o) for o in outs])[:-1])]


def plan_marginals(x, y, res: SinkhornResult, a=None, b=None,
                   opts: SinkhornOptions | None = None) -> tuple[np.ndarray, np.ndarray]:
    """Row and column sums (float64) of the plan of `res` between x (n, d) and y (m, d) with weights a, b
    (default uniform), without forming the n x m plan. opts selects backend and kernel as for sinkhorn():
    kernel="hip" (or "auto" on a ROCm GPU) runs two fused half-step launches."""
    opts = opts or SinkhornOptions()
    xs, ys = _normalised(x, y, res)
    log_a, log_b = _log_weights(a, len(xs), "a"), _log_weights(b, len(ys), "b")
    f, g, eps = np.asarray(res.f, np.float64), np.asarray(res.g, np.float64), float(res.eps)
    xx, yy = np.einsum("ij,ij->i", xs, xs), np.einsum("ij,ij->i", ys, ys)
    if _use_hip(opts, xs.shape[1]):
        plan = _HipPlan(xs, log_a, ys, log_b, eps, opts)
        lse_r, lse_c = plan.read(plan.lse(0, g - yy), plan.lse(1, f - xx))
    else:
        lse_r = _lse_torch(xs, ys, g - yy, log_b, eps, opts.backend)
        lse_c = _lse_torch(ys, xs, f - xx, log_a, eps, opts.backend)
    rows = np.exp(log_a + (f - xx) / eps + lse_r)
    cols = np.exp(log_b + (g - yy) / eps + lse_c)
    return rows, cols


def pull_back(x, y, res: SinkhornResult, v, a=None, b=None, opts: SinkhornOptions | None = None) -> np.ndarray:
    """log of P v, normalised to a distribution over x's points (log p with sum p = 1): wot's ancestor step
    p_t0 ∝ T_t0,t1 p_t1 for a distribution v (m,) on y's points. With uniform a, b it is the reference's
    pull_back_potentials (examples/singlecell_figures.py:35-47)."""
    opts = opts or SinkhornOptions()
    xs, ys = _normalised(x, y, res)
    log_a, log_b = _log_weights(a, len(xs), "a"), _log_weights(b, len(ys), "b")
    log_bv = np.maximum(log_b + _log_vector(v, len(ys)), _NEG)
    f, g, eps = np.asarray(res.f, np.float64), np.asarray(res.g, np.float64), float(res.eps)
    xx, yy = np.einsum("ij,ij->i", xs, xs), np.einsum("ij,ij->i", ys, ys)
    if _use_hip(opts, xs.shape[1]):
        plan = _HipPlan(xs, log_a, ys, log_bv, eps, opts)
        (lse,) = plan.read(plan.lse(0, g - yy))
    else:
        lse = _lse_torch(xs, ys, g - yy, log_bv, eps, opts.backend)
    out = log_a + (f - xx) / eps + lse
    mx = out.max()
    return out - (mx + np.log(np.exp(out - mx).sum()))
