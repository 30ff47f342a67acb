"""The calls whose speed this framework is judged by: one pass of each through the public entry points, on the sizes of
the repository's own benchmark and tests, with float64 answers in plain torch to hold the results to.

Kinds of calls (a case's "kind"):
  half_step  hip_sinkhorn.half_step: one fused half-step on packed clouds, as a program that drives its own loop calls it
  row_lse    hip_sinkhorn.row_lse: the row log-sum-exp of the augmented rows [x, 1] . [2y/eps, g/eps + log b]
  loop       hip_sinkhorn.DeviceLoop on clouds already on the GPU: a fixed number of iterations from zero potentials
  solve      sinkhorn() on host arrays, end to end: preparation, packing, the loop with its checks, the read-back
  pairs      wot_transport_maps: the maps between consecutive time points of a single-cell experiment, end to end
  median     normalization(how="median") of two clouds, the exact median over all pairs taken on the GPU
  marginals  plan_marginals of a result: the row and column sums of the plan without forming it
  pull_back  pull_back of a distribution through a result's plan

Clouds ("cloud"): "normal" is N(0, 1) against N(0, 1) + 0.5; "tests" the small clouds of the tests; "pca" anisotropic
Gaussians with per-axis std 1/sqrt(k + 1), shifted by 0.3 std per time point; "mixture" 20 blobs (centres N(0, 9)) per
cloud; "blobs8" eight blobs of std 0.5 shared by both clouds, the cost divided by its typical value. Points are float32
values, so that every path starts from the same numbers.
"""

import math
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = str(Path(__file__).resolve().parent.parent / "trainium-sinkhorn_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from trnopt import Backend, SinkhornOptions, SinkhornResult, plan_marginals, pull_back, sinkhorn  # noqa: E402
from trnopt import hip_sinkhorn as hk  # noqa: E402
from trnopt.singlecell import wot_transport_maps  # noqa: E402
from trnopt.sinkhorn import normalization  # noqa: E402

DEV = "cuda"


def listed():
    return [
        # The smallest call: the tests' clouds through one half-step with a marginal target and a KL penalty. Launches.
        dict(name="half_step_tests", kind="half_step", cloud="tests", n=137, m=91, d=5, eps=0.1, rho=1.0, off=True,
             role=0, log2=False),
        # One f update of the 10,000-point benchmark problem, x's log2-unit copy kept by the caller.
        dict(name="half_step_10k", kind="half_step", cloud="normal", n=10_000, m=10_000, d=64, eps=0.1, rho=0.0,
             off=False, role=0, log2=True),
        # One g update of the largest problem the benchmark has, the widest points the kernels take.
        dict(name="half_step_65k", kind="half_step", cloud="blobs8", n=65_536, m=65_536, d=128, eps=0.05, rho=0.0,
             off=False, role=1, log2=True),
        # The row log-sum-exp of augmented rows, the kernel-level check of the reference (d 64 and the ones column).
        dict(name="row_lse_4k", kind="row_lse", cloud="normal", n=4_096, m=3_796, d=64, eps=0.1),
        # A small solve to convergence from host arrays: latency of the whole call.
        dict(name="solve_700x500", kind="solve", cloud="tests", n=700, m=500, d=16, eps=0.1, rho_x=0.0, rho_y=0.0,
             eps_start=0.0, normalize="mean", tol=1e-5, max_iters=2000, fixed=False, its=60),
        # 100 fixed iterations of the balanced 2,048-point problem (the correctness workload).
        dict(name="solve_2048", kind="solve", cloud="normal", n=2_048, m=2_048, d=64, eps=0.1, rho_x=0.0, rho_y=0.0,
             eps_start=0.0, normalize="none", tol=1e-4, max_iters=100, fixed=True, its=100),
        # The headline: iterations of the 10,000-point problem with everything resident.
        dict(name="loop_10k", kind="loop", cloud="normal", n=10_000, m=10_000, d=64, eps=0.1, its=20),
        # The single-cell solve: unbalanced, growth-weighted row target, median-normalised cost, to convergence.
        dict(name="solve_cells", kind="solve", cloud="pca", n=7_355, m=8_962, d=30, eps=0.05, rho_x=1.0, rho_y=50.0,
             eps_start=0.0, normalize="median", tol=1e-4, max_iters=2000, fixed=False, its=140),
        # The published mixture problem with eps-scaling (a new eps in every one of the first iterations).
        dict(name="solve_schedule", kind="solve", cloud="mixture", n=10_000, m=10_000, d=64, eps=0.05, rho_x=0.0,
             rho_y=0.0, eps_start=1.0, normalize="mean", tol=1e-4, max_iters=2000, fixed=False, its=50),
        # Consecutive pairs of a single-cell experiment, wot's stages, solved together.
        dict(name="pairs_6", kind="pairs", cloud="pca", pairs=6, n=1_500, m=9_000, d=30, eps=0.05, its=400),
        # The exact median normalisation of the single-cell clouds alone.
        dict(name="median_cells", kind="median", cloud="pca", n=7_355, m=8_962, d=30),
        # What follows a solve of one such pair: its plan's marginals.
        dict(name="marginals_3k", kind="marginals", cloud="pca", n=3_001, m=3_507, d=30, eps=0.05),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["half_step", "half_step", "row_lse", "loop", "solve", "solve", "pairs", "median", "marginals",
                       "pull_back"])
    c = dict(kind=kind, cloud=rng.choice(["normal", "pca", "mixture"]), n=size(60, 12_000), m=size(60, 12_000),
             d=rng.randint(2, 128))
    if kind == "half_step":
        c.update(eps=rng.choice([0.05, 0.1, 0.5]), rho=rng.choice([0.0, 1.0, 50.0]), off=rng.random() < 0.5,
                 role=rng.randrange(2), log2=rng.random() < 0.5)
    elif kind == "row_lse":
        c.update(d=rng.randint(2, 127), eps=rng.choice([0.1, 0.5]))
    elif kind == "loop":
        c.update(eps=rng.choice([0.05, 0.1, 0.5]), its=rng.randint(5, 40))
    elif kind == "solve":
        unbalanced, sched = rng.random() < 0.4, rng.random() < 0.3
        its = rng.randint(20, 120)
        c.update(eps=rng.choice([0.05, 0.1, 0.2]), rho_x=1.0 if unbalanced else 0.0, rho_y=50.0 if unbalanced else 0.0,
                 eps_start=1.0 if sched else 0.0, normalize=rng.choice(["mean", "median"]), tol=1e-4, max_iters=its,
                 fixed=True, its=its)
    elif kind == "pairs":
        c.update(cloud="pca", pairs=rng.randint(2, 5), n=size(200, 1_500), m=size(1_600, 6_000), d=rng.randint(10, 50),
                 eps=0.05, its=400)
    elif kind == "median":
        c.update(n=size(60, 7_355), m=size(60, 8_962), d=rng.randint(2, 30))
    else:
        c.update(eps=rng.choice([0.05, 0.1]))
    return c


# ---------------------------------------------------------------------------------------------------------
# Inputs

def _f32(a):
    return a.astype(np.float32).astype(np.float64)


def _points(case, seed, t0=0, t1=1, n=None, m=None):
    n, m, d = n or case["n"], m or case["m"], case["d"]
    rx, ry = np.random.default_rng([seed, 11, t0]), np.random.default_rng([seed, 12, t1])
    zx = rx.standard_normal((n, d), dtype=np.float32)
    zy = ry.standard_normal((m, d), dtype=np.float32)
    kind = case["cloud"]
    if kind == "normal":
        x, y = zx, zy + np.float32(0.5)
    elif kind == "tests":
        x, y = zx, zy * np.float32(0.8) + np.float32(0.5)
    elif kind == "pca":
        sig = (1.0 / np.sqrt(np.arange(d) + 1.0)).astype(np.float32)
        x, y = zx * sig + np.float32(0.3 * t0) * sig, zy * sig + np.float32(0.3 * t1) * sig
    elif kind == "mixture":
        cx, cy = (r.normal(scale=3.0, size=(20, d)).astype(np.float32) for r in (rx, ry))
        x, y = cx[rx.integers(20, size=n)] + zx, cy[ry.integers(20, size=m)] + zy + np.float32(0.3)
    else:                                  # blobs8, in units of its typical cost
        mu = 2.0 * np.random.default_rng([seed, 13]).standard_normal((8, d)).astype(np.float32)
        x, y = mu[rx.integers(8, size=n)] + np.float32(0.5) * zx, mu[ry.integers(8, size=m)] + np.float32(0.5) * zy
        s = np.float32(1.0 / math.sqrt(7.5 * d))
        x, y = x * s, y * s
    return x.astype(np.float64), y.astype(np.float64)


def _step_inputs(case, seed):
    """Clouds, log weights, offset and the other side's shifted potential of one half-step: the state after one
    iteration from zero potentials (float64, rounded to float32)."""
    x, y = _points(case, seed)
    rows, cols = (x, y) if case["role"] == 0 else (y, x)
    r = np.random.default_rng([seed, 14])
    w = r.uniform(0.5, 1.5, len(cols))
    lw_rows, lw_cols = np.full(len(rows), -math.log(len(rows))), _f32(np.log(w / w.sum()))
    off = _f32(r.normal(scale=0.3, size=len(rows))) if case["off"] else None
    R, C = _dev(rows), _dev(cols)
    h = _update64(R, C, torch.zeros(len(cols), dtype=torch.float64, device=R.device), _dev(lw_cols), case["eps"])
    h = _update64(C, R, h, _dev(lw_rows), case["eps"])
    return rows, cols, lw_rows, lw_cols, off, h.float()


def _result_inputs(case, seed):
    """Clouds and potentials of a plan: the float64 potentials after four iterations."""
    x, y = _points(case, seed)
    c = float(np.square(x[:: max(1, len(x) // 512)][:, None, :] - y[:: max(1, len(y) // 512)][None]).sum(2).mean())
    center = np.concatenate([x, y]).mean(axis=0)
    X, Y = _dev((x - center) / math.sqrt(c)), _dev((y - center) / math.sqrt(c))
    la, lb = (torch.full((len(v),), -math.log(len(v)), dtype=torch.float64, device=v.device) for v in (X, Y))
    gh = torch.zeros(len(Y), dtype=torch.float64, device=Y.device)
    for _ in range(4):
        fh = _update64(X, Y, gh, lb, case["eps"])
        gh = _update64(Y, X, fh, la, case["eps"])
    f, g = fh + (X * X).sum(1), gh + (Y * Y).sum(1)
    v = np.random.default_rng([seed, 15]).uniform(0.0, 1.0, len(y))
    res = SinkhornResult(f=f.cpu().numpy(), g=g.cpu().numpy(), iterations=4, error=float("nan"), converged=False,
                         cost=float("nan"), seconds=0.0, eps=case["eps"], rho=None, center=center, cost_scale=c)
    return x, y, res, v / v.sum()


def _pair_sizes(case):
    """Sizes of the time points: spread over [n, m] on a logarithmic scale, large and small in turn."""
    k = case["pairs"] + 1
    s = [int(round(case["n"] * (case["m"] / case["n"]) ** (i / (k - 1)))) for i in range(k)]
    return [s[i // 2] if i % 2 == 0 else s[k - 1 - i // 2] for i in range(k)]


def _options(case):
    rho = (case["rho_x"], case["rho_y"]) if case["rho_x"] else None
    return SinkhornOptions(eps=case["eps"], rho=rho, max_iters=case["max_iters"], tol=case["tol"],
                           eps_start=case["eps_start"] or None, fixed_iters=case["fixed"],
                           normalize=False if case["normalize"] == "none" else case["normalize"],
                           kernel="hip", backend=Backend.preset("rocm"))


def _targets(case, seed, n, m):
    w = np.random.default_rng([seed, 16]).lognormal(0.0, 0.5, n)
    return w / w.sum(), np.full(m, 1.0 / m)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "half_step":
        rows, cols, lw_rows, lw_cols, off, h = _step_inputs(case, seed)
        R = hk.HipCloud(rows, lw_rows, DEV, off=off, role=case["role"])
        C = hk.HipCloud(cols, lw_cols, DEV, role=1 - case["role"])
        hp = torch.zeros(C.npad, dtype=torch.float32, device=DEV)
        hp[:C.n] = h
        rho = case["rho"]
        sc = hk.scalars(case["eps"], rho / (rho + case["eps"]) if rho else 1.0, DEV)
        if case["log2"]:
            hk.bake_log2(*((R, C) if case["role"] == 0 else (C, R)), sc)
        return dict(case=case, R=R, C=C, h=hp, sc=sc)
    if kind == "row_lse":
        xa, ya = _augmented(case, seed)
        return dict(case=case, xa=torch.from_numpy(xa).to(DEV), ya=torch.from_numpy(ya).to(DEV))
    if kind == "loop":
        x, y = _points(case, seed)
        X = hk.HipCloud(x, np.full(len(x), -math.log(len(x))), torch.device(DEV), role=0)
        Y = hk.HipCloud(y, np.full(len(y), -math.log(len(y))), torch.device(DEV), role=1)
        loop = hk.DeviceLoop(X, Y, eps=case["eps"], rho_x=None, rho_y=None, sched=[], stages=[], tol=1e-4,
                             stage_tol=1e-5, max_iters=case["its"], check_every=10, stage_max_iters=1000,
                             fixed_iters=True, balanced=True)
        return dict(case=case, loop=loop)
    if kind == "solve":
        x, y = _points(case, seed)
        at, bt = _targets(case, seed, len(x), len(y)) if case["rho_x"] else (None, None)
        return dict(case=case, x=x, y=y, at=at, bt=bt, opts=_options(case))
    if kind == "pairs":
        s = _pair_sizes(case)
        clouds = [_points(case, seed, t, t + 1, s[t], s[t + 1]) for t in range(case["pairs"])]
        growth = [np.random.default_rng([seed, 17, t]).lognormal(0.0, 0.3, s[t]) for t in range(case["pairs"])]
        opts = SinkhornOptions(check_every=5, max_iters=50_000, kernel="hip", backend=Backend.preset("rocm"))
        return dict(case=case, clouds=clouds, growth=growth, opts=opts)
    if kind == "median":
        x, y = _points(case, seed)
        return dict(case=case, x=x, y=y)
    x, y, res, v = _result_inputs(case, seed)
    return dict(case=case, x=x, y=y, res=res, v=v, opts=SinkhornOptions(kernel="hip", backend=Backend.preset("rocm")))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "half_step":
        return hk.half_step(state["R"], state["C"], state["h"], state["sc"])[:state["R"].n]
    if kind == "row_lse":
        return hk.row_lse(state["xa"], state["ya"])
    if kind == "loop":
        loop = state["loop"]
        loop.fh.zero_()
        loop.gh.zero_()
        loop.init()
        loop.enqueue(case["its"])
        return loop.fh[:case["n"]], loop.gh[:case["m"]]
    if kind == "solve":
        r = sinkhorn(state["x"], state["y"], opts=state["opts"], a_target=state["at"], b_target=state["bt"])
        return _solved(r)
    if kind == "pairs":
        maps = wot_transport_maps(state["clouds"], growth=state["growth"], eps=case["eps"], opts=state["opts"])
        return [_solved(t.result) for t in maps]
    if kind == "median":
        return normalization(state["x"], state["y"], how="median", device=DEV)
    if kind == "marginals":
        return plan_marginals(state["x"], state["y"], state["res"], opts=state["opts"])
    return pull_back(state["x"], state["y"], state["res"], state["v"], opts=state["opts"])


def _solved(r):
    out = dict(f=r.f, g=r.g)
    if r.rho is None:
        out["cost"] = r.cost
    else:
        out.update(row_mass=r.row_mass, col_mass=r.col_mass)
    return out


def work(case):
    """The augmented contraction, 2 (d + 1) per pair and half-step, each input and output once per call."""
    kind, n, m, d = case["kind"], case["n"], case["m"], case["d"]
    if kind == "pairs":
        s = _pair_sizes(case)
        cells = sum(s[t] * s[t + 1] for t in range(case["pairs"]))
        points = sum(s[t] + s[t + 1] for t in range(case["pairs"]))
        return {"bytes": points * (8 * d + 24), "flops": cells * (2 * case["its"] * 2 * (d + 1) + 2 * d)}
    if kind in ("half_step", "row_lse"):
        return {"bytes": 4 * (n + m) * (d + 2), "flops": 2 * n * m * (d + 1)}
    if kind == "median":
        return {"bytes": 8 * (n + m) * d, "flops": 2 * n * m * (d + 1)}
    if kind == "pull_back":
        return {"bytes": 8 * (n + m) * (d + 2), "flops": 2 * n * m * (d + 1)}
    if kind == "marginals":
        return {"bytes": 8 * (n + m) * (d + 2), "flops": 4 * n * m * (d + 1)}
    host = 8 if kind == "solve" else 4
    return {"bytes": host * (n + m) * (d + 2), "flops": case["its"] * 4 * n * m * (d + 1)}


# About four times the largest error against the float64 answer over 80 drawn cases and the listed ones: half-steps 1.9e-7,
# row log-sum-exps 1.7e-7, pull-backs 1.8e-7, marginals 8.6e-7 (exponentials of float32 potentials over eps); fixed loops
# 2.2e-5 (shifted potentials of raw clouds, smaller than the squared norms they are carried against), solves 4.4e-6 (a
# check may end them one cadence apart), staged pairs 2.3e-5 (as solves, stage by stage); the median is float64.
_REL = dict(half_step=8e-7, row_lse=7e-7, loop=9e-5, solve=2e-5, pairs=1e-4, median=1e-12, marginals=4e-6, pull_back=8e-7)


def tolerance(case):
    return {"rel": _REL[case["kind"]]}


# ---------------------------------------------------------------------------------------------------------
# The float64 answers

def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda" if torch.cuda.is_available() else "cpu")


def _lse64(R, C, h, lw, eps):
    """LSE_j((2 r_i . c_j + h_j) / eps + lw_j) by blocks of rows."""
    out = torch.empty(len(R), dtype=torch.float64, device=R.device)
    step = max(1, (1 << 26) // len(C))
    Ct, q = (C * (2.0 / eps)).T.contiguous(), h / eps + lw
    for s in range(0, len(R), step):
        z = R[s:s + step] @ Ct
        z += q
        out[s:s + step] = torch.logsumexp(z, dim=1)
    return out


def _update64(R, C, h, lw, eps, kappa=1.0, off=None):
    lse = _lse64(R, C, h, lw, eps)
    sq = (R * R).sum(1)
    return kappa * (sq + (0.0 if off is None else eps * off) - eps * lse) - sq


def _median64(x, y):
    X, Y = _dev(x), _dev(y)
    c = ((X * X).sum(1)[:, None] + (Y * Y).sum(1)[None, :] - 2.0 * (X @ Y.T)).clamp_(min=0.0).flatten()
    c = c.sort().values
    return float((c[(len(c) - 1) // 2] + c[len(c) // 2]) * 0.5)


def _normalise64(x, y, how):
    if how == "none":
        return np.zeros(x.shape[1]), 1.0
    center = np.concatenate([x, y]).mean(axis=0)
    if how == "median" and len(x) * len(y) <= 100_000_000:
        return center, _median64(x - center, y - center)
    rng = np.random.default_rng(0)
    i, j = rng.integers(len(x), size=20_000), rng.integers(len(y), size=20_000)
    dd = ((x[i] - y[j]) ** 2).sum(axis=1)
    return center, float(np.median(dd) if how == "median" else dd.mean())


def _solve64(x, y, how, eps, rho, stages, sched, tol, max_iters, check_every, fixed, at, bt):
    """The iteration in float64: eps stages or schedule, the checks at their cadence, the unbalanced masses."""
    n, m = len(x), len(y)
    center, scale = _normalise64(x, y, how)
    X, Y = _dev((x - center) / math.sqrt(scale)), _dev((y - center) / math.sqrt(scale))
    la, lb = (torch.full((k,), -math.log(k), dtype=torch.float64, device=X.device) for k in (n, m))
    ox = None if at is None else _dev(np.log(at)) - la
    oy = None if bt is None else _dev(np.log(bt)) - lb
    gh = torch.zeros(m, dtype=torch.float64, device=X.device)
    it = stage = stage_it = 0
    while it < max_iters:
        e = (stages[stage] if stage < len(stages) else eps) if stages else (sched[it] if it < len(sched) else eps)
        kx, ky = (1.0, 1.0) if rho is None else (rho[0] / (rho[0] + e), rho[1] / (rho[1] + e))
        fh = _update64(X, Y, gh, lb, e, kx, ox)
        new = _update64(Y, X, fh, la, e, ky, oy)
        it, stage_it = it + 1, stage_it + 1
        change = new - gh
        gh = new
        if stages and stage < len(stages):
            if stage_it % check_every == 0 and (float(change.abs().max()) / e < 1e-5 or stage_it >= 1000):
                stage, stage_it = stage + 1, 0
            continue
        if not fixed and (stages or it > len(sched)) and stage_it % check_every == 0:
            err = (float((torch.exp(lb) * (torch.exp((-change / e).clamp(max=50.0)) - 1.0)).abs().sum()) if rho is None
                   else float(change.abs().max()) / e)
            if err < tol:
                break
    f, g = fh + (X * X).sum(1), gh + (Y * Y).sum(1)
    out = dict(f=f.cpu().numpy(), g=g.cpu().numpy())
    if rho is None:
        out["cost"] = float(f.mean() + g.mean())
    else:
        fb = _update64(X, Y, gh, lb, eps)
        gb = _update64(Y, X, fh, la, eps)
        out["row_mass"] = torch.exp(la + (fh - fb) / eps).cpu().numpy()
        out["col_mass"] = torch.exp(lb + (gh - gb) / eps).cpu().numpy()
    return out


def _augmented(case, seed):
    x, y = _points(case, seed)
    r, eps = np.random.default_rng([seed, 14]), case["eps"]
    x, y = x * 0.15, y * 0.15
    gh = -(y * y).sum(1) + r.normal(scale=0.05, size=len(y))
    xa = np.hstack([x, np.ones((len(x), 1))]).astype(np.float32)
    ya = np.hstack([2.0 / eps * y, (gh / eps - math.log(len(y)))[:, None]]).astype(np.float32)
    return xa, ya


def exact(case, seed):
    kind, eps = case["kind"], case.get("eps")
    if kind == "half_step":
        rows, cols, _, lw_cols, off, h = _step_inputs(case, seed)
        rho = case["rho"]
        out = _update64(_dev(rows), _dev(cols), h.double(), _dev(lw_cols), eps, rho / (rho + eps) if rho else 1.0,
                        None if off is None else _dev(off))
        return out.cpu().numpy()
    if kind == "row_lse":
        xa, ya = _augmented(case, seed)
        zero = torch.zeros(len(ya), dtype=torch.float64, device=_dev(np.zeros(1)).device)
        return _lse64(_dev(xa), _dev(ya), zero, zero, 2.0).cpu().numpy()
    if kind == "loop":
        x, y = _points(case, seed)
        X, Y = _dev(x), _dev(y)
        la, lb = (torch.full((len(v),), -math.log(len(v)), dtype=torch.float64, device=v.device) for v in (X, Y))
        gh = torch.zeros(len(Y), dtype=torch.float64, device=Y.device)
        for _ in range(case["its"]):
            fh = _update64(X, Y, gh, lb, eps)
            gh = _update64(Y, X, fh, la, eps)
        return fh.cpu().numpy(), gh.cpu().numpy()
    if kind == "solve":
        x, y = _points(case, seed)
        at, bt = _targets(case, seed, len(x), len(y)) if case["rho_x"] else (None, None)
        sched, e = [], case["eps_start"]
        while e > eps and len(sched) < case["max_iters"]:
            sched.append(e)
            e *= 0.9
        rho = (case["rho_x"], case["rho_y"]) if case["rho_x"] else None
        return _solve64(x, y, case["normalize"], eps, rho, [], sched, case["tol"], case["max_iters"], 10, case["fixed"],
                        at, bt)
    if kind == "pairs":
        s = _pair_sizes(case)
        sf = math.exp(-math.log(eps) / 5)
        stages = [v for v in (sf ** -k for k in range(5)) if v > eps]
        out = []
        for t in range(case["pairs"]):
            x, y = _points(case, seed, t, t + 1, s[t], s[t + 1])
            g = np.random.default_rng([seed, 17, t]).lognormal(0.0, 0.3, s[t])
            out.append(_solve64(x, y, "median", eps, (1.0, 50.0), stages, [], 5e-6, 50_000, 5, False, g / len(g),
                                np.full(len(y), g.mean() / len(y))))
        return out
    if kind == "median":
        return _normalise64(*_points(case, seed), "median")
    x, y, res, v = _result_inputs(case, seed)
    X, Y = (_dev((p - res.center) / math.sqrt(res.cost_scale)) for p in (x, y))
    f, g = _dev(res.f), _dev(res.g)
    la, lb = (torch.full((len(p),), -math.log(len(p)), dtype=torch.float64, device=p.device) for p in (X, Y))
    fh, gh = f - (X * X).sum(1), g - (Y * Y).sum(1)
    if kind == "marginals":
        rows = torch.exp(la + fh / eps + _lse64(X, Y, gh, lb, eps))
        cols = torch.exp(lb + gh / eps + _lse64(Y, X, fh, la, eps))
        return rows.cpu().numpy(), cols.cpu().numpy()
    p = la + fh / eps + _lse64(X, Y, gh, lb + _dev(np.log(v)), eps)
    return (p - torch.logsumexp(p, 0)).cpu().numpy()
