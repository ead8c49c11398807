"""The work that a user of this framework has it do, as timed cases.

``listed()`` names the cases, ``draw()`` gives more of the same ranges.  A case
is one call (or one burst of calls) of the Python view of the C ABI on host
arrays, as a program that holds mu, Sigma and the portfolio weights makes it:
the factor, the paths, the reductions and the result copies are all inside a
pass.  Inputs come from a seeded factor model of daily returns (B ~ U(0.2,
0.8), 1 %/day factor and idiosyncratic volatility, sample mean and ddof-1
covariance).  ``exact()`` repeats the same stream in float64 with torch.
"""
from __future__ import annotations

import importlib.util
import math
import os
import sys
from fractions import Fraction

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    name = "gpu_montecarlo_risk_amd"
    if name not in sys.modules:
        pkg = os.path.join(_ROOT, "gpu-montecarlo-risk_amd")
        spec = importlib.util.spec_from_file_location(name, os.path.join(pkg, "__init__.py"),
                                                      submodule_search_locations=[pkg])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


mcr = _package()
_PRECISION = {"fp32": mcr.PREC_FP32, "bf16x3": mcr.PREC_BF16X3, "auto": mcr.PREC_AUTO}


# ------------------------------------------------------------------- cases ---
# kind "run": one risk query (mcr.run); "simulate": the prototype's function
# with the per-path crash counts; "factor": the covariance factor alone;
# "batch": uneven portfolios in one call; "serve": a burst of queries into the
# serving loop.  VaR levels are var_levels of (0.99, 0.999, 0.95, 0.5).
def listed():
    return [
        # the smallest query: an interactive check, all latency and launches
        {"name": "tiny_n8_4k", "kind": "run", "n": 8, "paths": 4096, "precision": "fp32",
         "var_levels": 1, "hist": False, "near": False, "weighted": False},
        # the prototype's function on a small portfolio, S values wanted
        {"name": "plain_n20_1M", "kind": "simulate", "n": 20, "paths": 1_000_000,
         "precision": "fp32"},
        # the driver's own setup: 15 indices, 1e8 paths, the default precision
        {"name": "driver_n15_100M", "kind": "run", "n": 15, "paths": 100_000_000,
         "precision": "fp32", "var_levels": 0, "hist": False, "near": False, "weighted": False},
        # the benchmark's headline: 50 assets, 1e8 paths, VaR99
        {"name": "fused_n50_100M", "kind": "run", "n": 50, "paths": 100_000_000,
         "precision": "bf16x3", "var_levels": 1, "hist": False, "near": False, "weighted": False},
        # a mid-sized odd portfolio with every option of the default precision
        {"name": "options_n143_1M", "kind": "run", "n": 143, "paths": 1_000_003,
         "precision": "fp32", "var_levels": 2, "hist": True, "near": True, "weighted": True},
        # a mid-sized odd portfolio on the matrix cores
        {"name": "mid_n301_1M", "kind": "run", "n": 301, "paths": 1_000_000,
         "precision": "bf16x3", "var_levels": 1, "hist": False, "near": False, "weighted": True},
        # the largest benchmark workload
        {"name": "large_n600_10M", "kind": "run", "n": 600, "paths": 10_000_000,
         "precision": "bf16x3", "var_levels": 2, "hist": False, "near": False, "weighted": False},
        # the same portfolio in the default precision
        {"name": "large_n600_fp32_1M", "kind": "run", "n": 600, "paths": 1_000_000,
         "precision": "fp32", "var_levels": 1, "hist": False, "near": False, "weighted": False},
        # the largest portfolio a query takes
        {"name": "widest_n1024_1M", "kind": "run", "n": 1024, "paths": 1_000_000,
         "precision": "auto", "var_levels": 1, "hist": False, "near": False, "weighted": False},
        # the factor alone, as a program that keeps it asks for it
        {"name": "factor_n600", "kind": "factor", "n": 600},
        # a book of uneven portfolios revalued in one call
        {"name": "batch_64_uneven", "kind": "batch", "count": 64, "n_lo": 5, "n_hi": 600,
         "paths_lo": 100_000, "paths_hi": 10_000_000, "mix": 1004},
        # queries that arrive together at the serving loop, some covariances reused
        {"name": "serve_burst_48", "kind": "serve", "count": 48, "n_lo": 5, "n_hi": 600,
         "paths_lo": 100_000, "paths_hi": 1_000_000, "mix": 1005},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    r = rng.random()
    if r < 0.10:
        return {"kind": "factor", "n": _log_int(rng, 8, 1024)}
    if r < 0.20:
        return {"kind": "simulate", "n": _log_int(rng, 2, 64), "paths": _log_int(rng, 1e4, 4e6),
                "precision": "fp32"}
    if r < 0.32:
        return {"kind": rng.choice(["batch", "serve"]), "count": rng.randint(4, 48), "n_lo": 5,
                "n_hi": _log_int(rng, 40, 600), "paths_lo": 100_000, "paths_hi": 1_000_000,
                "mix": rng.randrange(1 << 20)}
    precision = rng.choice(["fp32", "fp32", "bf16x3", "bf16x3", "auto"])
    n = _log_int(rng, 2, 1024)
    # no dearer than the largest listed query of that arithmetic
    most = 1e12 if precision == "fp32" or n > 767 else 3.6e12
    paths = _log_int(rng, 4096, min(1e8, most / (n * n + 40 * n)))
    return {"kind": "run", "n": n, "paths": paths, "precision": precision,
            "var_levels": rng.choice([0, 1, 1, 2, 4]), "hist": rng.random() < 0.2,
            "near": precision == "fp32" and rng.random() < 0.3, "weighted": rng.random() < 0.5}


# ------------------------------------------------------------------ inputs ---
_LEVELS = (0.99, 0.999, 0.95, 0.5)


def _returns_model(n, rng):
    """Sample mean and covariance of seeded factor-model returns."""
    K, T = int(min(20, max(1, n // 30))), 2 * n + 200
    B = rng.uniform(0.2, 0.8, (n, K))
    R = 2e-4 + 0.01 * (rng.standard_normal((T, K)) @ B.T + rng.standard_normal((T, n)))
    mu = R.mean(axis=0)
    R -= mu
    return mu, (R.T @ R) / (T - 1)


def _portfolio(n, paths, levels, weighted, rng, model=None):
    mu, sigma = model if model is not None else _returns_model(n, rng)
    return {"mu": mu, "sigma": sigma, "x": float(rng.uniform(0.01, 0.04)), "k": max(1, (n + 9) // 10),
            "paths": int(paths), "seed": int(rng.integers(0, 2**62)),
            "weights": rng.dirichlet(np.ones(n)) if weighted else None,
            "alphas": _LEVELS[:levels], "precision": mcr.PREC_BF16X3}


def _portfolios(case, seed):
    """The queries of a batch or a burst: their sizes belong to the case (a
    book keeps its shape from day to day), their data to the seed.  In a burst
    three in ten reuse an earlier query's covariance."""
    mix, rng = np.random.default_rng(case["mix"]), np.random.default_rng(seed)

    def size(lo, hi):
        return int(round(math.exp(mix.uniform(math.log(lo), math.log(hi)))))

    out = []
    for i in range(case["count"]):
        n = size(case["n_lo"], case["n_hi"])
        m = size(case["paths_lo"], case["paths_hi"])
        reuse, which = mix.uniform() < 0.3, int(mix.integers(0, max(i, 1)))
        model = None
        if case["kind"] == "serve" and i and reuse:
            model = (out[which]["mu"], out[which]["sigma"])
            n = model[0].shape[0]
        out.append(_portfolio(n, m, 1, True, rng, model))
    return out


def _query(case, seed):
    rng = np.random.default_rng(seed)
    return _portfolio(case["n"], case["paths"], case.get("var_levels", 0),
                      case.get("weighted", False), rng)


class _Server(mcr.Server):
    """A serving loop that ends with the state that holds it."""

    def __del__(self):
        if getattr(self, "_h", None):
            self.close()


def prepare(case, seed):
    mcr.init()
    state = {"case": case}
    if case["kind"] == "factor":
        state["sigma"] = _returns_model(case["n"], np.random.default_rng(seed))[1]
    elif case["kind"] in ("run", "simulate"):
        state["query"] = _query(case, seed)
    else:
        state["portfolios"] = _portfolios(case, seed)
        if case["kind"] == "serve":
            state["server"] = _Server(hbm_budget=512 << 20)
    return state


# -------------------------------------------------------------------- pass ---
def _many(results):
    return {"count": np.array([r.count for r in results], dtype=np.int64),
            "p_hat": np.array([r.p_hat for r in results]),
            "std_error": np.array([r.std_error for r in results]),
            "var": np.array([r.var for r in results]),
            "es": np.array([r.es for r in results]),
            "tail_sum": np.array([r.tail_sum_fixed for r in results], dtype=np.int64),
            "loss_mean": np.array([r.loss_mean for r in results]),
            "loss_sd": np.array([r.loss_sd for r in results])}


def run(state):
    case = state["case"]
    if case["kind"] == "factor":
        L, attempts, jitter, clamped = mcr.factor(state["sigma"])
        return {"L": L, "attempts": attempts, "jitter": jitter, "clamped": clamped}
    if case["kind"] == "simulate":
        q = state["query"]
        p, count, S = mcr.monte_carlo_crash_simulation(q["x"], case["n"], q["k"], q["mu"],
                                                       q["sigma"], q["paths"], q["seed"],
                                                       _PRECISION[case["precision"]])
        return {"p_hat": p, "count": count, "S": S}
    if case["kind"] == "batch":
        return _many(mcr.run_batch(state["portfolios"])[0])
    if case["kind"] == "serve":
        srv = state["server"]
        return _many([srv.wait(t)[0] for t in [srv.submit(p) for p in state["portfolios"]]])
    q = state["query"]
    r = mcr.run(q["mu"], q["sigma"], q["x"], q["k"], q["paths"], q["seed"], weights=q["weights"],
                precision=_PRECISION[case["precision"]], alphas=q["alphas"], near=case["near"],
                want_hist=case["hist"])
    out = {"count": r.count, "p_hat": r.p_hat, "std_error": r.std_error,
           "ci": [r.ci_lower, r.ci_upper], "loss_mean": r.loss_mean, "loss_sd": r.loss_sd,
           "attempts": r.factor_attempts}
    if case["near"]:
        out["near"] = r.near_threshold
    if case["hist"]:
        out["S_hist"] = r.s_hist
    if q["alphas"]:
        out.update(var=np.array(r.var), es=np.array(r.es),
                   tail_sum=np.array(r.tail_sum_fixed, dtype=np.int64))
    return out


def work(case):
    """Bytes: Sigma, mu and the weights in, the results out.  Operations: the
    factor, the triangular product, and per normal about 30 for its transform
    (logarithm, root, sine and cosine)."""
    def query(n, m, out):
        return 8 * (n * n + 2 * n) + out, n**3 / 3 + m * (n * (n + 1) + 30 * n)

    if case["kind"] == "factor":
        n = case["n"]
        return {"bytes": 16 * n * n, "flops": n**3 / 3}
    if case["kind"] in ("run", "simulate"):
        n, m = case["n"], case["paths"]
        out = 200 + (4 * m if case["kind"] == "simulate" else 0)
        b, f = query(n, m, out + (8 * (n + 1) if case.get("hist") else 0))
        return {"bytes": b, "flops": f}
    # sizes only: the mix generator gives them without the data
    mix, total, sizes = np.random.default_rng(case["mix"]), [0, 0], []
    for i in range(case["count"]):
        n = int(round(math.exp(mix.uniform(math.log(case["n_lo"]), math.log(case["n_hi"])))))
        m = int(round(math.exp(mix.uniform(math.log(case["paths_lo"]), math.log(case["paths_hi"])))))
        reuse, which = mix.uniform() < 0.3, int(mix.integers(0, max(i, 1)))
        if case["kind"] == "serve" and i and reuse:
            n = sizes[which]
        sizes.append(n)
        b, f = query(n, m, 200)
        total[0] += b
        total[1] += f
    return {"bytes": total[0], "flops": total[1]}


# ------------------------------------------------------------------- exact ---
# The stream is Philox4x32-10 (Salmon et al., SC'11) keyed by the seed with
# counter (block, 0, path id), two Box-Muller pairs to a block.
def _philox(block, path, seed):
    mask = 0xFFFFFFFF
    k0, k1 = seed & mask, seed >> 32
    x, y, z, w = block, torch.zeros_like(block), path & mask, path >> 32
    for _ in range(10):
        p0, p1 = x * 0xD2511F53, z * 0xCD9E8D57  # the low 64 bits; products are unsigned
        x, y, z, w = ((p1 >> 32) & mask) ^ y ^ k0, p1 & mask, ((p0 >> 32) & mask) ^ w ^ k1, p0 & mask
        k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
    return x, y, z, w


def _normals(seed, path0, count, n):
    nb = (n + 3) // 4
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    path = (path0 + torch.arange(count, dtype=torch.int64, device=dev)).repeat_interleave(nb)
    block = torch.arange(nb, dtype=torch.int64, device=dev).repeat(count)
    x, y, z, w = _philox(block, path, seed)
    out = torch.empty(count * nb, 4, dtype=torch.float64, device=dev)
    for i, (a, b) in enumerate(((x, y), (z, w))):
        r = torch.sqrt(-2.0 * torch.log(((a >> 8) + 1).double() * 2.0**-24))
        theta = b.double() * (2.0 * math.pi * 2.0**-32)
        out[:, 2 * i] = r * torch.cos(theta)
        out[:, 2 * i + 1] = r * torch.sin(theta)
    return out.view(count, 4 * nb)[:, :n]


def _exact_query(q, want_loss):
    """(exceedance count, losses or None, loss mean, loss sd) in float64."""
    n, m = q["mu"].shape[0], q["paths"]
    L = np.linalg.cholesky(q["sigma"])
    w = q["weights"] if q["weights"] is not None else np.full(n, 1.0 / n)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    Lt, mu = torch.from_numpy(np.ascontiguousarray(L.T)).to(dev), torch.from_numpy(q["mu"]).to(dev)
    v, mp = torch.from_numpy(L.T @ w).to(dev), float(w @ q["mu"])
    losses = torch.empty(m if want_loss else 0, dtype=torch.float64, device=dev)
    count, step = 0, max(1, (1 << 27) // max(n, 8))
    for s in range(0, m, step):
        z = _normals(q["seed"], s, min(step, m - s), n)
        if want_loss:
            losses[s:s + z.shape[0]] = -(z @ v) - mp
        count += int((((z @ Lt + mu) < -q["x"]).sum(1) >= q["k"]).sum())
    return count, losses if want_loss else None, -mp, float(np.sqrt(w @ q["sigma"] @ w))


def _tail(losses, alpha):
    m = losses.shape[0]
    rank = min(max(math.ceil(Fraction(alpha) * m), 1), m)
    top = torch.topk(losses, m - rank + 1, sorted=False).values if m - rank < m // 8 else \
        torch.sort(losses).values[rank - 1:]
    return float(top.min()), float(top.mean())


def _interval(count, m):
    p = count / m
    se = math.sqrt(p * (1 - p) / m)
    return p, se, [max(0.0, p - 1.96 * se), min(1.0, p + 1.96 * se)]


def exact(case, seed):
    if work(case)["flops"] > 1e13:
        return None  # over about 20 seconds
    if case["kind"] == "factor":
        sigma = _returns_model(case["n"], np.random.default_rng(seed))[1]
        return {"L": np.linalg.cholesky(sigma), "attempts": None, "jitter": None, "clamped": None}
    if case["kind"] == "simulate":
        q = _query(case, seed)
        return {"p_hat": _exact_query(q, False)[0] / q["paths"], "count": None, "S": None}
    if case["kind"] == "run":
        q = _query(case, seed)
        count, losses, mean, sd = _exact_query(q, bool(q["alphas"]))
        p, se, ci = _interval(count, q["paths"])
        out = {"count": None, "p_hat": p, "std_error": se, "ci": ci, "loss_mean": mean,
               "loss_sd": sd, "attempts": None}
        if q["alphas"]:
            t = np.array([_tail(losses, a) for a in q["alphas"]])
            out.update(var=t[:, 0], es=t[:, 1], tail_sum=None)
        return out
    rows = []
    for q in _portfolios(case, seed):
        count, losses, mean, sd = _exact_query(q, True)
        rows.append(_interval(count, q["paths"])[:2] + _tail(losses, q["alphas"][0]) + (mean, sd))
    r = np.array(rows)
    return {"count": None, "p_hat": r[:, 0], "std_error": r[:, 1], "var": r[:, 2:3], "es": r[:, 3:4],
            "tail_sum": None, "loss_mean": r[:, 4], "loss_sd": r[:, 5]}
