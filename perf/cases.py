"""Timed cases: the work a user of stan_amd has it do, through its Python entry points.

What a posterior costs here is log density + gradient evaluations and the NUTS transitions
between them, so the cases are single evaluations (what the drop-in model class does at every
leapfrog step), batched evaluations in each precision, and whole sampler runs of the three
forms (host service, device chains on a GLM, device chains on the hierarchical model).  Sizes
are those of the benchmark, the tests and the smoke run, or odd ones of the same range.

A case holds:  kind  (eval | batch | service | nuts),  family (logit | normal | hier),
N, K (rows, columns; hier: J groups of about `rows` rows each instead of N), C chains,
prec (fp64 | bf16 | fp32: the precision the context is created with), and for the sampler
runs the iterations and the largest tree depth.
"""
import math

import numpy as np
import torch

import stan_amd as S

FAMILY = {"logit": S.LOGIT, "normal": S.NORMAL, "hier": S.HIER_LOGIT}
PREC = {"fp64": S.FP64, "fp32": S.FP32, "bf16": S.BF16X2}
# (alpha_sd, beta_sd, sigma_sd, tau_sd); alpha_sd 0 is a flat prior
PRIOR = {"logit": (5.0, 2.0, 2.0, 1.0), "normal": (0.0, 1.0, 2.0, 1.0),
         "hier": (5.0, 2.0, 2.0, 1.0)}


def listed():
    return [
        # the smallest call: one leapfrog's gradient of a small model, all latency
        dict(name="eval_logit_small", kind="eval", family="logit", N=3000, K=37, C=1,
             prec="fp64"),
        # an ordinary single-chain gradient at sizes that divide nothing
        dict(name="eval_normal_odd", kind="eval", family="normal", N=100003, K=129, C=1,
             prec="fp64"),
        # the plain drop-in at the benchmark's size: one gradient of N=1e6, K=100
        dict(name="eval_logit_large", kind="eval", family="logit", N=1000000, K=100, C=1,
             prec="fp64"),
        # several chains' points at once at the default precision (FP64)
        dict(name="batch_logit_fp64", kind="batch", family="logit", N=200003, K=60, C=32,
             prec="fp64"),
        # the benchmark's mixed-precision batches: 256 chains, logistic and normal
        dict(name="batch_logit_bf16", kind="batch", family="logit", N=1000000, K=100, C=256,
             prec="bf16"),
        dict(name="batch_normal_bf16", kind="batch", family="normal", N=200000, K=256, C=256,
             prec="bf16"),
        # a serving job with many columns and one tile of chains
        dict(name="batch_logit_wide", kind="batch", family="logit", N=48176, K=468, C=64,
             prec="bf16"),
        # hierarchical model, ragged groups: one chain in FP64 (the drop-in), 64 in FP32
        dict(name="eval_hier", kind="eval", family="hier", J=1000, rows=400, K=20, C=1,
             prec="fp64"),
        dict(name="batch_hier_fp32", kind="batch", family="hier", J=1000, rows=400, K=20, C=64,
             prec="fp32"),
        # the reference's service: one chain on the host, its gradients on the GPU
        dict(name="service_logit", kind="service", family="logit", N=10000, K=50, C=1,
             prec="fp64", warmup=20, samples=20, depth=10),
        # device-resident chains: 256 on a logistic model in mixed precision
        dict(name="nuts_logit_bf16", kind="nuts", family="logit", N=20000, K=100, C=256,
             prec="bf16", warmup=20, samples=20, depth=10),
        # device-resident chains: 64 on the hierarchical model (11,022 parameters each)
        dict(name="nuts_hier_fp32", kind="nuts", family="hier", J=1000, rows=100, K=10, C=64,
             prec="fp32", warmup=10, samples=10, depth=6),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["eval", "batch64", "bf16", "bf16", "eval_hier", "hier32", "service",
                       "nuts64", "nuts16", "nuts_hier"])
    family = rng.choice(["logit", "normal"])
    if what == "eval":
        K = _log(rng, 1, 256)
        return dict(kind="eval", family=family, N=_log(rng, 500, min(1e6, 1e8 / K)), K=K, C=1,
                    prec="fp64")
    if what == "batch64":
        K, C = _log(rng, 2, 200), _log(rng, 2, 64)
        return dict(kind="batch", family=family, N=_log(rng, 1000, min(4e5, 3.8e8 / (K * C))),
                    K=K, C=C, prec="fp64")
    if what == "bf16":
        K, C = _log(rng, 8, 512), _log(rng, 8, 256)
        return dict(kind="batch", family=family, N=_log(rng, 2000, min(1e6, 6e7 / K)), K=K, C=C,
                    prec="bf16")
    if what in ("eval_hier", "hier32"):
        return dict(kind="eval" if what == "eval_hier" else "batch", family="hier",
                    J=_log(rng, 20, 1000), rows=_log(rng, 20, 400), K=rng.randint(1, 20),
                    C=1 if what == "eval_hier" else _log(rng, 4, 64),
                    prec="fp64" if what == "eval_hier" else "fp32")
    if what == "service":
        return dict(kind="service", family=family, N=_log(rng, 500, 10000), K=_log(rng, 3, 50),
                    C=1, prec="fp64", warmup=20, samples=20, depth=8)
    if what == "nuts_hier":
        return dict(kind="nuts", family="hier", J=_log(rng, 50, 1000), rows=_log(rng, 20, 100),
                    K=rng.randint(1, 10), C=_log(rng, 8, 64), prec="fp32", warmup=10, samples=10,
                    depth=6)
    small = what == "nuts64"
    return dict(kind="nuts", family=family, N=_log(rng, 500, 10000 if small else 20000),
                K=_log(rng, 3, 50 if small else 100), C=_log(rng, 4, 32 if small else 256),
                prec="fp64" if small else "bf16", warmup=20, samples=20, depth=8)


def _groups(case, seed):
    """Row offsets of ragged groups: sizes round(LogNormal(ln rows, 1)), at least 1."""
    rng = np.random.Generator(np.random.PCG64(seed))
    sizes = np.maximum(1, np.round(rng.lognormal(math.log(case["rows"]), 1.0, case["J"])))
    return np.concatenate([[0], np.cumsum(sizes.astype(np.int64))])


def _data(case, seed):
    """Inputs from the seed alone, as GPU tensors: X (unit-variance linear predictors), y from
    the model itself, and the points: the generating parameters plus a normal step of sd 0.3,
    as chains meet them in warm-up."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    dev = dict(generator=g, device="cuda", dtype=torch.float64)
    K, C = case["K"], case["C"]
    off = _groups(case, seed) if case["family"] == "hier" else None
    N = case["N"] if off is None else int(off[-1])
    X = torch.randn(N, K, **dev).mul_(1.0 / math.sqrt(K))
    beta = torch.randn(K, **dev)
    alpha = torch.full((1,), 0.5, device="cuda", dtype=torch.float64)
    d = dict(X=X, off=off, N=N)
    if off is None:
        eta = X @ beta + alpha
        if case["family"] == "logit":
            y = (torch.rand(N, **dev) < torch.sigmoid(eta)).to(torch.int32)
            truth = torch.cat([alpha, beta])
        else:
            y = eta + torch.randn(N, **dev)
            truth = torch.cat([alpha, beta, torch.zeros_like(alpha)])
    else:
        J = case["J"]
        v = -0.7 + 0.3 * torch.randn(K + 1, **dev)
        z = torch.randn(J, K + 1, **dev)
        gid = _group_ids(off)
        w = torch.cat([alpha, beta]) + torch.exp(v) * z
        eta = w[gid, 0] + (X * w[gid, 1:]).sum(1)
        y = (torch.rand(N, **dev) < torch.sigmoid(eta)).to(torch.int32)
        truth = torch.cat([alpha, beta, v, z.reshape(-1)])
    d["y"] = y
    d["theta"] = truth + 0.3 * torch.randn(C, truth.numel(), **dev)
    return d


def _group_ids(off):
    sizes = torch.as_tensor(np.diff(off), device="cuda")
    return torch.repeat_interleave(torch.arange(len(off) - 1, device="cuda"), sizes)


def prepare(case, seed):
    """The context a program creates once per data set, and the points it evaluates at."""
    d = _data(case, seed)
    m = S.GlmModel(FAMILY[case["family"]], d["X"].cpu().numpy(), d["y"].cpu().numpy(),
                   offsets=d["off"], precision=PREC[case["prec"]], prior=PRIOR[case["family"]])
    state = dict(case=case, model=m, seed=int(seed) % (1 << 31))
    if case["kind"] in ("eval", "batch"):
        theta = d["theta"].cpu().numpy()
        state["theta"] = theta[0] if case["kind"] == "eval" else theta
        if case["kind"] == "batch" and case["prec"] != "fp64":
            # mixed-precision evaluations carry FP32 accuracy (their last FP64 digits hang on
            # the summation order the autotuner picked): this program keeps them as FP32
            state["lp"] = np.zeros(theta.shape[0], np.float32)
            state["grad"] = np.zeros(theta.shape, np.float32)
    d.clear()
    torch.cuda.empty_cache()
    return state


def run(state):
    case, m = state["case"], state["model"]
    if case["kind"] == "eval":
        lp, g = m.log_prob_grad(state["theta"])
        return {"lp": lp, "grad": g}
    if case["kind"] == "batch":
        lp, g = m.log_prob_grad_batch(state["theta"])
        if "grad" in state:
            np.copyto(state["lp"], lp, casting="same_kind")
            np.copyto(state["grad"], g, casting="same_kind")
            lp, g = state["lp"], state["grad"]
        return {"lp": lp, "grad": g}
    cfg = dict(random_seed=state["seed"], chain=1, num_warmup=case["warmup"],
               num_samples=case["samples"], max_depth=case["depth"])
    if case["kind"] == "service":
        r = S.hmc_nuts_diag_e_adapt(m, **cfg)
        keep = ("rc", "draws", "stepsize", "inv_metric", "n_grad")
    else:
        r = S.hmc_nuts_diag_e_adapt_batch(m, case["C"], grad_precision=PREC[case["prec"]], **cfg)
        keep = ("draws", "rows", "status", "stepsize", "inv_metric", "n_grad")
    return {k: r[k] for k in keep}  # without the wall-clock and scheduling figures


def _dims(case):
    """Rows (hier: the expected number), parameters."""
    K = case["K"]
    if case["family"] == "hier":
        return case["J"] * case["rows"] * math.exp(0.5), 2 * K + 2 + case["J"] * (K + 1)
    return case["N"], K + (2 if case["family"] == "normal" else 1)


def work(case):
    """Bytes: X and y read once in the width the evaluation's precision holds them in (FP64 8,
    BF16 hi + lo 4, FP32 4 bytes), points read and results written once.  Flops: the two
    products with X per chain.  Sampler runs: at least one gradient per iteration and chain,
    the draws written once."""
    N, D = _dims(case)
    K, C = case["K"], case["C"]
    x = N * K * (8 if case["prec"] == "fp64" else 4)
    y = N * (8 if case["family"] == "normal" else 1)
    if case["kind"] in ("eval", "batch"):
        return {"bytes": x + y + 8.0 * C * (2 * D + 1), "flops": 4.0 * N * K * C}
    it = case["warmup"] + case["samples"]
    return {"bytes": x + y + 8.0 * C * case["samples"] * (D + 7), "flops": 4.0 * N * K * C * it}


def exact(case, seed):
    """Log density (priors without constants, Jacobian included) and gradient in 64 bits; a
    sampler run has no closed form."""
    if case["kind"] not in ("eval", "batch"):
        return None
    d = _data(case, seed)
    X, y, theta, K = d["X"], d["y"].to(torch.float64), d["theta"], case["K"]
    alpha_sd, beta_sd, sigma_sd, tau_sd = PRIOR[case["family"]]
    lps, grads = [], []
    for th in theta:  # one chain at a time: the largest temporary is a few rows' worth of X
        beta = th[1:1 + K]
        lp = -0.5 * (beta / beta_sd).square().sum()
        g = torch.zeros_like(th)
        g[1:1 + K] = -beta / beta_sd ** 2
        if alpha_sd > 0:
            lp = lp - 0.5 * (th[0] / alpha_sd) ** 2
            g[0] = -th[0] / alpha_sd ** 2
        if case["family"] == "hier":
            v, z = th[1 + K:2 + 2 * K], th[2 + 2 * K:].reshape(-1, K + 1)
            tau, gid = torch.exp(v), _group_ids(d["off"])
            w = th[:1 + K] + tau * z
            eta = w[gid, 0] + (X * w[gid, 1:]).sum(1)
        else:
            eta = X @ beta + th[0]
        if case["family"] == "normal":
            s2 = torch.exp(-2 * th[K + 1])
            r = (y - eta)
            ss = r.square().sum()
            sig = torch.exp(th[K + 1])
            lp = lp - 0.5 * ss * s2 - case["N"] * th[K + 1] - 0.5 * (sig / sigma_sd) ** 2 + th[K + 1]
            g[K + 1] = ss * s2 - case["N"] - (sig / sigma_sd) ** 2 + 1
            r = r * s2
        else:
            t = (2 * y - 1) * eta
            lp = lp + torch.nn.functional.logsigmoid(t).sum()
            r = (2 * y - 1) * torch.sigmoid(-t)
        if case["family"] == "hier":
            seg = torch.zeros_like(z)
            seg[:, 0].index_add_(0, gid, r)
            seg[:, 1:] = torch.zeros_like(z[:, 1:]).index_add_(0, gid, X * r[:, None])
            tot = seg.sum(0)
            g[:1 + K] += tot
            g[1 + K:2 + 2 * K] = tau * (z * seg).sum(0) - (tau / tau_sd) ** 2 + 1
            g[2 + 2 * K:] = (tau * seg - z).reshape(-1)
            lp = lp - 0.5 * z.square().sum() - 0.5 * (tau / tau_sd).square().sum() + v.sum()
        else:
            g[0] += r.sum()
            g[1:1 + K] += X.T @ r
        lps.append(lp)
        grads.append(g)
    lp, grad = torch.stack(lps).cpu().numpy(), torch.stack(grads).cpu().numpy()
    if case["kind"] == "eval":
        return {"lp": float(lp[0]), "grad": grad[0]}
    return {"lp": lp, "grad": grad}
