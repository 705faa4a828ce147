"""Device-resident chains bound the phase turns of one launch where a batched
gradient is cheap (FP32 / BF16 gradients, at least 32 coordinates and 2048
over all chains, N K chains <= 2^30).  A yield changes neither the arithmetic
nor the random stream: draws and diagnostics are bitwise those of an
unbounded run on both sides of the rule, and only a bounded run takes more
steps."""
import os

import numpy as np
import pytest

import stan_amd as S

pytestmark = pytest.mark.gpu


def _model(family, N, K, precision):
    rng = np.random.default_rng(11)
    X = rng.standard_normal((N, K)) / np.sqrt(K)
    beta = rng.standard_normal(K)
    if family == S.LOGIT:
        y = (rng.random(N) < 1 / (1 + np.exp(-(X @ beta)))).astype(np.int32)
    else:
        y = X @ beta + rng.standard_normal(N)
    prior = (5.0, 2.0, 2.0, 1.0) if family == S.LOGIT else (0.0, 1.0, 2.0, 1.0)
    return S.GlmModel(family, X, y, precision=precision, prior=prior)


def _run(m, chains, precision, budget):
    if budget is not None:
        os.environ["STANX_NUTS_PHASE_BUDGET"] = budget
    try:
        b = S.NutsBatch(m, chains, grad_precision=precision, random_seed=3, chain=1,
                        num_warmup=15, num_samples=10, max_depth=7, save_warmup=1)
    finally:
        os.environ.pop("STANX_NUTS_PHASE_BUDGET", None)
    n = 0
    while True:
        steps, done = b.run(max_steps=256)
        n += steps
        if done >= chains or steps == 0:
            break
    r = b.results()
    b.close()
    return r, n


@pytest.mark.parametrize("family,N,K,chains,precision,bounded", [
    ("logit", 500, 31, 64, "bf16", True),    # D = 32, 2048 coordinates: the smallest
    ("logit", 500, 30, 67, "bf16", False),   # D = 31
    ("logit", 500, 31, 63, "bf16", False),   # 2016 coordinates
    ("normal", 700, 100, 24, "bf16", True),
    ("logit", 500, 31, 64, "fp64", False),
])
def test_bounded_launches_leave_draws_unchanged(family, N, K, chains, precision, bounded):
    prec = S.BF16X2 if precision == "bf16" else S.FP64
    m = _model(S.LOGIT if family == "logit" else S.NORMAL, N, K, prec)
    got, n = _run(m, chains, prec, None)
    ref, nref = _run(m, chains, prec, "4096")
    assert np.all(got["status"] == 0)
    for key in ("draws", "rows", "status", "stepsize", "inv_metric", "n_grad"):
        assert np.array_equal(got[key], ref[key]), key
    assert n > nref if bounded else n == nref
    m.close()
