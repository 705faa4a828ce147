"""With few device chains no launch is bounded in its phase turns: hardly ever
is one of them closing a subtree while others wait, and a yield only adds a
gradient; likewise where a gradient is dear for the few chains it serves.  The
lines (hierarchical model 8 chains from 500 coordinates on and 16 below, the
others 24; 2^17 rows per chain of a padded tile) show in the number of steps:
equal to an unbounded run's below, more above; draws bitwise the same."""
import os

import numpy as np
import pytest

import stan_amd as S

pytestmark = pytest.mark.gpu


def _glm(N, K):
    rng = np.random.default_rng(11)
    X = rng.standard_normal((N, K)) / np.sqrt(K)
    y = (rng.random(N) < 1 / (1 + np.exp(-(X @ rng.standard_normal(K))))).astype(np.int32)
    return S.GlmModel(S.LOGIT, X, y, precision=S.BF16X2)


def _hier(J, K):
    rng = np.random.default_rng(12)
    off = np.concatenate([[0], np.cumsum(rng.integers(1, 20, J))])
    X = rng.standard_normal((off[-1], K)) / np.sqrt(K)
    y = rng.integers(0, 2, off[-1]).astype(np.int32)
    return S.GlmModel(S.HIER_LOGIT, X, y, offsets=off, precision=S.FP32)


def _run(m, chains, precision, budget):
    if budget is not None:
        os.environ["STANX_NUTS_PHASE_BUDGET"] = budget
    try:
        b = S.NutsBatch(m, chains, grad_precision=precision, random_seed=3, chain=1,
                        num_warmup=12, num_samples=8, max_depth=6)
    finally:
        os.environ.pop("STANX_NUTS_PHASE_BUDGET", None)
    n, done = b.run(max_steps=40_000)
    assert done == chains
    r = b.results()
    b.close()
    return r, n


@pytest.mark.parametrize("kind,size,chains,bounded", [
    ("glm", (300, 100), 23, False), ("glm", (300, 100), 24, True),
    ("glm", (300, 511), 5, False),
    ("glm", (65_000, 31), 64, True), ("glm", (65_000, 31), 70, True),
    ("glm", (132_000, 31), 64, False), ("glm", (75_000, 31), 70, False),
    ("hier", (90, 4), 15, False), ("hier", (90, 4), 16, True),     # D = 460
    ("hier", (100, 4), 7, False), ("hier", (100, 4), 8, True),     # D = 510
    ("hier", (498, 4), 1, False)])                                 # D = 2500
def test_few_chains_are_not_bounded(kind, size, chains, bounded):
    print(f"phase turns {kind} {size} chains={chains}", flush=True)
    m = _glm(*size) if kind == "glm" else _hier(*size)
    precision = S.BF16X2 if kind == "glm" else S.FP32
    got, n = _run(m, chains, precision, None)
    ref, nref = _run(m, chains, precision, "4096")
    assert np.all(got["status"] == 0)
    for key in ("draws", "rows", "status", "stepsize", "inv_metric", "n_grad"):
        assert np.array_equal(got[key], ref[key]), key
    assert n > nref if bounded else n == nref
    m.close()
