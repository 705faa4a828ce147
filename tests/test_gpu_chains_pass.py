"""FP64 batches around the lines between the several-chains pass and the
single-chain pass over a grid of chains (more than five chains per group of
eight on average, or 2^26 products with wide rows or the normal family; from
2^23 products with one lane per row, 1.5 and 3 times that with two and four):
either way each chain is bitwise its single evaluation, and the first is
within 1e-12 of the FP64 oracle, the bound of every FP64 evaluation."""
import numpy as np
import pytest

import oracle as O
import stan_amd as S
from stan_amd import workloads as W

pytestmark = pytest.mark.gpu
TOL = 1e-12


@pytest.mark.parametrize("family,N,K,L,cap,blocks,C", [
    (S.LOGIT, 20_001, 32, 1, 32, 77, 18), (S.NORMAL, 20_001, 32, 1, 32, 300, 18),
    (S.LOGIT, 100_033, 17, 2, 12, 256, 8), (S.NORMAL, 400_001, 3, 2, 4, 2048, 12),
    (S.LOGIT, 400_001, 3, 2, 4, 513, 12), (S.LOGIT, 32_003, 101, 4, 28, 255, 8),
    (S.LOGIT, 236_001, 32, 1, 32, 512, 9), (S.NORMAL, 1_700_003, 4, 1, 4, 1024, 10),
    # the other side
    (S.LOGIT, 900_000, 1, 1, 4, 512, 10), (S.LOGIT, 24_001, 127, 4, 32, 512, 8),
    (S.NORMAL, 40_001, 20, 1, 20, 512, 9)])
def test_either_pass_is_the_single_evaluation(family, N, K, L, cap, blocks, C):
    print(f"family={family} N={N} K={K} L={L} blocks={blocks} C={C}", flush=True)
    d = W.logistic(N, K, 1.0 / np.sqrt(K), 0.5, seed=K) if family == S.LOGIT \
        else W.normal(N, K, seed=K)
    m = S.GlmModel(family, d["X"], d["y"], prior=d["prior"],
                   tuning=dict(lanes_per_row=L, slots_cap=cap, blocks=blocks, autotune=0))
    th = W.random_thetas(m.D, C, seed=N) * 0.5
    lp, g = m.log_prob_grad_batch(th)
    for c in range(C):
        lp1, g1 = m.log_prob_grad(th[c])
        assert lp1 == lp[c] and np.array_equal(g1, g[c]), c
    ref = O.GlmData(family, d["X"], d["y"], prior=d["prior"])
    st, lp_r, g_r = ref.lpgrad(th[0], mode=1)
    assert st == 0
    assert abs(lp[0] - lp_r) <= TOL * max(1.0, abs(lp_r))
    assert np.linalg.norm(g[0] - g_r) <= TOL * max(1.0, np.linalg.norm(g_r))
    m.close()


@pytest.mark.parametrize("family,N,K,L,cap", [(S.LOGIT, 60_000, 20, 1, 20), (S.NORMAL, 40_000, 60, 4, 16),
                                              (S.LOGIT, 50_001, 33, 2, 20)])
def test_device_chains_share_tiles(family, N, K, L, cap, monkeypatch):
    """16 device chains, whose captured steps hold the several-chains pass, are
    bitwise those of batches of 2 (the single-chain pass), and of the same 16
    with the steps launched directly."""
    print(f"device chains family={family} N={N} K={K} L={L}", flush=True)
    assert 2 * N * K < 1 << 23 and 16 * N * K >= {1: 2, 2: 3, 4: 6}[L] << 22
    d = W.logistic(N, K, 1.0 / np.sqrt(K), 0.5, seed=K) if family == S.LOGIT \
        else W.normal(N, K, seed=K)
    m = S.GlmModel(family, d["X"], d["y"], prior=d["prior"],
                   tuning=dict(lanes_per_row=L, slots_cap=cap, blocks=512, autotune=0))
    cfg = dict(random_seed=5, num_warmup=15, num_samples=10, max_depth=5, save_warmup=1)
    keys = ("draws", "rows", "status", "stepsize", "inv_metric", "n_grad")
    many = S.hmc_nuts_diag_e_adapt_batch(m, 16, chain=1, **cfg)
    assert np.all(many["status"] == 0)
    for first in (1, 9, 15):
        two = S.hmc_nuts_diag_e_adapt_batch(m, 2, chain=first, **cfg)
        for key in keys:
            np.testing.assert_array_equal(two[key], many[key][first - 1:first + 1])
    monkeypatch.setenv("STANX_BATCH_NO_GRAPH", "1")
    direct = S.hmc_nuts_diag_e_adapt_batch(m, 16, chain=1, **cfg)
    for key in keys:
        np.testing.assert_array_equal(direct[key], many[key])
    m.close()
