"""Single FP64 evaluations: theta carried by the launch (up to 440
parameters) or copied, the cross-block reduction spread over blocks, and
results stored straight to pinned host memory.  Against the FP64 oracle
(1e-12, the plain path's bound) at the edges of each: around 440 parameters,
one to five columns (two per wave, three waves beside the first), block
counts around the reduction's 512-block step, and a run of calls whose
results must not be an earlier call's."""
import numpy as np
import pytest

import oracle as O
import stan_amd as S
from stan_amd import workloads as W

pytestmark = pytest.mark.gpu
TOL = 1e-12


def _check(m, ref, th):
    lp, g = m.log_prob_grad(th)
    st, lp_r, g_r = ref.lpgrad(th, mode=1)
    assert st == 0
    assert abs(lp - lp_r) <= TOL * max(1.0, abs(lp_r))
    assert np.linalg.norm(g - g_r) <= TOL * max(1.0, np.linalg.norm(g_r))


@pytest.mark.parametrize("family", [S.LOGIT, S.NORMAL])
@pytest.mark.parametrize("N,K,blocks", [(50, 1, 0), (300, 2, 0), (300, 3, 0), (64, 4, 0),
                                        (700, 5, 0), (900, 437, 0), (900, 438, 0),
                                        (900, 439, 0), (900, 440, 0), (40_000, 7, 511),
                                        (140_000, 6, 513), (300_000, 3, 1024)])
def test_eval_edges(family, N, K, blocks):
    print(f"eval family={family} N={N} K={K} blocks={blocks}", flush=True)
    d = W.logistic(N, K, 1.0 / np.sqrt(K), 0.5, seed=K) if family == S.LOGIT \
        else W.normal(N, K, seed=K)
    m = S.GlmModel(family, d["X"], d["y"], prior=d["prior"],
                   tuning=dict(blocks=blocks, autotune=0))
    ref = O.GlmData(family, d["X"], d["y"], prior=d["prior"])
    for th in W.random_thetas(m.D, 3, seed=N) * 0.5:
        _check(m, ref, th)
    # the batched call's chains are the single evaluations
    th = W.random_thetas(m.D, 2, seed=N + 1) * 0.5
    lp, g = m.log_prob_grad_batch(th)
    for c in range(2):
        lp1, g1 = m.log_prob_grad(th[c])
        assert lp1 == lp[c] and np.array_equal(g1, g[c])
    m.close()


def test_consecutive_evaluations_are_fresh():
    """500 different points in a row, then the same in reverse."""
    d = W.hier_logistic(J=30, K=4, seed=5, mean_log_size=np.log(30.0))
    h = S.GlmModel(S.HIER_LOGIT, d["X"], d["y"], offsets=d["offsets"], prior=d["prior"])
    e = W.logistic(500, 9, 0.3, 0.5, seed=2)
    m = S.GlmModel(S.LOGIT, e["X"], e["y"], prior=e["prior"])
    for model in (m, h):
        ths = W.random_thetas(model.D, 500, seed=3) * 0.5
        first = [model.log_prob_grad(t) for t in ths]
        again = [model.log_prob_grad(t) for t in ths[::-1]][::-1]
        assert len({lp for lp, _ in first}) == 500
        for (la, ga), (lb, gb) in zip(first, again):
            assert la == lb and np.array_equal(ga, gb)
        with pytest.raises(S.DomainError):
            model.log_prob_grad(np.full(model.D, 1e308))
        lp, g = model.log_prob_grad(ths[0])
        assert lp == first[0][0] and np.array_equal(g, first[0][1])
        model.close()


@pytest.mark.parametrize("family", [S.LOGIT, S.NORMAL])
@pytest.mark.parametrize("N,K,L,cap,blocks,C", [
    (120_011, 9, 1, 12, 384, 8), (70_001, 13, 1, 16, 300, 11), (50_000, 32, 1, 32, 77, 9),
    (64_033, 17, 2, 12, 256, 8), (61_007, 37, 2, 20, 513, 17), (300_001, 3, 2, 4, 2048, 10),
    (60_005, 60, 4, 16, 512, 8), (33_333, 63, 4, 16, 1024, 13), (30_001, 101, 4, 28, 255, 8),
    (21_000, 128, 4, 32, 512, 16), (66_000, 29, 4, 8, 64, 33)])
def test_chains_pass_is_the_single_pass(family, N, K, L, cap, blocks, C):
    """Batches large enough for the several-chains pass: every chain bitwise
    its single evaluation, over its forms (1, 2 and 4 lanes per row; slots
    odd, even and full; X values held and read again; one tile per sequence,
    odd and even tile counts; a partial last tile; block counts that do and do
    not divide by 8; a last group of 1, 2, 3 or 8 chains), and the first
    against the oracle (1e-12)."""
    print(f"chains family={family} N={N} K={K} L={L} blocks={blocks} C={C}", flush=True)
    assert N * K * C >= 1 << 23
    d = W.logistic(N, K, 1.0 / np.sqrt(K), 0.5, seed=K) if family == S.LOGIT \
        else W.normal(N, K, seed=K)
    m = S.GlmModel(family, d["X"], d["y"], prior=d["prior"],
                   tuning=dict(lanes_per_row=L, slots_cap=cap, blocks=blocks, autotune=0))
    th = W.random_thetas(m.D, C, seed=N) * 0.5
    th[3, 1] = 1e308  # eta overflows: this chain alone has no density
    lp, g = m.log_prob_grad_batch(th)
    assert np.isneginf(lp[3])
    for c in range(C):
        if c == 3:
            continue
        lp1, g1 = m.log_prob_grad(th[c])
        assert lp1 == lp[c], c
        assert np.array_equal(g1, g[c]), c
    ref = O.GlmData(family, d["X"], d["y"], prior=d["prior"])
    st, lp_r, g_r = ref.lpgrad(th[0], mode=1)
    assert abs(lp[0] - lp_r) <= TOL * abs(lp_r)
    assert np.linalg.norm(g[0] - g_r) <= TOL * np.linalg.norm(g_r)
    m.close()


def test_batch_of_a_non_finite_point():
    """A chain at a non-finite theta: -inf, its gradient row left alone, the
    others unaffected."""
    d = W.normal(900, 5, seed=3)
    m = S.GlmModel(S.NORMAL, d["X"], d["y"], prior=d["prior"])
    th = W.random_thetas(m.D, 3, seed=1) * 0.3
    th[1, 2] = np.nan
    lp, g = m.log_prob_grad_batch(th)
    assert np.isneginf(lp[1]) and np.all(g[1] == 0.0)
    for c in (0, 2):
        lp1, g1 = m.log_prob_grad(th[c])
        assert lp1 == lp[c] and np.array_equal(g1, g[c])
    m.close()


@pytest.mark.parametrize("J,C", [(3, 5), (60, 40), (60, 300), (3000, 140)])
def test_batch_staging_sizes(J, C):
    """Batches whose points go through the pinned buffer (small, and large on
    several threads), around it (between 64 KB and 1 MB), and in two slabs
    (70 MB): chains bitwise their single evaluations."""
    d = W.hier_logistic(J=J, K=20, seed=J, mean_log_size=np.log(4.0))
    m = S.GlmModel(S.HIER_LOGIT, d["X"], d["y"], offsets=d["offsets"], prior=d["prior"])
    th = W.random_thetas(m.D, C, seed=C) * 0.3
    print(f"staging J={J} C={C}: {th.nbytes} bytes", flush=True)
    lp, g = m.log_prob_grad_batch(th)
    for c in sorted({0, 1, C // 2, C - 9 if C > 9 else 0, C - 1}):
        lp1, g1 = m.log_prob_grad(th[c])
        assert lp1 == lp[c] and np.array_equal(g1, g[c]), c
    m.close()
