"""FP32 batches of the hierarchical model take the row chunks from the
longest to the shortest, in rounds of one wave per SIMD (FP32 products) or
one block of four chunks per CU (BF16 splits), every other round from its
end.  Every chunk must be taken exactly once whatever the number of items
in the last round: against the compensated oracle with the bars of the
FP32 batches (1e-5 log density, 1e-4 gradient, relative), a second set of
points on the same context, and chains bitwise as in a batch of their own."""
import numpy as np
import pytest

import oracle as O
import stan_amd as S
from stan_amd import workloads as W

pytestmark = pytest.mark.gpu

LP_TOL, GRAD_TOL = 1e-5, 1e-4


# chunks x blocks of 32 chains on 1024 SIMDs: 3, 1023, 1025 (an odd last
# round of one), 1402 (odd), 2049 and 2202 (even), 3302 (odd)
@pytest.mark.parametrize("J,C", [(3, 1), (1023, 5), (1025, 32), (701, 33), (683, 70), (1101, 64),
                                 (1651, 40)])
@pytest.mark.parametrize("kernel", [1, 2])
def test_every_chunk_is_taken_once(J, C, kernel):
    K = 3
    rng = np.random.default_rng(J + C)
    sizes = rng.integers(1, 40, J)
    off = np.concatenate([[0], np.cumsum(sizes)])
    X = rng.standard_normal((off[-1], K))
    y = rng.integers(0, 2, off[-1]).astype(np.int32)
    prior = (5.0, 2.0, 2.0, 1.0)
    m = S.GlmModel(S.HIER_LOGIT, X, y, offsets=off, prior=prior, precision=S.FP32,
                   tuning=dict(hier_kernel=kernel))
    ref = O.GlmData(O.HIER, X, y, offsets=off, prior=prior)
    for seed in (1, 2):
        th = np.ascontiguousarray(W.random_thetas(m.D, C, seed=seed) * 0.5)
        lp, g = m.log_prob_grad_batch(th)
        for c in sorted({0, C // 2, C - 1}):
            st, lp_r, g_r = ref.lpgrad(th[c], mode=1)
            assert st == 0
            assert abs(lp[c] - lp_r) <= LP_TOL * abs(lp_r)
            assert np.linalg.norm(g[c] - g_r) <= GRAD_TOL * np.linalg.norm(g_r)
            lp1, g1 = m.log_prob_grad_batch(th[c:c + 1])
            assert lp1[0] == lp[c] and np.array_equal(g1[0], g[c])
    m.close()


# FP64: the same rounds per chain; above 8192 chunks a wave takes several
@pytest.mark.parametrize("J", [1, 1025, 2048, 2051, 8192, 8193, 9300, 17500])
def test_every_chunk_is_taken_once_fp64(J):
    K = 2
    rng = np.random.default_rng(J)
    sizes = rng.integers(1, 6, J)
    sizes[J // 2] = 700  # three chunks
    off = np.concatenate([[0], np.cumsum(sizes)])
    X = rng.standard_normal((off[-1], K))
    y = rng.integers(0, 2, off[-1]).astype(np.int32)
    prior = (5.0, 2.0, 2.0, 1.0)
    m = S.GlmModel(S.HIER_LOGIT, X, y, offsets=off, prior=prior, precision=S.FP64)
    ref = O.GlmData(O.HIER, X, y, offsets=off, prior=prior)
    th = np.ascontiguousarray(W.random_thetas(m.D, 2, seed=J) * 0.5)
    lps, gs = m.log_prob_grad_batch(th)
    for c in range(2):
        st, lp_r, g_r = ref.lpgrad(th[c], mode=1)
        assert st == 0
        lp, g = m.log_prob_grad(th[c])
        assert lp == lps[c] and np.array_equal(g, gs[c])
        assert abs(lp - lp_r) <= 1e-12 * max(1.0, abs(lp_r))
        assert np.linalg.norm(g - g_r) <= 1e-12 * max(1.0, np.linalg.norm(g_r))
    m.close()
