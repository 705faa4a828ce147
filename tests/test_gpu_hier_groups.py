"""Sums over the groups of the hierarchical model at the edges of their
blocks: 8 groups side by side, 64 groups per row of blocks; 16 threads per
group up to K = 13, 32 up to K = 29, two entries per thread above; groups
of more chunks than one round of loads takes, and empty groups.  FP64,
against the compensated oracle within 1e-12 relative (normwise for the
gradient), the bar of every FP64 evaluation; a chain of a batch is bitwise
its single evaluation."""
import numpy as np
import pytest

import oracle as O
import stan_amd as S
from stan_amd import workloads as W

pytestmark = pytest.mark.gpu

TOL = 1e-12


@pytest.mark.parametrize("J", [1, 8, 9, 64, 71])
@pytest.mark.parametrize("K", [0, 13, 14, 29, 30])
def test_group_sums_at_block_edges(J, K):
    rng = np.random.default_rng(100 * J + K)
    sizes = rng.integers(0, 60, J)
    sizes[0] = 2400 + 17 * K  # about ten chunks
    off = np.concatenate([[0], np.cumsum(sizes)])
    X = rng.standard_normal((off[-1], K))
    y = rng.integers(0, 2, off[-1]).astype(np.int32)
    prior = (5.0, 2.0, 2.0, 1.0)
    m = S.GlmModel(S.HIER_LOGIT, X, y, offsets=off, prior=prior, precision=S.FP64)
    ref = O.GlmData(O.HIER, X, y, offsets=off, prior=prior)
    thetas = np.ascontiguousarray(W.random_thetas(m.D, 5, seed=J + K) * 0.3)
    lps, gs = m.log_prob_grad_batch(thetas)
    for c in range(len(thetas)):
        st, lp_r, g_r = ref.lpgrad(thetas[c], mode=1, propto=True, jacobian=True)
        assert st == 0
        lp, g = m.log_prob_grad(thetas[c])
        assert lp == lps[c] and np.array_equal(g, gs[c])
        assert abs(lp - lp_r) <= TOL * max(1.0, abs(lp_r))
        assert np.linalg.norm(g - g_r) <= TOL * max(1.0, np.linalg.norm(g_r))
    m.close()
