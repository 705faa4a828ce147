"""Mixed-precision batches at the edges of their column blocks: the reduction
in four column blocks per chain (up to 64 chains) or one (more), and, above K
= 256, the adjoint in blocks of 128 columns with and without a last one of
64.  Each chain bitwise the same in a batch of 64, alone and in a batch of
70; the first within the mixed-precision bounds (lp 2e-6, gradient 2e-5) of
the FP64 oracle."""
import numpy as np
import pytest

import oracle as O
import stan_amd as S
from stan_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("family", [S.LOGIT, S.NORMAL])
@pytest.mark.parametrize("N,K", [(33, 1), (700, 32), (5000, 33), (900, 96), (40_000, 97),
                                 (1100, 160), (2000, 200), (600, 225), (3000, 256), (900, 257),
                                 (4100, 320), (1500, 321), (700, 384), (2100, 400), (1000, 448),
                                 (9000, 449), (1200, 512)])
def test_column_blocks(family, N, K):
    print(f"mfma blocks family={family} N={N} K={K}", flush=True)
    d = W.logistic(N, K, 1.0 / np.sqrt(K), 0.5, seed=K) if family == S.LOGIT \
        else W.normal(N, K, seed=K)
    m = S.GlmModel(family, d["X"], d["y"], prior=d["prior"], precision=S.BF16X2)
    th = W.random_thetas(m.D, 70, seed=N) * 0.5
    lp, g = m.log_prob_grad_batch(th)
    lp64, g64 = m.log_prob_grad_batch(th[:64])
    np.testing.assert_array_equal(lp64, lp[:64])
    np.testing.assert_array_equal(g64, g[:64])
    lp1, g1 = m.log_prob_grad_batch(th[69:])
    assert lp1[0] == lp[69] and np.array_equal(g1[0], g[69])
    ref = O.GlmData(family, d["X"], d["y"], prior=d["prior"])
    st, lp_r, g_r = ref.lpgrad(th[0], mode=1)
    assert abs(lp[0] - lp_r) <= 2e-6 * abs(lp_r)
    assert np.linalg.norm(g[0] - g_r) <= 2e-5 * np.linalg.norm(g_r)
    m.close()
