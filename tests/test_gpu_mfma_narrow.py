"""Mixed-precision batches of one 32-column row: the reduction in four column
blocks per chain up to 16 chains and in one above.  Each chain bitwise the
same on either side of the line, the first within the mixed-precision bounds
(lp 2e-6, gradient 2e-5) of the FP64 oracle."""
import numpy as np
import pytest

import oracle as O
import stan_amd as S
from stan_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("family", [S.LOGIT, S.NORMAL])
@pytest.mark.parametrize("N,K", [(40, 1), (3001, 31), (100_003, 30), (50_000, 32)])
def test_narrow_rows(family, N, K):
    print(f"narrow family={family} N={N} K={K}", flush=True)
    d = W.logistic(N, K, 1.0 / np.sqrt(K), 0.5, seed=K) if family == S.LOGIT \
        else W.normal(N, K, seed=K)
    m = S.GlmModel(family, d["X"], d["y"], prior=d["prior"], precision=S.BF16X2)
    th = W.random_thetas(m.D, 64, seed=N) * 0.5
    lp, g = m.log_prob_grad_batch(th)
    for C in (1, 16, 17):
        lpc, gc = m.log_prob_grad_batch(th[:C])
        np.testing.assert_array_equal(lpc, lp[:C])
        np.testing.assert_array_equal(gc, g[:C])
    ref = O.GlmData(family, d["X"], d["y"], prior=d["prior"])
    st, lp_r, g_r = ref.lpgrad(th[0], mode=1)
    assert st == 0
    assert abs(lp[0] - lp_r) <= 2e-6 * abs(lp_r)
    assert np.linalg.norm(g[0] - g_r) <= 2e-5 * np.linalg.norm(g_r)
    m.close()
