"""Single hierarchical evaluations store their results straight to pinned host
memory, in two launches, while the host watches.  Every call must return its
own gradient: consecutive calls at many points, with 21,042 parameters (most
of them stored by the launch before the last) and with a few hundred, bitwise
what the batched call, which waits for its stream, returns for them."""
import numpy as np
import pytest

import stan_amd as S
from stan_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("J,K,calls", [(1000, 20, 300), (3, 1, 500), (90, 32, 300)])
def test_every_word_is_this_calls(J, K, calls):
    print(f"fresh J={J} K={K}", flush=True)
    d = W.hier_logistic(J=J, K=K, seed=J, mean_log_size=np.log(30.0))
    m = S.GlmModel(S.HIER_LOGIT, d["X"], d["y"], offsets=d["offsets"], prior=d["prior"])
    th = W.random_thetas(m.D, 7, seed=K) * 0.4
    lp, g = m.log_prob_grad_batch(th)
    order = np.random.default_rng(J).integers(0, 7, calls)
    for i in order:
        lp1, g1 = m.log_prob_grad(th[i])
        assert lp1 == lp[i] and np.array_equal(g1, g[i])
    m.close()
