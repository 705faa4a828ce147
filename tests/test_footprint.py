"""A serving job's footprint is an upper bound of the device bytes it holds
(no GPU needed: the estimate is arithmetic on its sizes)."""
import numpy as np

import stan_amd as S


def _footprint(N, J, K=0, chains=1):
    spec, keep = S.job_spec(S.HIER_LOGIT, np.zeros((N, K)), np.zeros(N, np.int32), chains,
                            offsets=np.linspace(0, N, J + 1).astype(np.int64),
                            grad_precision=S.FP64, num_warmup=0, num_samples=1)
    del keep
    return S.job_footprint(spec)


def test_hierarchical_chunk_tables_are_counted():
    """Per chunk: its entry in the sorted table (first row, rows, group, id
    and padding: 24 bytes) and its K + 3 partial sums for the context and
    every chain; per row its y."""
    chunks, chains = 4096, 3  # of 128 rows, the smallest that is tuned for
    more = _footprint(2 * 128 * chunks, 10, chains=chains) - _footprint(128 * chunks, 10, chains=chains)
    assert more >= chunks * (128 + 24 + 8 * 3 * (chains + 1))
