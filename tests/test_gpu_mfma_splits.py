"""The row splits of the mixed-precision pass that a tuned context may choose:
4 to 128 tiles of 32 rows per split, and those that give half, one and two
splits per CU, forced one after the other through a tuning file.  Against the
FP64 oracle with the mixed-precision bounds (lp 2e-6, gradient 2e-5); a chain
of a batch of 3 bitwise as in a batch of 70."""
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle as O
import stan_amd as S
from stan_amd import workloads as W

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHILD = """
import sys
import numpy as np
sys.path.insert(0, sys.argv[1])
import stan_amd as S
from stan_amd import workloads as W
out = {}
for i, (fam, N, K, want) in enumerate(eval(sys.argv[3])):
    d = W.logistic(N, K, 1.0 / np.sqrt(K), 0.5, seed=K) if fam == S.LOGIT else W.normal(N, K, seed=K)
    m = S.GlmModel(fam, d["X"], d["y"], prior=d["prior"], precision=S.BF16X2, tuning=dict(autotune=1))
    print(fam, N, K, want, m.tuning_log().strip().splitlines()[-1], flush=True)
    th = W.random_thetas(m.D, 70, seed=N) * 0.5
    out[f"lp{i}"], out[f"g{i}"] = m.log_prob_grad_batch(th)
    out[f"lq{i}"], out[f"h{i}"] = m.log_prob_grad_batch(th[:3])
    m.close()
np.savez(sys.argv[2], **out)
"""


def _run(tmp_path, cases, cache):
    npz = str(tmp_path / f"out{len(cases)}.npz")
    r = subprocess.run([sys.executable, "-c", CHILD, ROOT, npz, repr(cases)], capture_output=True,
                       text=True, timeout=100, env={**os.environ, "STANX_TUNING_CACHE": str(cache)})
    assert r.returncode == 0, r.stdout + r.stderr
    return np.load(npz), r.stdout


def test_forced_splits(tmp_path):
    cache = tmp_path / "tuning"
    # one tuned context names the device in the file
    _run(tmp_path, [(S.LOGIT, 700, 5, 0)], cache)
    device = cache.read_text().split()[0]
    # rows (odd sizes), columns, kernel variant, tiles per split
    forced = [(S.LOGIT, 9_001, 100, 2, 1), (S.LOGIT, 9_002, 100, 0, 2), (S.NORMAL, 9_003, 100, 0, 3),
              (S.LOGIT, 9_004, 64, 2, 25), (S.NORMAL, 20_005, 256, 1, 5), (S.LOGIT, 20_006, 256, 0, 49),
              (S.NORMAL, 9_007, 468, 0, 3), (S.LOGIT, 9_008, 468, 0, 13), (S.LOGIT, 40_009, 30, 0, 128)]
    with open(cache, "a") as f:
        for fam, N, K, variant, tps in forced:
            f.write(f"{device} {100 + fam} {N} {K} {variant} {tps} 0 0\n")
    cases = [(fam, N, K, tps) for fam, N, K, _, tps in forced]
    out, log = _run(tmp_path, cases, cache)
    print(log, flush=True)
    assert log.count("MFMA pass cached") == len(cases), log
    for i, (fam, N, K, tps) in enumerate(cases):
        d = W.logistic(N, K, 1.0 / np.sqrt(K), 0.5, seed=K) if fam == S.LOGIT \
            else W.normal(N, K, seed=K)
        ref = O.GlmData(fam, d["X"], d["y"], prior=d["prior"])
        th = W.random_thetas(K + (1 if fam == S.LOGIT else 2), 70, seed=N) * 0.5
        np.testing.assert_array_equal(out[f"lq{i}"], out[f"lp{i}"][:3])
        np.testing.assert_array_equal(out[f"h{i}"], out[f"g{i}"][:3])
        for c in (0, 69):
            st, lp_r, g_r = ref.lpgrad(th[c], mode=1)
            assert st == 0
            assert abs(out[f"lp{i}"][c] - lp_r) <= 2e-6 * abs(lp_r), (N, K, tps)
            assert np.linalg.norm(out[f"g{i}"][c] - g_r) <= 2e-5 * np.linalg.norm(g_r), (N, K, tps)
