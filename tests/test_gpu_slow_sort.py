"""The slow path's sort of probability keys: rows without top-k or top-p whose
uniform asks for the last entries, so that every positive probability is
sorted, at the edges of its rounds (8192 keys) and of a wave's share (512),
with ties (stable in the index) and with probabilities from 1 down to
subnormals (all three digits), against the oracle bit for bit."""
import numpy as np
import pytest

import llmk
from gpu_util import assert_bit_exact, run_gpu, workload
from oracle import llmk_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [5000, 8191, 8192, 8193, 8705, 16385, 33001])
def test_every_probability_sorted(V):
    rng = np.random.default_rng(V)
    lg = rng.normal(0.0, 2.5, (4, V)).astype(np.float32)
    lg[1] = np.round(lg[1] * 4) / 4  # ties in hundreds
    lg[2] = rng.uniform(-100.0, 0.0, V)  # 2^-145 .. 1
    lg[2, V // 2] = 0.0
    lg[3] = 1.0  # all equal
    hist = [rng.integers(0, V, 300) for _ in range(4)]
    w = workload(lg, T=0.9, R=1.1, hists=hist, u=[0.9999, 0.9999, 0.5, 0.9999])
    s = llmk.HipSampler(max_batch=4, max_vocab=V)
    try:
        print(f"[case] V={V}", flush=True)
        gpu = run_gpu(s, w, 256)
        assert_bit_exact(w, gpu, O.sample_workload(O.MIRROR, w, out_cap=256, nthreads=8), 256, f"V={V}")
        assert s.status() == 0
    finally:
        s.close()
