"""The slow path's sort of probability keys: rows without top-k or top-p whose
uniform asks for the last entries, so that every positive probability is
sorted, at the edges of its rounds (8192 keys) and of a wave's share (512),
with ties (stable in the index) and with probabilities from 1 down to
subnormals (all three digits), against the oracle bit for bit."""
import numpy as np
import pytest
import torch

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


def _call_us(lg):
    """Median time of a call that sorts every probability of every row."""
    B, V = lg.shape
    s = llmk.HipSampler(max_batch=B, max_vocab=V)
    try:
        db = llmk.DeviceBatch(logits=lg, uniforms=torch.full((B,), 0.9999, device=lg.device))
        args = s.prepare(db, torch.empty(B, dtype=torch.int32, device=lg.device))
        st, times = torch.cuda.current_stream(), []
        for _ in range(12):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record(st)
            s.launch_prepared(args, st)
            b.record(st)
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b) * 1e3)
        return float(np.median(times[2:]))
    finally:
        s.close()


@pytest.mark.parametrize("odd", [0.0, 0.05])
def test_rows_of_equal_logits_cost_no_more_than_spread_ones(odd):
    """An idle slot's row (equal logits, or all but one in twenty) has nearly
    every key in one bin of each digit.  The histogram's adds to one address
    take their turns: with every lane adding by itself such rows took 1.01
    and 1.05 of a spread row's time, added once a wave 0.73 and 0.80; the line
    lies between."""
    g = torch.Generator(device="cuda")
    g.manual_seed(7)
    B, V = 8, 151936
    spread = torch.randn(B, V, generator=g, device="cuda") * 0.02
    equal = 1.0 - (torch.rand(B, V, generator=g, device="cuda") < odd).float() * 0.1
    print(f"[case] odd={odd}", flush=True)
    a, b = _call_us(equal), _call_us(spread)
    print(f"equal {a:.0f} us, spread {b:.0f} us", flush=True)
    assert a < 0.9 * b
