"""The slow path's sort of probability keys: rows whose draw lies past the
candidate path's reach and whose uniform leaves no probability out, so that
every positive one is sorted, at the edges of its rounds (8192 keys) and of a
wave's share (512), with ties (stable in the index) and with probabilities
from 1 down to subnormals and zero (all three digits), in every dtype, with a
mask and with a history past the LDS tables; and a row that is sorted twice.
Against the oracle bit for bit."""
import numpy as np
import pytest
import torch

import band_util as BU
import llmk
from gpu_util import assert_bit_exact, run_gpu, workload
from oracle import llmk_oracle as O

pytestmark = pytest.mark.gpu
CANDIDATES = 1024  # a row without top-k that draws past these takes the slow path
U = 0.9999  # within 0.002 of 1: every bin of the row is chosen


def _rows(V, rng):
    lg = rng.normal(0.0, 2.5, (4, V)).astype(np.float32)
    lg[1] = np.round(lg[1] * 4) / 4  # ties in hundreds
    lg[2] = rng.uniform(-100.0, 0.0, V)  # 2^-160 .. 1 at T 0.9: subnormals and zeros too
    lg[2, rng.permutation(V)[:2000]] = rng.uniform(-2.0, 0.0, 2000)
    lg[2, V // 2] = 0.0
    lg[3] = 1.0  # all equal
    return lg


def _check(w, label):
    """Every row's draw lies past the candidates, and the outputs are the oracle's."""
    full = O.sample_workload(O.MIRROR, w, out_cap=w.V, nthreads=8)
    for b in range(w.B):
        assert int(np.nonzero(full[2][b] == full[1][b])[0][0]) > CANDIDATES, (label, b)
    s = llmk.HipSampler(max_batch=w.B, max_vocab=w.V)
    try:
        print(f"[case] {label}", flush=True)
        gpu = run_gpu(s, w, 256)
        assert_bit_exact(w, gpu, O.sample_workload(O.MIRROR, w, out_cap=256, nthreads=8), 256, label)
        return s.status()
    finally:
        s.close()


@pytest.mark.parametrize("V", [5000, 8191, 8192, 8193, 8705, 16385, 33001])
def test_every_probability_sorted(V):
    rng = np.random.default_rng(V)
    hist = [rng.integers(0, V, 300) for _ in range(4)]
    w = workload(_rows(V, rng), T=0.9, R=1.1, hists=hist, u=U)
    assert _check(w, f"V={V}") == 0


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_half_precision_rows_under_a_mask(dtype):
    V = 17001
    rng = np.random.default_rng(V)
    mask = rng.integers(0, 1 << 32, (4, (V + 31) // 32), dtype=np.uint64).astype(np.uint32)
    hist = [rng.integers(0, V, 300) for _ in range(4)]
    w = workload(_rows(V, rng), T=0.9, R=1.1, hists=hist, u=U, mask=mask, dtype=dtype)
    assert _check(w, f"masked {dtype}") == 0


def test_materialised_rows():
    """More distinct history tokens than the LDS tables hold: the row's logits
    lie beside the sort's lists."""
    V = 17001
    rng = np.random.default_rng(V)
    hist = [rng.permutation(V)[:9000] for _ in range(4)]
    w = workload(_rows(V, rng), T=0.9, R=1.1, FR=0.1, hists=hist, u=U)
    assert _check(w, "materialised") == llmk._lib.LLMK_STATUS_HISTORY_OVERFLOW


def test_rows_sorted_twice():
    """top-k above the candidate path's 1024, with a uniform between the
    cumulatives of S = 1 and of the reference's S at one entry: no band can
    prove that draw, so S is computed and the row gathered and sorted again,
    after the first sort has overwritten the history's token table."""
    V, K = 17001, 2000
    rng = np.random.default_rng(V)
    lg = rng.normal(0.0, 2.5, (12, V)).astype(np.float32)
    w = workload(lg, T=0.9, K=K, R=1.1, hists=[rng.integers(0, V, 300) for _ in range(12)])
    hit = 0
    for b in range(w.B):
        prm = BU.row_params(w, b)
        es, ix = O.sorted_e(w.logits[b], prm, BU.row_hist(w, b), None, n=K + 1)
        ref = BU.cumulative(BU.kept(O.REF, w, b, prm, 0.5, K)[3][:K])
        one = BU.cumulative(BU.kept("s1", w, b, prm, 0.5, K, es, ix)[3][:K])
        between = [u for u in map(BU.grid_between, ref[100:1900], one[100:1900]) if u is not None]
        if between:
            w.uniforms[b] = np.float32(between[len(between) * b // w.B])
            hit += 1
    assert hit >= 4
    s = llmk.HipSampler(max_batch=w.B, max_vocab=V)
    try:
        print(f"[case] {hit} rows sorted twice", flush=True)
        gpu = run_gpu(s, w, 256)
        assert_bit_exact(w, gpu, O.sample_workload(O.MIRROR, w, out_cap=256, nthreads=8), 256, "sorted twice")
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
