"""device_batch_from_params without a GPU: every array of the batch is a view
of one packed buffer, so each is compared with one built by itself."""
import numpy as np
import pytest
import torch

import llmk
from llmk.sampler import device_batch_from_params


@pytest.mark.parametrize("B", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("masked", [False, True])
def test_fields_equal_arrays_built_one_by_one(B, masked):
    rng = np.random.default_rng(10 * B + masked)
    V = 100  # four mask words a row
    params = [llmk.SampleParams(temperature=0.5 + b, top_k=7 * b, top_p=0.9 - 0.01 * b, min_p=0.01 * b,
                                repetition_penalty=1.0 + 0.1 * b, presence_penalty=0.2 * b,
                                frequency_penalty=-0.3 * b) for b in range(B)]
    hists = [list(map(int, rng.integers(0, 2**32, n))) for n in (0, 5, 1, 0, 14, 3, 0, 2)[:B]]
    uniforms = [float(u) for u in rng.random(B)]
    mask = rng.integers(0, 2**32, (B, 8), dtype=np.uint64).astype(np.uint32)[:, ::2] if masked else None
    db = device_batch_from_params(torch.zeros(B, V), params, hists, uniforms, mask)

    want = {"uniforms": np.asarray(uniforms, np.float32),
            "top_k": np.asarray([p.top_k for p in params], np.int32),
            "hist_offsets": np.cumsum([0] + [len(h) for h in hists]).astype(np.int32),
            "hist_tokens": np.asarray(sum(hists, []) or [0], np.uint32).view(np.int32)}
    for name in ("temperature", "top_p", "min_p", "repetition_penalty", "presence_penalty",
                 "frequency_penalty"):
        want[name] = np.asarray([getattr(p, name) for p in params], np.float32)
    if masked:
        want["allow_mask"] = np.ascontiguousarray(mask).view(np.int32)
    else:
        assert db.allow_mask is None
    spans = []
    for name, x in want.items():
        t = getattr(db, name)
        assert t.dtype == (torch.float32 if x.dtype == np.float32 else torch.int32), name
        assert tuple(t.shape) == x.shape and t.is_contiguous(), name
        assert np.array_equal(t.numpy().view(np.int32), x.view(np.int32)), name
        assert (t.data_ptr() - db.uniforms.untyped_storage().data_ptr()) % 16 == 0, name
        spans.append((t.data_ptr(), t.data_ptr() + 4 * t.numel()))
    spans.sort()
    assert all(a[1] <= b[0] for a, b in zip(spans, spans[1:]))  # no array reaches into another
