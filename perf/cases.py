"""The sampling work a program gives this framework, as measurable cases.

A case is a dict of plain values that describes one call (or the few calls of
one decode step) through the public entry points:

  kind      "row"     HipSampler.sample, one row from host parameters
            "sample"  a batched sampling call
            "verify"  a sampling call and HipSampler.verify_batch on its lists
            "top_k", "top_p"  the mask forms on a copy of the logits
  B, V      rows and vocabulary
  dtype     "f32", "bf16" or "f16"
  law       how a row's logits are distributed (_logits)
  sigma     the standard deviation of the bulk of a row's logits
  T, top_k, top_p, min_p, rep, pres, freq
            the sampling parameters of every row; None leaves the array out
            (SampleParams defaults); T "mixed" draws every parameter per row
  hist, form  history tokens per row, as "csr" or as (token, "counts") tables
  mask      a grammar's allow-bitmask
  softcap   final_logit_softcapping fused into the reads (0 = off)
  pad       elements between rows past V (odd: rows at any alignment)
  cap       entries of the processed distribution returned per row (0 = none)
  plan      True: the checked arguments are kept from step to step
            (HipSampler.prepare), False: HipSampler.launch on each step

Results are the reference's bit for bit (tokens, kept counts, ids and
probabilities), whatever the order of the work, so nearly every tolerance is
"exact"; see tolerance().
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llm-rs_amd"))

import llmk  # noqa: E402

_DT = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}

_BASE = dict(kind="sample", dtype="f32", law="spikes", sigma=3.0, T=None, top_k=None, top_p=None,
             min_p=None, rep=None, pres=None, freq=None, hist=0, form="csr", mask=False,
             softcap=0.0, pad=0, cap=16, plan=True)


def _case(**kw):
    return dict(_BASE, **kw)


def listed():
    return [
        # LlmBackend::sample as a program without a scheduler calls it: one
        # row, its parameters and history on the host, the token back
        _case(name="one_row_call", kind="row", B=1, V=32000, T=0.7, top_k=40, top_p=0.9, rep=1.1,
              hist=200, cap=0, plan=False),
        # one user decoding: the smallest batched call, all latency
        _case(name="decode_1", B=1, V=151936, T=0.8, top_k=40, top_p=0.95, rep=1.1, hist=64),
        # SampleParams' own defaults (T 1, no top-k, no top-p): a draw from the
        # whole distribution, a few users, f16 straight from the lm_head
        _case(name="defaults_8", B=8, V=32000, dtype="f16", law="peaked", sigma=2.5, plan=False),
        # a scheduler's batch of requests with every kind of parameters
        _case(name="mixed_64", B=64, V=151936, dtype="bf16", sigma=2.5, T="mixed", hist=640),
        # the benchmark's shape: a full batch with top-k, top-p and penalties
        _case(name="topk_256", B=256, V=151936, law="heavy", T=0.7, top_k=50, top_p=0.95, rep=1.1,
              pres=0.5, freq=0.3, hist=2048),
        # structured output: a grammar's allow-bitmask and top-p alone
        _case(name="grammar_128", B=128, V=128256, law="flat", T=1.0, top_k=0, top_p=0.9, rep=1.1,
              hist=512, mask=True),
        # the largest: a wide vocabulary, top-k 200, min-p and device-resident
        # count-table histories
        _case(name="wide_512", B=512, V=256000, dtype="bf16", sigma=4.0, T=0.9, top_k=200,
              top_p=0.98, min_p=0.02, rep=1.0, freq=0.5, hist=4096, form="counts"),
        # the usual chat request: temperature and top-p, no top-k
        _case(name="chat_64", B=64, V=128256, dtype="bf16", law="peaked", sigma=2.5, T=0.8,
              top_p=0.95, rep=1.1, hist=300, plan=False),
        # the last position of a [batch, sequence, vocabulary] lm_head output
        # at an odd vocabulary (rows at any alignment), softcapped f16 logits
        _case(name="ragged_33", B=33, V=50257, dtype="f16", law="peaked", sigma=4.0, T=1.0,
              top_k=64, top_p=0.95, hist=96, softcap=30.0, pad=50257, plan=False),
        # speculative decoding: eight sequences' four draft positions sampled
        # and verified against the draft model's probabilities
        _case(name="verify_32", kind="verify", B=32, V=32000, law="peaked", sigma=2.5, T=0.8,
              top_k=50, top_p=0.95, hist=128, cap=64, plan=False),
        # the mask forms on a copy (the raw logits are kept for log-probabilities)
        _case(name="mask_top_k_64", kind="top_k", B=64, V=151936, law="heavy", top_k=50, cap=0),
        _case(name="mask_top_p_128", kind="top_p", B=128, V=128256, law="peaked", top_p=0.9, cap=0),
    ]


def draw(rng):
    """One more case of the ranges above: any batch and vocabulary whose
    logits are at most a third of the largest case's (a sixteenth where
    nothing bounds the tokens a row keeps), any parameters."""
    kind = rng.choice(["sample"] * 7 + ["verify", "top_k", "top_p", "row"])
    v = int(round(math.exp(rng.uniform(math.log(2000), math.log(256000)))))
    if rng.random() < 0.5:
        v = max(2048, v // 1024 * 1024)
    most = min(512, 40_000_000 // v) if kind == "sample" else min(256, 20_000_000 // v)
    b = 1 if kind == "row" else int(round(math.exp(rng.uniform(0.0, math.log(most)))))
    c = _case(kind=kind, B=b, V=v, dtype=rng.choice(["f32", "bf16", "f16"]),
              law=rng.choice(["spikes", "heavy", "peaked", "flat"]), sigma=rng.choice([2.5, 3.0, 4.0]),
              cap=rng.choice([0, 16, 64]), plan=rng.random() < 0.5)
    h = rng.choice([0, 100, 500, 2000])
    if kind == "top_p":
        c["B"] = max(1, min(b, 8_000_000 // v))
    if kind in ("top_k", "top_p"):
        c.update(dtype="f32", cap=0, **({"top_k": rng.choice([1, 20, 50, 200])} if kind == "top_k"
                                        else {"top_p": round(rng.uniform(0.8, 0.98), 3)}))
        return c
    c.update(T=round(rng.uniform(0.5, 1.2), 3), top_k=rng.choice([None, 0, 20, 50, 100, 200]),
             top_p=rng.choice([None, round(rng.uniform(0.8, 0.99), 3)]),
             min_p=rng.choice([None, None, 0.05]), hist=h)
    if h:
        c.update(rep=1.1, freq=rng.choice([None, 0.3]), pres=rng.choice([None, 0.5]),
                 form=rng.choice(["csr", "counts"]))
    if kind == "row":
        c.update(dtype="f32", cap=0, plan=False, form="csr", hist=min(h, 500),
                 top_k=c["top_k"] or 0, top_p=c["top_p"] or 1.0)
    elif kind == "verify":
        c.update(top_k=c["top_k"] or 50, cap=256)
    else:
        c.update(mask=rng.random() < 0.2, softcap=rng.choice([0.0, 0.0, 0.0, 30.0]),
                 pad=rng.choice([0, 0, 0, 1, 64]))
        if rng.random() < 0.2:
            c.update(T="mixed", rep=None, pres=None, freq=None, top_k=None, top_p=None, min_p=None)
        if not c["top_k"]:
            c["B"] = max(1, min(b, 8_000_000 // v))
    return c


# ---- inputs, made on the GPU from the seed alone ---------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _uniform(g, lo, hi, *shape):
    return torch.rand(*shape, generator=g, device="cuda") * (hi - lo) + lo


def _places(c, g, k):
    """[B, k] distinct tokens: one in each of k equal stretches of the vocabulary."""
    step = c["V"] // k
    at = torch.randint(0, step, (c["B"], k), generator=g, device="cuda")
    return at + torch.arange(k, device="cuda")[None, :] * step


def _logits(c, g):
    """float32 [B, V]: a bulk of normal logits and the tokens that stand out."""
    B, V = c["B"], c["V"]
    lg = torch.randn(B, V, generator=g, device="cuda").mul_(c["sigma"])
    if c["law"] == "heavy":  # one token in a thousand from N(8, 2^2)
        at = _places(c, g, max(1, V // 1000))
        lg.scatter_(1, at, torch.randn(at.shape, generator=g, device="cuda") * 2.0 + 8.0)
    elif c["law"] == "spikes":  # sixteen tokens raised well above the bulk
        lg.scatter_add_(1, _places(c, g, 16), _uniform(g, 6.0, 15.0, B, 16))
    elif c["law"] == "peaked":
        # rows from sure to undecided, as a model's are: a falling series of
        # tokens from a level of its own on each row
        k = min(64, V // 2)
        level = _uniform(g, 4.0, 9.0, B, 1) * c["sigma"]
        slope = _uniform(g, 0.05, 0.4, B, 1)
        order = torch.rand(B, k, generator=g, device="cuda").argsort(1).float()
        noise = torch.randn(B, k, generator=g, device="cuda") * 0.5
        lg.scatter_(1, _places(c, g, k), level - order * slope + noise)
    return lg  # "flat": the bulk alone


def _zipf(c, g):
    """[B, hist] token ids, Zipf(1) ranks of one permuted vocabulary."""
    u = torch.rand(c["B"], c["hist"], generator=g, device="cuda", dtype=torch.float64)
    rank = (torch.exp(u * math.log(c["V"] + 1)).long() - 1).clamp_(0, c["V"] - 1)
    return torch.randperm(c["V"], generator=g, device="cuda")[rank]


def _grammar(c, g):
    """int32 [B, words]: runs of 8..64 allowed tokens, a few per cent of the row."""
    B, V = c["B"], c["V"]
    runs = max(1, V * 3 // 100 // 36)
    s = torch.randint(0, max(1, V - 64), (B, runs), generator=g, device="cuda")
    n = torch.randint(8, 65, (B, runs), generator=g, device="cuda")
    words = (V + 31) // 32
    d = torch.zeros(B, words * 32 + 1, dtype=torch.int32, device="cuda")
    one = torch.ones(B, runs, dtype=torch.int32, device="cuda")
    d.scatter_add_(1, s, one)
    d.scatter_add_(1, (s + n).clamp_(max=V), -one)
    bits = (d.cumsum(1)[:, :-1] > 0).view(B, words, 32)
    out = torch.zeros(B, words, dtype=torch.int64, device="cuda")
    for i in range(32):
        out += bits[:, :, i].long() << i
    return torch.where(out >= 2**31, out - 2**32, out).int()


def _inputs(c, seed):
    """Everything a call reads, as tensors on the GPU."""
    g = _gen(seed)
    B, V = c["B"], c["V"]
    x = {"logits": _logits(c, g).to(_DT[c["dtype"]])}
    x["uniforms"] = torch.randint(0, 1 << 24, (B,), generator=g, device="cuda").float() * 2.0**-24
    full = lambda v: torch.full((B,), float(v), device="cuda")  # noqa: E731
    if c["T"] == "mixed":
        greedy = torch.rand(B, generator=g, device="cuda") < 0.25
        x["temperature"] = torch.where(greedy, full(0.0), _uniform(g, 0.5, 1.2, B))
        ks = torch.tensor([0, 20, 50, 100], dtype=torch.int32, device="cuda")
        x["top_k"] = ks[torch.randint(0, 4, (B,), generator=g, device="cuda")]
        x["top_p"] = _uniform(g, 0.8, 1.0, B)
        x["min_p"] = (torch.rand(B, generator=g, device="cuda") < 0.5).float() * 0.05
        x["repetition_penalty"] = torch.where(greedy, full(1.0), full(1.1))
        quarter = (torch.arange(B, device="cuda") % 4 == 3).float()
        x["presence_penalty"], x["frequency_penalty"] = quarter * 0.2, quarter * 0.1
    else:
        for key, name in (("T", "temperature"), ("top_p", "top_p"), ("min_p", "min_p"),
                          ("rep", "repetition_penalty"), ("pres", "presence_penalty"),
                          ("freq", "frequency_penalty")):
            if c[key] is not None:
                x[name] = full(c[key])
        if c["top_k"] is not None:
            x["top_k"] = torch.full((B,), c["top_k"], dtype=torch.int32, device="cuda")
    if c["hist"]:
        x["history"] = _zipf(c, g)
    if c["mask"]:
        x["allow_mask"] = _grammar(c, g)
    if c["kind"] == "verify":
        # the draft model: the target's logits seen through noise
        q = x["logits"].float() + torch.randn(B, V, generator=g, device="cuda") * 0.7
        x["draft_probs"] = torch.softmax(q, 1)
        x["draft_tokens"] = torch.multinomial(x["draft_probs"], 1, generator=g)[:, 0].int()
        x["u_accept"], x["u_resample"] = (_uniform(g, 0.0, 1.0, B) for _ in range(2))
    return x


def prepare(case, seed):
    c = dict(_BASE, **case)
    B, V = c["B"], c["V"]
    x = _inputs(c, seed)
    s = {"case": c, "sampler": llmk.HipSampler(max_batch=B, max_vocab=V)}
    if c["kind"] == "row":
        s["logits"] = x["logits"][0].contiguous()
        s["params"] = llmk.SampleParams(temperature=c["T"], top_k=c["top_k"], top_p=c["top_p"],
                                        repetition_penalty=c["rep"] or 1.0, min_p=c["min_p"] or 0.0,
                                        presence_penalty=c["pres"] or 0.0,
                                        frequency_penalty=c["freq"] or 0.0)
        s["history"] = x["history"][0].tolist() if c["hist"] else []
        s["u"] = float(x["uniforms"][0])
        return s
    if c["kind"] in ("top_k", "top_p"):
        s["logits"], s["param"] = x["logits"], x[c["kind"]]
        s["masked"] = torch.empty_like(x["logits"])
        return s
    lg = x["logits"]
    if c["pad"]:
        wide = torch.zeros(B, V + c["pad"], dtype=lg.dtype, device="cuda")
        wide[:, c["pad"]:] = lg
        lg = wide[:, c["pad"]:]
    db = llmk.DeviceBatch(logits=lg, uniforms=x["uniforms"], vocab=V, softcap=c["softcap"],
                          allow_mask=x.get("allow_mask"))
    for name in ("temperature", "top_k", "top_p", "min_p", "repetition_penalty", "presence_penalty",
                 "frequency_penalty"):
        setattr(db, name, x.get(name))
    if c["hist"] and c["form"] == "csr":
        db.hist_offsets = (torch.arange(B + 1, device="cuda") * c["hist"]).int()
        db.hist_tokens = x["history"].reshape(-1).int()
    elif c["hist"]:
        rows = torch.arange(B, device="cuda")[:, None]
        key, n = torch.unique(rows * V + x["history"], return_counts=True)
        bound = torch.arange(B + 1, device="cuda") * V
        db.hist_offsets = torch.searchsorted(key, bound).int()
        db.hist_tokens, db.hist_counts = (key % V).int(), n.int()
    s["batch"] = db
    s["tok"] = torch.zeros(B, dtype=torch.int32, device="cuda")
    s["cnt"] = torch.zeros(B, dtype=torch.int32, device="cuda")
    s["ids"] = s["probs"] = None
    if c["cap"]:
        s["ids"] = torch.zeros(B, c["cap"], dtype=torch.int32, device="cuda")
        s["probs"] = torch.zeros(B, c["cap"], device="cuda")
    if c["plan"]:
        s["args"] = s["sampler"].prepare(db, s["tok"], s["ids"], s["probs"], s["cnt"])
        s["stream"] = torch.cuda.current_stream()
    if c["kind"] == "verify":
        s["verify"] = [x[k] for k in ("draft_tokens", "draft_probs", "u_accept", "u_resample")]
    return s


def run(state):
    c, sampler = state["case"], state["sampler"]
    if c["kind"] == "row":
        return sampler.sample(state["logits"], state["params"], state["history"], state["u"])
    if c["kind"] in ("top_k", "top_p"):
        out = state["masked"]
        out.copy_(state["logits"])
        (sampler.apply_top_k if c["kind"] == "top_k" else sampler.apply_top_p)(out, state["param"])
        return out
    if c["plan"]:
        sampler.launch_prepared(state["args"], state["stream"])
    else:
        sampler.launch(state["batch"], state["tok"], state["ids"], state["probs"], state["cnt"])
    out = {"tokens": state["tok"], "count": state["cnt"]}
    if c["cap"]:
        out["ids"], out["probs"] = state["ids"], state["probs"]
    if c["kind"] == "verify":
        d, q, ua, ur = state["verify"]
        out["verified"], out["accepted"] = sampler.verify_batch(
            state["ids"], state["probs"], state["cnt"], d, q, ua, ur)
    return out


def work(case):
    """The logits once, histories, mask, parameters and results; per logit the
    division, subtraction, exponential and addition of a softmax."""
    c = dict(_BASE, **case)
    B, V = c["B"], c["V"]
    n = B * V * (4 if c["dtype"] == "f32" else 2) + 36 * B
    if c["kind"] in ("top_k", "top_p"):
        return {"bytes": n + 4 * B * V, "flops": (4 if c["kind"] == "top_p" else 1) * B * V}
    n += 4 * B * c["hist"] + 8 * B * c["cap"]
    if c["mask"]:
        n += 4 * B * ((V + 31) // 32)
    if c["kind"] == "verify":  # the draft's probabilities of the listed tokens
        n += 4 * B * c["cap"] + 16 * B
    return {"bytes": n, "flops": 4 * B * V}


def tolerance(case):
    """Tokens, kept counts, ids and masks are the reference's sequential f32
    arithmetic bit for bit, in whatever order the work is done.  Only a row
    that top-k renormalises may be sampled with another normaliser (it cancels
    up to rounding): its few divisions and sums of 2^-24 each show 2e-7."""
    c = dict(_BASE, **case)
    if c["kind"] in ("sample", "verify") and c["cap"] and (c["top_k"] or c["T"] == "mixed"):
        return {"rel": 8e-7, "max": 4e-6, "differ": 0.0}
    return "exact"


# ---- the same results in 64 bits, with plain torch --------------------------

def _row64(c, x, b):
    """The processed distribution of row b: (probabilities, descending)."""
    v = x["logits"][b].double()
    get = lambda k, d: float(x[k][b]) if k in x else d  # noqa: E731
    if c["softcap"]:
        v = c["softcap"] * torch.tanh(v / c["softcap"])
    if c["hist"]:
        t, n = torch.unique(x["history"][b], return_counts=True)
        rp = get("repetition_penalty", 1.0)
        y = v[t]
        y = torch.where(y > 0, y / rp, y * rp)
        v[t] = y - (get("presence_penalty", 0.0) + n.double() * get("frequency_penalty", 0.0))
    if c["mask"]:
        e = torch.arange(c["V"], device="cuda")
        v = torch.where((x["allow_mask"][b][e >> 5].long() >> (e & 31)) & 1 == 1, v, float("-inf"))
    T = get("temperature", 1.0)
    if T <= 1e-5:
        return torch.ones(1, dtype=torch.float64, device="cuda")
    p = torch.softmax(v / T, 0).sort(descending=True, stable=True).values
    mp = get("min_p", 0.0)
    if mp > 0:
        p = p[p >= mp * p[0]]
        p = p / p.sum()
    k = int(get("top_k", 0))
    if 0 < k < p.numel():
        p = p[:k] / p[:k].sum()
    tp = get("top_p", 1.0)
    if tp < 1:
        cum = p.cumsum(0)
        n = int(torch.searchsorted(cum, torch.tensor(tp, dtype=torch.float64, device="cuda"))) + 1
        p = p[:n] / p[:n].sum()
    return p


def exact(case, seed):
    c = dict(_BASE, **case)
    if c["kind"] == "row":
        return None  # a token alone
    x = _inputs(c, seed)
    B, V = c["B"], c["V"]
    if c["kind"] == "top_k":
        k = min(max(c["top_k"], 1), V)
        kth = x["logits"].topk(k, 1).values[:, -1:]
        lg = x["logits"].double()
        return torch.where(x["logits"] < kth, float("-inf"), lg)
    if c["kind"] == "top_p":
        lg = x["logits"].double()
        for b in range(B):
            p, i = torch.softmax(lg[b], 0).sort(descending=True, stable=True)
            tp = torch.tensor(c["top_p"], dtype=torch.float64, device="cuda")
            lg[b, i[int(torch.searchsorted(p.cumsum(0), tp)) + 1:]] = float("-inf")
        return lg
    if not c["cap"]:
        return None  # whole numbers alone
    probs = torch.zeros(B, c["cap"], dtype=torch.float64, device="cuda")
    for b in range(B):
        p = _row64(c, x, b)[: c["cap"]]
        probs[b, : p.numel()] = p
    out = {"tokens": None, "count": None, "ids": None, "probs": probs}
    if c["kind"] == "verify":
        out["verified"] = out["accepted"] = None
    return out
