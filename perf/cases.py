"""Performance cases of the sampler: what a decode or prefill step asks of this library,
through its public Python entry points (which call the C ABI with device pointers).

Kinds of call:
  sample    GpuSampler.sample_device with finite pools (top-k / top-p / temperature per row)
  nucleus   GpuSampler.sample_device with top-k 0: top-p over the whole vocabulary
  argmax    GpuSampler.argmax_device, greedy decoding
  lmhead    LmHeadQ4.logits, the int4 lm_head product
  fused     GpuSampler.sample_lmhead_q4_device, the lm_head fused with sampling
  softmax   softmax_rows, the attention scores' row softmax

Each case is a dict of plain values; ``prepare`` makes its inputs on the GPU from a seed,
``run`` is one call, ``exact`` the same outputs in 64 bits by plain torch.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from tabby_amd import sampler as S

MASK32 = 0xFFFFFFFF


# ---------------------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------------------

def _sample(name, rows, vocab, dtype="f32", values="spiky", k="50", k_max=64, t="0.7", p="0.9", lists=0):
    return {"name": name, "kind": "sample", "rows": rows, "vocab": vocab, "dtype": dtype, "values": values,
            "k": k, "k_max": k_max, "t": t, "p": p, "lists": lists}


def listed():
    return [
        # One sequence's decode step over a large vocabulary: latency.
        _sample("one_row", 1, 151936, t="0.8"),
        # A serving batch of ordinary size; half-precision logits as most engines emit them.
        _sample("batch32_f16", 32, 128000, dtype="f16", k="40"),
        # A full serving batch, each sequence with its own parameters (one row per CU).
        _sample("batch256", 256, 151936, k="1,20,50,100", k_max=128, t="0.5,0.7,1.0", p="0.8,0.95,1.0"),
        # A batch that divides evenly into nothing: odd vocabulary, more rows than CUs, and the
        # top-20 log-probability lists that an API with `logprobs` returns.
        _sample("ragged_lists", 391, 50257, k="20,40,64", t="0.7,1.0", p="0.9,1.0", lists=20),
        # Constrained decoding: a third of the vocabulary masked to -inf, coarse (tied) logits,
        # large pools.
        _sample("masked_pool1024", 512, 151936, values="tied", k="1024", k_max=1024, t="1.0", p="0.98"),
        # Nucleus sampling with top-k off, cold and f16: almost all mass in a few tokens.
        {"name": "nucleus_cold_f16", "kind": "nucleus", "rows": 64, "vocab": 151936, "dtype": "f16", "sigma": 3.0,
         "t": "0.3", "p": "0.95"},
        # Nucleus sampling with top-k off at chat temperatures: some rows' cuts lie deep in the
        # sorted vocabulary.
        {"name": "nucleus_warm", "kind": "nucleus", "rows": 16, "vocab": 151936, "dtype": "f32", "sigma": 2.5,
         "t": "0.7,1.0", "p": "0.9,0.95"},
        # Greedy decoding of a small batch.
        {"name": "argmax32", "kind": "argmax", "rows": 32, "vocab": 151936, "dtype": "f32"},
        # The last layer of a decode step, one sequence: lm_head and sampling in one call.
        {"name": "lmhead_fused1", "kind": "fused", "rows": 1, "vocab": 151936, "hidden": 896, "block": 32},
        # The lm_head of eight sequences decoded together.
        {"name": "lmhead_logits8", "kind": "lmhead", "rows": 8, "vocab": 151936, "hidden": 896, "block": 32},
        # Attention softmax, prefill: 14 heads x 512 causal queries over 512 positions.
        {"name": "softmax_prefill", "kind": "softmax", "heads": 14, "queries": 512, "cache": 0},
        # Attention softmax, decode: one query per head over a 4,096-token cache.
        {"name": "softmax_decode", "kind": "softmax", "heads": 14, "queries": 1, "cache": 4095},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the listed ranges: 1-512 rows, vocabularies of 32,000-151,936 (odd
    ones included), both logit types, pools of 1-1,024 and the whole vocabulary, lm_heads of
    1-16 rows, softmaxes from one decode query to a 1,024-token prefill."""
    kind = rng.choice(["sample", "sample", "pool", "nucleus", "argmax", "lmhead", "fused", "prefill", "decode"])
    vocab = _log_int(rng, 32000, 151936)
    dtype = rng.choice(["f32", "f16"])
    if rng.random() < 0.6:
        vocab -= vocab % 64
    if kind == "sample":
        k = rng.choice(["1", "20", "40", "50", "1,20,50,100", "64", "100"])
        c = _sample("", _log_int(rng, 1, 512), vocab, dtype=dtype, values=rng.choice(["spiky", "spiky", "tied"]), k=k,
                    k_max=128 if "100" in k else 64, t=rng.choice(["0.7", "1.0", "0.5,0.7,1.0", "0.0,0.8"]),
                    p=rng.choice(["0.9", "0.95", "1.0", "0.8,0.95,1.0"]), lists=rng.choice([0, 0, 5, 20]))
    elif kind == "pool":
        k = rng.randint(257, 1024)
        c = _sample("", _log_int(rng, 1, 512), vocab, dtype=dtype, values=rng.choice(["spiky", "tied"]), k=str(k),
                    k_max=1024, t=rng.choice(["0.7", "1.0"]), p=rng.choice(["0.95", "0.98", "1.0"]))
    elif kind == "nucleus":
        c = {"kind": "nucleus", "rows": _log_int(rng, 1, 64), "vocab": vocab, "dtype": dtype,
             "sigma": rng.choice([2.0, 2.5, 3.0]), "t": rng.choice(["0.3", "0.7", "0.7,1.0", "1.0"]),
             "p": rng.choice(["0.9", "0.95", "0.8,0.95"])}
    elif kind == "argmax":
        c = {"kind": "argmax", "rows": _log_int(rng, 1, 512), "vocab": vocab, "dtype": dtype}
    elif kind in ("lmhead", "fused"):
        block = rng.choice([32, 32, 64, 128])
        c = {"kind": kind, "rows": rng.randint(1, 16) if kind == "lmhead" else rng.randint(1, 4), "vocab": vocab,
             "hidden": block * rng.randint(-(-512 // block), 1536 // block), "block": block}
    elif kind == "prefill":
        c = {"kind": "softmax", "heads": rng.choice([8, 14, 16]), "queries": _log_int(rng, 17, 1024),
             "cache": rng.choice([0, 0, rng.randint(1, 512)])}
    else:
        c = {"kind": "softmax", "heads": rng.randint(8, 64), "queries": rng.choice([1, 1, 2, 4]),
             "cache": _log_int(rng, 127, 8191)}
    c.pop("name", None)
    return c


# ---------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _handle(vocab, rows, k_max):
    """The handle a program creates once for its shape and keeps."""
    return S.GpuSampler(vocab_max=vocab, rows_max=rows, k_max=k_max)


def _floats(text):
    return [float(v) for v in text.split(",")]


def _rng(seed, purpose):
    return torch.Generator(device="cuda").manual_seed((seed * 1000003 + purpose) & MASK32)


def _logits(case, seed):
    """Logits of [rows, vocab]: N(0, sigma^2) with eight spikes a row of +12..+18 (the peaky
    output of an lm_head), or N(0, 2^2) rounded to quarters with 30 % of entries -inf."""
    rows, vocab, g = case["rows"], case["vocab"], _rng(seed, 1)
    if case.get("values") == "tied":
        x = torch.empty((rows, vocab), device="cuda").normal_(0.0, 2.0, generator=g)
        x = torch.round(x * 4.0) * 0.25
        x[torch.rand((rows, vocab), device="cuda", generator=g) < 0.3] = -math.inf
    else:
        x = torch.empty((rows, vocab), device="cuda").normal_(0.0, case.get("sigma", 3.0), generator=g)
        at = torch.randint(0, vocab, (rows, 8), device="cuda", generator=g)
        x.scatter_add_(1, at, 12.0 + 6.0 * torch.rand((rows, 8), device="cuda", generator=g))
    return x.half() if case.get("dtype") == "f16" else x


def _params(case, seed):
    """Per-row parameters: each of k, T and p drawn from the case's choices, one 32-bit
    uniform per row (SeededRandom's resolution)."""
    rows = case["rows"]
    r = np.random.RandomState((seed * 7919 + 3) & MASK32)
    params = np.zeros(rows, dtype=S.PARAMS_DTYPE)
    params["top_k"] = r.choice(np.array([int(v) for v in case.get("k", "40").split(",")]), rows)
    if case["kind"] == "nucleus":
        params["top_k"] = 0
    params["temperature"] = r.choice(np.array(_floats(case.get("t", "0.7"))), rows)
    params["top_p"] = r.choice(np.array(_floats(case.get("p", "0.9"))), rows)
    params["uniform"] = r.randint(0, 1 << 32, rows, dtype=np.int64) / 4294967296.0
    return params


def _results(rows):
    """A results buffer and views of its fields."""
    buf = torch.zeros(rows * S.RESULT_DTYPE.itemsize, dtype=torch.uint8, device="cuda")
    i4, f4, f8 = (buf.view(t).view(rows, -1) for t in (torch.int32, torch.float32, torch.float64))
    out = {"id": i4[:, 0], "considered": i4[:, 1], "probability": f8[:, 1], "pool_mass": f8[:, 2],
           "max_logit": f4[:, 6], "pool_exhausted": i4[:, 7], "sum_exp": f8[:, 4], "status": i4[:, 10],
           "topk_count": i4[:, 11]}
    return buf, out


def _head_inputs(case, seed):
    """Random int4 codes and block scales in the reference's layout, and hidden states that
    put the logits near N(0, 3^2)."""
    vocab, hidden, block, g = case["vocab"], case["hidden"], case["block"], _rng(seed, 2)
    words = torch.randint(-(1 << 31), 1 << 31, (vocab * hidden // 8,), device="cuda", generator=g, dtype=torch.int64)
    words = words.to(torch.int32)
    n = vocab * hidden // block
    mag = (0.04 + 0.01 * torch.rand(n, device="cuda", generator=g)) / 8.0
    sign = torch.where(torch.rand(n, device="cuda", generator=g) < 0.5, 1.0, -1.0)
    scales = (mag * sign).half()
    x = (torch.rand((case["rows"], hidden), device="cuda", generator=g) * 2.0 - 1.0) * (6.0 * math.sqrt(896.0 / hidden))
    return words, scales, x


def _softmax_shape(case):
    """(rows, row length, causal period, causal offset) of an attention block: `queries` new
    positions after `cache` old ones."""
    return case["heads"] * case["queries"], case["cache"] + case["queries"], case["queries"], case["cache"]


def _softmax_input(case, seed):
    rows, n, _, _ = _softmax_shape(case)
    return torch.empty(rows * n, device="cuda").normal_(0.0, 3.0, generator=_rng(seed, 4))


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "softmax":
        s["x"] = _softmax_input(case, seed)
        s["out"] = torch.empty_like(s["x"])
        s["shape"] = _softmax_shape(case)
        return s
    rows, vocab = case["rows"], case["vocab"]
    if kind in ("lmhead", "fused"):
        words, scales, s["x"] = _head_inputs(case, seed)
        s["head"] = S.LmHeadQ4(words, scales.view(torch.int16), vocab, case["hidden"], case["block"])
        if kind == "lmhead":
            s["out"] = torch.empty((rows, vocab), device="cuda")
            return s
    else:
        s["logits"] = _logits(case, seed)
    s["g"] = _handle(vocab, rows, case.get("k_max", 64))
    if kind == "argmax":
        s["ids"] = torch.zeros(rows, dtype=torch.int32, device="cuda")
        s["max"] = torch.zeros(rows, device="cuda")
        return s
    s["params"] = torch.from_numpy(_params(case, seed).view(np.uint8).copy()).cuda()
    s["results"], s["fields"] = _results(rows)
    s["flags"] = S.TABBY_FLAG_FULL_VOCAB if kind == "nucleus" else 0
    s["lists"] = s["list_ids"] = s["list_logits"] = None
    if case.get("lists"):
        s["list_ids"] = torch.zeros((rows, case["lists"]), dtype=torch.int32, device="cuda")
        s["list_logits"] = torch.zeros((rows, case["lists"]), device="cuda")
        s["fields"] = dict(s["fields"], list_ids=s["list_ids"], list_logits=s["list_logits"])
    return s


def run(s):
    kind = s["kind"]
    if kind in ("sample", "nucleus"):
        s["g"].sample_device(s["logits"], s["params"], s["results"], s["list_ids"], s["list_logits"],
                             flags=s["flags"])
        return s["fields"]
    if kind == "argmax":
        s["g"].argmax_device(s["logits"], s["ids"], s["max"])
        return {"ids": s["ids"], "max": s["max"]}
    if kind == "lmhead":
        return {"logits": s["head"].logits(s["x"], out=s["out"])}
    if kind == "fused":
        s["g"].sample_lmhead_q4_device(s["head"], s["x"], s["params"], s["results"])
        return s["fields"]
    rows, n, period, offset = s["shape"]
    return {"out": S.softmax_rows(s["x"], rows, n, period, offset, out=s["out"])}


# ---------------------------------------------------------------------------------------
# What a pass cannot do without, and what it must give
# ---------------------------------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "softmax":
        rows, n, period, offset = _softmax_shape(case)
        covered = case["heads"] * sum(offset + q + 1 for q in range(period))
        return {"bytes": 4 * (covered + rows * n), "flops": 4 * covered}
    rows, vocab = case["rows"], case["vocab"]
    if kind in ("lmhead", "fused"):
        hidden = case["hidden"]
        b = vocab * hidden // 2 + 2 * vocab * hidden // case["block"] + 4 * rows * hidden
        b += 4 * rows * vocab if kind == "lmhead" else 80 * rows
        return {"bytes": b, "flops": 2 * rows * vocab * hidden}
    b = rows * vocab * (2 if case["dtype"] == "f16" else 4)
    if kind == "argmax":
        return {"bytes": b + 8 * rows, "flops": rows * vocab}
    return {"bytes": b + rows * (80 + 8 * case.get("lists", 0)), "flops": 3 * rows * vocab}


def tolerance(case):
    """The softmax, the lm_head and the argmax are the CPU reference's bit for bit. Sampling
    gives ids, counts and lists exactly; its probabilities come from sums of f32 exps (at most
    6e-8 from 64 bits, and 2.6e-8 between two calls whose waves took chunks in another order).
    The fused lm_head's logits are f32 sums: 9e-7 from 64 bits in a probability."""
    if case["kind"] in ("softmax", "lmhead", "argmax"):
        return "exact"
    return {"rel": 4e-6 if case["kind"] == "fused" else 4e-7, "max": 1e-5}


def _exact_head(case, seed):
    words, scales, x = _head_inputs(case, seed)
    vocab, hidden, block = case["vocab"], case["hidden"], case["block"]
    out = torch.empty((case["rows"], vocab), dtype=torch.float64, device="cuda")
    shifts = torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)
    words, scales = words.view(vocab, hidden // 8), scales.view(vocab, hidden // block)
    for v0 in range(0, vocab, 16384):
        v1 = min(vocab, v0 + 16384)
        q = ((words[v0:v1, :, None] >> shifts) & 15).reshape(v1 - v0, hidden // block, block).double() - 8.0
        w = (q * scales[v0:v1, :, None].double()).reshape(v1 - v0, hidden)
        out[:, v0:v1] = x.double() @ w.t().contiguous()
    return out


def _exact_sample(case, logits, params):
    """The sampling outputs in 64 bits: full sort, softmax, nucleus cut and draw of each row."""
    rows, vocab = logits.shape
    lists = case.get("lists", 0)
    out = {"probability": torch.zeros(rows, dtype=torch.float64), "pool_mass": torch.zeros(rows, dtype=torch.float64),
           "max_logit": torch.zeros(rows, dtype=torch.float64), "sum_exp": torch.zeros(rows, dtype=torch.float64)}
    tops = torch.zeros((rows, lists), dtype=torch.float64)
    for r in range(rows):
        x, _ = torch.sort(logits[r].double(), descending=True, stable=True)
        p = params[r]
        k = int(p["top_k"]) if 0 < int(p["top_k"]) < vocab else vocab
        top = x[:k]
        e = torch.exp(x - x[0])
        total = e.sum()
        chosen = 0
        if p["temperature"] > 0:
            run_sum = torch.cumsum(torch.exp((top - x[0]) / float(p["temperature"])), 0)
            c = run_sum / run_sum[-1]
            cut = k
            if p["top_p"] < 1.0:
                cut = min(k, int((c < float(p["top_p"])).sum()) + 1)
            chosen = min(cut - 1, int((c[:cut] <= float(p["uniform"]) * c[cut - 1]).sum()))
        out["probability"][r], out["pool_mass"][r] = float(e[chosen] / total), float(e[:k].sum() / total)
        out["max_logit"][r], out["sum_exp"][r] = float(x[0]), float(total)
        n = min(lists, k)
        tops[r, :n] = top[:n].cpu()
    out.update(id=None, considered=None, pool_exhausted=None, status=None, topk_count=None)
    if lists:
        out.update(list_ids=None, list_logits=tops)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "softmax":
        rows, n, period, offset = _softmax_shape(case)
        x = _softmax_input(case, seed).double().view(rows, n)
        valid = offset + 1 + torch.arange(rows, device="cuda") % period
        x[torch.arange(n, device="cuda")[None, :] >= valid[:, None]] = -math.inf
        return {"out": torch.softmax(x, dim=1).view(-1)}
    if kind == "argmax":
        return {"ids": None, "max": _logits(case, seed).double().max(dim=1).values}
    if kind == "lmhead":
        return {"logits": _exact_head(case, seed)}
    if kind == "fused":
        return _exact_sample(case, _exact_head(case, seed), _params(case, seed))
    return _exact_sample(case, _logits(case, seed), _params(case, seed))
