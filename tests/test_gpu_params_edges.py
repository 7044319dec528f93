"""Temperatures and top-p values outside the usual range, on every launch shape, through the
C ABI's device form (per-row statuses).

sampler.ts (sampleFromTopK, src/engine/sampler.ts:147-212) takes any number: `temperature <=
0` is greedy (-0 and -inf included), `topP < 1` cuts at the first running sum reaching it (the
first candidate for topP <= 0; NaN and >= 1 never cut). Those rows must give the oracle's
answer on every path. A NaN or +inf temperature is refused with TABBY_EINVAL on every path
(the reference would sample NaN weights), and the other rows of the batch are still sampled.
The hosts refuse such a row before drawing a uniform."""
import math

import numpy as np
import pytest

from tabby_amd import sampler as S
from tabby_amd import synth

from parity import REL_TOL, rel

pytestmark = pytest.mark.gpu

T_GRID = (math.nan, math.inf, -0.0, 1e-300, -math.inf, 0.7, 5e-324, 1e300)
P_GRID = (math.nan, -1.0, 0.0, math.inf, 0.9, -math.inf)


def _edge_params(w, seed):
    """Every (temperature, top_p) pair of the grids, cycled over the rows."""
    n = len(T_GRID) * len(P_GRID)
    order = np.random.default_rng(seed).permutation(max(w.rows, n))[: w.rows] % n
    w.temperature[:] = [T_GRID[i % len(T_GRID)] for i in order]
    w.top_p[:] = [P_GRID[i // len(T_GRID)] for i in order]
    p = np.zeros(w.rows, dtype=S.PARAMS_DTYPE)
    p["temperature"], p["top_p"], p["uniform"], p["top_k"] = w.temperature, w.top_p, w.uniform, w.top_k
    return p


def _run_device(w, params, k_max, flags=0):
    import torch
    x = torch.from_numpy(np.ascontiguousarray(w.logits)).cuda()
    pd = torch.from_numpy(params.view(np.uint8).copy()).cuda()
    rd = torch.zeros(w.rows * S.RESULT_DTYPE.itemsize, dtype=torch.uint8, device="cuda")
    with S.GpuSampler(vocab_max=w.vocab, rows_max=w.rows, k_max=k_max) as g:
        g.sample_device(x, pd, rd, flags=flags)
        return rd.cpu().numpy().view(S.RESULT_DTYPE).copy()


def _check(oracle, logits, params, res, ctx):
    refused = checked = 0
    for r in range(len(params)):
        T, p, k, u = (float(params[r]["temperature"]), float(params[r]["top_p"]), int(params[r]["top_k"]),
                      float(params[r]["uniform"]))
        c = f"{ctx} row {r}: k={k} T={T!r} p={p!r} u={u!r}"
        g = res[r]
        if not T < math.inf:
            assert int(g["status"]) == S.TABBY_EINVAL, c
            refused += 1
            continue
        o = oracle.sample_row(logits[r], k, T, p, u)
        assert int(g["status"]) == o["status"] == 0, f"{c}: status {int(g['status'])}"
        assert int(g["id"]) == o["id"], f"{c}: id gpu={int(g['id'])} oracle={o['id']}"
        assert int(g["considered"]) == o["considered"], f"{c}: consideredCount {int(g['considered'])} vs {o['considered']}"
        assert np.float32(g["max_logit"]) == np.float32(o["max_logit"]), c
        for f in ("probability", "pool_mass", "sum_exp"):
            assert rel(float(g[f]), o[f]) < REL_TOL, (c, f, float(g[f]), o[f])
        if not abs(o["pool_mass"] - p) <= REL_TOL * abs(p):  # clear of the flag's boundary (or NaN)
            assert bool(g["pool_exhausted"]) == o["pool_exhausted"], f"{c}: poolExhausted"
        checked += 1
    assert refused > 0 and checked > 0
    print(f"[edges] {ctx}: {checked} rows as the oracle, {refused} refused", flush=True)


# (name, rows, vocab, k choices, k_max, ties / -inf): one case per launch shape of the device
# form -- the per-row kernel's small-pool tail and its sorted merge (256, 200 rows), parts of
# rows merged by the wave-merge kernel (5 rows of 100,000), one workgroup per row among few
# rows (5 rows of 33,000), one-wave slices and their merge (61 short rows), the large-pool
# streaming kernel, as many rows as CUs (256) and few (8, "slice kernel" for what served them
# before), and whole-vocabulary rows (the head kernels, beside finite rows).
SHAPES = [
    ("row kernel", 256, 12000, (1, 50, 100, 200, 256), 256, False),
    ("row kernel 200 rows", 200, 12000, (1, 50, 256), 256, True),
    ("parts", 5, 100000, (1, 50, 256), 256, True),
    ("one workgroup per row", 5, 33000, (1, 40, 100), 256, False),
    ("wave kernel", 61, 12000, (1, 20, 50, 256), 256, True),
    ("pool row kernel", 256, 20000, (300, 1024), 1024, True),
    ("slice kernel", 8, 20000, (512, 1024), 1024, False),
    ("whole vocabulary", 48, 20000, (0, 0, 0, 50), 64, True),
]


@pytest.mark.parametrize("name,rows,vocab,ks,k_max,ties", SHAPES, ids=[s[0] for s in SHAPES])
def test_parameter_edges_every_launch_shape(oracle, name, rows, vocab, ks, k_max, ties):
    w = synth.random_workload(rows=rows, vocab=vocab, seed=rows * 7 + vocab, k_choices=ks, ties=ties,
                              neg_inf_frac=0.05 if ties else 0.0)
    params = _edge_params(w, rows + vocab)
    flags = S.TABBY_FLAG_FULL_VOCAB if 0 in ks else 0
    print(f"[edges] {name}: {rows} x {vocab}, k {ks}", flush=True)
    res = _run_device(w, params, k_max, flags)
    _check(oracle, w.logits_f32(), params, res, name)


def test_parameter_edges_fused_lm_head(oracle):
    import torch
    vocab, hidden = 4096, 64
    words, f16, f32 = synth.lm_head_q4(vocab, hidden, 32, seed=3)
    head = S.LmHeadQ4(words, f16, vocab, hidden, 32)
    n = len(T_GRID) * len(P_GRID)
    x = synth.hidden_states(8, hidden, seed=17)
    logits = oracle.matmul_quantized(words, f32, x, vocab, hidden)
    with S.GpuSampler(vocab_max=vocab, rows_max=8, k_max=64) as g:
        for call in range((n + 7) // 8):
            w = synth.Workload("lm_head", logits, np.resize(np.array([1, 7, 40, 64], np.int32), 8),
                               np.zeros(8), np.zeros(8), synth.mulberry32_stream(call + 1, 8))
            p = np.zeros(8, dtype=S.PARAMS_DTYPE)
            idx = (np.arange(8) + 8 * call) % n
            p["temperature"] = [T_GRID[i % len(T_GRID)] for i in idx]
            p["top_p"] = [P_GRID[i // len(T_GRID)] for i in idx]
            p["uniform"], p["top_k"] = w.uniform, w.top_k
            res = g.sample_lmhead_q4(head, torch.from_numpy(x).cuda(), p)
            if any(not t < math.inf for t in p["temperature"]) and any(t < math.inf for t in p["temperature"]):
                _check(oracle, logits, p, res, f"fused lm_head call {call}")


def test_host_forms_refuse_nan_and_inf_temperature():
    import torch
    x = torch.zeros((2, 1000), dtype=torch.float32, device="cuda")
    with S.GpuSampler(vocab_max=1000, rows_max=2, k_max=64) as g:
        for t in (math.nan, math.inf):
            p = np.zeros(2, dtype=S.PARAMS_DTYPE)
            p["temperature"], p["top_p"], p["top_k"], p["uniform"] = [0.7, t], 0.9, 40, 0.5
            with pytest.raises(S.SamplingError) as e:
                g.sample_params(x, p)
            assert "temperature" in str(e.value)
            rng = S.SeededRandom(5)
            with pytest.raises(ValueError):
                S.make_params([S.SamplingParams(0.7, 40, 0.9), S.SamplingParams(t, 40, 0.9)], 2, rng)
