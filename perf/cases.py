"""Performance cases: the calls a serving program makes on this package's kernels.

A serving step of a Qwen3 model runs, per layer, the FP8 block-scaled linears
(qkv, o, gate/up, down), the fused q/k RMSNorm + RoPE + KV store and an
attention call over the paged FP8 cache (decode, speculative rows and prompt
chunks), and once per step the sampler.  The cases are those calls at the
shapes of the repository's benchmark and tests (Qwen3-0.6B, 8B and 32B heads
and projections), from a single sequence to the largest batch; ``draw`` gives
other sizes of the same ranges.

  listed()             the named cases
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  inputs, weights and caches on the GPU
  run(state)           one pass through the public entry points
  work(case)           bytes and flops the pass cannot do without
  tolerance(case)      how far two correct implementations may differ
  exact(case, seed)    the result in 64 bits, in plain torch
"""
import math
import os
import random
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "my-nano-vllm_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from nanovllm_amd.kernels.fp8_attention import fp8_decode_attention, fp8_prefill_attention  # noqa: E402
from nanovllm_amd.kernels.fp8_linear import fp8_block_linear  # noqa: E402
from nanovllm_amd.layers.qk_norm_rope import qk_norm_rope_store  # noqa: E402
from nanovllm_amd.layers.sampler import sample_tokens  # noqa: E402

D = 128                    # head_dim of every Qwen3 model
SCALE = D ** -0.5
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}

# (query heads, kv heads) of Qwen3-0.6B, 8B and 32B
HEADS = [(16, 8), (32, 8), (64, 8)]

# (in, out) features of their projections: qkv, o, gate/up, down
PROJECTIONS = [
    (1024, 4096), (2048, 1024), (1024, 6144), (3072, 1024),
    (4096, 6144), (4096, 4096), (4096, 24576), (12288, 4096),
    (5120, 10240), (8192, 5120), (5120, 51200), (25600, 5120),
]

VOCAB = 151936             # Qwen3 vocabulary

# the largest drawn work, that of the largest listed case of each kind
MAX_KV_TOKENS = 2_500_000                  # decode: keys over all sequences
MAX_LINEAR = 8192 * 4096 * 24576           # linear: multiply-adds
MAX_PREFILL = 304_447_750_144              # prefill: flops


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # one user's stream on the small model: launches and latency
        {"name": "decode_0p6b_b1", "kind": "decode", "hq": 16, "hkv": 8, "batch": 1, "lo": 777, "hi": 777,
         "lens": 1, "block": 256, "dtype": "bf16", "outliers": 0.0},
        # a full serving batch of ragged contexts, the headline decode
        {"name": "decode_8b_b192", "kind": "decode", "hq": 32, "hkv": 8, "batch": 192, "lo": 256, "hi": 4096,
         "lens": 4, "block": 256, "dtype": "bf16", "outliers": 0.0},
        # long documents on the large model, with outlier channels
        {"name": "decode_32b_b32_long", "kind": "decode", "hq": 64, "hkv": 8, "batch": 32, "lo": 32768, "hi": 131072,
         "lens": 5, "block": 256, "dtype": "bf16", "outliers": 0.01},
        # a chat prompt that arrives alone (no cached prefix: contiguous K/V)
        {"name": "prefill_8b_prompt_1003", "kind": "prefill", "hq": 32, "hkv": 8, "spec": 0, "spec_rows": 1,
         "chunks": 1, "chunk": 1003, "lo": 0, "hi": 0, "lens": 1, "paged": False, "block": 256, "dtype": "bf16"},
        # a step that mixes speculative verification rows and prompt chunks
        {"name": "prefill_8b_mixed", "kind": "prefill", "hq": 32, "hkv": 8, "spec": 32, "spec_rows": 5,
         "chunks": 3, "chunk": 512, "lo": 256, "hi": 4096, "lens": 4, "paged": True, "block": 256, "dtype": "bf16"},
        # a step of prompt chunks over cached prefixes: throughput of prefill
        {"name": "prefill_8b_16x512", "kind": "prefill", "hq": 32, "hkv": 8, "spec": 0, "spec_rows": 1,
         "chunks": 16, "chunk": 512, "lo": 0, "hi": 4096, "lens": 3, "paged": True, "block": 256, "dtype": "bf16"},
        # the qkv projections of 16 layers for one token (weights from HBM,
        # as in a model step, where every layer has its own)
        {"name": "linear_8b_qkv_m1_x16", "kind": "linear", "k": 4096, "n": 6144, "m": 1, "layers": 16, "dtype": "bf16"},
        # gate/up of the full decode batch, three layers
        {"name": "linear_8b_gate_up_m192_x3", "kind": "linear", "k": 4096, "n": 24576, "m": 192, "layers": 3,
         "dtype": "bf16"},
        # down of a mixed step (decode rows + speculative rows + three chunks)
        {"name": "linear_8b_down_m1888", "kind": "linear", "k": 12288, "n": 4096, "m": 1888, "layers": 1,
         "dtype": "bf16"},
        # gate/up of a full prefill step
        {"name": "linear_8b_gate_up_m8192", "kind": "linear", "k": 4096, "n": 24576, "m": 8192, "layers": 1,
         "dtype": "bf16"},
        # q/k norm, rotary embedding and KV store of a full prefill step
        {"name": "qk_norm_rope_8b_n8192", "kind": "qk_norm_rope", "hq": 32, "hkv": 8, "tokens": 8192, "lens": 3},
        # one token for every row of a mixed step
        {"name": "sample_355", "kind": "sample", "rows": 355, "vocab": VOCAB, "dtype": "bf16"},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "linear", "linear", "linear", "qk_norm_rope", "sample"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    hq, hkv = rng.choice(HEADS)
    if kind == "decode":
        hi = _log_int(rng, 64, 131072)
        batch = max(1, min(_log_int(rng, 1, 512), MAX_KV_TOKENS // hi))
        return {"kind": kind, "hq": hq, "hkv": hkv, "batch": batch, "lo": max(1, hi // rng.choice([1, 4, 16])),
                "hi": hi, "lens": rng.randrange(1 << 16), "block": rng.choice([256, 256, 64, 16]), "dtype": dtype,
                "outliers": rng.choice([0.0, 0.01])}
    if kind == "prefill":
        paged = rng.random() < 0.7
        case = {"kind": kind, "hq": hq, "hkv": hkv, "spec": 0, "spec_rows": 1, "chunks": _log_int(rng, 1, 16),
                "chunk": _log_int(rng, 33, 2048), "lo": 0, "hi": 0, "lens": rng.randrange(1 << 16), "paged": paged,
                "block": rng.choice([256, 256, 64, 16]), "dtype": dtype}
        if paged:
            case["hi"] = _log_int(rng, 16, 8192)
            if rng.random() < 0.5:
                case["spec"], case["spec_rows"] = _log_int(rng, 1, 64), rng.randrange(2, 32 * hkv // hq + 1)
        while _flops(case) > MAX_PREFILL:
            case["chunk"] = max(33, case["chunk"] // 2)
            case["hi"] //= 2
        return case
    if kind == "linear":
        k, n = rng.choice(PROJECTIONS)
        m = min(_log_int(rng, 1, 8192), MAX_LINEAR // (k * n))
        layers = max(1, min(16, (400 << 20) // (k * n))) if m <= 256 else 1
        return {"kind": kind, "k": k, "n": n, "m": m, "layers": layers, "dtype": dtype}
    if kind == "qk_norm_rope":
        return {"kind": kind, "hq": hq, "hkv": hkv, "tokens": _log_int(rng, 1, 8192), "lens": rng.randrange(1 << 16)}
    return {"kind": kind, "rows": _log_int(rng, 1, 355), "vocab": VOCAB, "dtype": dtype}


# ---------------------------------------------------------------------------
# shapes (from the case alone)
# ---------------------------------------------------------------------------
def _decode_lens(case):
    rng = random.Random(case["lens"])
    return [rng.randint(case["lo"], case["hi"]) for _ in range(case["batch"])]


def _prefill_seqs(case):
    """(query tokens, cached keys) of each sequence, speculative ones first."""
    rng = random.Random(case["lens"])
    spec = [(case["spec_rows"], rng.randint(case["lo"], case["hi"])) for _ in range(case["spec"])]
    return spec + [(case["chunk"], rng.randint(case["lo"], case["hi"])) for _ in range(case["chunks"])]


def _flops(case):
    return 4 * D * case["hq"] * sum(lq * c + lq * (lq + 1) // 2 for lq, c in _prefill_seqs(case))


def work(case):
    kind = case["kind"]
    if kind == "decode":
        lens = _decode_lens(case)
        q = case["batch"] * case["hq"] * D * 2
        tables = sum(4 * -(-c // case["block"]) + 4 for c in lens)
        return {"bytes": 2 * sum(lens) * case["hkv"] * D + 2 * q + tables, "flops": 4 * D * case["hq"] * sum(lens)}
    if kind == "prefill":
        seqs = _prefill_seqs(case)
        q = sum(lq for lq, _ in seqs) * case["hq"] * D * 2
        return {"bytes": 2 * sum(lq + c for lq, c in seqs) * case["hkv"] * D + 2 * q, "flops": _flops(case)}
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        one = k * n + 2 * (k // 128) * (n // 128) + 2 * m * k + 2 * m * n
        return {"bytes": case["layers"] * one, "flops": case["layers"] * 2 * m * k * n}
    if kind == "qk_norm_rope":
        hq, hkv, t = case["hq"], case["hkv"], case["tokens"]
        return {"bytes": t * ((hq + 2 * hkv) * D * 2 + hq * D * 2 + 2 * hkv * D + 8 + 4), "flops": t * (hq + hkv) * D * 10}
    size = 2
    return {"bytes": case["rows"] * (case["vocab"] * size + 4 + 8), "flops": case["rows"] * case["vocab"] * 4}


def tolerance(case):
    """About four times what is seen against 64 bits: 1.7e-3 where the rounding
    of the output to bf16 is all there is (attention, the rotated q), up to
    6e-3 in a linear, whose FP8 matrix instructions align the products of a
    128-wide block to its largest one and drop what lies 14 bits below."""
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        return {"rel": 8e-3}
    if kind == "linear":
        return {"rel": 2.4e-2}
    if kind == "qk_norm_rope":  # E4M3 bytes: a value at a rounding boundary moves by one of 8 steps of its binade
        return {"rel": 8e-3, "max": 0.2}
    return {"rel": 0.0, "differ": 0.01}  # tokens: ties within the sums' rounding


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1009 + salt)


def _normal(g, shape, dtype):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).to(dtype)


def _fp8_values(g, rows, hkv, outliers):
    """[rows, hkv, 128] K or V values as the store leaves them in the cache."""
    out = torch.empty(rows, hkv, D, dtype=torch.float8_e4m3fn, device="cuda")
    step = 1 << 18
    for a in range(0, rows, step):
        b = min(rows, a + step)
        x = torch.randn((b - a, hkv, D), generator=g, device="cuda", dtype=torch.float32)
        if outliers > 0:
            mask = torch.rand(x.shape, generator=g, device="cuda") < outliers
            x = torch.where(mask, x * 20.0, x).clamp_(-448.0, 448.0)
        out[a:b] = x.to(torch.bfloat16).to(torch.float8_e4m3fn)
    return out


def _pool(g, lens, block):
    """Shuffled physical blocks of a pool 1.25x the blocks needed: (blocks in
    the pool, table [S, width], -1 padded), on the GPU."""
    nb = [max(1, -(-c // block)) for c in lens]
    pool = int(math.ceil(1.25 * sum(nb)))
    ids = torch.randperm(pool, generator=g, device="cuda").to(torch.int32)
    table = torch.full((len(lens), max(nb)), -1, dtype=torch.int32, device="cuda")
    o = 0
    for i, n in enumerate(nb):
        table[i, :n] = ids[o:o + n]
        o += n
    return pool, table


def _cumsum(values):
    out = [0]
    for v in values:
        out.append(out[-1] + v)
    return torch.tensor(out, dtype=torch.int32, device="cuda")


def _linear_inputs(case, seed):
    """Per layer (x, weight, weight_scale); weights span the E4M3 range under
    a per-block scale, as quantised checkpoints have them."""
    g = _gen(seed, 3)
    m, k, n = case["m"], case["k"], case["n"]
    layers = []
    for _ in range(case["layers"]):
        w = torch.randn((n, k), generator=g, device="cuda", dtype=torch.float32) * (448.0 / 4.5)
        w = w.clamp_(-448.0, 448.0).to(torch.float8_e4m3fn)
        scale = torch.rand((n // 128, k // 128), generator=g, device="cuda") * 2e-4 + 1e-4
        x = _normal(g, (m, k), DTYPES[case["dtype"]])
        layers.append((x, w, scale.to(torch.bfloat16)))
    return layers


def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode":
        g = _gen(seed, 1)
        lens = _decode_lens(case)
        pool, table = _pool(g, lens, case["block"])
        shape = (pool, case["block"], case["hkv"], D)
        k = _fp8_values(g, pool * case["block"], case["hkv"], case["outliers"]).view(shape)
        v = _fp8_values(g, pool * case["block"], case["hkv"], case["outliers"]).view(shape)
        q = _normal(g, (case["batch"], case["hq"], D), DTYPES[case["dtype"]])
        return {"kind": kind, "q": q, "k": k, "v": v, "table": table,
                "lens": torch.tensor(lens, dtype=torch.int32, device="cuda")}
    if kind == "prefill":
        g = _gen(seed, 2)
        seqs = _prefill_seqs(case)
        lk = [lq + c for lq, c in seqs]
        state = {"kind": kind, "cu_q": _cumsum([lq for lq, _ in seqs]), "cu_k": _cumsum(lk),
                 "max_q": max(lq for lq, _ in seqs), "max_k": max(lk), "table": None}
        if case["paged"]:
            pool, state["table"] = _pool(g, lk, case["block"])
            rows, shape = pool * case["block"], (pool, case["block"], case["hkv"], D)
        else:
            rows, shape = sum(lk), (sum(lk), case["hkv"], D)
        state["k"] = _fp8_values(g, rows, case["hkv"], 0.0).view(shape)
        state["v"] = _fp8_values(g, rows, case["hkv"], 0.0).view(shape)
        state["q"] = _normal(g, (sum(lq for lq, _ in seqs), case["hq"], D), DTYPES[case["dtype"]])
        return state
    if kind == "linear":
        return {"kind": kind, "layers": _linear_inputs(case, seed)}
    if kind == "qk_norm_rope":
        g = _gen(seed, 4)
        hq, hkv, t = case["hq"], case["hkv"], case["tokens"]
        blocks = -(-t // 256) + 1
        qkv = _normal(g, (t, (hq + 2 * hkv) * D), torch.bfloat16)
        inv_freq = 1.0 / (1_000_000.0 ** (torch.arange(0, D, 2, dtype=torch.float, device="cuda") / D))
        angles = torch.outer(torch.arange(8192, dtype=torch.float, device="cuda"), inv_freq)
        rng = random.Random(case["lens"])
        first = rng.randint(0, 8191)
        return {"kind": kind, "hq": hq, "hkv": hkv, "qkv": qkv,
                "positions": (torch.arange(t, device="cuda") + first) % 8192,
                "wq": _normal(g, (D,), torch.bfloat16) * 0.1 + 1.0, "wk": _normal(g, (D,), torch.bfloat16) * 0.1 + 1.0,
                "cos_sin": torch.cat((angles.cos(), angles.sin()), dim=-1),
                "k": torch.zeros(blocks, 256, hkv, D, dtype=torch.uint8, device="cuda").view(torch.float8_e4m3fn),
                "v": torch.zeros(blocks, 256, hkv, D, dtype=torch.uint8, device="cuda").view(torch.float8_e4m3fn),
                "slots": torch.randperm(blocks * 256, generator=g, device="cuda")[:t].to(torch.int32)}
    g = _gen(seed, 5)
    dtype = DTYPES[case["dtype"]]
    logits = torch.empty(case["rows"], case["vocab"], dtype=dtype, device="cuda")
    for i in range(0, case["rows"], 64):
        n = min(64, case["rows"] - i)
        logits[i:i + n] = _normal(g, (n, case["vocab"]), dtype) * 3.0
    temperatures = torch.rand(case["rows"], generator=g, device="cuda") + 0.5
    return {"kind": kind, "logits": logits, "temperatures": temperatures, "seed": int(seed) * 7919 + 17}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "decode":
        return fp8_decode_attention(state["q"], state["k"], state["v"], state["table"], state["lens"], SCALE)
    if kind == "prefill":
        return fp8_prefill_attention(q=state["q"], k=state["k"], v=state["v"], block_tables=state["table"],
                                     cu_seqlens_q=state["cu_q"], cu_seqlens_k=state["cu_k"],
                                     max_seqlen_q=state["max_q"], max_seqlen_k=state["max_k"], softmax_scale=SCALE)
    if kind == "linear":
        return [fp8_block_linear(x, w, scale) for x, w, scale in state["layers"]]
    if kind == "qk_norm_rope":
        q = qk_norm_rope_store(state["positions"], state["qkv"], state["wq"], state["wk"], 1e-6, state["cos_sin"],
                               state["k"], state["v"], state["slots"], state["hq"], state["hkv"])
        return [q, state["k"], state["v"]]
    return sample_tokens(state["logits"], state["temperatures"], seed=state["seed"])


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _attend(q, k, v, cached):
    """q [Lq, Hq, D], k / v [Lk, Hkv, D] (E4M3 values) -> float64 [Lq, Hq, D];
    query row i sees the keys before cached + i + 1."""
    lq, hq, _ = q.shape
    lk, hkv, _ = k.shape
    g = hq // hkv
    out = torch.empty(lq, hq, D, dtype=torch.float64, device=q.device)
    hidden = torch.arange(lk, device=q.device)[None, :] > torch.arange(lq, device=q.device)[:, None] + cached
    for j in range(hkv):
        kk, vv = k[:, j].to(torch.float32).double(), v[:, j].to(torch.float32).double()
        for h in range(j * g, (j + 1) * g) if lq > 1 else [slice(j * g, (j + 1) * g)]:
            if lq > 1:
                s = (q[:, h].double() @ kk.T) * SCALE
                s.masked_fill_(hidden, -math.inf)
                out[:, h] = torch.softmax(s, dim=-1) @ vv
            else:
                out[0, h] = torch.softmax((q[0, h].double() @ kk.T) * SCALE, dim=-1) @ vv
    return out


def _gather(cache, table, n, block):
    nb = max(1, -(-n // block))
    return cache.view(torch.uint8)[table[:nb].long()].flatten(0, 1)[:n].view(torch.float8_e4m3fn)


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        return None
    s = prepare(case, seed)
    if kind == "decode":
        rows = [_attend(s["q"][i:i + 1], _gather(s["k"], s["table"][i], n, case["block"]),
                        _gather(s["v"], s["table"][i], n, case["block"]), n - 1)
                for i, n in enumerate(_decode_lens(case))]
        return torch.cat(rows)
    if kind == "prefill":
        rows, q0, k0 = [], 0, 0
        for i, (lq, c) in enumerate(_prefill_seqs(case)):
            if case["paged"]:
                k = _gather(s["k"], s["table"][i], lq + c, case["block"])
                v = _gather(s["v"], s["table"][i], lq + c, case["block"])
            else:
                k, v = s["k"][k0:k0 + lq + c], s["v"][k0:k0 + lq + c]
            rows.append(_attend(s["q"][q0:q0 + lq], k, v, c))
            q0, k0 = q0 + lq, k0 + lq + c
        return torch.cat(rows)
    if kind == "linear":
        outs = []
        for x, w, ws in s["layers"]:
            m, k = x.shape
            groups = x.float().view(m, k // 128, 128)
            scale = groups.abs().amax(-1, keepdim=True) / 448.0   # the quantisation is part of the layer
            scale = torch.where(scale > 0, scale, torch.ones_like(scale))
            xq = (groups / scale).clamp(-448.0, 448.0).to(torch.float8_e4m3fn).float().double()
            xd = (xq * scale.to(torch.bfloat16).double()).view(m, k)
            out = torch.empty(m, w.shape[0], dtype=torch.float64, device=x.device)
            for a in range(0, w.shape[0], 4096):
                b = min(a + 4096, w.shape[0])
                wd = w[a:b].float().double() * ws[a // 128:b // 128].double().repeat_interleave(128, 0).repeat_interleave(
                    128, 1)
                out[:, a:b] = xd @ wd.T
            outs.append(out)
        return outs
    hq, hkv, t = case["hq"], case["hkv"], case["tokens"]
    x = s["qkv"].double().view(t, hq + 2 * hkv, D)
    cs = s["cos_sin"].double()[s["positions"]].unsqueeze(1)
    cos, sin = cs[..., :D // 2], cs[..., D // 2:]

    def norm_rope(y, weight):
        y = y * torch.rsqrt(y.square().mean(-1, keepdim=True) + 1e-6) * weight.double()
        a, b = y[..., :D // 2], y[..., D // 2:]
        return torch.cat((a * cos - b * sin, b * cos + a * sin), dim=-1)

    out = [norm_rope(x[:, :hq], s["wq"])]
    for values in (norm_rope(x[:, hq:hq + hkv], s["wk"]), x[:, hq + hkv:]):
        cache = torch.zeros(s["k"].shape, dtype=torch.float64, device="cuda")
        cache.view(-1, hkv, D)[s["slots"].long()] = values
        out.append(cache)
    return out
