"""What a user of this library has it do, as cases that can be timed and compared.

One pass is one full-attention layer of the served model (24 query heads, 4 KV heads, head_dim 256, hidden width
5,120, Q8_0 weights, q8_0 or q4_0 caches) over what one step of an engine brings it, through the entry points of
`hipml_amd.attn` in the order in which the engine issues them: the Q, K and V projections, the front end (q|gate split,
head norms, RoPE) with the append of the new rows, the attention over the cache with the output gate, the output
projection.  Kinds of step:

  token   one sequence, one new token
  verify  one sequence, 2 to 4 drafted tokens that are checked against one cache
  batch   many sequences of different depths, one token each, the first of them with 3 drafted tokens to verify
  chunk   a piece of a prompt, behind what the cache holds already
  core    the benchmark's headline: the attention core of a prompt alone (RoPE, append, attention, gate)
"""
import math
import random

import torch

from hipml_amd import attn

H, KV, HD, N_ROT = 24, 4, 256, 64
SECTIONS = (11, 11, 10, 0)
THETA, EPS, SCALE = 1e7, 1e-6, 1.0 / 16.0
HIDDEN, Q_ROWS, KV_ROWS, O_COLS = 5120, 2 * H * HD, KV * HD, H * HD
N_CTX = 131_328  # positions the RoPE table is registered for, once per process
DRAFTED = 3      # rows of a batch's verify slots


def listed():
    return [
        # the first answer tokens of a short chat: every launch is small
        {"name": "token_673", "kind": "token", "depth": 673, "fmt": "q8_0"},
        # the benchmark's decode depth, over both cache formats
        {"name": "token_32k", "kind": "token", "depth": 32_768, "fmt": "q8_0"},
        {"name": "token_q4_32k", "kind": "token", "depth": 32_768, "fmt": "q4_0"},
        # the deepest context the benchmark decodes at
        {"name": "token_131k", "kind": "token", "depth": 131_072, "fmt": "q8_0"},
        # speculative decoding: three drafted tokens over one long sequence
        {"name": "verify3_32k", "kind": "verify", "depth": 32_768, "rows": 3, "fmt": "q8_0"},
        # the benchmark's served batch: 16 sequences, four of them with drafted tokens
        {"name": "batch16_mtp", "kind": "batch", "slots": 16, "verify": 4, "low": 512, "high": 16_384, "fmt": "q8_0"},
        # a server full of short sequences, nothing drafted
        {"name": "batch32_short", "kind": "batch", "slots": 32, "verify": 0, "low": 64, "high": 2_048, "fmt": "q8_0"},
        # the headline prompt of 672 tokens: its attention core, and the whole layer
        {"name": "core_672", "kind": "core", "tokens": 672, "fmt": "q8_0"},
        {"name": "chunk_672", "kind": "chunk", "tokens": 672, "pos0": 0, "fmt": "q8_0", "shadow": False},
        # a follow-up question of a chat: few tokens, a prefix of no round length
        {"name": "turn_117_at_5003", "kind": "chunk", "tokens": 117, "pos0": 5_003, "fmt": "q8_0", "shadow": False},
        # a document read in pieces into a q4_0 cache
        {"name": "chunk_1024_q4_at_8k", "kind": "chunk", "tokens": 1_024, "pos0": 8_192, "fmt": "q4_0", "shadow": False},
        # a long document at the benchmark's depth, the cache registered with its f16 copy
        {"name": "chunk_2048_at_100k", "kind": "chunk", "tokens": 2_048, "pos0": 100_000, "fmt": "q8_0", "shadow": True},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("token", "token", "verify", "batch", "batch", "core", "chunk", "chunk", "chunk"))
    fmt = "q4_0" if rng.random() < 0.25 else "q8_0"
    if kind == "token":
        return {"kind": kind, "depth": _log(rng, 16, 131_072), "fmt": fmt}
    if kind == "verify":
        return {"kind": kind, "depth": _log(rng, 16, 131_000), "rows": rng.randint(2, 4), "fmt": fmt}
    if kind == "batch":
        slots = _log(rng, 2, 32)
        low = _log(rng, 16, 512)
        return {"kind": kind, "slots": slots, "verify": rng.randint(0, min(4, slots)), "low": low,
                "high": low + _log(rng, 64, 16_384), "fmt": fmt}
    if kind == "core":
        return {"kind": kind, "tokens": _log(rng, 32, 2_048), "fmt": fmt}
    tokens = _log(rng, 16, 2_048)
    pos0 = 0 if rng.random() < 0.3 else _log(rng, 64, 90_000)
    return {"kind": kind, "tokens": tokens, "pos0": pos0, "fmt": fmt, "shadow": pos0 > 0 and rng.random() < 0.4}


def _depths(case):
    """Rows that each sequence of a batch has cached already: part of the case, the same for every seed."""
    r = random.Random(case["slots"] * 1_000_003 + case["low"] * 1_009 + case["high"])
    return [r.randint(case["low"], case["high"]) for _ in range(case["slots"])]


def _cols(case):
    return [DRAFTED if s < case["verify"] else 1 for s in range(case["slots"])]


# ---- inputs --------------------------------------------------------------------------------------------------------

def _weights(m, k, gen):
    """m rows of k/32 Q8_0 blocks of a normal matrix with variance 1/k: what quantizing a trained projection gives."""
    q = (torch.randn((m, k // 32, 32), device="cuda", generator=gen) * 40.0).round_().clamp_(-127, 127).to(torch.int8)
    d = (1.0 + 0.2 * torch.rand((m, k // 32, 1), device="cuda", generator=gen)) * (0.9 / (40.0 * math.sqrt(k)))
    return torch.cat((d.to(torch.float16).view(torch.uint8), q.view(torch.uint8)), dim=2).contiguous()


def _fill(dtype, k, v, stride, rows, gen):
    """Rows [0, rows) of a cache, quantized by the library itself from normal values."""
    for start in range(0, rows, 16_384):
        n = min(16_384, rows - start)
        kf = torch.randn((n, KV, HD), device="cuda", generator=gen)
        vf = torch.randn((n, KV, HD), device="cuda", generator=gen)
        attn.kv_encode_bulk(dtype, kf, vf, k, v, KV, HD, stride, start, 0, n)


def _norm(gen):
    return 1.0 + 0.1 * torch.randn(HD, device="cuda", generator=gen)


def prepare(case, seed):
    attn.init(0)
    attn.rope_table(THETA, N_ROT, N_CTX)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind, dtype = case["kind"], 1 if case["fmt"] == "q4_0" else 0
    s = {"kind": kind, "dtype": dtype}

    if kind == "core":
        tokens = s["tokens"] = case["tokens"]
        s["stride"] = (tokens + 63) // 64 * 64
        s["kv"] = attn.DeepKv(H, KV, HD, s["stride"], dtype=dtype)
        s["q"] = torch.randn((tokens, H, HD), device="cuda", generator=gen)
        s["k"] = torch.randn((tokens, KV, HD), device="cuda", generator=gen)
        s["v"] = torch.randn((tokens, KV, HD), device="cuda", generator=gen)
        s["gate"] = torch.randn((tokens, H, HD), device="cuda", generator=gen)
        s["out"] = torch.empty((tokens, H, HD), device="cuda")
        s["splits"] = attn.chunk_splits(0, tokens, KV)
        s["acc"], s["ml"] = attn.chunk_scratch(tokens, H, s["splits"]) if s["splits"] >= 2 else (None, None)
        return s

    if kind == "token":
        rows, depth = 1, case["depth"]
        s["stride"] = stride = depth + 64
        kv = attn.DeepKv(H, KV, HD, stride, dtype=dtype)
        _fill(dtype, kv.k, kv.v, stride, depth, gen)
        s["splits"] = kv.splits(depth + 1)
        s["step"] = torch.tensor([depth, depth + 1, 0, 0] + [depth] * 4, dtype=torch.int32, device="cuda")
    elif kind == "verify":
        rows, depth = case["rows"], case["depth"]
        s["stride"] = stride = depth + 64
        kv = attn.DeepKv(H, KV, HD, stride, max_cols=rows, dtype=dtype)
        _fill(dtype, kv.k, kv.v, stride, depth, gen)
        s["splits"] = kv.max_splits
        s["pos"] = torch.tensor([[depth + c, depth + c + 1] for c in range(rows)], dtype=torch.int32, device="cuda")
    elif kind == "batch":
        depths, cols = _depths(case), _cols(case)
        rows, s["cols"], s["verify"] = sum(cols), cols, case["verify"]
        s["stride"] = stride = (case["high"] + DRAFTED + 63) // 64 * 64
        kv = attn.BatchKv(case["slots"], H, KV, HD, stride, max_rows=rows, dtype=dtype)
        for b, depth in enumerate(depths):
            _fill(dtype, kv.k[b], kv.v[b], stride, depth, gen)
        s["pos"] = torch.tensor([[d + c, d + c + 1] for d, n in zip(depths, cols) for c in range(n)],
                                dtype=torch.int32, device="cuda")
    else:
        rows, pos0 = case["tokens"], case["pos0"]
        s["tokens"], s["pos0"] = rows, pos0
        s["stride"] = stride = (pos0 + rows + 63) // 64 * 64
        kv = attn.DeepKv(H, KV, HD, stride, dtype=dtype)
        if case["shadow"]:
            kv.attach_f16()
        _fill(dtype, kv.k, kv.v, stride, pos0, gen)
        s["splits"] = attn.chunk_splits(pos0, rows, KV)
        if case["shadow"] and s["splits"] >= 2:
            s["splits"] = attn.chunk_slices(pos0, rows, KV)  # the rows live in the registered copy, not in the scratch
        s["acc"], s["ml"] = attn.chunk_scratch(rows, H, s["splits"]) if s["splits"] >= 2 else (None, None)
        s["out16"] = torch.empty((rows, H, HD), dtype=torch.float16, device="cuda")
    s["rows"], s["kv"] = rows, kv
    s["x"] = torch.randn((rows, HIDDEN), device="cuda", generator=gen)
    s["wq"], s["wk"] = _weights(Q_ROWS, HIDDEN, gen), _weights(KV_ROWS, HIDDEN, gen)
    s["wv"], s["wo"] = _weights(KV_ROWS, HIDDEN, gen), _weights(HIDDEN, O_COLS, gen)
    s["q_norm"], s["k_norm"] = _norm(gen), _norm(gen)
    s["qg"] = torch.empty((rows, H, 2 * HD), device="cuda")
    s["q"] = torch.empty((rows, H, HD), device="cuda")
    s["gate"] = torch.empty((rows, H, HD), device="cuda")
    s["k"] = torch.empty((rows, KV, HD), device="cuda")
    s["v"] = torch.empty((rows, KV, HD), device="cuda")
    s["out"] = torch.empty((rows, H, HD), device="cuda")
    s["y"] = torch.empty((rows, HIDDEN), device="cuda")
    if kind == "batch" and s["verify"]:
        # which rows are appended where: the drafted rows of a slot to consecutive positions of its cache (slot_bytes
        # 0), the rows of the other slots to a cache each
        s["appends"] = [(s["k"][DRAFTED * b:], s["v"][DRAFTED * b:], kv.k[b], kv.v[b], s["pos"][DRAFTED * b:], 0, DRAFTED)
                        for b in range(s["verify"])]
        b, at = s["verify"], DRAFTED * s["verify"]
        if rows > at:
            s["appends"].append((s["k"][at:], s["v"][at:], kv.k[b], kv.v[b], s["pos"][at:], kv.slot_bytes, rows - at))
    return s


# ---- one pass ------------------------------------------------------------------------------------------------------

def _core(s):
    kv, t = s["kv"], s["tokens"]
    if s["splits"] == 0:  # the attention rotates the query rows where it loads them
        attn.rope_encode_chunk(None, s["k"], s["v"], kv.k, kv.v, H, KV, HD, N_ROT, THETA, 0, t, s["dtype"], s["stride"])
        attn.chunk_attention_rope_q8(s["q"], kv.k, kv.v, s["gate"], s["out"], None, H, KV, HD, N_ROT, THETA, 0, t,
                                     s["dtype"] + 1, s["stride"], None, None, 0)
    else:
        attn.rope_encode_chunk(s["q"], s["k"], s["v"], kv.k, kv.v, H, KV, HD, N_ROT, THETA, 0, t, s["dtype"],
                               s["stride"])
        attn.chunk_attention_q8_split_gate(s["q"], kv.k, kv.v, s["gate"], s["out"], H, KV, HD, 0, t, s["dtype"] + 1,
                                           s["stride"], s["acc"], s["ml"], s["splits"])
    return {"out": s["out"], "k": s["k"], "k_cache": kv.k, "v_cache": kv.v}


def _chunk(s):
    kv, t = s["kv"], s["tokens"]
    attn.gemm_q8_0_f16(s["wq"], s["x"], s["qg"], Q_ROWS, HIDDEN, t)
    attn.gemm_q8_0_f16(s["wk"], s["x"], s["k"], KV_ROWS, HIDDEN, t)
    attn.gemm_q8_0_f16(s["wv"], s["x"], s["v"], KV_ROWS, HIDDEN, t)
    attn.chunk_front_encode(s["dtype"], s["qg"], s["k"], s["v"], s["q"], s["gate"], s["q_norm"], s["k_norm"], kv.k, kv.v,
                            H, KV, HD, N_ROT, THETA, EPS, s["pos0"], t, s["stride"])
    attn.chunk_attention_q8_split_gate_f16(s["q"], kv.k, kv.v, s["gate"], s["out"], s["out16"], H, KV, HD, s["pos0"], t,
                                           s["dtype"] + 1, s["stride"], s["acc"], s["ml"], s["splits"])
    attn.output_chunk_q8_0(s["wo"], None, None, s["y"], HIDDEN, O_COLS, t, s["out16"])
    return {"y": s["y"], "attention": s["out16"], "k": s["k"], "k_cache": kv.k, "v_cache": kv.v}


def run(s):
    kind = s["kind"]
    if kind == "core":
        return _core(s)
    if kind == "chunk":
        return _chunk(s)
    kv, rows, dtype, stride = s["kv"], s["rows"], s["dtype"], s["stride"]
    attn.gemv_q8_0_rows(s["wq"], s["x"], s["qg"], Q_ROWS, HIDDEN, rows)
    attn.gemv_q8_0_rows(s["wk"], s["x"], s["k"], KV_ROWS, HIDDEN, rows)
    attn.gemv_q8_0_rows(s["wv"], s["x"], s["v"], KV_ROWS, HIDDEN, rows)
    if kind == "token":
        attn.attn_front_encode(s["step"], dtype, s["qg"], s["q"], s["gate"], s["k"], s["v"], s["q_norm"], s["k_norm"],
                               kv.k, kv.v, H, KV, HD, N_ROT, SECTIONS, THETA, EPS, stride)
        attn.attn_decode_kv_gate(s["step"], dtype, s["q"], kv.k, kv.v, kv.part_acc, kv.part_ml, s["out"], s["gate"], H,
                                 KV, HD, stride, SCALE, s["splits"])
    elif kind == "verify":  # slot_bytes 0: the rows are consecutive positions of one cache
        attn.front_rows_encode(dtype, s["qg"], s["k"], s["v"], s["q"], s["gate"], s["q_norm"], s["k_norm"], kv.k, kv.v,
                               H, KV, HD, N_ROT, THETA, EPS, stride, s["pos"], 0, rows)
        attn.attn_decode_kv_cols(dtype, s["pos"], s["q"], kv.k, kv.v, kv.part_acc, kv.part_ml, s["out"], H, KV, HD,
                                 stride, SCALE, s["splits"], rows, H * s["splits"] * HD, H * s["splits"] * 2, H * HD)
        attn.q_gate(s["out"], s["gate"], s["out"])
    elif s["verify"] == 0:
        kv.front_append(s["qg"], s["k"], s["v"], s["q"], s["gate"], s["q_norm"], s["k_norm"], N_ROT, THETA, EPS,
                        s["pos"])
        kv.decode(s["pos"], s["q"], s["out"], SCALE, gate=s["gate"])
    else:
        attn.front_rows(s["qg"], s["k"], s["q"], s["gate"], s["q_norm"], s["k_norm"], H, KV, HD, N_ROT, THETA, EPS,
                        s["pos"], rows)
        for k, v, k_cache, v_cache, pos, slot_bytes, n in s["appends"]:
            attn.kv_encode_rows(dtype, k, v, k_cache, v_cache, KV, HD, stride, pos, slot_bytes, n)
        kv.decode(s["pos"], s["q"], s["out"], SCALE, s["cols"], s["gate"])
    attn.gemv_q8_0_rows(s["wo"], s["out"], s["y"], HIDDEN, O_COLS, rows)
    return {"y": s["y"], "attention": s["out"], "k": s["k"], "k_cache": kv.k, "v_cache": kv.v}


# ---- what a pass cannot do without ---------------------------------------------------------------------------------

def work(case):
    kind, row = case["kind"], 144 if case["fmt"] == "q4_0" else 272
    if kind == "core":
        t = case["tokens"]
        pairs = t * (t + 1) // 2
        return {"bytes": 4 * t * HD * (3 * H + 3 * KV) + 2 * KV * t * row, "flops": 4 * HD * H * pairs}
    if kind == "token":
        rows, cached, pairs = 1, case["depth"], case["depth"] + 1
    elif kind == "verify":
        rows, cached = case["rows"], case["depth"]
        pairs = sum(cached + c + 1 for c in range(rows))
    elif kind == "batch":
        depths, cols = _depths(case), _cols(case)
        rows, cached = sum(cols), sum(depths)
        pairs = sum(d + c + 1 for d, n in zip(depths, cols) for c in range(n))
    else:
        rows, cached = case["tokens"], case["pos0"]
        pairs = rows * cached + rows * (rows + 1) // 2
    values = (Q_ROWS + 2 * KV_ROWS) * HIDDEN + HIDDEN * O_COLS  # of the four weight matrices
    return {"bytes": values // 32 * 34 + 2 * KV * (cached + rows) * row + 2 * 4 * rows * HIDDEN,
            "flops": 2 * rows * values + 4 * HD * H * pairs}


def tolerance(case):
    # Cache bytes: a value quantized from a sum in another order may fall on the other side of a rounding border.
    if case["kind"] in ("chunk", "core"):
        return {"rel": 2e-3, "differ": 2e-3}  # f16 operands in the projections, the scores and the probabilities
    return {"rel": 1e-3, "differ": 1e-3}      # fp32 sums; the softmax weights enter the PV product as f16
