"""Performance cases of the attention path: what a serving program asks of this library.

A case is one pass through the public entry points (``Attention``, ``MatMul3``, ``MatMulAdd``,
``KVCache``), with what such a program keeps between calls (operators, weights, caches) made
beforehand.  Five kinds of call:

  attend        attention over a cache with one capacity: a single-token step (interval 1), the
                short last chunk of a prompt, a whole prompt, a chunk appended to a long cache
  attend_ragged one new token for sequences of different lengths, on a cache with a capacity per
                sequence
  token_layer   the attention block of a layer for one new token per sequence: Q/K/V projection
                and attention as one call, then the output projection with its residual
  chunk_layer   the same block for a chunk of prompt positions, as three calls
  other_heads   attention on head sizes other than 128 or in binary32

Model shapes are those of the repository's configurations: 32 query / 4 key-value heads on 2048
hidden elements, 32 / 32 on 4096, and 64 / 8 on 8192, all with 128-wide heads.
"""
import math
import random

import torch

import ellm_amd

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
CACHE_CODES = {"f16": ellm_amd.DTYPE_F16, "bf16": ellm_amd.DTYPE_BF16}
# (hidden size, query heads, key-value heads)
SHAPES = [(2048, 32, 4), (4096, 32, 32), (8192, 64, 8)]


def listed():
    return [
        # The reference's published operating point: one conversation, a few hundred tokens in.
        # Latency of the calls and of short launches.
        dict(name="token_layer_1x512", kind="token_layer", dtype="f16", hidden=2048, q_heads=32,
             kv_heads=4, batch=1, cached=512, per_sequence=False),
        # A serving batch in steady state: 16 conversations at 8k tokens, with its projections.
        dict(name="token_layer_16x8192", kind="token_layer", dtype="f16", hidden=2048, q_heads=32,
             kv_heads=4, batch=16, cached=8192, per_sequence=True),
        # One user on a very long document.
        dict(name="decode_1x131072", kind="attend", dtype="f16", q_heads=32, kv_heads=4, batch=1,
             start=131071, interval=1, lse=False),
        # Continuous batching: 32 conversations between 1k and 128k tokens.
        dict(name="decode_32_of_1k_to_128k", kind="attend_ragged", dtype="f16", q_heads=32, kv_heads=4,
             batch=32, shortest=1024, longest=131072, len_seed=7),
        # Continuous batching of short conversations, lengths odd.
        dict(name="decode_100_of_100_to_4k", kind="attend_ragged", dtype="f16", q_heads=32, kv_heads=4,
             batch=100, shortest=100, longest=4096, len_seed=11),
        # What is left of 24 prompts after their full chunks: 13 tokens each, nothing aligned.
        dict(name="last_chunk_13x24_on_8191", kind="attend", dtype="f16", q_heads=32, kv_heads=4,
             batch=24, start=8191, interval=13, lse=False),
        # The reference's serving chunk: 64 positions of 24 sequences, the whole attention block.
        dict(name="chunk_layer_64x24_on_4096", kind="chunk_layer", dtype="f16", hidden=2048, q_heads=32,
             kv_heads=4, batch=24, start=4096, interval=64),
        # A medium prompt, multi-head attention without grouping, 512 of 4096 cache positions.
        dict(name="prompt_512_mha", kind="attend", dtype="f16", q_heads=32, kv_heads=32, batch=1,
             start=0, interval=512, lse=True),
        # The attention block of a layer on a long prompt, odd length.
        dict(name="chunk_layer_8000x1", kind="chunk_layer", dtype="bf16", hidden=2048, q_heads=32,
             kv_heads=4, batch=1, start=0, interval=8000),
        # A chunk appended to a very long cache: the largest call.
        dict(name="chunk_8192_on_120000", kind="attend", dtype="bf16", q_heads=64, kv_heads=8, batch=1,
             start=120000, interval=8192, lse=False),
        # A prompt of a model with 64-wide heads.
        dict(name="prompt_2048_head64", kind="other_heads", dtype="bf16", head_size=64, q_heads=32,
             kv_heads=8, batch=1, start=0, interval=2048),
        # A single-token step in binary32 (the element type of the reference's own operator test).
        dict(name="decode_8x4096_f32", kind="other_heads", dtype="f32", head_size=128, q_heads=32,
             kv_heads=4, batch=8, start=4095, interval=1),
    ]


def _log_int(rng, lo, hi):
    """A whole number between lo and hi, uniform over its logarithm (odd ones as likely as even)."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the same ranges; none costs more than the largest listed one."""
    kind = rng.choice(["token_layer", "decode", "attend_ragged", "last_chunk", "chunk_layer", "prompt",
                       "append", "other_step", "other_chunk"])
    dtype = rng.choice(["f16", "bf16"])
    hidden, hq, hkv = rng.choice(SHAPES)
    heads = dict(dtype=dtype, q_heads=hq, kv_heads=hkv)
    if kind == "token_layer":
        batch = _log_int(rng, 1, 48)
        return dict(kind=kind, hidden=hidden, batch=batch, cached=_log_int(rng, 128, 262144 // batch // hkv * 4),
                    per_sequence=rng.random() < 0.5, **heads)
    if kind == "decode":
        batch = _log_int(rng, 1, 64)
        return dict(kind="attend", batch=batch, start=_log_int(rng, 256, 1048576 // batch // hkv) - 1, interval=1,
                    lse=False, **heads)
    if kind == "attend_ragged":
        batch = _log_int(rng, 8, 128)
        longest = _log_int(rng, 2048, min(131072, 16777216 // batch // hkv))
        return dict(kind=kind, batch=batch, shortest=_log_int(rng, 64, longest // 2), longest=longest,
                    len_seed=rng.randrange(1 << 20), **heads)
    if kind == "last_chunk":
        batch = _log_int(rng, 4, 24)
        return dict(kind="attend", batch=batch, start=_log_int(rng, 1024, 1048576 // batch // hkv),
                    interval=rng.randint(2, 63), lse=False, **heads)
    if kind == "chunk_layer":
        batch = _log_int(rng, 1, 24)
        return dict(kind=kind, hidden=hidden, batch=batch, start=rng.choice([0, _log_int(rng, 64, 8192)]),
                    interval=_log_int(rng, 64, 8192 // batch), **heads)
    if kind == "prompt":
        batch = _log_int(rng, 1, 4)
        return dict(kind="attend", batch=batch, start=0, interval=_log_int(rng, 128, 32768 // batch),
                    lse=rng.random() < 0.5, **heads)
    if kind == "append":
        return dict(kind="attend", batch=1, start=_log_int(rng, 4096, 65536), interval=_log_int(rng, 128, 8192),
                    lse=False, **heads)
    other = dict(kind="other_heads", q_heads=32, kv_heads=rng.choice([4, 8, 32]))
    other["dtype"], other["head_size"] = rng.choice(
        [(d, h) for d in ("f16", "bf16") for h in (64, 80, 96, 192, 256)] + [("f32", 64), ("f32", 128)])
    if kind == "other_step":
        batch = _log_int(rng, 1, 16)
        return dict(batch=batch, start=_log_int(rng, 128, 65536 // batch) - 1, interval=1, **other)
    batch = _log_int(rng, 1, 4)
    interval = _log_int(rng, 16, 2048 // batch)
    return dict(batch=batch, start=rng.choice([0, _log_int(rng, 64, 2048)]), interval=interval, **other)


# ---------------------------------------------------------------------------------------------
# inputs and operators
# ---------------------------------------------------------------------------------------------
def _normal(gen, shape, dtype, scale=1.0):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, scale, generator=gen)


def _rotary_table(positions, head_size, dtype):
    j = torch.arange(head_size // 2, device="cuda", dtype=torch.float64)
    angle = torch.arange(positions, device="cuda", dtype=torch.float64)[:, None] * (1.0e6 ** (-2.0 * j / head_size))
    return torch.stack((torch.cos(angle), torch.sin(angle)), dim=-1).reshape(positions, head_size).to(dtype)


def _lengths(case):
    r = random.Random(case["len_seed"])
    return [r.randint(case["shortest"], case["longest"]) for _ in range(case["batch"])]


def _token_positions(case):
    """Positions of the new tokens: all alike, or a batch of conversations up to `cached` tokens
    long (the longest reaches it)."""
    if not case["per_sequence"]:
        return [case["cached"] - 1] * case["batch"]
    r = random.Random(case["batch"] * 1000003 + case["cached"])
    return [case["cached"] - 1] + [r.randint(case["cached"] * 3 // 4, case["cached"]) - 1
                                   for _ in range(case["batch"] - 1)]


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    hq, hkv, batch = case["q_heads"], case["kv_heads"], case["batch"]
    kind = case["kind"]
    if kind in ("attend", "other_heads"):
        d = case.get("head_size", 128)
        interval = case["interval"]
        capacity = (case["start"] + interval + 255) // 256 * 256
        q = _normal(gen, (interval, batch, hq, d), dtype)
        k = _normal(gen, (batch, hkv, capacity, d), dtype)
        v = _normal(gen, (batch, hkv, capacity, d), dtype)
        out = torch.zeros_like(q)
        lse = torch.zeros((interval, batch, hq), dtype=torch.float32, device="cuda") if case.get("lse") else None
        op = ellm_amd.Attention(q, k, v, out, batch, hq, hkv, d, k.stride(), 1.0 / math.sqrt(d), lse=lse)
        return dict(case=case, op=op, out=out, lse=lse)
    d = 128
    if kind == "attend_ragged":
        lengths = _lengths(case)
        cache = ellm_amd.KVCache.ragged(1, [n + 64 for n in lengths], hkv, CACHE_CODES[case["dtype"]])
        k, v = cache.layer_flat_tensors(0, dtype)
        k.normal_(generator=gen)
        v.normal_(generator=gen)
        view = cache.layer_ragged(0)
        q = _normal(gen, (1, batch, hq, d), dtype)
        out = torch.zeros_like(q)
        op = ellm_amd.Attention(q, k, v, out, batch, hq, hkv, d, view.strides, 1.0 / math.sqrt(d), seq_table=view)
        positions = torch.tensor([n - 1 for n in lengths], dtype=torch.int32, device="cuda")
        return dict(case=case, op=op, out=out, positions=positions, longest=max(lengths) - 1, cache=cache)

    hidden = case["hidden"]
    interval = case.get("interval", 1)
    end = case["start"] + interval if kind == "chunk_layer" else case["cached"]
    capacity = (end + 255) // 256 * 256
    # the cache in buffers of the caller's own: their rows are among the outputs, which outlive the operators
    k = _normal(gen, (batch, hkv, capacity, d), dtype)
    v = _normal(gen, (batch, hkv, capacity, d), dtype)
    strides = k.stride()
    x = _normal(gen, (interval, batch, hidden), dtype)
    residual = _normal(gen, (interval, batch, hidden), dtype)
    wq = _normal(gen, (hq * d, hidden), dtype, hidden ** -0.5)
    wk = _normal(gen, (hkv * d, hidden), dtype, hidden ** -0.5)
    wv = _normal(gen, (hkv * d, hidden), dtype, hidden ** -0.5)
    wo = _normal(gen, (hidden, hq * d), dtype, (hq * d) ** -0.5)
    q = torch.zeros((interval, batch, hq, d), dtype=dtype, device="cuda")
    att = torch.zeros_like(q)
    y = torch.zeros_like(x)
    rope = _rotary_table(capacity, d, dtype)
    state = dict(case=case, q=q, k=k, v=v, att=att, y=y)
    state["qkv"] = ellm_amd.MatMul3(x, wq, q, wk, k, wv, v, rope, d, batch, hq, hkv, strides, capacity)
    state["op"] = ellm_amd.Attention(q, k, v, att, batch, hq, hkv, d, strides, 1.0 / math.sqrt(d),
                                     sequence_capacity=capacity, max_position_interval=interval)
    state["proj"] = ellm_amd.MatMulAdd(att.view(interval, batch, hq * d), wo, residual, y)
    if kind == "token_layer":
        where = _token_positions(case)
        state["positions"] = (torch.tensor(where, dtype=torch.int32, device="cuda")
                              if case["per_sequence"] else None)
    return state


def run(state):
    case = state["case"]
    kind, batch = case["kind"], case["batch"]
    if kind in ("attend", "other_heads"):
        state["op"].run(case["start"], case["interval"], batch)
        return {"out": state["out"]} if state.get("lse") is None else {"out": state["out"], "lse": state["lse"]}
    if kind == "attend_ragged":
        state["op"].run_ragged(state["positions"], state["longest"], batch)
        return {"out": state["out"]}
    if kind == "token_layer":
        state["qkv"].run_with_attention(state["op"], case["cached"] - 1, batch, positions=state["positions"])
        state["proj"].run(0, 1, batch)
    else:
        state["qkv"].run(case["start"], case["interval"], batch)
        state["op"].run(case["start"], case["interval"], batch)
        state["proj"].run(0, case["interval"], batch)
    return {"q": state["q"], "k": state["k"], "v": state["v"], "attention": state["att"], "out": state["y"]}


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without, and how exact it is
# ---------------------------------------------------------------------------------------------
def work(case):
    size = 4 if case["dtype"] == "f32" else 2
    d = case.get("head_size", 128)
    hq, hkv, batch = case["q_heads"], case["kv_heads"], case["batch"]
    kind = case["kind"]
    if kind == "attend_ragged":
        keys = seen = sum(_lengths(case))
        tokens = batch
    elif kind == "token_layer":
        keys = seen = sum(p + 1 for p in _token_positions(case))
        tokens = batch
    else:
        s, p0 = case["interval"], case["start"]
        keys = batch * (p0 + s)
        seen = batch * (s * p0 + s * (s + 1) // 2)   # (query position, visible key) pairs of a head
        tokens = batch * s
    nbytes = 2 * keys * hkv * d * size               # keys and values
    nbytes += 2 * tokens * hq * d * size             # queries in, attention rows out
    flops = 4 * d * hq * seen
    if case.get("lse"):
        nbytes += 4 * tokens * hq
    if kind in ("token_layer", "chunk_layer"):
        hidden = case["hidden"]
        nbytes += hidden * (2 * hq + 2 * hkv) * d * size   # the four weight matrices
        nbytes += 3 * tokens * hidden * size               # hidden rows and residual in, rows out
        flops += 2 * tokens * hidden * (2 * hq + 2 * hkv) * d
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Relative 2-norm, about four times what the path shows against 64-bit arithmetic on the same
    inputs: 3e-4 in binary16 (16-bit probabilities and outputs), 2.4e-3 in bfloat16, 6e-7 in
    binary32 on one row of 4096 keys and up to twice that where values cancel."""
    if case["dtype"] == "f32":
        return {"rel": 5e-6}
    return {"rel": 1.2e-3 if case["dtype"] == "f16" else 1e-2}
