"""What is timed of this framework: the calls that a program with a model around them makes, at the sizes it makes them.

Three kinds of pass cover the path:

  steps    one forward of a few new tokens through every layer's cache behind a cached context: rotary positions, append
           (quantized caches: quantize), attention; the new rows are trimmed off again at the end (what a rejected draft
           does), so that a pass can be repeated on the same caches.
  prompt   one request from the start: a fresh cache, the prompt in balanced chunks of at most 512 rows, then single tokens.
  convert  a full-precision prompt cache turned into a quantized one and its state read out, as for a saved prompt cache.

Arrays are made on the device from the seed.  Keys and values carry a few channels of eight times the spread of the
others, as those of trained models do; scores have a standard deviation of a little over one.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "mlx-swift-lm_amd"))

import kvhip  # noqa: E402

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
CHUNK = 2048     # rows per update while a cached context is laid down
RAGGED_MIN = 16  # a ragged batch's lengths are uniform in [context / 16, context]


def _case(name, kind, **given):
    case = dict(name=name, kind=kind, cache="simple", dtype="f16", bits=0, group=64, batch=1, q_heads=32, kv_heads=8,
                key_dim=128, value_dim=128, layers=1, context=0, new=1, ragged=False, rope=False, tokens=0, window=0, keep=0)
    case.update(given)
    return case


def listed():
    return [
        # A small model's chat turn: one sequence, one token through 16 layers of 8-bit caches.  Nothing but latency and
        # launches.
        _case("chat_small", "steps", cache="quantized", bits=8, q_heads=16, kv_heads=4, key_dim=64, value_dim=64, layers=16,
              context=512, rope=True),
        # One user's long chat with an 8B-class model, 4-bit cache: a token through four of its layers over 30 000 keys.
        _case("chat_long_q4", "steps", cache="quantized", bits=4, layers=4, context=30011, rope=True),
        # Serving: a batch of 32 at a context of 32768 from a 4-bit cache, one token, one layer.
        _case("serve_q4", "steps", cache="quantized", bits=4, batch=32, context=32768),
        # Serving from a full-precision bfloat16 cache: a batch of 8 at 8191 keys, two layers.
        _case("serve_bf16", "steps", dtype="bf16", batch=8, layers=2, context=8191),
        # Serving a model with eight query heads to a kv head, 4-bit cache, two layers.
        _case("serve_gqa8_q4", "steps", cache="quantized", bits=4, dtype="bf16", batch=8, q_heads=64, layers=2, context=8000, rope=True),
        # Speculative decoding: a ragged, left-padded batch of 16, four draft tokens scored and rejected.
        _case("speculate_q4", "steps", cache="quantized", bits=4, batch=16, context=16384, new=4, ragged=True),
        # A sliding-window layer (window 4096, four pinned tokens): a prompt that wraps the ring, then tokens in it.
        _case("ring_request", "prompt", cache="rotating", dtype="bf16", batch=4, q_heads=8, kv_heads=4, key_dim=256,
              value_dim=256, context=6000, tokens=48, window=4096, keep=4),
        # One sequence's prompt into a full-precision cache, 8B-class layer.
        _case("prompt_bf16", "prompt", dtype="bf16", context=8192, rope=True),
        # The same into a 4-bit cache, with the first tokens of the answer.
        _case("prompt_q4", "prompt", cache="quantized", bits=4, context=6001, tokens=8, rope=True),
        # A full-attention layer of head size 512 (Gemma 4): prompt and answer.
        _case("head512_request", "prompt", dtype="bf16", q_heads=8, kv_heads=2, key_dim=512, value_dim=512, context=2048,
              tokens=32, rope=True),
        # A model run in float32: a short prompt and the start of the answer.
        _case("float32_request", "prompt", dtype="f32", q_heads=16, kv_heads=4, key_dim=64, value_dim=64, context=1500,
              tokens=16, rope=True),
        # Four layers of a prompt cache converted to 4 bits and read out to be saved.
        _case("convert_q4", "convert", bits=4, batch=2, layers=4, context=5000),
    ]


# head layouts met in use: (query heads, kv heads, key size, value size)
LAYOUTS = [(16, 4, 64, 64), (32, 8, 64, 64), (32, 8, 128, 128), (64, 8, 128, 128), (28, 4, 128, 128), (16, 8, 128, 128),
           (8, 4, 256, 256), (32, 32, 96, 96), (16, 16, 192, 128), (8, 2, 512, 512)]
LARGEST_BYTES, LARGEST_FLOPS = 1.1e9, 5.0e11  # a drawn case costs no more than the largest listed ones


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    while True:
        kind = rng.choice(["steps", "steps", "steps", "prompt", "prompt", "convert"])
        hq, hkv, dk, dv = rng.choice(LAYOUTS)
        case = _case("", kind, q_heads=hq, kv_heads=hkv, key_dim=dk, value_dim=dv, dtype=rng.choice(["f16", "bf16"]),
                     batch=_log_uniform(rng, 1, 32), context=_log_uniform(rng, 64, 32768), rope=rng.random() < 0.5)
        del case["name"]
        quantized = kind == "convert" or rng.random() < 0.55
        if quantized:
            case.update(bits=rng.choice([4, 4, 4, 8, 8, 6, 3]), group=32 if dk % 64 or dv % 64 else 64)
        if kind == "steps":
            case["cache"] = "quantized" if quantized else "simple"
            case.update(layers=rng.choice([1, 1, 2, 4, 8]), new=rng.choice([1, 1, 1, 2, 3, 4, 5]))
            case["ragged"] = case["batch"] > 1 and rng.random() < 0.25
            if not quantized and rng.random() < 0.15:
                case["dtype"] = "f32"
        elif kind == "prompt":
            case.update(tokens=rng.choice([0, 4, 16, 32]))
            if quantized:
                case["cache"] = "quantized"
            elif rng.random() < 0.3:
                case.update(cache="rotating", window=_log_uniform(rng, 256, 4096), keep=rng.choice([0, 4]))
            elif rng.random() < 0.2:
                case["dtype"] = "f32"
        else:
            case.update(rope=False, layers=rng.choice([1, 2, 4]))
        w = work(case)
        slow = case["dtype"] == "f32" or dk > 256
        if w["bytes"] <= LARGEST_BYTES / (4 if slow else 1) and w["flops"] <= LARGEST_FLOPS / (20 if slow else 1):
            return case


# ---- inputs -------------------------------------------------------------------------------------------------------
def _rows(gen, case, heads, n, size, channels=None):
    x = torch.randn(case["batch"], heads, n, size, generator=gen, device="cuda")
    if channels is not None:
        x *= channels
    return x.to(DTYPES[case["dtype"]])


def _channels(gen, size):
    """Per-channel spread: 1 % of the channels eight times the others."""
    c = torch.ones(size, device="cuda")
    c[torch.randperm(size, generator=gen, device="cuda")[:max(1, size // 100)]] = 8.0
    return c


def _new_cache(case):
    if case["cache"] == "quantized":
        return kvhip.QuantizedKVCache(case["group"], case["bits"])
    if case["cache"] == "rotating":
        return kvhip.RotatingKVCache(case["window"], keep=case["keep"])
    return kvhip.KVCacheSimple()


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    hq, hkv, dk, dv = case["q_heads"], case["kv_heads"], case["key_dim"], case["value_dim"]
    ck, cv = _channels(gen, dk), 0.5 * _channels(gen, dv)
    state = {"case": case, "scale": dk ** -0.5, "rope": kvhip.RoPE(dk, base=500000.0) if case["rope"] else None}

    def call(n):
        return _rows(gen, case, hq, n, dk), _rows(gen, case, hkv, n, dk, ck), _rows(gen, case, hkv, n, dv, cv)

    if case["kind"] == "prompt":
        chunks = []
        total = case["context"]
        kvhip.PrefillParameters().for_each_chunk(total, lambda r: chunks.append(len(r)), reserving=0)
        state["chunks"] = [call(n) for n in chunks]
        state["tokens"] = [call(1) for _ in range(case["tokens"])]
        return state

    state["caches"] = []
    for _ in range(case["layers"]):
        cache = kvhip.KVCacheSimple() if case["kind"] == "convert" else _new_cache(case)
        for at in range(0, case["context"], CHUNK):
            n = min(CHUNK, case["context"] - at)
            k, v = _rows(gen, case, hkv, n, dk, ck), _rows(gen, case, hkv, n, dv, cv)
            if case["cache"] == "quantized" and case["kind"] == "steps":
                cache.update_quantized(k, v, fetch=False)
            else:
                cache.update(k, v, fetch=False)
        state["caches"].append(cache)
    if case["kind"] == "steps":
        state["calls"] = [call(case["new"]) for _ in range(case["layers"])]
        state["left_pad"] = None
        if case["ragged"]:
            low = max(1, case["context"] // RAGGED_MIN)
            lengths = torch.randint(low, case["context"] + 1, (case["batch"],), generator=gen, device="cuda", dtype=torch.int32)
            state["left_pad"] = case["context"] - lengths
    return state


# ---- one pass -----------------------------------------------------------------------------------------------------
def _attend(state, cache, call, mask):
    q, k, v = call
    if state["rope"] is not None:
        return kvhip.attention_with_rope_and_cache_update(state["rope"], q, k, v, cache, state["scale"], mask)
    return kvhip.attention_with_cache_update(q, k, v, cache, state["scale"], mask)


def run(state):
    case = state["case"]
    if case["kind"] == "steps":
        caches, n = state["caches"], case["new"]
        if state["left_pad"] is not None:
            mask = kvhip.MaskMode.window_mask(caches[0].offset, 0, left_pad=state["left_pad"])
        else:
            mask = kvhip.create_attention_mask(n, caches[0])
        out = [_attend(state, cache, call, mask) for cache, call in zip(caches, state["calls"])]
        kvhip.trim_prompt_cache(caches, n)
        return out
    if case["kind"] == "prompt":
        cache = _new_cache(case)
        out = []
        for call in state["chunks"] + state["tokens"]:
            mask = kvhip.create_attention_mask(call[0].shape[2], cache, case["window"] or None)
            out.append(_attend(state, cache, call, mask))
        return out
    caches = list(state["caches"])
    kvhip.maybe_affine_quantize_kv_cache(caches, case["bits"], case["group"], 0)
    return [cache.state for cache in caches]


# ---- what a pass cannot do without --------------------------------------------------------------------------------
def _row_bytes(case, quantized):
    """Bytes of one cached token of one kv head, keys and values."""
    width = case["key_dim"] + case["value_dim"]
    es = DTYPES[case["dtype"]].itemsize
    return width * case["bits"] / 8 + width / case["group"] * 2 * es if quantized else width * es


def work(case):
    b, hq, hkv, dk, dv = (case[k] for k in ("batch", "q_heads", "kv_heads", "key_dim", "value_dim"))
    es = DTYPES[case["dtype"]].itemsize
    cached = b * hkv * _row_bytes(case, case["cache"] == "quantized")  # of one token, all kv heads
    dense = b * (hkv + hq) * (dk + dv) * es                           # new rows, queries and outputs of one token
    per_key = 2.0 * b * hq * (dk + dv)                                # flops of one query row and one key
    t = case["context"]
    if case["kind"] == "steps":
        n, mean = case["new"], (1 + 1 / RAGGED_MIN) / 2 if case["ragged"] else 1.0
        keys = t * mean + n
        return {"bytes": case["layers"] * (cached * keys + dense * n), "flops": case["layers"] * per_key * n * (keys - (n - 1) / 2)}
    if case["kind"] == "prompt":
        w, steps = case["window"] or 1 << 60, case["tokens"]
        prompt_keys = sum(min(i + 1, w) for i in range(t))
        step_keys = sum(min(t + i + 1, w) for i in range(steps))
        return {"bytes": dense * (t + steps) + cached * (min(t, w) + step_keys), "flops": per_key * (prompt_keys + step_keys)}
    full, packed = b * hkv * t * _row_bytes(case, False), b * hkv * t * _row_bytes(case, True)
    return {"bytes": case["layers"] * (full + 2 * packed), "flops": case["layers"] * 4.0 * b * hkv * t * (dk + dv)}


def tolerance(case):
    """Four times the distance from a float64 evaluation over the same cached rows (2-norms): float16 1.3e-3, bfloat16
    2.2e-3, float32 0.6e-6 and up to twice that over long contexts; bfloat16 scores of a quantized cache 1.0e-2, since
    they are rounded to bfloat16 before the softmax as the unfused quantized attention does."""
    if case["kind"] == "convert":
        return "exact"
    if case["dtype"] == "bf16" and case["cache"] == "quantized":
        return {"rel": 3e-2, "max": 0.99}
    return {"f16": {"rel": 5e-3}, "bf16": {"rel": 1e-2}, "f32": {"rel": 5e-6}}[case["dtype"]]
