"""GPU parity of the rotary embedding in front of the cache write.

`kvhip_rope_apply` is held to one unit in the last place of a 16-bit array dtype against the
CPU restatement (angles are the same float32 values on both sides; the device rounds its
float32 products, the restatement works in float64: which intermediate roundings MLX's own
CPU path makes is parity unpinned).  The fused rotate-and-append must equal rotate-then-append
on the device bit for bit, for every cache kind, since both run the same element function.
"""
import ctypes as C

import numpy as np
import pytest
import torch

import kvhip
from kvhip.cache import _DT as DT
from oracle import kv_oracle as O
from oracle import rope as OR
from tests.util import NAME, dev, err_stats, np32, randn

pytestmark = pytest.mark.gpu

# float32 arrays: the device's three float32 roundings and its sincosf against float64, a few ulp
ULP = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7, torch.float32: 2.0 ** -19}


def within_one_ulp(got, want, dtype, pair_norm):
    """|got - want| <= one ulp of dtype at the magnitude of the rotated pair (an element of a
    pair may be tiny while its error scales with the pair)."""
    d = np.abs(got.astype(np.float64) - want.astype(np.float64))
    return bool((d <= ULP[dtype] * np.maximum(pair_norm, 1e-30) * 1.001 + 1e-30).all()), float(d.max())


def pair_norms(x, dims, traditional):
    n = np.abs(x).astype(np.float64).copy()
    half = dims // 2
    if traditional:
        m = np.maximum(np.abs(x[..., 0:dims:2]), np.abs(x[..., 1:dims:2]))
        n[..., 0:dims:2] = m
        n[..., 1:dims:2] = m
    else:
        m = np.maximum(np.abs(x[..., :half]), np.abs(x[..., half:dims]))
        n[..., :half] = m
        n[..., half:dims] = m
    return n * np.sqrt(2.0)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("traditional", [False, True])
@pytest.mark.parametrize("D,dims,offset", [(128, 128, 0), (128, 128, 4097), (64, 32, 100000), (256, 256, 17)])
def test_rope_apply_matches_the_restatement(dtype, traditional, D, dims, offset):
    rng = np.random.default_rng(0)
    x32, xd = randn(rng, (2, 3, 5, D), dtype)
    rope = kvhip.RoPE(dims, traditional=traditional, base=500000.0, scale=1.0)
    got = np32(kvhip.apply_rotary_position(rope, xd, offset))
    want = OR.rope(x32, dims, traditional, 500000.0, 1.0, offset, dtype=NAME[dtype])
    ok, mx = within_one_ulp(got, want, dtype, pair_norms(x32, dims, traditional))
    assert ok, f"max diff {mx:.3e}"
    if offset == 0:
        assert np.array_equal(got[:, :, 0], x32[:, :, 0])   # position 0 is the identity
    assert np.array_equal(got[..., dims:], x32[..., dims:])


def test_rope_scale_freqs_and_batch_offsets():
    rng = np.random.default_rng(1)
    dtype = torch.float16
    x32, xd = randn(rng, (3, 2, 4, 64), dtype)
    freqs = (1.0 / OR.inv_freqs(64, 10000.0) * np.linspace(1.0, 8.0, 32)).astype(np.float32)
    rope = kvhip.RoPE(64, traditional=False, scale=0.5, freqs=freqs)
    offs = torch.tensor([0, 9, 1234], dtype=torch.int32)
    got = np32(kvhip.apply_rotary_position(rope, xd, offs))
    want = OR.rope(x32, 64, False, 10000.0, 0.5, offs.numpy(), freqs=freqs, dtype="float16")
    ok, mx = within_one_ulp(got, want, dtype, pair_norms(x32, 64, False))
    assert ok, f"max diff {mx:.3e}"
    # in place
    y = xd.clone()
    r, keep = rope.to_c()
    import ctypes as C
    from kvhip import _lib as L
    L.check(kvhip.load().kvhip_rope_apply(C.byref(r), C.c_void_p(y.data_ptr()), C.c_void_p(y.data_ptr()), 3, 2, 4, 64,
                                          L.F16, 0, C.c_void_p(offs.cuda().data_ptr()), None))
    torch.cuda.synchronize()
    assert np.array_equal(np32(y), got)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_fused_append_equals_rotate_then_append_simple_and_ring(dtype):
    rng = np.random.default_rng(2)
    rope = kvhip.RoPE(64, traditional=False, base=10000.0)
    for make in (lambda: kvhip.KVCacheSimple(), lambda: kvhip.RotatingKVCache(24, keep=2)):
        fused, plain = make(), make()
        for Lq in (7, 1, 1, 9, 1, 12, 1):          # ring: multi-token writes, single-token writes, wraps
            _, k = randn(rng, (2, 2, Lq, 64), dtype)
            _, v = randn(rng, (2, 2, Lq, 64), dtype)
            off = plain.offset
            assert fused.rope_offset == off
            fused.update_rope(rope, k, v)
            plain.update(kvhip.apply_rotary_position(rope, k, off), v, fetch=False)
            assert fused.offset == plain.offset
            fk, fv = fused.fetch()
            pk, pv = plain.fetch()
            assert torch.equal(fk, pk) and torch.equal(fv, pv)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("traditional", [False, True])
@pytest.mark.parametrize("Dk,Dv,dims", [(128, 128, 128), (192, 128, 64)])
def test_fused_prompt_sized_append_equals_rotate_then_append(dtype, traditional, Dk, Dv, dims):
    """Whole-tile appends rotate inside the tile kernel."""
    rng = np.random.default_rng(7)
    rope = kvhip.RoPE(dims, traditional=traditional, base=500000.0)
    fused, plain = kvhip.KVCacheSimple(), kvhip.KVCacheSimple()
    for Lq in (5, 200, 130):
        _, k = randn(rng, (2, 2, Lq, Dk), dtype)
        _, v = randn(rng, (2, 2, Lq, Dv), dtype)
        off = plain.offset
        fused.update_rope(rope, k, v)
        plain.update(kvhip.apply_rotary_position(rope, k, off), v, fetch=False)
    fk, fv = fused.fetch()
    pk, pv = plain.fetch()
    assert torch.equal(fk, pk) and torch.equal(fv, pv)


@pytest.mark.parametrize("bits,gs,D,dims", [(4, 64, 128, 96), (8, 32, 128, 96), (4, 32, 96, 96), (8, 32, 96, 48),
                                            (4, 64, (192, 128), 64), (8, 32, (192, 128), 192)])
def test_fused_quantize_on_append_equals_rotate_then_append(bits, gs, D, dims):
    rng = np.random.default_rng(3)
    dtype = torch.float16
    Dk, Dv = D if isinstance(D, tuple) else (D, D)
    rope = kvhip.RoPE(dims, traditional=True, base=1e6)          # (partial rotation of a 128-wide head)
    fused, plain = kvhip.QuantizedKVCache(gs, bits), kvhip.QuantizedKVCache(gs, bits)
    for Lq in (70, 1, 1, 3, 190):
        _, k = randn(rng, (2, 2, Lq, Dk), dtype)
        _, v = randn(rng, (2, 2, Lq, Dv), dtype)
        off = plain.offset
        fused.update_rope(rope, k, v)
        plain.update_quantized(kvhip.apply_rotary_position(rope, k, off), v, fetch=False)
    for a, b in zip(fused.state, plain.state):
        assert torch.equal(a, b)
    # and the codes are what the restatement gives for the rotated keys (bit-exact quantizer)
    assert fused.offset == 265


def test_layer_sequence_against_the_restatement():
    """rope(q), rope(k) at the cache offset, append, attend -- the sequence of an attention
    layer -- against rope + sdpa of the restatement, prefill chunk then decode steps."""
    rng = np.random.default_rng(4)
    dtype = torch.float16
    B, Hq, Hkv, D = 2, 8, 2, 64
    rope = kvhip.RoPE(D, traditional=False, base=10000.0)
    cache = kvhip.KVCacheSimple()
    ks, vs = [], []
    for step, Lq in enumerate((33, 1, 1, 1)):
        q32, q = randn(rng, (B, Hq, Lq, D), dtype)
        k32, k = randn(rng, (B, Hkv, Lq, D), dtype)
        v32, v = randn(rng, (B, Hkv, Lq, D), dtype)
        off = cache.offset
        mask = kvhip.MaskMode.causal() if Lq > 1 else kvhip.MaskMode.none()
        out = kvhip.attention_with_rope_and_cache_update(rope, q, k, v, cache, D ** -0.5, mask)
        ks.append(OR.rope(k32, D, offset=off, dtype="float16"))
        vs.append(v32)
        ref = O.sdpa(OR.rope(q32, D, offset=off, dtype="float16"), np.concatenate(ks, 2), np.concatenate(vs, 2),
                     D ** -0.5, O.Mask.CAUSAL if Lq > 1 else O.Mask.NONE, "float16")
        mx, mean = err_stats(np32(out), ref)
        assert mx <= 1e-2 and mean <= 1e-3, f"step {step}: {mx:.3e} {mean:.3e}"
    assert cache.offset == 36


def test_staged_round_positions_count_the_staged_rows():
    rng = np.random.default_rng(5)
    dtype = torch.float16
    rope = kvhip.RoPE(64)
    live = kvhip.RotatingKVCache(16, keep=0)
    _, k0 = randn(rng, (1, 2, 10, 64), dtype)
    live.update_rope(rope, k0, k0)
    staged = kvhip.RotatingStagedKVCache(live)
    _, k1 = randn(rng, (1, 2, 2, 64), dtype)
    _, k2 = randn(rng, (1, 2, 1, 64), dtype)
    assert staged.rope_offset == 10
    staged.update_rope(rope, k1, k1)
    assert staged.rope_offset == 12
    staged.update_rope(rope, k2, k2)
    sk, _ = staged.staged_arrays
    want = torch.cat([kvhip.apply_rotary_position(rope, k1, 10), kvhip.apply_rotary_position(rope, k2, 12)], 2)
    assert torch.equal(sk, want)
    staged.commit(3)
    assert live.offset == 13


def test_rope_argument_errors():
    _, x = randn(np.random.default_rng(6), (1, 1, 1, 64), torch.float16)
    for bad in (kvhip.RoPE(63), kvhip.RoPE(66), kvhip.RoPE(0), kvhip.RoPE(64, base=0.0)):
        with pytest.raises(kvhip.KVHipError):
            kvhip.apply_rotary_position(bad, x, 0)
    c = kvhip.KVCacheSimple()
    with pytest.raises(kvhip.KVHipError):
        c.update_rope(kvhip.RoPE(130), x, x)
    assert c.offset == 0


def _cache_of(kind):
    if kind == "simple":
        return kvhip.KVCacheSimple()
    return kvhip.RotatingKVCache(150, keep=4) if kind == "ring" else kvhip.QuantizedKVCache(32, kind)


@pytest.mark.parametrize("kind", ["simple", "ring", 4, 3, 8])
@pytest.mark.parametrize("dtype,Hq,Hkv,Dk,Dv,dims,traditional", [
    (torch.float16, 8, 2, 128, 128, 128, False), (torch.bfloat16, 40, 4, 64, 64, 64, False),
    (torch.float16, 6, 2, 96, 96, 64, True), (torch.bfloat16, 8, 4, 256, 256, 256, False), (torch.float16, 4, 4, 128, 128, 32, True), (torch.bfloat16, 4, 4, 192, 128, 64, False),
    (torch.float16, 4, 2, 128, 128, 72, False),     # pairs cut through 16-byte chunks: a launch of its own
    (torch.bfloat16, 4, 1, 512, 512, 512, False), (torch.float32, 4, 2, 64, 64, 64, False)])
def test_queries_in_the_appends_launch_equal_separate_calls(kind, dtype, Hq, Hkv, Dk, Dv, dims, traditional):
    """Bit for bit: the one call runs the same rotation, append and attention as the three (and a single token's decode
    kernel, which rotates its rows itself, the same arithmetic)."""
    B = 3
    rope = kvhip.RoPE(dims, traditional=traditional, base=1e6)
    one, three = _cache_of(kind), _cache_of(kind)
    gen = torch.Generator(device="cuda").manual_seed(11)
    positions = torch.tensor([5, 0, 1000], dtype=torch.int32, device="cuda")
    for step, Lq in enumerate((70, 1, 5, 131, 2, 1, 1, 1)):
        q, k, v = (torch.randn(B, h, Lq, d, generator=gen, device="cuda").to(dtype) for h, d in ((Hq, Dk), (Hkv, Dk), (Hkv, Dv)))
        at = positions if step in (2, 6) else None
        mask = kvhip.create_attention_mask(Lq, one)
        got = kvhip.attention_with_rope_and_cache_update(rope, q, k, v, one, Dk ** -0.5, mask, at)
        turned = kvhip.apply_rotary_position(rope, q, at if at is not None else three.offset)
        three.update_rope(rope, k, v, at)
        assert torch.equal(got, three.attend(turned, Dk ** -0.5, mask)), f"step {step}"
    for a, b in zip(one.state, three.state):
        assert torch.equal(a, b)


@pytest.mark.parametrize("bits,gs", [(4, 32), (8, 32), (3, 32)])
@pytest.mark.parametrize("Hq,Hkv,Dk,Dv,dims,traditional", [
    (40, 8, 96, 96, 96, False), (32, 32, 96, 96, 64, False), (32, 8, 96, 96, 96, True), (24, 24, 192, 128, 192, False),
    (128, 16, 192, 128, 192, False), (16, 16, 192, 128, 64, False), (16, 8, 192, 128, 192, True)])
def test_every_query_head_turns_in_the_quantizers_launch(bits, gs, Hq, Hkv, Dk, Dv, dims, traditional):
    """Head counts that the query workgroups beside rows of 96 and 192 elements (three quarters of the usual width) pass
    over more than once, below and above the number of row positions from which one workgroup takes every head.  Each row
    position has its own values, so that a head left as an earlier call had it shows."""
    B, dtype = 3, torch.bfloat16
    rope = kvhip.RoPE(dims, traditional=traditional, base=1e6)
    one, three = kvhip.QuantizedKVCache(gs, bits), kvhip.QuantizedKVCache(gs, bits)
    gen = torch.Generator(device="cuda").manual_seed(13)
    for Lq in (90, 12, 13, 5, 91):
        q, k, v = (torch.randn(B, h, Lq, d, generator=gen, device="cuda").to(dtype) for h, d in ((Hq, Dk), (Hkv, Dk), (Hkv, Dv)))
        got = kvhip.attention_with_rope_and_cache_update(rope, q, k, v, one, Dk ** -0.5, kvhip.MaskMode.causal())
        turned = kvhip.apply_rotary_position(rope, q, three.offset)
        three.update_rope(rope, k, v)
        assert torch.equal(got, three.attend(turned, Dk ** -0.5, kvhip.MaskMode.causal())), Lq


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("D,dims", [(64, 64), (40, 32), (128, 72)])
def test_one_call_in_a_staged_round_counts_the_staged_rows(dtype, D, dims):
    """Queries and keys turn at the offset plus the rows staged so far, as `ropeOffset` has it in an open round (40: a
    head size stored zero-padded; 72: pairs that cut through 16-byte chunks)."""
    B, Hq, Hkv = 2, 4, 2
    rope = kvhip.RoPE(dims, base=1e4)
    gen = torch.Generator(device="cuda").manual_seed(3)

    def rows(n):
        return [torch.randn(B, h, n, D, generator=gen, device="cuda").to(dtype) for h in (Hq, Hkv, Hkv)]

    rings = [kvhip.RotatingKVCache(48, keep=2) for _ in range(2)]
    _, k, v = rows(30)
    for ring in rings:
        ring.update(k, v, fetch=False)
    staged = [kvhip.RotatingStagedKVCache(ring) for ring in rings]
    for Lq in (2, 1, 3):
        q, k, v = rows(Lq)
        turned = kvhip.apply_rotary_position(rope, q, staged[1].rope_offset)
        staged[1].update_rope(rope, k, v)
        want = staged[1].attend(turned, D ** -0.5, kvhip.MaskMode.causal())
        got = rings[0].update_attend_rope(rope, q, k, v, D ** -0.5, kvhip.MaskMode.causal())
        assert torch.equal(got, want), Lq
    assert all(torch.equal(a, b) for a, b in zip(staged[0].staged_arrays, staged[1].staged_arrays))


@pytest.mark.parametrize("traditional", [False, True])
@pytest.mark.parametrize("dims", [64, 56])  # (56: pairs that cut through 16-byte chunks)
def test_angles_of_any_size(dims, traditional):
    """Frequencies and a scale that give angles from 10^-3 to 10^38 (all finite): float32 sines and cosines of the float32 angle."""
    rng = np.random.default_rng(8)
    x32, xd = randn(rng, (1, 2, 9, 64), torch.float32)
    freqs = np.logspace(0., -34., dims // 2).astype(np.float32)
    rope = kvhip.RoPE(dims, traditional=traditional, scale=0.5, freqs=freqs)
    for offset in (0, 3, 4000):
        got = np32(kvhip.apply_rotary_position(rope, xd, offset))
        want = OR.rope(x32, dims, traditional, 10000.0, 0.5, offset, freqs=freqs, dtype="float32")
        ok, mx = within_one_ulp(got, want, torch.float32, pair_norms(x32, dims, traditional))
        assert ok, f"offset {offset}: max diff {mx:.3e}"


@pytest.mark.parametrize("kind,dtype,D,Lq", [("simple", torch.float16, 128, 5), ("simple", torch.bfloat16, 512, 1), ("simple", torch.float32, 64, 1),
                                             ("simple", torch.float16, 128, 1), (4, torch.float16, 128, 5), (4, torch.bfloat16, 128, 1)])
def test_one_call_is_captured_where_the_separate_calls_are(kind, dtype, D, Lq):
    """Pages reserved and attention scratch there from calls without the rotation: the one call allocates nothing of its
    own, so it can be captured, and each replay equals the separate calls on the same rows."""
    B, Hq, Hkv = 2, 8, 2
    rope = kvhip.RoPE(D, base=1e4)
    gen = torch.Generator(device="cuda").manual_seed(5)

    def rows(n):
        return [torch.randn(B, h, n, D, generator=gen, device="cuda").to(dtype) for h in (Hq, Hkv, Hkv)]

    cache = kvhip.KVCacheSimple() if kind == "simple" else kvhip.QuantizedKVCache(64, kind)
    cache.reserve(B, Hkv, D, D, dtype, 600)
    _, k, v = rows(300)
    cache._update(k, v)
    mask = kvhip.create_attention_mask(Lq, cache)
    q, k, v = rows(Lq)

    def separate():
        turned = kvhip.apply_rotary_position(rope, q, cache.rope_offset)
        cache.update_rope(rope, k, v)
        out = cache.attend(turned, D ** -0.5, mask)
        cache.trim(Lq)
        return out

    separate()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = kvhip.attention_with_rope_and_cache_update(rope, q, k, v, cache, D ** -0.5, mask)
    cache.trim(Lq)
    for _ in range(3):
        for t, new in zip((q, k, v), rows(Lq)):
            t.copy_(new)
        graph.replay()
        got = out.clone()
        torch.cuda.synchronize()
        assert torch.equal(got, separate())
        torch.cuda.synchronize()


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 512), (torch.float16, 512), (torch.float32, 64), (torch.float32, 128), (torch.float16, 128)])
@pytest.mark.parametrize("ring", [False, True])
def test_a_captured_token_that_turns_in_the_attention_kernel_needs_no_scratch(dtype, D, ring):
    """The first rotary call of a cache, captured, through the C entry without `q_rotated`: the kernel that attends turns
    the queries itself, so there is nothing to refuse."""
    B, Hq, Hkv = 2, 8, 2
    rope = kvhip.RoPE(D, base=1e4)
    gen = torch.Generator(device="cuda").manual_seed(6)

    def rows(n):
        return [torch.randn(B, h, n, D, generator=gen, device="cuda").to(dtype) for h in (Hq, Hkv, Hkv)]

    _, k, v = rows(300)
    warm = [rows(1) for _ in range(2)]  # (the ring at its size, the attention scratch there)
    caches = [kvhip.RotatingKVCache(256, keep=4) if ring else kvhip.KVCacheSimple() for _ in range(4)]
    for c in caches:
        c.update(k, v, fetch=False)
        for row in warm:
            c.update_attend(*row, D ** -0.5)
        if not ring:
            c.trim(2)
    one, others = caches[0], caches[1:]
    q, k, v = rows(1)
    out = torch.empty_like(q)
    r, keep = rope.to_c()
    lib, mask = kvhip.load(), kvhip.MaskMode.none().to_c(B, Hq, 1)[0]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        status = lib.kvhip_cache_update_attend_rope(one._h, C.byref(r), None, q.data_ptr(), k.data_ptr(), v.data_ptr(), B, Hq, Hkv, 1, D, D, DT[dtype],
                                                    D ** -0.5, C.byref(mask), None, out.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert status == 0, lib.kvhip_last_error_message()
    for other in others:
        for t, new in zip((q, k, v), rows(1)):
            t.copy_(new)
        graph.replay()
        got = out.clone()
        torch.cuda.synchronize()
        turned = kvhip.apply_rotary_position(rope, q, other.rope_offset)
        other.update_rope(rope, k, v)
        assert torch.equal(got, other.attend(turned, D ** -0.5))
        torch.cuda.synchronize()


def test_one_call_across_the_lengths_at_which_the_float32_kernel_changes():
    """One token of 128 pairs of 128 columns in float32: from 512 rows on the vector-ALU kernel, which neither writes nor
    turns rows, takes the step, and the call sees that before it decides whether the queries need room."""
    B, Hq, Hkv, D = 16, 8, 8, 128
    rope = kvhip.RoPE(D, base=1e4)
    gen = torch.Generator(device="cuda").manual_seed(7)

    def rows(n):
        return [torch.randn(B, h, n, D, generator=gen, device="cuda") for h in (Hq, Hkv, Hkv)]

    for ring in (False, True):
        one, three = (kvhip.RotatingKVCache(514, keep=4) if ring else kvhip.KVCacheSimple() for _ in range(2))
        _, k, v = rows(507)
        for c in (one, three):
            c.update(k, v, fetch=False)
        for _ in range(10):
            q, k, v = rows(1)
            got = one.update_attend_rope(rope, q, k, v, D ** -0.5)
            turned = kvhip.apply_rotary_position(rope, q, three.rope_offset)
            three.update_rope(rope, k, v)
            assert torch.equal(got, three.attend(turned, D ** -0.5)), one.offset


def test_one_call_refuses_queries_that_do_not_go_with_the_keys():
    """The library reads the queries as the keys' dtype and row count; the method itself says so, before any write."""
    rope = kvhip.RoPE(64, base=1e4)
    cache = kvhip.KVCacheSimple()
    k = torch.randn(1, 2, 3, 64, device="cuda").bfloat16()
    with pytest.raises(TypeError):
        cache.update_attend_rope(rope, torch.randn(1, 4, 3, 64, device="cuda"), k, k, 0.125)
    for shape in [(1, 4, 5, 64), (2, 4, 3, 64), (1, 4, 3, 128)]:
        with pytest.raises(ValueError):
            cache.update_attend_rope(rope, torch.randn(shape, device="cuda").bfloat16(), k, k, 0.125)
    assert cache.offset == 0
    q = torch.randn(1, 4, 3, 64, device="cuda").bfloat16()
    assert cache.update_attend_rope(rope, q, k, k, 0.125).shape == q.shape and cache.offset == 3
