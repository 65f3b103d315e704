"""Single-token steps whose kernel writes the step's new row itself, at the slots where that can go wrong: the first and
the last row of a tile and of a page, the new row in the first tile of its wavefront and in a later one.  Against the
same step as separate calls (rotate, append, attend), which read the row from the page: the same bits in the cache and in
the output."""
import pytest
import torch

import kvhip

pytestmark = pytest.mark.gpu

# rows cached before the step: tile (64) and page (256) edges, one tile per wavefront, several, several workgroups
CONTEXTS = [1, 63, 64, 255, 256, 300, 511, 1023, 1024, 2047, 5000]


def _rows(gen, B, heads, n, D, dtype):
    return torch.randn(B, heads, n, D, generator=gen, device="cuda").to(dtype)


def _caches(kind, gs):
    return [kvhip.KVCacheSimple() if kind == "simple" else kvhip.QuantizedKVCache(gs, kind) for _ in range(2)]


def _compare(caches, q, k, v, rope):
    D = q.shape[3]
    one, two = caches
    if rope is None:
        got = kvhip.attention_with_cache_update(q, k, v, one, D ** -0.5)
        two._update(k, v)
        turned = q
    else:
        got = kvhip.attention_with_rope_and_cache_update(rope, q, k, v, one, D ** -0.5)
        turned = kvhip.apply_rotary_position(rope, q, two.rope_offset)
        two.update_rope(rope, k, v)
    assert torch.equal(got, two.attend(turned, D ** -0.5))


@pytest.mark.parametrize("rotary", [False, True])
@pytest.mark.parametrize("kind,gs,dtype,B,Hq,Hkv,Dk,Dv", [
    (4, 64, torch.float16, 1, 8, 2, 128, 128), (8, 64, torch.float16, 2, 16, 4, 64, 64), (4, 32, torch.bfloat16, 1, 4, 2, 64, 64),
    (8, 128, torch.bfloat16, 1, 4, 1, 256, 256), (4, 64, torch.float16, 70, 4, 2, 128, 128),
    (4, 64, torch.bfloat16, 2, 16, 2, 128, 128), (6, 64, torch.float16, 1, 8, 2, 128, 128), (3, 64, torch.bfloat16, 2, 4, 4, 256, 256),
    (4, 32, torch.float16, 1, 8, 8, 96, 96), (8, 64, torch.bfloat16, 1, 4, 4, 192, 128),
    ("simple", 0, torch.float16, 1, 8, 2, 64, 64), ("simple", 0, torch.bfloat16, 2, 16, 2, 128, 128), ("simple", 0, torch.float16, 1, 4, 1, 256, 256),
    ("simple", 0, torch.bfloat16, 1, 8, 2, 512, 512), ("simple", 0, torch.float16, 2, 16, 1, 512, 512),
    ("simple", 0, torch.float32, 1, 16, 4, 64, 64), ("simple", 0, torch.float32, 1, 4, 4, 96, 96), ("simple", 0, torch.float32, 2, 16, 1, 128, 128),
    ("simple", 0, torch.float32, 1, 8, 2, 256, 256), ("simple", 0, torch.float32, 1, 4, 2, 192, 128)])
def test_a_step_equals_its_separate_calls(kind, gs, dtype, B, Hq, Hkv, Dk, Dv, rotary):
    gen = torch.Generator(device="cuda").manual_seed(17)
    rope = kvhip.RoPE(Dk, base=1e4) if rotary else None
    for T in CONTEXTS if B < 64 else (63, 300, 511):
        caches = _caches(kind, gs)
        k, v = _rows(gen, B, Hkv, T, Dk, dtype), _rows(gen, B, Hkv, T, Dv, dtype)
        for c in caches:
            c._update(k, v)
        for _ in range(2):
            _compare(caches, _rows(gen, B, Hq, 1, Dk, dtype), _rows(gen, B, Hkv, 1, Dk, dtype), _rows(gen, B, Hkv, 1, Dv, dtype), rope)
        for a, b in zip(caches[0].state, caches[1].state):
            assert torch.equal(a, b), T


@pytest.mark.parametrize("rotary", [False, True])
@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (128, torch.bfloat16), (256, torch.bfloat16), (512, torch.bfloat16), (128, torch.float32), (256, torch.float32)])
def test_a_ring_step_equals_its_separate_calls(D, dtype, rotary):
    """The ring's write cursor goes round: the new row lies in any tile of any wavefront."""
    gen = torch.Generator(device="cuda").manual_seed(18)
    rope = kvhip.RoPE(D, base=1e4) if rotary else None
    caches = [kvhip.RotatingKVCache(1400, keep=4) for _ in range(2)]
    k, v = _rows(gen, 1, 2, 1300, D, dtype), _rows(gen, 1, 2, 1300, D, dtype)
    for c in caches:
        c._update(k, v)
    for i in range(400):
        q, k, v = (_rows(gen, 1, h, 1, D, dtype) for h in (8, 2, 2))
        _compare(caches, q, k, v, rope)
    for a, b in zip(caches[0].state, caches[1].state):
        assert torch.equal(a, b)
