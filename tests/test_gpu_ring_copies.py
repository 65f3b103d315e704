"""Rows gathered from a ring (a copy, a ring laid out again for a longer write) and key-range parts merged over many rows."""
import numpy as np
import pytest
import torch

import kvhip
from tests.util import randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("window,keep", [(70, 0), (70, 4), (150, 3), (300, 1), (513, 4)])
@pytest.mark.parametrize("dtype,Dk,Dv", [(torch.float16, 64, 64), (torch.bfloat16, 256, 256), (torch.float16, 192, 128),
                                         (torch.bfloat16, 300, 301), (torch.float32, 64, 64), (torch.float32, 30, 7)])
def test_gathered_rows_are_the_rows_written(window, keep, dtype, Dk, Dv):
    """Every shift of the ring against 16-byte chunks, runs that end inside one, chunks across pages, columns beyond 256."""
    rng = np.random.default_rng(window + Dk)
    B, H = 2, 3
    cache = kvhip.RotatingKVCache(window, keep=keep)
    rows = [[], []]
    held = None

    def write(n):
        nonlocal held
        new = [randn(rng, (B, H, n, d), dtype)[1] for d in (Dk, Dv)]
        cache.update(*new, fetch=False)
        for side in range(2):
            rows[side].append(new[side])
        return new

    write(window)
    for n in (1, 1, 1, 2, 4, 1, 7):  # the ring turns by single tokens: odd and even shifts
        for _ in range(n):
            write(1)
        cp = cache.copy()
        assert (cp.offset, cp.meta_state) == (cache.offset, cache.meta_state)
        for a, b in zip(cp.state, cache.state):
            assert torch.equal(a, b)
    # a longer write puts the ring into temporal order first: pinned rows, the newest before it, the new ones
    every = [torch.cat(r, dim=2) for r in rows]
    new = [randn(rng, (B, H, 9, d), dtype)[1] for d in (Dk, Dv)]
    for got, old, n in zip(cache.update(*new), every, new):
        tail = got.shape[2] - keep - 9
        assert torch.equal(got, torch.cat([old[:, :, :keep], old[:, :, old.shape[2] - tail:], n], dim=2))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [64, 80, 96, 128, 256])
@pytest.mark.parametrize("keys,parts", [(200, 1), (700, 2), (900, 3), (1100, 4), (1500, 5), (2100, 8), (3001, 11)])
def test_parts_of_many_rows_merge(dtype, D, keys, parts):
    """One part (no merge), the two to eight of combine_rows_kernel, each of its instances at its last count and at one
    below, and a count above (combine_kernel); rows that do not fill the last workgroup, parts that a row's mask leaves
    empty.  These few workgroups get an eighth of the 32-key tiles each."""
    assert (keys + 31) // 32 // 8 in (parts, parts - 1) and max(1, (keys + 31) // 32 // 8) == parts
    rng = np.random.default_rng(D + keys)
    B, Hq, Hkv, L = 2, 6, 2, 131
    cache = kvhip.KVCacheSimple()
    q = randn(rng, (B, Hq, L, D), dtype)[1]
    k, v = (randn(rng, (B, Hkv, keys, D), dtype)[1] for _ in range(2))
    cache.update(k[:, :, :keys - L].contiguous(), v[:, :, :keys - L].contiguous(), fetch=False)
    window = 150
    mask = kvhip.MaskMode.window_mask(cache.offset, window)
    out = kvhip.attention_with_cache_update(q, k[:, :, keys - L:].contiguous(), v[:, :, keys - L:].contiguous(), cache, D ** -0.5, mask)
    q, k, v = (x.double().cpu() for x in (q, k, v))
    at = torch.arange(keys - L, keys)[:, None]
    keep = (torch.arange(keys)[None] <= at) & (torch.arange(keys)[None] > at - window)
    kk, vv = (x.repeat_interleave(Hq // Hkv, dim=1) for x in (k, v))
    ref = torch.softmax((q @ kk.transpose(2, 3).contiguous() * D ** -0.5).masked_fill(~keep, -float("inf")), dim=-1) @ vv
    # probabilities and outputs round once each: 2 u of the largest value, u = 2^-11 (float16), 2^-8 (bfloat16)
    u = 2.0 ** (-11 if dtype == torch.float16 else -8)
    assert (out.double().cpu() - ref).abs().max() <= 2 * u * v.abs().max()
