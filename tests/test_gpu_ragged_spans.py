"""Batches of rows of very different lengths: the decode kernels share their spans out by length (2 to 64 rows, where a
workgroup has more than one step over the longest) or give every row the same number.  Against the plain kernel, which
knows nothing of spans, over the same cache."""
import pytest
import torch

import kvhip

pytestmark = pytest.mark.gpu

T, D, HKV = 1700, 128, 2


def _pads(how, B, gen):
    if how == "one long":
        pad = torch.full((B,), T - 1, dtype=torch.int32)
        pad[B // 2] = 0
    elif how == "equal":
        pad = torch.full((B,), 37, dtype=torch.int32)
    elif how == "steps":  # lengths around whole tiles and wavefront steps
        edges = [1, 63, 64, 65, 255, 256, 257, 511, 513, 1023, 1025, T]
        pad = T - torch.tensor([edges[i % len(edges)] for i in range(B)], dtype=torch.int32)
    else:
        pad = torch.randint(0, T, (B,), generator=gen, dtype=torch.int32)
    return pad


@pytest.mark.parametrize("how", ["one long", "equal", "steps", "random"])
@pytest.mark.parametrize("B", [2, 3, 16, 64, 65])
@pytest.mark.parametrize("many", [False, True])  # (batch, kv head) pairs: few, a step to a workgroup; 120 and more, several
@pytest.mark.parametrize("kind,Hq,L", [(4, 8, 1), (8, 4, 2), (4, 8, 4), (5, 4, 1), ("bf16", 8, 1), ("f16", 4, 4)])
def test_ragged_rows_equal_the_plain_kernel(kind, Hq, L, many, B, how):
    hkv = {2: 64, 3: 40, 16: 8}.get(B, HKV) if many else HKV
    Hq = Hq // HKV * hkv
    gen = torch.Generator(device="cuda").manual_seed(3)
    dtype = torch.bfloat16 if kind == "bf16" else torch.float16
    cache = kvhip.KVCacheSimple() if isinstance(kind, str) else kvhip.QuantizedKVCache(64, kind)
    rows = lambda h, n: torch.randn(B, h, n, D, generator=gen, device="cuda").to(dtype)
    cache._update(rows(hkv, T), rows(hkv, T))
    pad = _pads(how, B, torch.Generator().manual_seed(4))
    for lengths in (None, torch.clamp(pad + 700, max=T)):
        mask = kvhip.MaskMode.window_mask(T - L, 0, left_pad=pad, lengths=lengths)
        q = rows(Hq, L)
        lib = kvhip.load()
        got = [cache.attend(q, D ** -0.5, mask), cache.attend(q, D ** -0.5, mask, static_scratch=True)]
        assert lib.kvhip_last_attend_kernel() in (1, 2)
        lib.kvhip_set_kernel_policy(1)
        try:
            want = cache.attend(q, D ** -0.5, mask)
        finally:
            lib.kvhip_set_kernel_policy(0)
        # scores and probabilities of a quantized cache are rounded to the dtype on both sides, at different points: a score
        # of up to 8 by 2^-11 (float16) of itself moves a weight by 2^-8; the full-precision kernels differ by output roundings
        for g in got:
            diff = (g.float() - want.float()).abs().max().item()
            assert diff <= (2 ** -8 if dtype == torch.float16 else 2 ** -6) * max(1.0, want.float().abs().max().item()), (how, diff)
