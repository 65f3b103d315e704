"""One token over float32 caches and caches of head size 512: tiles at the edges of what the token sees (under no mask, a
window, left padding, lengths) and, at head size 512, sequences of more than 64 tiles, a tile to a part.  Against the plain
kernel, over the same cache."""
import pytest
import torch

import kvhip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,dtype", [(512, torch.bfloat16), (512, torch.float16), (64, torch.float32), (128, torch.float32), (256, torch.float32)])
@pytest.mark.parametrize("B,Hkv", [(1, 2), (2, 1)])
@pytest.mark.parametrize("T", [33, 1500, 2049, 2080, 4095, 4200])
def test_against_the_plain_kernel(D, dtype, B, Hkv, T):
    gen = torch.Generator(device="cuda").manual_seed(T + D)
    rand = lambda h, n: torch.randn(B, h, n, D, generator=gen, device="cuda").to(dtype)
    c = kvhip.KVCacheSimple()
    c._update(rand(Hkv, T), rand(Hkv, T))
    q, lib = rand(4 * Hkv, 1), kvhip.load()
    W = kvhip.MaskMode.window_mask
    ends, pads = (torch.tensor([x, y][:B], dtype=torch.int32) for x, y in ((T - 17, max(1, T - 40)), (T // 2 + 1, 7)))
    for mask in (kvhip.MaskMode.none(), kvhip.MaskMode.causal(), W(T - 1, 16), W(T - 1, 17), W(T - 1, 0, lengths=ends), W(T - 1, 0, left_pad=pads)):
        got = c.attend(q, D ** -0.5, mask)
        assert lib.kvhip_last_attend_kernel() == 5
        try:
            lib.kvhip_set_kernel_policy(1)
            want = c.attend(q, D ** -0.5, mask)
        finally:
            lib.kvhip_set_kernel_policy(0)
        # one rounding of the output on either side, of values up to 5 (float32: sums of D products and of T probabilities)
        tol = {torch.float16: 2.0 ** -8, torch.bfloat16: 2.0 ** -5, torch.float32: 1e-5}[dtype]
        assert (got.double() - want.double()).abs().max() <= tol, mask
