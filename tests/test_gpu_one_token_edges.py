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
@pytest.mark.parametrize("spread", [1., .1])
def test_against_the_plain_kernel(D, dtype, B, Hkv, T, spread):
    """`spread` of the keys: at 0.1 all weigh nearly the same, and one of N more or less moves an output row by its
    N^-1/2-th part (0.015 of 4200), twice the bfloat16 bound below."""
    gen = torch.Generator(device="cuda").manual_seed(T + D)
    rand = lambda h, n, by=1.: (torch.randn(B, h, n, D, generator=gen, device="cuda") * by).to(dtype)
    c = kvhip.KVCacheSimple()
    c._update(rand(Hkv, T, spread), rand(Hkv, T))
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
        # Of a row, in 2-norms: the probabilities and either output are rounded once, by up to eps of an element and 0.4 eps
        # in the mean (float32: sums of D products and of T probabilities).
        eps = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 5e-6}[dtype]
        got, want = got.double(), want.double()
        assert ((got - want).norm(dim=-1) <= 2 * eps * want.norm(dim=-1)).all(), mask
