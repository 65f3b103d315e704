"""Array masks of every element type in the float32 and head-size-512 attention kernels (family 5), whose instances for
them read whole tiles' elements at once: tiles that end inside, rows of odd length, rings whose rows lie in pieces, masks
with and without batch and head extents.  Against the plain kernel, which reads element by element."""
import pytest
import torch

import kvhip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,D", [(torch.float16, 512), (torch.bfloat16, 512), (torch.float32, 64), (torch.float32, 96), (torch.float32, 256)])
@pytest.mark.parametrize("mask_dtype", [torch.bool, torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,n,ring", [(33, 1, False), (64, 2, False), (1001, 3, False), (1030, 40, False), (300, 1, True), (777, 9, True)])
def test_against_the_plain_kernel(dtype, D, mask_dtype, T, n, ring):
    B, Hkv, r = 2, 2, 4
    gen = torch.Generator(device="cuda").manual_seed(T + n + D)

    def rand(*shape):
        return torch.randn(*shape, generator=gen, device="cuda")

    c = kvhip.RotatingKVCache(T, keep=4) if ring else kvhip.KVCacheSimple()
    c.update(rand(B, Hkv, T, D).to(dtype), rand(B, Hkv, T, D).to(dtype), fetch=False)
    for _ in range(21 if ring else 0):  # (the ring wraps: its rows are in several pieces)
        c.update(rand(B, Hkv, 1, D).to(dtype), rand(B, Hkv, 1, D).to(dtype), fetch=False)
    if ring and n > 1:
        c.update(rand(B, Hkv, n, D).to(dtype), rand(B, Hkv, n, D).to(dtype), fetch=False)
    q, keys = rand(B, Hkv * r, n, D).to(dtype), c.presented_length
    lib = kvhip.load()
    for shape in ((n, keys), (B, 1, n, keys), (B, Hkv * r, n, keys)):
        keep = rand(*shape) < 0.5
        keep[..., :keys // 2] &= rand(*shape[:-1], 1) > 0  # (half the rows see nothing of the first half)
        keep[..., -1] = True
        array = keep if mask_dtype == torch.bool else torch.where(keep, rand(*shape), float("-inf")).to(mask_dtype)
        mask = kvhip.MaskMode.from_array(array)
        got = c.attend(q, D ** -0.5, mask)
        assert lib.kvhip_last_attend_kernel() == 5
        try:
            lib.kvhip_set_kernel_policy(1)
            want = c.attend(q, D ** -0.5, mask)
        finally:
            lib.kvhip_set_kernel_policy(0)
        # one rounding of the output on either side, of values up to 4 (float32: sums of 512 products, T probabilities)
        tol = {torch.float16: 2.0 ** -9, torch.bfloat16: 2.0 ** -6, torch.float32: 1e-5}[dtype]
        assert (got.double() - want.double()).abs().max() <= tol, shape
