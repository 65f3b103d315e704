"""Prompt chunks of 256 query rows per kv head and more over full-precision caches of head sizes up to 128 (128 rows a
workgroup, 32 a wavefront): query rows that end inside a wavefront, odd and even numbers of 32-key blocks, blocks that end
inside, key ranges in parts, every mask, rings whose rows lie in pieces.  Against the plain kernel, over the same cache."""
import pytest
import torch

import kvhip

pytestmark = pytest.mark.gpu


def _compare(c, q, scale, mask):
    lib = kvhip.load()
    got = c.attend(q, scale, mask)
    assert lib.kvhip_last_attend_kernel() == 3
    try:
        lib.kvhip_set_kernel_policy(1)
        want = c.attend(q, scale, mask)
    finally:
        lib.kvhip_set_kernel_policy(0)
    # Of a row, in 2-norms: the probabilities (float16: their sum too) and either output are rounded once, each by at most eps
    # of an element.
    eps = 2.0 ** -11 if q.dtype == torch.float16 else 2.0 ** -8
    got, want = got.double(), want.double()
    worst = ((got - want).norm(dim=-1) / want.norm(dim=-1).clamp_min(1e-30)).max().item()
    assert worst <= 4 * eps, worst / eps


# (kv heads, query heads to one, new rows): 256 rows; ends inside a wavefront; rows of several heads in a workgroup; a
# grid that fills the chip without parts.  The others' key ranges are in parts: behind 300 rows in two that a workgroup takes at
# once, behind 700 in three, behind 1601 in seven, or three times two (the second set), behind 2300 in nine, or five times two.
ROWS = [(2, 1, 256), (2, 4, 75), (1, 2, 257), (8, 8, 520)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [64, 80, 96, 128])
@pytest.mark.parametrize("before", [0, 1, 31, 33, 300, 700, 1601, 2300])
@pytest.mark.parametrize("hkv,r,n", ROWS)
def test_masks_and_edges(dtype, D, before, hkv, r, n):
    B, T = 2, before + n
    gen = torch.Generator(device="cuda").manual_seed(T + n + D)
    rand = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")
    c = kvhip.KVCacheSimple()
    # (half of the pairs' keys with a spread of two, half of 0.1: of N keys that weigh nearly the same, one more or less moves a
    # row by its N^-1/2-th part, five bfloat16 roundings of 2500)
    spread = torch.where(torch.arange(B * hkv, device="cuda") % 2 == 0, 2., .1).view(B, hkv, 1, 1)
    c.update((rand(B, hkv, T, D) * spread).to(dtype), rand(B, hkv, T, D).to(dtype), fetch=False)
    q, scale = rand(B, hkv * r, n, D).to(dtype), D ** -0.5
    W = kvhip.MaskMode.window_mask
    ends = torch.tensor([T, max(1, T - 45)], dtype=torch.int32)
    pads = torch.tensor([0, min(before, 40)], dtype=torch.int32)
    masks = [kvhip.MaskMode.none(), kvhip.MaskMode.causal(), W(before, 100), W(before, 0, lengths=ends), W(before, 0, left_pad=pads)]
    if hkv < 8:  # (the plain kernel is slow)
        keep = rand(B, 1, n, T) < 0.5
        keep[..., 0] = True
        masks += [kvhip.MaskMode.from_array(keep), kvhip.MaskMode.from_array(torch.where(keep, rand(n, T), float("-inf")).to(dtype))]
    elif before not in (33, 300, 1601, 2300):
        masks = masks[1:2]
    for mask in masks:
        _compare(c, q, scale, mask)
    _compare(c, q, -scale, kvhip.MaskMode.causal())


@pytest.mark.parametrize("dtype,D", [(torch.float16, 128), (torch.bfloat16, 128), (torch.bfloat16, 64), (torch.float16, 96)])
@pytest.mark.parametrize("window,n", [(300, 128), (512, 131), (700, 256)])
def test_rings(dtype, D, window, n):
    B, hkv, r = 2, 2, 4
    gen = torch.Generator(device="cuda").manual_seed(window + D)
    rand = lambda h, m: torch.randn(B, h, m, D, generator=gen, device="cuda").to(dtype)
    c = kvhip.RotatingKVCache(window, keep=4)
    for _ in range(9):
        mask = c.make_mask(n, window, False)
        c.update(rand(hkv, n), rand(hkv, n), fetch=False)
        _compare(c, rand(hkv * r, n), D ** -0.5, mask)
    for _ in range(21):  # (single tokens: the ring's rows are in pieces)
        c.update(rand(hkv, 1), rand(hkv, 1), fetch=False)
    mask = c.make_mask(n, window, False)
    c.update(rand(hkv, n), rand(hkv, n), fetch=False)
    _compare(c, rand(hkv * r, n), D ** -0.5, mask)
    _compare(c, rand(hkv * r, n), D ** -0.5, kvhip.MaskMode.from_array(mask.array))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [64, 80, 96, 128])
@pytest.mark.parametrize("hkv,r,n,before", [(8, 8, 67, 0), (2, 4, 75, 450), (2, 4, 75, 1601)])  # whole; in two halves; in parts
def test_an_output_that_starts_anywhere(dtype, D, hkv, r, n, before):
    """The caller's array is aligned as its elements are: the same rows as into one aligned to 256 bytes, and nothing beside them."""
    B, T = 2, before + n
    gen = torch.Generator(device="cuda").manual_seed(T + D)
    rand = lambda h, m: torch.randn(B, h, m, D, generator=gen, device="cuda").to(dtype)
    c = kvhip.KVCacheSimple()
    c.update(rand(hkv, T), rand(hkv, T), fetch=False)
    q, mask = rand(hkv * r, n), kvhip.MaskMode.causal()
    want = c.attend(q, D ** -0.5, mask)
    assert kvhip.load().kvhip_last_attend_kernel() == 3
    for ahead in (1, 3, 4):
        room = torch.full((want.numel() + 16,), 7., dtype=dtype, device="cuda")
        c.attend(q, D ** -0.5, mask, out=room[ahead:ahead + want.numel()].view_as(want))
        assert torch.equal(room[ahead:ahead + want.numel()].view_as(want), want)
        assert (room[:ahead] == 7).all() and (room[ahead + want.numel():] == 7).all()
