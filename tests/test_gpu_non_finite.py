"""Infinite and NaN elements in the float32 and head-size-512 attention kernels (family 5): an infinite value reaches its
output column with its sign, a key whose score is NaN weighs nothing, and tiles that no row sees under a boolean array
mask are not read.  The other columns against float64 at the dtype's own rounding."""
import pytest
import torch

import kvhip

pytestmark = pytest.mark.gpu

INF, NAN = float("inf"), float("nan")
KINDS = [(torch.float16, 512), (torch.bfloat16, 512), (torch.float32, 64), (torch.float32, 128), (torch.float32, 256)]
# one rounding of the output, of values up to about 5 (float32: sums of D products and T probabilities)
TOL = {torch.float16: 2.0 ** -8, torch.bfloat16: 2.0 ** -5, torch.float32: 1e-5}


def tensors(dtype, D, T, n, seed=1):
    gen = torch.Generator(device="cuda").manual_seed(seed + T + n + D)
    return [torch.randn(2, h, m, D, generator=gen, device="cuda").to(dtype) for h, m in ((8, n), (2, T), (2, T))]


def attend(q, k, v, mask, ring=False):
    c = kvhip.RotatingKVCache(k.shape[2], keep=4) if ring else kvhip.KVCacheSimple()
    c.update(k, v, fetch=False)
    out = c.attend(q, q.shape[3] ** -0.5, mask)
    assert kvhip.load().kvhip_last_attend_kernel() == 5
    return out.double()


def exact(q, k, v, keep, add=None):
    """float64, infinite values left out (`keep`: keys that weigh something)."""
    k, v = (torch.nan_to_num(x.double(), 0., 0., 0.).repeat_interleave(4, 1) for x in (k, v))
    s = torch.matmul(torch.nan_to_num(q.double()), k.transpose(2, 3).contiguous()) * q.shape[3] ** -0.5
    s = s if add is None else s + add.double()
    p = torch.softmax(s.masked_fill(~keep, -INF), -1)
    return torch.matmul(torch.nan_to_num(p), v)


@pytest.mark.parametrize("dtype,D", KINDS)
@pytest.mark.parametrize("T,n", [(40, 1), (40, 9), (3000, 1), (3000, 9)])
def test_infinite_values_reach_the_output(dtype, D, T, n):
    q, k, v = tensors(dtype, D, T, n)
    add = torch.zeros(1, T, device="cuda")
    add[0, 9] = -60.  # weights down to 2^-100: nothing beside the others, but not zero
    v[:, :, 7, 3], v[:, :, 7, 6], v[:, :, 9, 5], v[:, :, 9, D - 1] = INF, -INF, INF, -INF
    out = attend(q, k, v, kvhip.MaskMode.from_array(add.expand(n, T)))
    for col, want in ((3, INF), (6, -INF), (5, INF), (D - 1, -INF)):
        assert (out[..., col] == want).all(), col
        out[..., col] = 0.
    ref = exact(q, k, v, torch.ones(1, T, dtype=torch.bool, device="cuda"), add)
    ref[..., [3, 5, 6, D - 1]] = 0.
    assert (out - ref).abs().max() <= TOL[dtype]


@pytest.mark.parametrize("dtype,D", KINDS)
@pytest.mark.parametrize("T,n", [(40, 1), (40, 9), (3000, 1), (3000, 9)])
def test_keys_whose_score_is_nan_weigh_nothing(dtype, D, T, n):
    q, k, v = tensors(dtype, D, T, n)
    k[0, :, 7, 3] = NAN
    k[0, 1, T - 2, D - 1] = NAN
    q[1, 5, 0, 2] = NAN  # every score of one row: zeros, as where every key is excluded
    out = attend(q, k, v, kvhip.MaskMode.none())
    keep = torch.ones(2, 8, n, T, dtype=torch.bool, device="cuda")
    keep[0, :, :, 7] = False
    keep[0, 4:, :, T - 2] = False
    keep[1, 5, 0] = False
    assert (out - exact(q, k, v, keep)).abs().max() <= TOL[dtype]
    assert (out[1, 5, 0] == 0).all()


@pytest.mark.parametrize("dtype,D", KINDS)
@pytest.mark.parametrize("T,n,seen", [(300, 1, 70), (3000, 1, 6), (3000, 9, 200), (700, 70, 64), (5000, 1, 4000)])
@pytest.mark.parametrize("ring", [False, True])
def test_tiles_nobody_sees_are_not_read(dtype, D, T, n, seen, ring):
    """A boolean window over the last keys: values in front of the first tile with a visible key do not matter."""
    q, k, v = tensors(dtype, D, T, n)
    i, j = torch.arange(n, device="cuda")[:, None] + T - n, torch.arange(T, device="cuda")[None]
    keep = (j <= i) & (j > i - seen)
    hidden = (T - n - seen + 1) // 64 * 64  # whole tiles of 64 in front of every row's window
    v[:, :, :hidden] = NAN
    out = attend(q, k, v, kvhip.MaskMode.from_array(keep), ring)
    assert (out - exact(q, k, v, keep)).abs().max() <= TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("Dk,Dv", [(512, 512), (576, 512), (320, 64), (320, 96), (1024, 128), (320, 256)])
@pytest.mark.parametrize("n", [1, 5, 40])
def test_infinite_values_of_a_range_with_a_denormal_weight_reach_the_output(dtype, Dk, Dv, n):
    """The merge of key ranges: one range's maximum lies 90 above another's, which leaves that a weight of 2^-130 -- not
    zero in float32, so its infinite value stays infinite."""
    T = 2048
    q, k, v = torch.zeros(1, 2, n, Dk), torch.zeros(1, 1, T, Dk), torch.ones(1, 1, T, Dv)
    q[..., 0] = 1.
    k[0, 0, :, 0] = -90.
    k[0, 0, 5, 0] = 0.
    v[0, 0, 1500, 3], v[0, 0, 1500, Dv - 1] = INF, -INF
    c = kvhip.KVCacheSimple()
    c.update(k.to(dtype).cuda(), v.to(dtype).cuda(), fetch=False)
    out = c.attend(q.to(dtype).cuda(), 1.0, kvhip.MaskMode.none())
    assert kvhip.load().kvhip_last_attend_kernel() == 5
    assert (out[..., 3] == INF).all() and (out[..., Dv - 1] == -INF).all()
    out[..., 3] = out[..., Dv - 1] = 1.
    assert (out.double() - 1.).abs().max() <= TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,T", [(1, 40), (1, 64), (1, 3000), (70, 300)])  # (the new row in its part's only tile, or in the tenth)
@pytest.mark.parametrize("rotary", [False, True])
def test_a_step_that_reads_its_own_row_again(dtype, B, T, rotary):
    """One token at head size 512 whose kernel writes the new row: an infinite value, in the new row or behind it, sends the
    workgroup through its tiles once more, and there the row is read from the page.  Against separate calls."""
    D = 512
    gen = torch.Generator(device="cuda").manual_seed(T)
    rand = lambda h, n: torch.randn(B, h, n, D, generator=gen, device="cuda").to(dtype)
    rope = kvhip.RoPE(D, base=1e4) if rotary else None
    k, v = rand(4, T), rand(4, T)
    v[:, :, T - 1, 3] = INF
    one, two = kvhip.KVCacheSimple(), kvhip.KVCacheSimple()
    for c in (one, two):
        c.update(k, v, fetch=False)
    for i in range(2):
        q, nk, nv = rand(8, 1), rand(4, 1), rand(4, 1)
        nv[..., 5], nv[..., D - 1] = -INF, INF
        if rotary:
            got = kvhip.attention_with_rope_and_cache_update(rope, q, nk, nv, one, D ** -0.5)
            q = kvhip.apply_rotary_position(rope, q, two.rope_offset)
            two.update_rope(rope, nk, nv)
        else:
            got = kvhip.attention_with_cache_update(q, nk, nv, one, D ** -0.5)
            two._update(nk, nv)
        assert kvhip.load().kvhip_last_attend_kernel() == 5
        assert (got[..., 3] == INF).all() and (got[..., 5] == -INF).all() and (got[..., D - 1] == INF).all()
        assert torch.equal(got, two.attend(q, D ** -0.5))
    for a, b in zip(one.state, two.state):
        assert torch.equal(a, b)
