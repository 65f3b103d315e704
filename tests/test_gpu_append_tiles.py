"""Full-precision appends of a tile and more at the head sizes and types that share the tile kernel: pieces that begin and
end inside tiles, and rows whose memory begins at an odd element, give the bits that single rows give (moved, not computed;
the rotation is the same elementwise function of position and pair)."""
import pytest
import torch

import kvhip

pytestmark = pytest.mark.gpu

PIECES = [64, 5, 65, 130, 64, 200]  # a whole tile, then starts and ends inside tiles and pages
BATCH, HEADS = 4, 8  # (pieces of a tile and more are past the 512 KB of rows from which tiles take them, at every size)


def _shifted(x):
    """`x` in memory that begins one element behind a 16-byte boundary."""
    flat = torch.empty(x.numel() + 1, dtype=x.dtype, device="cuda")[1:].view(x.shape)
    return flat.copy_(x)


@pytest.mark.parametrize("dtype,D", [(torch.float16, 80), (torch.bfloat16, 80), (torch.float16, 512), (torch.bfloat16, 512),
                                     (torch.float32, 64), (torch.float32, 96), (torch.float32, 128), (torch.float32, 256)])
@pytest.mark.parametrize("rotary", ["none", "halves", "pairs", "part", "odd", "queries"])
def test_tiles_equal_single_rows(dtype, D, rotary):
    gen = torch.Generator(device="cuda").manual_seed(D)
    rope = {"none": None, "halves": kvhip.RoPE(D, base=5e5), "pairs": kvhip.RoPE(D, traditional=True), "part": kvhip.RoPE(D // 2),
            "odd": kvhip.RoPE(20), "queries": kvhip.RoPE(D)}[rotary]
    tiled, single = kvhip.KVCacheSimple(), kvhip.KVCacheSimple()
    for piece, n in enumerate(PIECES):
        q, k, v = (torch.randn(BATCH, h, n, D, generator=gen, device="cuda").to(dtype) for h in (2 * HEADS, HEADS, HEADS))
        kk, vv = (k, v) if piece % 2 == 0 else (_shifted(k), _shifted(v))
        if rotary == "queries":
            tiled.update_attend_rope(rope, q, kk, vv, D ** -0.5)
        elif rope is not None:
            tiled.update_rope(rope, kk, vv)
        else:
            tiled.update(kk, vv, fetch=False)
        assert kvhip.load().kvhip_last_append_kernel() == (n >= 64)
        for i in range(n):
            row = k[:, :, i:i + 1].contiguous(), v[:, :, i:i + 1].contiguous()
            if rope is not None:
                single.update_rope(rope, *row)
            else:
                single.update(*row, fetch=False)
        assert kvhip.load().kvhip_last_append_kernel() == 0
    for a, b in zip(tiled.state, single.state):
        assert a.shape == b.shape and torch.equal(a, b)


@pytest.mark.parametrize("bits,gs,dtype,Dk,Dv", [(4, 64, torch.float16, 128, 128), (8, 32, torch.bfloat16, 64, 64), (4, 128, torch.float16, 256, 256),
                                                 (3, 32, torch.float16, 96, 96), (4, 64, torch.bfloat16, 192, 128), (0, 0, torch.float16, 128, 128),
                                                 (0, 0, torch.bfloat16, 64, 64), (0, 0, torch.float32, 128, 128)])
@pytest.mark.parametrize("n", [2, 3, 4, 5, 12, 15, 16, 33, 63])
def test_few_rows_equal_single_rows(bits, gs, dtype, Dk, Dv, n):
    """Either side of the row counts from which tiles take over, in many (batch, head) pairs, from slots that leave the
    rows in one tile, in two, and in two pages."""
    gen = torch.Generator(device="cuda").manual_seed(n)
    for rope in (None, kvhip.RoPE(Dk)):
        for at in (3, 256 - n // 2):
            caches = [kvhip.QuantizedKVCache(gs, bits) if bits else kvhip.KVCacheSimple() for _ in range(2)]
            k0, v0, k, v = (torch.randn(5, 16, m, d, generator=gen, device="cuda").to(dtype) for m in (at, n) for d in (Dk, Dv))
            for c in caches:
                c._update(k0, v0)
            rows = [(k, v)], [(k[:, :, i:i + 1].contiguous(), v[:, :, i:i + 1].contiguous()) for i in range(n)]
            for c, parts in zip(caches, rows):
                for part in parts:
                    c.update_rope(rope, *part) if rope is not None else c._update(*part)
            for a, b in zip(caches[0].state, caches[1].state):
                assert a.shape == b.shape and torch.equal(a, b)
