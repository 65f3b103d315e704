"""Appends that begin and end inside 64-token tiles: the tile kernels write the rows they are given and nothing else.

A cache filled by pieces that start at odd slots must hold, bit for bit, what one filled a row at a time holds (the row
kernels), rows before and behind a piece included.
"""
import numpy as np
import pytest
import torch

import kvhip
from tests.util import randn

pytestmark = pytest.mark.gpu

# a first piece inside one tile, one that ends on a tile's edge, one of a whole tile at an odd slot, one that begins on an
# edge and crosses a 256-row page; pieces on both sides of the counts from which the tile kernels take over (quantized 3 to 12
# by size and rotation, full precision 16 and 512 KB of rows); at the end one whose two halves lie below them, two rows
# either side of a tile's edge; 'trim' leaves older rows behind the end
PIECES = [(9, 0), (55, 0), (5, 0), (64, 3), (9, 0), (63, 20), (10, 0), (130, 1), (61, 0), (13, 0), (14, 0), (16, 0), (17, 0), (22, 0), (19, 0), (20, 0), (2, 0), (5, 0), (4, 0)]


def _fill(cache, k, v, pieces, rope, quantized, one_by_one):
    at, ran = 0, set()
    for n, trim in pieces:
        for lo in range(at, at + n) if one_by_one else [at]:
            kk, vv = (x[:, :, lo:lo + (1 if one_by_one else n)].contiguous() for x in (k, v))
            if rope is not None:
                cache.update_rope(rope, kk, vv)
            elif quantized:
                cache.update_quantized(kk, vv, fetch=False)
            else:
                cache.update(kk, vv, fetch=False)
            ran.add(kvhip.load().kvhip_last_append_kernel())
        at += n
        cache.trim(trim)
    assert ran == ({0} if one_by_one else {0, 1})
    return cache.state


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bits,dk,dv,gs", [(0, 64, 64, 0), (0, 96, 96, 0), (0, 128, 128, 0), (0, 256, 256, 0), (0, 192, 128, 0),
                                           (4, 64, 64, 64), (8, 96, 96, 32), (4, 128, 128, 64), (2, 128, 128, 128), (3, 64, 64, 32),
                                           (5, 96, 96, 32), (6, 256, 256, 64), (4, 192, 128, 64), (8, 192, 128, 32)])
@pytest.mark.parametrize("rotary", [None, False, True])
def test_pieces_at_odd_slots_equal_single_rows(dtype, bits, dk, dv, gs, rotary):
    rng = np.random.default_rng(bits * 1000 + dk)
    rows = sum(n for n, _ in PIECES)
    pairs = (2, 3) if bits else (8, 8)
    _, k = randn(rng, (*pairs, rows, dk), dtype, 2.0)
    _, v = randn(rng, (*pairs, rows, dv), dtype)
    rope = None if rotary is None else kvhip.RoPE(dk, traditional=rotary, base=500000.0)
    a, b = (_fill(kvhip.QuantizedKVCache(gs, bits) if bits else kvhip.KVCacheSimple(), k, v, PIECES, rope, bits != 0, one)
            for one in (False, True))
    for x, y in zip(a, b):
        assert x.shape == y.shape and torch.equal(x.view(torch.int16), y.view(torch.int16))
