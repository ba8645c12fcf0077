"""The longest union of two tiles' lists (csrc/attn.hip): 1024 blocks, every tile listing one
block 1024 times, adjacent tiles different ones and none its own, so that the pair's list
has 2048 entries. Attending a block n times is attending it once with n times the weight:
the output of one mention, the LSE plus ln n. One block's keys lie far closer to the
queries, so a tile that met the other tile's entries would follow them."""

import math

import pytest
import torch

from exp3_amd import _lib
from exp3_amd.upstream import flashprefill_native_forward as upstream

pytestmark = pytest.mark.gpu

LENGTH, BLOCKS, DIM = 131000, 1024, 128


@pytest.mark.parametrize("persistent", (True, False))
def test_disjoint_full_lists(gpu, persistent):
    gen = torch.Generator("cuda").manual_seed(71)
    q, k, v = (torch.randn(1, LENGTH, 1, DIM, generator=gen, device="cuda") for _ in range(3))
    q[..., 0] = 16.0
    k[:, :128, :, 0] = 16.0
    q, k, v = (x.to(torch.bfloat16) for x in (q, k, v))
    q = q.expand(1, LENGTH, 2, DIM).contiguous()
    tiles = upstream.attention_tiles(k, v)
    odd = torch.arange(BLOCKS, device="cuda") % 2        # the first tile of a pair: block 0
    idx = (1 - odd)[None, :, None, None].expand(1, BLOCKS, BLOCKS, 2).contiguous()
    cnt = torch.full((1, BLOCKS, 2), BLOCKS, dtype=torch.int32, device="cuda")
    out = torch.full(q.shape, float("nan"), dtype=q.dtype, device="cuda")
    lse = torch.full(q.shape[:3], float("nan"), device="cuda")
    queue = (torch.zeros(_lib.WORK_QUEUE_INTS, dtype=torch.int32, device="cuda")
             if persistent else None)
    _lib.call("spx_exact_attention", _lib.ptr(q), _lib.strides(q), _lib.ptr(tiles[0]),
              _lib.ptr(tiles[1]), _lib.ptr(idx), _lib.strides(idx), _lib.ptr(cnt),
              _lib.strides(cnt), 1, LENGTH, 2, 1, DIM, 128, DIM ** -0.5, _lib.ptr(out),
              _lib.strides(out), _lib.ptr(lse), _lib.strides(lse), _lib.ptr(queue),
              _lib.stream(q.device))
    torch.cuda.synchronize()
    peak = v[0, :256].double().abs().max()
    row_odd = odd[torch.arange(LENGTH, device="cuda") // 128].bool()
    for block, rows in ((0, row_odd), (1, ~row_odd)):
        keys, values = (x[0, block * 128:block * 128 + 128, 0].double() for x in (k, v))
        logits = q[0, rows, 0].double() @ keys.T * DIM ** -0.5
        want = torch.softmax(logits, -1) @ values
        want_lse = torch.logsumexp(logits, -1) + math.log(BLOCKS)
        for h in range(2):
            # P rounds to bf16 (half a step, 2^-9 of every share), the output by half a step
            # of itself; fp32 sums of 2^17 equal rounds leave at most 1024 x 2^-24 = 2^-14
            assert ((out[0, rows, h].double() - want).abs()
                    <= (2 ** -9 + 2 ** -13) * peak + 2 ** -8 * want.abs()).all()
            assert (lse[0, rows, h].double() - want_lse).abs().max() <= 1e-3
