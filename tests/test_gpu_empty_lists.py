"""Attention with a tail where a tile pair lists no block at all: nothing of the exact part
then runs between building the lists and building the tails (csrc/attn.hip). Persistent
grid and one workgroup per pair, block means and rescue tokens with and without remainder,
beside heads that list their own block, against the tail alone in float64."""

import math

import pytest
import torch

from exp3_amd import _lib, kernels, synthetic
from exp3_amd.upstream import flashprefill_native_forward as upstream

pytestmark = pytest.mark.gpu

LENGTH, HEADS, KV, DIM = 9100, 28, 4, 128     # 72 blocks: two tail tiles of 64 entries


def _tail(kind, q, k, v, desc, choice):
    """(output, LSE) of the tail entries of every history block, [S, Hq, D] / [S, Hq]."""
    blocks = desc.mean_k.shape[1]
    group = HEADS // KV
    tile = torch.arange(LENGTH, device="cuda") // 128
    out = torch.zeros(LENGTH, HEADS, DIM, dtype=torch.float64, device="cuda")
    lse = torch.full((LENGTH, HEADS), -math.inf, dtype=torch.float64, device="cuda")
    for t in range(1, blocks):
        rows = tile == t
        for h in range(HEADS):
            g = h // group
            mk, mv = (x[0, :t, g].double() for x in (desc.mean_k, desc.mean_v))
            if kind == "mean":
                keys, values, weight = mk, mv, torch.full((t,), 128.0, device="cuda")
            else:
                token = torch.arange(t, device="cuda") * 128 + choice[0, t, :t, h].long()
                keys, values = (x[0, token, g].double() for x in (k, v))
                weight = torch.ones(t, device="cuda")
                if kind == "rescue2":
                    keys, values = (torch.cat((x, (m * 128 - x) / 127))
                                    for x, m in ((keys, mk), (values, mv)))
                    weight = torch.cat((weight, weight * 127))
            logits = q[0, rows, h].double() @ keys.T * DIM ** -0.5 + weight.double().log()
            out[rows, h] = torch.softmax(logits, -1) @ values
            lse[rows, h] = torch.logsumexp(logits, -1)
    return out, lse


@pytest.mark.parametrize("persistent", (True, False))
@pytest.mark.parametrize("kind", ("mean", "rescue1", "rescue2"))
def test_pairs_without_entries(gpu, kind, persistent):
    assert _lib.load().spx_attention_queue_ints(1, LENGTH, HEADS, KV, DIM) > 0    # tile pairs
    q, k, v, _ = synthetic.make_inputs(LENGTH, seed=61, q_heads=HEADS, kv_heads=KV, device="cuda")
    blocks = (LENGTH + 127) // 128
    desc = kernels.block_descriptors(k, v)
    tiles = upstream.attention_tiles(k, v)
    choice = kernels.rescue_choice(q, tiles[0])
    # entries past the count are never read: ids of no block; every fourth head lists its tile
    idx = torch.full((1, blocks, blocks, HEADS), 1 << 40, dtype=torch.int64, device="cuda")
    idx[:, :, 0, ::4] = torch.arange(blocks, device="cuda")[None, :, None]
    cnt = torch.zeros(1, blocks, HEADS, dtype=torch.int32, device="cuda")
    cnt[:, :, ::4] = 1
    out = torch.full(q.shape, float("nan"), dtype=q.dtype, device="cuda")
    lse = torch.full(q.shape[:3], float("nan"), device="cuda")
    queue = (torch.zeros(_lib.WORK_QUEUE_INTS, dtype=torch.int32, device="cuda")
             if persistent else None)
    head = (_lib.ptr(q), _lib.strides(q), _lib.ptr(tiles[0]), _lib.ptr(tiles[1]), _lib.ptr(idx),
            _lib.strides(idx), _lib.ptr(cnt), _lib.strides(cnt))
    end = (1, LENGTH, HEADS, KV, DIM, 128, DIM ** -0.5, _lib.ptr(out), _lib.strides(out),
           _lib.ptr(lse), _lib.strides(lse), _lib.ptr(queue), _lib.stream(q.device))
    if kind == "mean":
        _lib.call("spx_sparse_attention_mean", *head, _lib.ptr(desc.mean_k), _lib.ptr(desc.mean_v),
                  _lib.ptr(desc.counts), *end)
    else:
        _lib.call("spx_sparse_attention_rescue", *head, _lib.ptr(choice), _lib.ptr(v),
                  _lib.strides(v), _lib.ptr(desc.mean_k), _lib.ptr(desc.mean_v),
                  int(kind == "rescue2"), *end)
    torch.cuda.synchronize()
    assert not torch.isnan(out).any() and not torch.isnan(lse).any()
    want, want_lse = _tail(kind, q, k, v, desc, choice)
    empty = torch.arange(HEADS, device="cuda") % 4 != 0
    got, want = out[0][:, empty].double(), want[:, empty]
    # P and the entries' values round to bf16, half a step (2^-9) each of every entry's
    # share, at most 2^-8 max |v| together; keys as bf16 hi + lo move a logit by 2^-17 of it
    # (under 2^-12 of a weight); the output rounds by half a step of itself
    peak = v.double().abs().max()
    assert ((got - want).abs() <= 1.1 * 2 ** -8 * peak + 2 ** -8 * want.abs()).all()
    got_lse, want_lse = lse[0][:, empty].double(), want_lse[:, empty]
    assert torch.equal(torch.isinf(got_lse), torch.isinf(want_lse)) and not got[:128].any()
    # fp32 logits and sums, and the keys' 2^-17
    assert (got_lse - want_lse)[128:].abs().max() <= 1e-3
