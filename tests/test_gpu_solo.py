"""The single-tile attention kernel (a launch without work queue whose shape
spx_attention_queue_ints answers with 0) against the tile-pair kernel (the same call with a
queue): the same bits on ascending lists, at the edges of its rule (12 blocks; pair items
up to 4/3 of the CUs) and of its loops (one block, a lone first tile, partial last blocks,
64-key halves, tails of more than one 64-entry tile; lists and tails past one, two and
more positions per thread), exact, with block means and with rescue tokens, LSE included; and unordered, repeated and future entries and empty rows
within rounding of it (the two add blocks in different orders there)."""

import pytest
import torch

from exp3_amd import _lib, kernels, synthetic
from exp3_amd.upstream import flashprefill_native_forward as upstream

pytestmark = pytest.mark.gpu


def _both(kind, q, k, v, idx, cnt, descriptors, choice):
    batch, seq, q_heads, dim = q.shape
    tiles = upstream.attention_tiles(k, v)
    results = []
    for queue in (None, torch.zeros(_lib.WORK_QUEUE_INTS, dtype=torch.int32, device="cuda")):
        out = torch.full(q.shape, float("nan"), dtype=q.dtype, device="cuda")
        lse = torch.full(q.shape[:3], float("nan"), device="cuda")
        head = (_lib.ptr(q), _lib.strides(q), _lib.ptr(tiles[0]), _lib.ptr(tiles[1]), _lib.ptr(idx),
                _lib.strides(idx), _lib.ptr(cnt), _lib.strides(cnt))
        tail = (batch, seq, q_heads, k.shape[2], dim, 128, dim ** -0.5, _lib.ptr(out),
                _lib.strides(out), _lib.ptr(lse), _lib.strides(lse), _lib.ptr(queue),
                _lib.stream(q.device))
        d = descriptors
        if kind == "exact":
            _lib.call("spx_exact_attention", *head, *tail)
        elif kind == "mean":
            _lib.call("spx_sparse_attention_mean", *head, _lib.ptr(d.mean_k), _lib.ptr(d.mean_v),
                      _lib.ptr(d.counts), *tail)
        else:
            _lib.call("spx_sparse_attention_rescue", *head, _lib.ptr(choice), _lib.ptr(v),
                      _lib.strides(v), _lib.ptr(d.mean_k), _lib.ptr(d.mean_v),
                      int(kind == "rescue2"), *tail)
        results.append((out, lse))
    torch.cuda.synchronize()
    return results


def _case(batch, length, q_heads, kv_heads, seed):
    q, k, v, _ = synthetic.make_inputs(length, seed=seed, q_heads=q_heads, kv_heads=kv_heads,
                                       batch=batch, device="cuda")
    q, k = ((x.float() * 3).to(torch.bfloat16) for x in (q, k))
    blocks = (length + 127) // 128
    lib = _lib.load()
    assert lib.spx_attention_queue_ints(batch, length, q_heads, kv_heads, 128) == 0
    return (q, k, v, blocks, kernels.block_descriptors(k, v),
            kernels.rescue_choice(q, upstream.attention_tiles(k, v)[0]))


@pytest.mark.parametrize("kind", ("exact", "mean", "rescue1", "rescue2"))
@pytest.mark.parametrize("batch,length,q_heads,kv_heads",
                         ((1, 1, 2, 1), (2, 127, 4, 2), (1, 128, 28, 4), (1, 129, 6, 3),
                          (3, 1000, 12, 4), (1, 1536, 28, 4), (1, 3072, 28, 4),
                          (1, 16300, 4, 1)))
def test_same_bits_as_tile_pairs(gpu, kind, batch, length, q_heads, kv_heads):
    q, k, v, blocks, d, choice = _case(batch, length, q_heads, kv_heads, 50 + length)
    gen = torch.Generator("cuda").manual_seed(length)
    keep = torch.rand(batch, blocks, blocks, q_heads, generator=gen, device="cuda") < 0.3
    ids = torch.arange(blocks, device="cuda")
    causal = (ids[None, :] <= ids[:, None])[None, :, :, None]
    keep = (keep | (ids[None, :] == ids[:, None])[None, :, :, None]) & causal
    idx, cnt = kernels.indices_from_mask(keep)
    solo, pair = _both(kind, q, k, v, idx, cnt, d, choice)
    assert not torch.isnan(solo[0]).any()
    assert torch.equal(solo[0], pair[0]) and torch.equal(solo[1], pair[1])
    if kind == "exact":          # every causal block
        solo, pair = _both(kind, q, k, v, None, None, d, choice)
        assert torch.equal(solo[0], pair[0]) and torch.equal(solo[1], pair[1])


@pytest.mark.parametrize("kind", ("exact", "mean", "rescue2"))
def test_lists_in_any_order(gpu, kind):
    q, k, v, blocks, d, choice = _case(2, 1100, 8, 2, 7)
    gen = torch.Generator("cuda").manual_seed(3)
    idx = torch.randint(-2, blocks + 2, (2, blocks, blocks, 8), generator=gen, device="cuda")
    cnt = torch.randint(0, blocks + 1, (2, blocks, 8), generator=gen, device="cuda",
                        dtype=torch.int32)
    cnt[0, 2] = 0
    solo, pair = _both(kind, q, k, v, idx, cnt, d, choice)
    assert torch.equal(torch.isinf(solo[1]), torch.isinf(pair[1]))
    # each side rounds P to bf16 (half a step: 2^-8 relative) at its own running max: the
    # weights sum to 1, so the two sums differ by at most 2 * 2^-8 of the largest |v|; then
    # two output roundings of 2^-8 each
    err = (solo[0].float() - pair[0].float()).abs() - 2.0 ** -7 * pair[0].float().abs()
    assert err.max() <= 2.0 ** -7 * v.float().abs().max()
    finite = torch.isfinite(pair[1])
    assert (solo[1] - pair[1])[finite].abs().max() <= 1e-4


@pytest.mark.parametrize("kind", ("exact", "mean", "rescue2"))
@pytest.mark.parametrize("length,q_heads,share", ((40000, 2, 0.3), (87000, 1, 0.6), (87000, 1, 0.02)))
def test_long_lists(gpu, kind, length, q_heads, share):
    """Few heads keep single tiles up to hundreds of blocks: more than 256 list positions
    and tail blocks, a thread taking several of each."""
    q, k, v, blocks, d, choice = _case(1, length, q_heads, 1, 9)
    gen = torch.Generator("cuda").manual_seed(length)
    keep = torch.rand(1, blocks, blocks, q_heads, generator=gen, device="cuda") < share
    ids = torch.arange(blocks, device="cuda")
    keep &= (ids[None, :] <= ids[:, None])[None, :, :, None]
    keep[:, -1] = True                      # every block of the last tile
    idx, cnt = kernels.indices_from_mask(keep)
    solo, pair = _both(kind, q, k, v, idx, cnt, d, choice)
    assert not torch.isnan(solo[0]).any()
    assert torch.equal(solo[0], pair[0]) and torch.equal(solo[1], pair[1])
    # a sampled tile against float64: its listed keys alone
    if kind == "exact":
        t = blocks - 7
        blocks_of = idx[0, t, :cnt[0, t, 0], 0]
        tokens = (blocks_of[:, None] * 128 + torch.arange(128, device="cuda")).flatten()
        rows = slice(t * 128, t * 128 + 128)
        logits = q[0, rows, 0].double() @ k[0, tokens, 0].double().T * 128 ** -0.5
        hidden = tokens[None, :] > torch.arange(t * 128, t * 128 + 128, device="cuda")[:, None]
        logits = logits.masked_fill(hidden, float("-inf"))
        want = torch.softmax(logits, -1).nan_to_num() @ v[0, tokens, 0].double()
        # P rounds to bf16 (half a step, 2^-9 of every share), the output by half a step of
        # itself, fp32 sums below that
        bound = 2 ** -8 * (v.double().abs().max() + want.abs())
        assert ((solo[0][0, rows, 0].double() - want).abs() <= bound).all()
