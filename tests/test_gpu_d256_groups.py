"""Head dim 256: short launches split each tile's keys over two groups of waves
(csrc/attn256.hip), long ones do not. The same sequence alone and within a batch that
makes the launch long: same lists, outputs and LSEs within the rounding of the
probabilities, for one to four blocks (two groups from three on), ragged ends, empty, unsorted and repeated lists
with entries outside the sequence, and every method's tail."""

import pytest
import torch

from exp3_amd import _lib, attention, kernels, synthetic
from exp3_amd.upstream import flashprefill_native_forward as upstream

pytestmark = pytest.mark.gpu

HEADS, KV, DIM = 16, 4, 256
LONG = 1536 // HEADS + 1          # batch from which any launch is long


def _inputs(length, seed):
    q, k, v, _ = synthetic.make_inputs(length, seed=seed, q_heads=HEADS, kv_heads=KV, head_dim=DIM,
                                       device="cuda")
    return ((q.float() * 4).bfloat16(), (k.float() * 4).bfloat16(), v)


def _batch(x):
    return x.expand(LONG, *x.shape[1:]).contiguous()


def _assert_close(got, want, v):
    # bf16 keeps 8 significant bits: a rounding moves a value by up to 2^-8 of it. In each
    # kernel P rounds against another running maximum (2^-8 of every key's share of the
    # output, at most 2^-8 max |v|), then the output: both sides, twice
    bound = 2 ** -7 * (v.float().abs().amax() + want.float().abs())
    assert ((got.float() - want.float()).abs() <= bound).all()


@pytest.mark.parametrize("length", (1, 31, 128, 129, 300, 512))
def test_lists(gpu, length):
    q, k, v = _inputs(length, 3 + length)
    blocks = (length + 127) // 128
    gen = torch.Generator().manual_seed(length)
    # ids -1 and NB are dropped; a list may hold a block twice or none
    idx = torch.randint(-1, blocks + 1, (1, blocks, blocks, HEADS), generator=gen)
    tile = torch.arange(blocks)[None, :, None, None]
    idx = torch.where((idx > tile) & (idx < blocks), tile, idx).cuda()
    cnt = torch.randint(0, blocks + 1, (1, blocks, HEADS), generator=gen, dtype=torch.int32)
    cnt[:, 0, 0] = 0
    cnt = cnt.cuda()
    out, lse = upstream.exact_attention(q, k, v, idx, cnt, DIM ** -0.5)
    many, many_lse = upstream.exact_attention(*(_batch(x) for x in (q, k, v, idx, cnt)), DIM ** -0.5)
    assert torch.equal(many[0], many[-1]) and not torch.isnan(out).any()
    _assert_close(out[0], many[-1], v)
    empty = torch.isinf(many_lse[-1])
    assert torch.equal(torch.isinf(lse[0]), empty) and not out[0][empty].any()
    # fp32 sums and base-2 logits of up to some 2^8
    assert torch.allclose(lse[0][~empty], many_lse[-1][~empty], rtol=1e-5, atol=1e-4)


@pytest.mark.parametrize("method", attention.METHODS)
@pytest.mark.parametrize("length", (1, 260, 1089))
def test_layers(gpu, method, length):
    q, k, v = _inputs(length, 5)
    backend = attention.AttentionBackend(alpha=0.6, register=False, dense_impl="hip", sink_blocks=1,
                                         window_blocks=1, last_full_blocks=0)
    backend.configure(method, 0.6)

    class Layer:
        layer_idx = 0

    args = [x.transpose(1, 2) for x in (q, k, v)]
    out, _ = backend.forward(Layer(), *args, None, DIM ** -0.5)
    many, _ = backend.forward(Layer(), *(_batch(x) for x in args), None, DIM ** -0.5)
    _assert_close(out[0], many[-1], v)


@pytest.mark.parametrize("length,seen", ((700, 1), (5000, 0), (5000, 3)))
def test_tails_alone(gpu, length, seen):
    """A launch of tails without exact blocks keeps one group (two were slower): the same
    bits alone and in a batch, with tails of one and of several steps."""
    q, k, v = _inputs(length, 8)
    blocks = (length + 127) // 128
    ids = torch.arange(blocks, device="cuda")
    near = (ids[None, :] <= ids[:, None]) & (ids[:, None] - ids[None, :] < seen)
    selected = near[None, :, :, None].expand(1, blocks, blocks, HEADS).contiguous()

    def tails(q, k, v, selected):
        return (kernels.mean_tail(q, kernels.block_descriptors(k, v), selected, DIM ** -0.5)
                + kernels.rescue_tail(q, k, v, selected, DIM ** -0.5, remainder=True))

    copies = 3 if length > 4096 else LONG     # past 1024 (tile, head) items
    many = tails(*(x.expand(copies, *x.shape[1:]).contiguous() for x in (q, k, v, selected)))
    for one, batch in zip(tails(q, k, v, selected), many):
        assert torch.equal(one[0], batch[0]) and torch.equal(one[0], batch[-1])


@pytest.mark.parametrize("batch,length", ((1, 100), (1, 256), (4, 731), (2, 4059)))
def test_where_one_group_stays(gpu, batch, length):
    """One or two blocks, few blocks of many heads and sequences of a batch: the bits of
    the one-group kernel."""
    q, k, v = _inputs(length, 9)
    blocks = (length + 127) // 128
    idx = torch.arange(blocks, device="cuda")[None, None, :, None].expand(1, blocks, blocks, HEADS)
    cnt = torch.arange(1, blocks + 1, device="cuda", dtype=torch.int32)[None, :, None]
    cnt = cnt.expand(1, blocks, HEADS)

    def outputs(count):
        args = (x.expand(count, *x.shape[1:]).contiguous() for x in (q, k, v, idx, cnt))
        return upstream.exact_attention(*args, DIM ** -0.5)

    many = outputs(5 if length > 4000 else LONG)
    for one, all_ in zip(outputs(batch), many):
        assert torch.equal(one[0], all_[0]) and torch.equal(one[-1], all_[-1])


@pytest.mark.parametrize("kind,q_heads,kv_heads,length", (("rescue2", 16, 4, 6113),
                                                          ("rescue1", 12, 2, 10800),
                                                          ("mean", 12, 2, 10800)))
def test_several_tail_steps(gpu, kind, q_heads, kv_heads, length):
    """Two groups take 32 tail entries each per step: sparse lists with up to 85 unlisted
    blocks make two and three steps. Alone (two groups) against a batch of two (one)."""
    q, k, v, _ = synthetic.make_inputs(length, seed=13, q_heads=q_heads, kv_heads=kv_heads,
                                       head_dim=DIM, device="cuda")
    q, k = (q.float() * 4).bfloat16(), (k.float() * 4).bfloat16()
    blocks = (length + 127) // 128
    ids = torch.arange(blocks, device="cuda")
    gen = torch.Generator("cuda").manual_seed(2)
    keep = torch.rand(1, blocks, blocks, q_heads, generator=gen, device="cuda") < 0.04
    keep &= (ids[None, :] <= ids[:, None])[None, :, :, None]
    keep[:, blocks // 2] = False            # a tile of its tail alone
    assert (ids[-1] - keep[0, -1].sum(0)).max() > 32 * 2 // (2 if kind == "rescue2" else 1)
    results = []
    for copies in (1, 2):
        q_, k_, v_, keep_ = (x.expand(copies, *x.shape[1:]).contiguous() for x in (q, k, v, keep))
        d = kernels.block_descriptors(k_, v_)
        tiles = upstream.attention_tiles(k_, v_)
        choice = kernels.rescue_choice(q_, tiles[0])
        idx, cnt = kernels.indices_from_mask(keep_)
        out = torch.full(q_.shape, float("nan"), dtype=q.dtype, device="cuda")
        lse = torch.full(q_.shape[:3], float("nan"), device="cuda")
        head = (_lib.ptr(q_), _lib.strides(q_), _lib.ptr(tiles[0]), _lib.ptr(tiles[1]),
                _lib.ptr(idx), _lib.strides(idx), _lib.ptr(cnt), _lib.strides(cnt))
        end = (copies, length, q_heads, kv_heads, DIM, 128, DIM ** -0.5, _lib.ptr(out),
               _lib.strides(out), _lib.ptr(lse), _lib.strides(lse), None, _lib.stream(q.device))
        if kind == "mean":
            _lib.call("spx_sparse_attention_mean", *head, _lib.ptr(d.mean_k), _lib.ptr(d.mean_v),
                      _lib.ptr(d.counts), *end)
        else:
            _lib.call("spx_sparse_attention_rescue", *head, _lib.ptr(choice), _lib.ptr(v_),
                      _lib.strides(v_), _lib.ptr(d.mean_k), _lib.ptr(d.mean_v),
                      int(kind == "rescue2"), *end)
        results.append((out[-1], lse[-1]))
    (two, two_lse), (one, one_lse) = results
    assert not torch.isnan(one).any() and not torch.isnan(two).any()
    _assert_close(two, one, v)
    empty = torch.isinf(one_lse)
    assert torch.equal(torch.isinf(two_lse), empty)
    assert torch.allclose(two_lse[~empty], one_lse[~empty], rtol=1e-5, atol=1e-4)
