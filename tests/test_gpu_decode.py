"""spx_decode_attention (one query row per head over a KV cache) against the same
attention in float64, at the edges of its key tiles (16 keys), wave steps (64 keys at
head dim 128, 32 at 256), workgroup steps (256 / 128), the single-launch limit (two
steps) and several steps per workgroup; every head layout incl. more than 16 q heads
per KV head; cache slices and [B, S, H, D] views as inputs.

Tolerance: fp32 scores and sums leave about 1e-6 of the largest value, the bf16 output
half a step, 2^-8 of its own: |got - want| <= 2^-8 |want| + 1e-4 admits both with room for
a sum of fp32 rounding over 10^5 keys."""

import pytest
import torch

from exp3_amd import attention

pytestmark = pytest.mark.gpu

LAYOUTS = ((28, 4, 128), (16, 4, 256), (8, 8, 128), (20, 1, 128), (34, 2, 256))


class _Layer:
    layer_idx = 0


def _inputs(batch, q_heads, kv_heads, dim, length, seed, sharp=1.0):
    gen = torch.Generator("cuda").manual_seed(seed)
    def draw(*shape):
        return torch.randn(*shape, generator=gen, device="cuda")
    q = (draw(batch, 1, q_heads, dim) * sharp).to(torch.bfloat16).transpose(1, 2)
    k = draw(batch, kv_heads, length, dim).to(torch.bfloat16)
    v = draw(batch, kv_heads, length, dim).to(torch.bfloat16)
    return q, k, v


def _want(q, k, v, scale):
    group = q.shape[1] // k.shape[1]
    logits = (k.double().repeat_interleave(group, 1) * q.double()).sum(-1) * scale
    weights = torch.softmax(logits, -1)
    return (weights[..., None] * v.double().repeat_interleave(group, 1)).sum(2)[:, None]


def _step(q, k, v, scale):
    backend = attention.AttentionBackend(register=False)
    backend.configure("mean_native", 0.08)
    assert attention._decode_kernel_takes(q, k, v, scale)
    return backend.forward(_Layer(), q, k, v, attention_mask=None, scaling=scale)[0]


def _close(got, want, what=""):
    err = (got.double() - want).abs() - 2.0 ** -8 * want.abs()
    assert torch.isfinite(got).all() and err.max() <= 1e-4, f"{what} {err.max().item()}"


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("length", (2, 15, 17, 32, 33, 63, 64, 65, 127, 129, 255, 256, 257, 511,
                                    512, 513, 769, 4097))
def test_lengths(gpu, layout, length):
    q, k, v = _inputs(2, *layout, length, seed=length)
    out = _step(q, k, v, layout[2] ** -0.5)
    assert out.shape == (2, 1, layout[0], layout[2]) and out.is_contiguous()
    _close(out, _want(q, k, v, layout[2] ** -0.5), f"{layout} S={length}")


# several steps per workgroup: more than 256 ranges, and more streams than workgroups
@pytest.mark.parametrize("batch,layout,length", ((1, (4, 2, 128), 131072), (1, (2, 1, 256), 70001),
                                                 (40, (8, 8, 128), 1900)))
def test_long_and_wide(gpu, batch, layout, length):
    q, k, v = _inputs(batch, *layout, length, seed=5, sharp=6.0)   # sharp: the max moves
    _close(_step(q, k, v, layout[2] ** -0.5), _want(q, k, v, layout[2] ** -0.5))


@pytest.mark.parametrize("scale", (-0.2, 0.0, 3.0))
def test_scales(gpu, scale):
    q, k, v = _inputs(1, 28, 4, 128, 700, seed=9)
    _close(_step(q, k, v, scale), _want(q, k, v, scale))


def test_layouts_and_special_values(gpu):
    q, k, v = _inputs(2, 28, 4, 128, 1000, seed=3)
    cache = torch.full((2, 4, 1500, 128), float("nan"), dtype=torch.bfloat16, device="cuda")
    cache[:, :, :1000] = k
    rows = v.transpose(1, 2).contiguous().transpose(1, 2)          # [B, S, H, D] storage
    want = _step(q, k, v, 0.1)
    assert torch.equal(_step(q, cache[:, :, :1000], rows, 0.1), want)
    # an infinite value in the last row reaches the outputs of its heads only, as inf
    # (the repeated rows past the end must not turn it into NaN)
    v[0, 1, -1, 5] = float("inf")
    out = _step(q, k, v, 0.1)
    assert torch.isinf(out[0, 0, 7:14, 5]).all() and not torch.isnan(out).any()
    assert torch.isfinite(out[0, 0, :7]).all() and torch.isfinite(out[1]).all()
    # a NaN key makes its heads' rows NaN, as SDPA's softmax does
    k[1, 3, 500, 0] = float("nan")
    out = _step(q, k, v, 0.1)
    assert torch.isnan(out[1, 0, 21:]).all() and not torch.isnan(out[1, 0, :21]).any()


def test_captured_step(gpu):
    q, k, v = _inputs(1, 28, 4, 128, 3000, seed=4)
    want = _step(q, k, v, 0.1).clone()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        _step(q, k, v, 0.1)
    stream.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = _step(q, k, v, 0.1)
    for _ in range(3):
        out.zero_()
        _step(q, v, k, 0.1)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


def test_what_stays_with_sdpa(gpu):
    q, k, v = _inputs(1, 28, 4, 128, 300, seed=6)
    takes = attention._decode_kernel_takes
    assert takes(q, k, v, 0.1)
    assert not takes(q.half(), k.half(), v.half(), 0.1)
    assert not takes(q.repeat(1, 1, 2, 1), k, v, 0.1) and not takes(q, k, v, None)
    assert not takes(q[..., :64], k[..., :64], v[..., :64], 0.1)
    assert not takes(q, k[..., 1:], v[..., 1:], 0.1) and not takes(q[:, :27], k, v, 0.1)
    assert not takes(q.cpu(), k.cpu(), v.cpu(), 0.1) and not takes(q, k, v[:, :, :-1], 0.1)
    assert not takes(q.clone().requires_grad_(), k, v, 0.1)
    with torch.no_grad():
        assert takes(q.clone().requires_grad_().detach(), k, v, 0.1)
    with torch.autocast("cuda", torch.float16):
        assert not takes(q, k, v, 0.1)
    with torch.nn.attention.sdpa_kernel(torch.nn.attention.SDPBackend.MATH):
        assert not takes(q, k, v, 0.1)
    with torch.device("cuda"):
        assert takes(q, k, v, 0.1)
    seen = []
    torch.vmap(lambda x: (seen.append(takes(x, k, v, 0.1)), x)[1])(q[None])
    assert seen == [False]
    # gradients still flow through the step
    backend = attention.AttentionBackend(register=False)
    leaf = q.float().requires_grad_()
    out, _ = backend.forward(_Layer(), leaf.to(torch.bfloat16), k, v, None, 0.1)
    out.sum().backward()
    assert leaf.grad is not None and torch.isfinite(leaf.grad).all()


# one range of three and of four steps per stream, whole and with a few keys in the last
@pytest.mark.parametrize("batch,layout,length", ((64, (8, 8, 128), 514), (49, (8, 8, 128), 1024),
                                                 (33, (32, 16, 256), 300), (26, (16, 16, 256), 511)))
def test_one_range_of_several_steps(gpu, batch, layout, length):
    q, k, v = _inputs(batch, *layout, length, seed=11, sharp=6.0)
    _close(_step(q, k, v, layout[2] ** -0.5), _want(q, k, v, layout[2] ** -0.5))
