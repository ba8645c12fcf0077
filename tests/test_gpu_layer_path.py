"""The prefill layer as bare launches over one allocation (AttentionBackend._prefill)
against the same layer through the stage tensors (taken when kernel events, profiles or
captures are asked for): the same bits for every method and both head dims, on inputs
whose selection drops blocks; also when its scratch comes from recently freed memory, on
another stream, and after the shape changed."""

import pytest
import torch

from exp3_amd import attention, synthetic
from exp3_amd.upstream import flashprefill_native_forward as upstream

pytestmark = pytest.mark.gpu


class _Layer:
    layer_idx = 0


@pytest.mark.parametrize("method", attention.METHODS)
@pytest.mark.parametrize("batch,length,q_heads,kv_heads,dim",
                         ((1, 1089, 28, 4, 128), (2, 2113, 8, 2, 128), (1, 5000, 28, 4, 128),
                          (2, 1500, 16, 4, 256), (1, 1, 4, 1, 128)))
def test_same_bits_as_stages(gpu, method, batch, length, q_heads, kv_heads, dim):
    q, k, v, _ = synthetic.make_inputs(length, seed=length, q_heads=q_heads, kv_heads=kv_heads,
                                       head_dim=dim, batch=batch, device="cuda")
    q, k = ((x.float() * 4).to(torch.bfloat16) for x in (q, k))
    args = [x.transpose(1, 2) for x in (q, k, v)]
    backend = attention.AttentionBackend(alpha=0.6, register=False, dense_impl="hip")
    backend.configure(method, 0.6)
    scale = dim ** -0.5
    torch.full((64 << 20,), 255, dtype=torch.uint8, device="cuda")   # freed: the next scratch is garbage
    out, _ = backend.forward(_Layer(), *args, None, scale)
    assert upstream.attention_tile_sizes()[1] == (128 if dim == 128 else 32)
    backend.kernel_events = []
    want, _ = backend.forward(_Layer(), *args, None, scale)
    assert len(backend.kernel_events) == 1
    backend.kernel_events = None
    assert torch.equal(out, want) and not torch.isnan(out).any()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        half, _ = backend.forward(_Layer(), *(x[:, :, :(length + 1) // 2] for x in args), None, scale)
        other, _ = backend.forward(_Layer(), *args, None, scale)
    stream.synchronize()
    assert half.shape[1] == (length + 1) // 2 and torch.equal(other, want)


def test_refusals(gpu):
    q, k, v, _ = synthetic.make_inputs(300, seed=1, device="cuda")
    for kwargs, cut, method in (({"block_size": 64}, 128, "mean_native"), ({}, 64, "fp_v1"),
                                ({}, 64, "cgf_mean"), ({}, 64, "dense")):
        backend = attention.AttentionBackend(register=False, dense_impl="hip", **kwargs)
        backend.configure(method)
        with pytest.raises(ValueError):
            backend.forward(_Layer(), *(x[..., :cut].transpose(1, 2) for x in (q, k, v)), None, 0.1)


@pytest.mark.parametrize("q_cut,k_cut", (((0, 1), (0, 2)), ((0, 2), (0, 1)), ((1, 3), (1, 2))))
def test_mismatched_keys_reach_the_stage_checks(gpu, q_cut, k_cut):
    """A selector layer whose Q and K differ in batch or do not divide in heads."""
    q, k, v, _ = synthetic.make_inputs(300, seed=2, q_heads=4, kv_heads=2, batch=2, device="cuda")
    q, k, v = (x.transpose(1, 2) for x in (q, k, v))
    backend = attention.AttentionBackend(alpha=0.1, register=False)
    backend.configure("cgf_mean", 0.1)
    cut = lambda x, c: x.narrow(c[0], 0, c[1])    # noqa: E731
    with pytest.raises(ValueError, match="does not match"):
        backend.forward(_Layer(), cut(q, q_cut), cut(k, k_cut), cut(v, k_cut), None, 0.1)
