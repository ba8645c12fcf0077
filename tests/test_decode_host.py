"""Decode steps on the host: the calls the kernel does not take still go to SDPA, and
the C entry points refuse what they cannot run before any launch."""

import ctypes
from pathlib import Path
import subprocess
import sys

import pytest
import torch

from exp3_amd import _lib, attention


class _Layer:
    layer_idx = 0


@pytest.mark.parametrize("dtype", (torch.float32, torch.bfloat16))
@pytest.mark.parametrize("rows", (1, 3))
def test_cpu_step_goes_to_sdpa(dtype, rows):
    gen = torch.Generator().manual_seed(1)
    q = torch.randn(2, 4, rows, 128, generator=gen).to(dtype)
    k = torch.randn(2, 2, 40, 128, generator=gen).to(dtype)
    v = torch.randn(2, 2, 40, 128, generator=gen).to(dtype)
    assert not attention._decode_kernel_takes(q, k, v, 0.1)
    backend = attention.AttentionBackend(register=False)
    backend.configure("fp_v1")
    out, _ = backend.forward(_Layer(), q, k, v, attention_mask=None, scaling=0.1)
    wide = [x.double().repeat_interleave(2, 1) for x in (k, v)]
    want = torch.softmax(q.double() @ wide[0].transpose(2, 3) * 0.1, -1) @ wide[1]
    torch.testing.assert_close(out.double(), want.transpose(1, 2), rtol=1e-2, atol=1e-2)


def test_entry_point_validation():
    lib = _lib.load()
    s4 = (ctypes.c_int64 * 4)(4096, 512, 128, 1)
    odd = (ctypes.c_int64 * 4)(4096, 512, 132, 1)
    fake, off = 1 << 20, (1 << 20) + 8

    def call(q=fake, k=fake, ks=s4, shape=(1, 600, 28, 4, 128), workspace=fake):
        return lib.spx_decode_attention(q, s4, k, ks, fake, s4, *shape, 0.1, workspace, fake, None)

    assert call(shape=(1, 600, 28, 4, 64)) == _lib.SPX_EUNSUPPORTED
    assert call(shape=(1, 600, 28, 3, 128)) == _lib.SPX_EINVAL
    assert call(shape=(1, 0, 28, 4, 128)) == _lib.SPX_EINVAL
    assert call(shape=(4096, 600, 28, 4, 128)) == _lib.SPX_EINVAL      # 114688 rows
    assert call(q=None) == call(k=off) == call(ks=odd) == _lib.SPX_EINVAL
    assert call(workspace=None) == _lib.SPX_EINVAL                     # three ranges
    # ranges x rows x (dim + 2) floats; none up to two steps (512 keys, 256 at dim 256)
    size = lib.spx_decode_workspace_bytes
    assert size(1, 512, 28, 4, 128) == 0 and size(1, 513, 28, 4, 128) == 3 * 28 * 130 * 4
    assert size(1, 256, 16, 4, 256) == 0 and size(2, 257, 16, 4, 256) == 3 * 32 * 258 * 4
    assert size(1, 131072, 28, 4, 128) == 256 * 28 * 130 * 4
    assert size(1, 512, 28, 4, 64) == size(0, 512, 28, 4, 128) == -1


def test_prefill_scratch_needs_matching_shapes():
    """Calls whose Q, K and V disagree stay with the stage functions and their checks."""
    def x(*shape):
        return torch.empty(*shape)

    def match(*shapes):
        return attention._layer_shapes_match(*(x(*s) for s in shapes))

    q, kv = (2, 8, 300, 128), (2, 4, 300, 128)
    assert match(q, kv, kv)
    for bad in ((1, 4, 300, 128), (2, 3, 300, 128), (2, 0, 300, 128), (2, 4, 300, 256),
                (2, 4, 299, 128), (4, 300, 128)):
        assert not match(q, bad, bad) and not match(q, kv, bad) and not match(q, bad, kv)
    assert not match((0, 8, 300, 128), (0, 4, 300, 128), (0, 4, 300, 128))
    assert not match(q[1:], kv, kv)


def test_decode_shapes():
    """Calls that the decode kernel cannot run stay with SDPA, empty ones among them."""
    def fit(q, k, v=None):
        return attention._decode_shapes_fit(*(torch.Size(s) for s in (q, k, v or k)))

    q, kv = (2, 8, 1, 128), (2, 4, 300, 128)
    assert fit(q, kv) and fit((2, 8, 1, 256), (2, 4, 1, 256)) and fit((4095, 16, 1, 128), (4095, 2, 3, 128))
    for empty in ((2, 0, 1, 128), (0, 8, 1, 128), (2, 8, 0, 128), (2, 8, 1, 0)):
        assert not fit(empty, kv)
    for bad in ((2, 0, 300, 128), (2, 4, 0, 128), (1, 4, 300, 128), (2, 3, 300, 128),
                (2, 4, 300, 256)):
        assert not fit(q, bad) and not fit(q, kv, bad)
    assert not fit((2, 8, 2, 128), kv) and not fit((2, 8, 1, 64), (2, 4, 300, 64))
    assert not fit((4096, 16, 1, 128), (4096, 2, 3, 128))       # 65536 rows
    assert not fit((1, 1, 1, 128), (1, 1, (1 << 30) + 1, 128))


def test_tensors_read_in_place():
    def reads(x):
        return attention._reads_in_place((x,), -1)       # the index of a CPU tensor

    x = torch.zeros(2, 4, 40, 128, dtype=torch.bfloat16)
    assert reads(x) and reads(x.transpose(1, 2)) and reads(x[:, :, 8:]) and reads(x.expand(2, 4, 40, 128))
    assert not reads(torch._neg_view(x))          # negated when read, not in storage
    assert not attention._reads_in_place((x,), 0)
    assert not reads(x.half()) and not reads(x[0]) and not reads(x.transpose(2, 3))
    assert not reads(x[..., 1:]) and not reads(torch.nn.Parameter(x))


@pytest.mark.parametrize("missing", ("torch.overrides._get_current_function_mode_stack",
                                     "torch.utils._device.DeviceContext",
                                     "torch._C._len_torch_dispatch_stack",
                                     "torch._C._functorch.maybe_current_level",
                                     "torch.autograd.forward_ad._current_level"))
def test_torch_without_private_names(missing):
    """The backend imports and leaves its decode steps to SDPA."""
    program = f"""
import torch, torch.overrides, torch.utils._device, torch.autograd.forward_ad
q, k = torch.randn(1, 4, 1, 128), torch.randn(1, 2, 40, 128)
want = torch.nn.functional.scaled_dot_product_attention(q, k, k, scale=0.1, enable_gqa=True)
del {missing}
from exp3_amd import attention
backend = attention.AttentionBackend(register=False)
assert not attention._decode_kernel_takes(q, k, k, 0.1)
out, _ = backend.forward(None, q, k, k, None, 0.1)
assert torch.equal(out, want.transpose(1, 2))
"""
    done = subprocess.run([sys.executable, "-c", program], cwd=Path(__file__).resolve().parent.parent,
                          capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stderr


def test_stream_without_raw_handle(monkeypatch):
    class Stream:
        cuda_stream = 1234

    monkeypatch.setattr(_lib, "_raw_stream", None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: Stream)
    assert _lib.stream(torch.device("cuda", 0)) == 1234


def test_few_steps_of_many_streams_are_one_range():
    """Three or four steps of a stream are not cut in two where the launch has a stream for
    most workgroups (no workspace: one range)."""
    size = _lib.load().spx_decode_workspace_bytes
    assert size(64, 600, 8, 8, 128) == size(43, 700, 8, 8, 128) == size(49, 1000, 8, 8, 128) == 0
    assert size(32, 300, 16, 16, 256) == size(128, 1024, 28, 4, 128) == 0
    for streams, keys, ranges in ((42, 700, 3), (48, 1000, 2), (64, 1100, 2), (49, 1100, 2)):
        assert size(streams, keys, 8, 8, 128) == ranges * streams * 8 * 130 * 4
