"""merge_exact_mean with 16-byte accesses and, for bases or strides that these do not
fit, with narrow ones, against the same merge in 64 bits: row counts around a workgroup's,
equal, far apart and empty (-inf) LSEs."""

import pytest
import torch

from exp3_amd import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", (128, 256))
@pytest.mark.parametrize("batch,length,heads", ((1, 1, 1), (1, 5, 3), (1, 16, 1), (3, 43, 7)))
@pytest.mark.parametrize("layout", ("aligned", "exact", "mean", "transposed"))
def test_against_64_bits(gpu, dim, batch, length, heads, layout):
    gen = torch.Generator("cuda").manual_seed(dim + length)

    def draw(*shape):
        return torch.randn(*shape, generator=gen, device="cuda")

    def place(x, shift):      # the same values, `shift` elements past an aligned base
        room = torch.empty(x.numel() + shift, dtype=x.dtype, device="cuda")
        return room[shift:].view(x.shape).copy_(x)

    exact, mean = draw(batch, length, heads, dim).bfloat16(), draw(batch, length, heads, dim)
    if layout == "exact":
        exact = place(exact, 2)
    elif layout == "mean":
        mean = place(mean, 1)
    elif layout == "transposed":
        exact, mean = (x.transpose(1, 2).contiguous().transpose(1, 2) for x in (exact, mean))
    el, ml = 4 * draw(batch, length, heads), 4 * draw(batch, length, heads)
    row = torch.arange(el.numel(), device="cuda").view(el.shape) % 5
    el = torch.where(row == 1, ml, torch.where(row == 2, -torch.inf, el))
    ml = torch.where(row == 3, -torch.inf, torch.where(row == 4, ml - 200, ml))
    out, lse = kernels.merge_exact_mean(exact, el, mean, ml)
    want_lse = torch.logaddexp(el.double(), ml.double())
    we, wm = (torch.exp(x.double() - want_lse)[..., None] for x in (el, ml))
    parts = (we * exact.double()).abs() + (wm * mean.double()).abs()
    want = we * exact.double() + wm * mean.double()
    # bf16 rounding (2^-8 of the value) and fp32 weights: LSEs of up to 200 in 2^-24
    # steps, so exp(le - total) is good to about 3e-5 of each part
    assert ((out.double() - want).abs() <= 2 ** -8 * want.abs() + 5e-5 * parts).all()
    assert torch.allclose(lse.double(), want_lse, rtol=1e-6, atol=1e-6)
