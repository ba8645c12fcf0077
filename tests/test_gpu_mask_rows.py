"""indices_from_mask by (batch, query tile) workgroups: chunk edges of the key blocks,
head groups that exceed the LDS lists, and the sizes past its limits (256 heads, 1024 key
blocks) that keep one workgroup per row; masks without any causal order, empty and full
rows, bytes other than 0 and 1."""

import pytest
import torch

from exp3_amd import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,query,keys,heads", (
    (1, 1, 1, 1), (2, 3, 63, 28), (1, 2, 64, 28), (1, 3, 65, 12), (2, 5, 129, 3), (1, 2, 256, 32),
    (1, 2, 257, 17), (1, 2, 513, 28), (1, 3, 1024, 64), (1, 2, 1024, 256), (1, 2, 130, 257),
    (1, 2, 1025, 4)))
def test_lists_of_any_mask(gpu, batch, query, keys, heads):
    gen = torch.Generator().manual_seed(keys * 7 + heads)
    share = torch.rand(batch, query, 1, heads, generator=gen)
    mask = torch.rand(batch, query, keys, heads, generator=gen) < share
    mask[:, 0, :, 0] = False
    mask[:, -1, :, -1] = True
    ids = torch.arange(keys)[None, None, :, None]
    want = torch.where(mask, ids, keys).sort(dim=2).values
    value = torch.randint(1, 256, mask.shape, generator=gen, dtype=torch.uint8)
    for given in (mask, value * mask):
        indices, counts = kernels.indices_from_mask(given.cuda())
        assert indices.dtype is torch.int64 and counts.dtype is torch.int32
        assert torch.equal(indices.cpu(), want)
        assert torch.equal(counts.cpu().long(), mask.sum(2))
