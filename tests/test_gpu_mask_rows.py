"""indices_from_mask by (batch, query tile) workgroups (64 tiles and 6 heads or more) and
with one workgroup per row: chunk edges of the key blocks, head groups that exceed the LDS
lists, and the sizes past the first form's limits (256 heads, 1024 key blocks); masks
without any causal order, empty and full rows, bytes other than 0 and 1."""

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


@pytest.mark.parametrize("batch,query,keys,heads", (
    (1, 63, 63, 28), (1, 64, 1, 8), (2, 43, 64, 6), (2, 43, 65, 5), (1, 64, 65, 7), (3, 30, 129, 17),
    (1, 64, 256, 32), (1, 70, 257, 9), (1, 65, 513, 28), (1, 64, 1024, 64), (1, 64, 1000, 256),
    (1, 64, 130, 257), (1, 64, 1025, 8)))
def test_lists_by_tile(gpu, batch, query, keys, heads):
    gen = torch.Generator("cuda").manual_seed(keys * 5 + heads)
    share = torch.rand(batch, query, 1, heads, generator=gen, device="cuda")
    mask = torch.rand(batch, query, keys, heads, generator=gen, device="cuda") < share
    mask[:, 0, :, 0] = False
    mask[:, -1, :, -1] = True
    ids = torch.arange(keys, device="cuda")[None, None, :, None]
    want = torch.where(mask, ids, keys).sort(dim=2).values
    value = torch.randint(1, 256, mask.shape, generator=gen, dtype=torch.uint8, device="cuda")
    for given in (mask, value * mask):
        indices, counts = kernels.indices_from_mask(given)
        assert torch.equal(indices, want) and torch.equal(counts.long(), mask.sum(2))


@pytest.mark.parametrize("shape", ((1, 2, 1024, 256), (1, 1, 1000, 64)))
def test_few_tiles_use_the_chip(gpu, shape):
    """One or two query tiles are spread over the CUs: 4 MB or less of lists in a few times
    what it takes to fill them (2 and 3 measured; with a workgroup per tile 13 and 60)."""
    mask = torch.rand(shape, device="cuda") < 0.5
    lists = torch.empty(shape, dtype=torch.int64, device="cuda")

    def best(call):
        times = []
        for _ in range(10):
            begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            begin.record()
            for _ in range(20):
                call()
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end))
        return min(times)

    assert best(lambda: kernels.indices_from_mask(mask)) <= 9 * best(lambda: lists.fill_(1))
