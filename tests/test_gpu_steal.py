"""Items drawn from other XCDs' shares (attention work queue, d = 128). Lists whose
length differs between KV groups by 50x leave most XCDs without items of their own
while one group's are still queued; what the other XCDs then take must give the same
bits as one workgroup per item, every item exactly once (outputs start as NaN), and the
counters the same final values as without steals: a draw past another share's end is
given back, and a workgroup that never drew a tail in vain does so when it ends."""

import numpy as np
import pytest
import torch

from exp3_amd import _lib, kernels, synthetic
from exp3_amd.upstream import flashprefill_native_forward as upstream
from tests.test_gpu_schedule import _call

pytestmark = pytest.mark.gpu


# (batch, q heads, KV heads, tokens): 2 / 1 XCDs per stream, an odd block count, three
# streams (one XCD each), and more streams than XCDs with enough items per share to steal
@pytest.mark.parametrize("layout", ((1, 28, 4, 9000), (1, 16, 8, 5000), (2, 8, 2, 300),
                                    (1, 12, 3, 6400), (2, 32, 8, 7000)))
@pytest.mark.parametrize("entry", ("exact", "mean"))
def test_unequal_groups(gpu, layout, entry):
    batch, q_heads, kv_heads, length = layout
    q, k, v, _ = synthetic.make_inputs(length, seed=43, q_heads=q_heads, kv_heads=kv_heads,
                                       batch=batch, device="cuda")
    blocks = (length + 127) // 128
    group = q_heads // kv_heads
    ids = torch.arange(blocks, device="cuda")
    causal = ids[None, :] <= ids[:, None]
    near = causal & (ids[:, None] - ids[None, :] < 1)
    mask = near[None, :, :, None].repeat(batch, 1, 1, q_heads)
    mask[..., :group] = causal[None, :, :, None]          # the first KV group lists all blocks
    idx, cnt = kernels.indices_from_mask(mask)
    desc = kernels.block_descriptors(k, v)
    tiles = upstream.attention_tiles(k, v)
    static = _call(entry, q, k, tiles, idx, cnt, desc, None)
    queue = torch.zeros(_lib.WORK_QUEUE_INTS, dtype=torch.int32, device="cuda")
    dynamic = _call(entry, q, k, tiles, idx, cnt, desc, queue)
    torch.cuda.synchronize()
    assert not torch.isnan(dynamic[0]).any()
    assert torch.equal(static[0], dynamic[0]) and torch.equal(static[1], dynamic[1])
    streams, pairs = batch * kv_heads, (blocks + 1) // 2
    xps = 8 // streams if streams <= 8 and 8 % streams == 0 else 1
    tp0 = pairs * 2 // 3
    while tp0 > 0 and xps > 1 and (tp0 * group) % xps:
        tp0 -= 1
    per_xcd = (pairs * group + xps - 1) // xps if xps > 1 else (pairs * streams + 7) // 8 * group
    grid = 8 * min(torch.cuda.get_device_properties(0).multi_processor_count // 8, per_xcd)
    counters = queue.cpu().numpy().astype(np.int64)
    assert counters[1:9].sum() == tp0 * streams * group + grid
    tails = counters[9:9 + streams] if xps > 1 else counters[:1]
    assert (tails == (pairs - tp0) * group * (1 if xps > 1 else streams) + grid).all()
