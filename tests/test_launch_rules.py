"""Rules by which a launch picks a kernel, as far as the host shows them."""

from exp3_amd import _lib


def test_single_tiles_or_pairs():
    """spx_attention_queue_ints: no queue (single tiles) for few blocks, fewer where no heads
    share K and V, and for few pair items (341 on 256 CUs); head dim 256 takes a queue."""
    ints = _lib.load().spx_attention_queue_ints
    for shape in ((80, 1536, 16, 8), (80, 768, 8, 8), (4, 1300, 8, 8), (1, 3072, 28, 4)):
        assert ints(*shape, 128) == 0, shape
    for shape in ((80, 1537, 16, 8), (80, 1507, 8, 8), (80, 769, 8, 8), (1, 3073, 28, 4)):
        assert ints(*shape, 128) == _lib.WORK_QUEUE_INTS, shape
    assert ints(1, 100, 16, 4, 256) == _lib.WORK_QUEUE_INTS
