"""What the attention launches are told about a ragged step, on the host."""

import pytest

from colossalai_amd.ops.ragged import RaggedBatch


@pytest.mark.parametrize("new,want", [([1, 1, 1], (0, 0, 0)), ([1], (0, 0, 0)), ([2], (1, 1, 1)), ([1, 33, 1], (4, 3, 3)), ([128, 129, 64], (11, 6, 4))])
def test_tiles_are_counted_once_a_step(new, want):
    batch = RaggedBatch.build(new, [5] * len(new), list(range(len(new))), "cpu")
    assert batch.tile_counts() == want and batch.num_tiles32 == want[0]
    assert batch.tile_counts() is batch.tile_counts()   # every layer of a step asks
