"""What the attention launches are told about a ragged step, on the host."""

import pytest

from colossalai_amd.ops.ragged import RaggedBatch


@pytest.mark.parametrize("new,want", [([1, 1, 1], (0, 0, 0)), ([1], (0, 0, 0)), ([2], (1, 1, 1)), ([1, 33, 1], (4, 3, 3)), ([128, 129, 64], (11, 6, 4))])
def test_tiles_are_counted_once_a_step(new, want):
    batch = RaggedBatch.build(new, [5] * len(new), list(range(len(new))), "cpu")
    assert batch.tile_counts() == want and batch.num_tiles32 == want[0]
    assert batch.tile_counts() is batch.tile_counts()   # every layer of a step asks


@pytest.mark.parametrize("new,start", [([1000], [0]), ([300, 64], [0, 500]), ([1, 400, 1], [16000, 100, 30]), ([33, 31], [10, 900]), ([1, 1, 2], [5, 9, 3])])
@pytest.mark.parametrize("window", [0, 200, 100000])
@pytest.mark.parametrize("fewest", [1, 2])
def test_key_lengths_of_tiles(new, start, window, fewest):
    """Counted tile by tile. A sequence's mean is its first and last tile's, or linear up to the window: half a tile apart at most at either end."""
    batch = RaggedBatch.build(new, start, list(range(len(new))), "cpu")
    keys = [s + min(t + 32, n) for n, s in zip(new, start) if n >= fewest for t in range(0, n, 32)]
    keys = [min(k, window) if window else k for k in keys]
    even, most = batch.key_lengths(window, fewest)
    assert most == max(keys) and abs(even - sum(keys) / len(keys) / most) <= 16 / most


def test_key_lengths_of_no_tiles():
    assert RaggedBatch.build([], [], [], "cpu").key_lengths() == (0.5, 0)
    assert RaggedBatch.build([1, 1], [5, 900], [0, 1], "cpu").key_lengths(0, 2) == (0.5, 0)
