"""The rows of a prefill step over several sequences, one of them behind a
cached prefix, and the lists that do not belong together, on the CPU."""

import pytest

from naivllm_amd.layers.qwen3 import prefill_rows


def test_rows_of_a_fresh_and_a_cached_sequence():
    toks = [[10, 11, 12, 13, 14], list(range(100, 107))]
    ids, pos, slots, last, bt, new, lens = prefill_rows(toks, [0, 4], [[7, 2], [5, 0, 9]], 4)
    assert ids.tolist() == [10, 11, 12, 13, 14, 104, 105, 106]
    assert pos.tolist() == [0, 1, 2, 3, 4, 4, 5, 6]
    assert slots.tolist() == [28, 29, 30, 31, 8, 0, 1, 2]
    assert last.tolist() == [4, 7] and new == [5, 3] and lens == [5, 7]
    assert bt.tolist() == [[7, 2, -1], [5, 0, 9]]


@pytest.mark.parametrize("starts,tables", [([0, 0], [[1]]), ([0], [[1], [2]]), ([0, 0, 0], [[1], [2]]),
                                           ([0, 0], [[1], [2], [3]])])
def test_lists_of_different_lengths_are_refused(starts, tables):
    with pytest.raises(ValueError, match="token lists"):
        prefill_rows([[1, 2], [3]], starts, tables, 4)


@pytest.mark.parametrize("start", [-1, 2, 3])
def test_starts_outside_the_sequence_are_refused(start):
    with pytest.raises(ValueError, match="outside"):
        prefill_rows([[1, 2]], [start], [[1]], 4)
