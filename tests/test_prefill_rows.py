"""The rows of a prefill step over several sequences, one of them behind a
cached prefix, and the lists that do not belong together, on the CPU."""

import pytest

from naivllm_amd.layers.attention import verify_serves_prefill
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


@pytest.mark.parametrize("new,keys,heads,page,width,taken", [
    ([24], [300], (16, 8), 16, 19, True), ([25], [4000], (16, 8), 16, 250, False),      # 48 packed rows, 8 pairs
    ([8], [300], (4, 2), 16, 19, True), ([9], [300], (4, 2), 16, 19, False),            # 16 with fewer pairs
    ([9] * 4, [300] * 4, (4, 2), 16, 19, True),
    ([9], [300], (16, 8), 8, 38, False), ([9], [300], (32, 8), 8, 38, True),            # pages the key-split kernel does not take
    ([9], [300], (16, 8), 16, 1024, True), ([9], [300], (16, 8), 16, 1025, False),      # its longest table
    ([16], [1536], (32, 8), 256, 6, True), ([16], [1535], (32, 8), 256, 6, False),      # 64 packed rows
    ([32], [4000], (16, 8), 256, 16, False), ([17], [4000], (32, 8), 256, 16, False),
    ([1], [1], (80, 1), 256, 1, False), ([4], [4], (32, 8), 1, 1 << 22, False),
])
def test_steps_of_few_rows(new, keys, heads, page, width, taken):
    assert verify_serves_prefill(new, keys, *heads, page, width) is taken
