"""The prefill kernel's work list (layers.attention.prefill_tiles) covers every
(row, key) pair of a causal prefill exactly once, on the CPU."""

import numpy as np
import pytest

from naivllm_amd.layers.attention import prefill_tiles


@pytest.mark.parametrize("heads,block_size", [((16, 8), 256), ((32, 8), 16), ((8, 8), 1), ((3, 1), 1), ((16, 8), None)])
@pytest.mark.parametrize("ql,kl", [([1], [1]), ([64], [64]), ([65, 1, 300], [65, 5000, 300]), ([40], [4136]),
                                   ([2900, 700], [7000, 700]), ([129, 128, 127], [4000, 4001, 127])])
def test_tiles_cover_every_pair_once(heads, block_size, ql, kl):
    tiles, merges, rows, slots = prefill_tiles(ql, kl, *heads, block_size, 256)
    group = heads[0] // heads[1]
    hw = 2 if group % 2 == 0 else 1
    assert rows * hw in (128, 256)
    seen = np.zeros((sum(ql), max(kl)), dtype=np.int32)
    q0, k0 = np.cumsum(ql) - ql, np.cumsum(kl) - kl
    parts = {}
    for seq, row0, nr, pos, kv0, begin, end, slot in tiles.tolist():
        assert 1 <= nr <= rows and begin % 64 == 0 and begin < end
        first = row0 - q0[seq]
        assert 0 <= first and first + nr <= ql[seq] and pos == kl[seq] - ql[seq] + first
        assert kv0 == (k0[seq] if block_size is None else 0)
        for r in range(nr):
            seen[row0 + r, begin:min(end, pos + r + 1)] += 1
        parts.setdefault((row0, nr), []).append((begin, end, slot))
    for i, n in enumerate(ql):
        for r in range(n):
            want = np.zeros(max(kl), dtype=np.int32)
            want[:kl[i] - n + r + 1] = 1
            assert np.array_equal(seen[q0[i] + r], want)
    cut = {k: sorted(v) for k, v in parts.items() if len(v) > 1}
    assert all(v[0][2] == -1 for v in parts.values() if len(v) == 1)
    assert sorted((v[0][2], len(v), *k) for k, v in cut.items()) == sorted(map(tuple, merges.tolist()))
    for v in cut.values():  # consecutive slots in key order
        assert [x[2] for x in v] == list(range(v[0][2], v[0][2] + len(v)))
    assert slots == sum(len(v) for v in cut.values())
    sizes = tiles[:, 6] - tiles[:, 5]
    assert np.all(sizes[:-1] >= sizes[1:])


def test_bad_lengths_are_refused():
    for ql, kl in (([0], [4]), ([5], [4]), ([4, 4], [4])):
        with pytest.raises(ValueError):
            prefill_tiles(ql, kl, 16, 8, 256, 256)


@pytest.mark.parametrize("heads", [(16, 8), (32, 8), (64, 8), (8, 8), (3, 1), (2, 1)])
@pytest.mark.parametrize("block_size", [1, 16, 256])
def test_partials_are_bounded(heads, block_size):
    # only a step whose tiles leave compute units idle is cut over keys (into
    # parts of two thirds of a compute unit's share of its key tiles or more),
    # whatever the page size: its partials stay within 2.5 workgroups' rows a
    # compute unit, 85 MB at 256
    for ql, kl in (([32000], [32000]), ([40000], [40000]), ([1], [40000]), ([300, 5], [20000, 33000]), ([128] * 8, [9000] * 8)):
        tiles, merges, rows, slots = prefill_tiles(ql, kl, *heads, block_size, 256)
        assert slots * heads[0] * rows * (128 + 2) * 4 <= 2.5 * 256 * 256 * (128 + 2) * 4, (ql, kl, slots)
    assert prefill_tiles([40000], [40000], *heads, 1, 256)[3] == prefill_tiles([40000], [40000], *heads, 256, 256)[3]
