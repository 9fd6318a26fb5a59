"""The 16-bit dK/dV work list's item length (CPU): ``balanced_chunk`` keeps
typical column walks whole, and the list built with it covers every column once,
in order, in items no longer than it."""

from __future__ import annotations

import pytest
import torch

from gki.lists import balanced_chunk, dkdv_items, long_walk_chunk


def _ptr(lens):
    return torch.tensor([0] + lens, dtype=torch.int32).cumsum(0).to(torch.int32)


@pytest.mark.parametrize("lens,group,bh,want", [
    ([128] + [17] * 127, 1, 64, 32),          # short walks, one long: the least chunk
    ([256] + [33] * 255, 1, 16, 33),          # walks just past 32 stay whole
    ([64] + [18] * 63, 4, 16, 72),            # grouped-query walks of 72
    ([128] + [18] * 127, 8, 4, 80),           # of 144: cut
    ([32] + [7] * 31, 1, 32, 16),             # a short grid: total / 512
    ([6] * 16, 1, 4, 8),                      # the shortest
    ([2048] + [66] * 2047, 16, 1, 268),       # a long grid: the library's own
    ([0, 0, 0], 1, 4, 0), ([], 1, 4, 0),
])
def test_chunk_and_list(lens, group, bh, want):
    ptr = _ptr(lens)
    chunk = balanced_chunk(ptr, group, bh)
    assert chunk == want
    if not chunk:
        return
    grid = max(bh, -(-8192 * chunk // (int(ptr[-1]) * group)))
    items, split, n_items, n_split, n_pslots = dkdv_items(ptr, group, grid, chunk)
    at, slots = {}, 0
    for kt, a, b, slot in items.tolist():
        assert a == at.get(kt, 0) and b - a <= chunk
        at[kt] = b
        assert (slot >= 0) == (lens[kt] * group > chunk)
        slots += slot >= 0
    assert at == {k: n * group for k, n in enumerate(lens)} and slots == n_pslots


@pytest.mark.parametrize("lens,group,want", [
    ([32] + [5] * 31, 1, 6),          # only the long one is cut
    ([128] + [17] * 127, 1, 21),      # a quarter above a typical walk
    ([16] + [9] * 30, 4, 45),         # grouped-query walks of 36
    ([5, 3, 3, 2, 1], 1, 5), ([0, 0, 0], 1, 5), ([1], 1, 5),
])
def test_fp32_long_walks(lens, group, want):
    assert long_walk_chunk(_ptr(lens), group) == want
