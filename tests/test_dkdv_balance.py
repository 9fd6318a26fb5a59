"""The 16-bit dK/dV work list's item length (CPU): ``balanced_chunk`` keeps
typical column walks whole, and the list built with it covers every column once,
in order, in items no longer than it."""

from __future__ import annotations

import pytest
import torch

from gki import _lib
from gki.lists import balanced_chunk, dkdv_items, dkdv_items_cut, long_walk_chunk
from oracle import streaming_oracle as so


def _ptr(lens):
    return torch.tensor([0] + lens, dtype=torch.int32).cumsum(0).to(torch.int32)


@pytest.mark.parametrize("lens,group,bh,want", [
    ([128] + [17] * 127, 1, 64, 32),          # short walks, one long: the least chunk
    ([256] + [33] * 255, 1, 16, 33),          # walks just past 32 stay whole
    ([64] + [18] * 63, 4, 16, 72),            # grouped-query walks of 72
    ([20] + [18] * 63, 4, 8, 72),             # 512 of them; their mean is a little less
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
    items, split, n_items, n_split, n_pslots = dkdv_items_cut(ptr, group, chunk)
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
    assert long_walk_chunk(_ptr(lens), group, 16) == want


@pytest.mark.parametrize("lens,group,bh", [
    ([512] * 50 + [5] * 462, 1, 16),          # a tenth of the columns over every row
    ([2048] * 200 + [5] * 1848, 1, 16), ([2048] + [65] * 2047, 1, 16), ([300] * 9 + [2] * 91, 8, 8),
])
def test_fp32_long_walks_bounded_partials(lens, group, bh):
    """Many long columns over short typical ones: still about 8192 items in all, each
    of which is 128 rows of fp32 partials."""
    ptr = _ptr(lens)
    chunk = long_walk_chunk(ptr, group, bh)
    n_pslots = dkdv_items(ptr, group, bh, chunk)[4]
    assert n_pslots * bh <= 8192 + len(lens) * bh


@pytest.mark.parametrize("lens,group,bh,want", [
    ([64] + [18] * 63, 4, 8, 32),             # 512 columns of 72: in pieces
    ([64] + [18] * 63, 4, 16, 72),            # 1024: whole
    ([128] + [18] * 127, 8, 4, 32), ([128] + [18] * 127, 8, 8, 80),
    ([64] + [33] * 63, 1, 8, 33),             # walks of up to 48: whole
    ([64] + [18] * 63, 4, 4, 38),             # fewer columns: total / 512
    ([16] * 16, 1, 16, 16), ([9, 7, 12] * 7, 1, 24, 16),   # even walks: whole
    ([16] * 16, 1, 7, 8),                     # too few of them
    ([32] + [9] * 31, 1, 8, 8),               # a long one among them
])
def test_chunk_where_more_workgroups_fit(lens, group, bh, want):
    for head_dim in (16, 32, 64):
        assert balanced_chunk(_ptr(lens), group, bh, head_dim) == want


@pytest.mark.parametrize("lens,bh,wide,narrow", [
    ([24] * 24, 8, 24, 9), ([16] * 16, 8, 16, 8), ([16] * 16, 12, 16, 16), ([17] * 17, 12, 17, 8),
])
def test_even_walks_by_head_dim(lens, bh, wide, narrow):
    for head_dim, want in ((16, narrow), (32, narrow), (64, wide), (128, wide)):
        assert balanced_chunk(_ptr(lens), 1, bh, head_dim) == want


@pytest.mark.parametrize("chunk", [1, 5, 32, 80, 1 << 20])
def test_cut_list_equals_the_oracle(chunk):
    """Any length, also above the least one of the library's own rule."""
    for lens, group in (([128] + [18] * 127, 8), ([0, 3, 0, 7], 1), ([1], 4)):
        ptr = _ptr(lens)
        items, split, n_items, n_split, n_pslots = dkdv_items_cut(ptr, group, chunk)
        want = so.dkdv_items(ptr.numpy(), group, 1, chunk=chunk)
        assert items.tolist() == want[0].tolist() and split[:n_split].tolist() == want[1].tolist()
        assert (n_items, n_pslots) == (len(want[0]), want[2])
        own = dkdv_items(ptr, group, 1, min(chunk, 32))
        assert dkdv_items_cut(ptr, group, min(chunk, 32))[0].tolist() == own[0].tolist()


def test_cut_refuses_what_the_rule_refuses():
    lib, ptr = _lib.load(), _ptr([3, 4])
    out = torch.zeros(3, dtype=torch.int32)
    refs = [out.data_ptr() + 4 * i for i in range(3)]
    falling = torch.tensor([0, 5, 3], dtype=torch.int32)
    for col_ptr, n_kt, group, chunk in ((ptr, 2, 1, 0), (ptr, 2, 1, -1), (ptr, 2, 0, 8), (ptr, 0, 1, 8),
                                        (falling, 2, 1, 8)):
        assert lib.gki_dkdv_items_cut(col_ptr.data_ptr(), n_kt, group, chunk, None, refs[0], None, refs[1], refs[2]) == 1
    assert lib.gki_dkdv_items_cut(None, 2, 1, 8, None, refs[0], None, refs[1], refs[2]) == 1
