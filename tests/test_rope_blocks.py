"""The block order of the prologue's rotary passes: every (row range, chunk of
heads) is one block, and the blocks of a chip of eight XCDs, which take blocks
in turn, cover them evenly whatever the number of ranges."""

from __future__ import annotations

import ctypes

import pytest

from repercep_runtime_amd import _capi


def _block(ranges: int, chunks: int, b: int) -> tuple[int, int]:
    r, c = ctypes.c_int64(), ctypes.c_int64()
    assert _capi.lib().rp_selftest_rope_block(ranges, chunks, b, ctypes.byref(r),
                                              ctypes.byref(c)) == 0
    return r.value, c.value


@pytest.mark.parametrize("ranges", [1, 2, 3, 7, 8, 9, 15, 16, 23, 440])
@pytest.mark.parametrize("chunks", [1, 2, 5, 8, 20, 128])
def test_each_block_once_and_every_xcd_alike(ranges: int, chunks: int) -> None:
    n = ranges * chunks
    at = [_block(ranges, chunks, b) for b in range(n)]
    assert sorted(at) == [(r, c) for r in range(ranges) for c in range(chunks)]
    # the ranges an XCD works on: as few as an even share allows (one more
    # where its run of the last ones begins inside a range)
    for x in range(min(8, n)):
        mine = at[x::8]
        assert n // 8 <= len(mine) <= -(-n // 8)
        assert len({r for r, _ in mine}) <= -(-len(mine) // chunks) + 1


def test_bad_arguments() -> None:
    r = ctypes.c_int64()
    L = _capi.lib()
    for args in ((0, 1, 0), (1, 0, 0), (2, 3, 6), (2, 3, -1), (1 << 31, 2, 0)):
        assert L.rp_selftest_rope_block(*args, ctypes.byref(r), ctypes.byref(r)) == 1
    assert L.rp_selftest_rope_block(2, 3, 0, None, ctypes.byref(r)) == 1
