"""Which bytes of C the lanes or waves of a kernel store (csrc/lane_ranges.hpp, compiled here for the host): every byte once where two lanes hold
different sums, and only bytes whose sum the lane has.  No GPU needed."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hopper_spmm_amd", "csrc")
SOURCE = """
#include "lane_ranges.hpp"
using namespace hspmm;
extern "C" unsigned begin(unsigned lane, unsigned bytes, unsigned row_len, int odd) { return entry_lane_begin(lane, bytes, row_len, odd); }
extern "C" unsigned stores(unsigned lane, unsigned bytes, unsigned row_len, int odd) { return entry_lane_stores(lane, bytes, row_len, odd); }
extern "C" unsigned first(unsigned tile, int odd) { return narrow_tile_first(tile, odd); }
extern "C" unsigned own(unsigned tile, int odd) { return narrow_tile_own(tile, odd); }
extern "C" unsigned end(unsigned tile, int odd) { return narrow_tile_end(tile, odd); }
"""


@pytest.fixture(scope="module")
def ranges(tmp_path_factory):
    at = tmp_path_factory.mktemp("ranges")
    (at / "ranges.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, "-o", str(at / "ranges.so"), str(at / "ranges.cpp")], check=True)
    return ctypes.CDLL(str(at / "ranges.so"))


def _lanes(bytes_):
    n = 1
    while n * 16 < bytes_:
        n *= 2
    return n


@pytest.mark.parametrize("N", range(9, 257, 2))
def test_odd_rows_of_the_entry_kernels(ranges, N):
    """A row, or a block of 16 k + 14 bytes of a longer one, that begins on a word and half a word behind one."""
    row_len = 2 * N
    lanes = _lanes(row_len)
    begin = [ranges.begin(i, 16, row_len, 1) for i in range(lanes)]
    stores = [ranges.stores(i, 16, row_len, 1) for i in range(lanes)]
    assert all(b >= 0 and b + 14 <= row_len for b in begin)
    written = [0] * N
    for odd in (0, 1):
        # features a lane holds after its load (eight from the word in front of an odd row's piece on) and the shift by half a word,
        # which takes the eighth from the next lane's first word
        loaded = [[b // 2 - odd + i for i in range(8)] for b in begin]
        for lane in range(lanes):
            behind = loaded[lane + 1][0] if lane + 1 < lanes else None
            held = loaded[lane][odd:] + ([behind] if odd else [])
            for i in range(stores[lane] // 2):
                assert held[i] == begin[lane] // 2 + i, "lane %d stores feature %d from %s" % (lane, begin[lane] // 2 + i, held[i])
                written[begin[lane] // 2 + i] += 1
    assert written == [2] * N                           # (once a parity)


@pytest.mark.parametrize("lane_bytes,lanes,elem", [(2, 1, 2), (4, 1, 2), (4, 2, 2), (8, 2, 2), (16, 2, 2), (16, 4, 2), (16, 8, 2), (16, 16, 2), (16, 32, 2),
                                                   (4, 1, 4), (8, 1, 4), (8, 2, 4), (16, 4, 4), (16, 32, 4)])
def test_whole_rows_of_the_entry_kernels(ranges, lane_bytes, lanes, elem):
    for row_len in range(max(lane_bytes, lane_bytes * lanes // 2 + elem if lanes > 1 else lane_bytes), lane_bytes * lanes + 1, elem):
        covered = set()
        for lane in range(lanes):
            b, n = ranges.begin(lane, lane_bytes, row_len, 0), ranges.stores(lane, lane_bytes, row_len, 0)
            assert b + lane_bytes <= row_len
            covered.update(range(b, b + n))
        assert covered == set(range(row_len))


@pytest.mark.parametrize("N", range(1, 33))
def test_a_feature_of_the_narrow_kernels_is_one_waves(ranges, N):
    """Also where it is summed again, for which a wave reads what it has stored: not what another wave may not have."""
    odd = N % 2
    if N > ranges.end(1, odd):
        pytest.skip("more than two tiles")
    tiles = 1 if N <= ranges.end(0, odd) else 2
    stored = [f for t in range(tiles) for f in range(ranges.own(t, odd), min(N, ranges.end(t, odd)))]
    assert stored == list(range(N))
    for t in range(tiles):
        assert ranges.first(t, odd) <= ranges.own(t, odd) and ranges.end(t, odd) <= ranges.first(t, odd) + 16      # (what its lanes have)
        assert ranges.first(t, odd) % 2 == 0
