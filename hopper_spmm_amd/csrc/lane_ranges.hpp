// Which bytes of a row of C a lane of the entry kernels stores, and which features a wave of the narrow kernels: what must not overlap
// where two of them may hold different values.  Plain C++, so that it can be checked without a GPU.
#pragma once
#include <stdint.h>

namespace hspmm {

// A block of `row_len` bytes of a row of B (or C), `lane_bytes` a lane.  Lanes whose bytes would reach past the block's end are moved
// back to end with it; of an odd number of 16-bit elements (`odd`, lanes of 16 bytes) that is 14 bytes, seven features.
constexpr bool entry_lane_last(uint32_t lane, uint32_t lane_bytes, uint32_t row_len) { return lane * lane_bytes + lane_bytes > row_len; }

constexpr uint32_t entry_lane_begin(uint32_t lane, uint32_t lane_bytes, uint32_t row_len, bool odd)
{
    return !entry_lane_last(lane, lane_bytes, row_len) ? lane * lane_bytes : row_len - (odd ? 14u : lane_bytes);
}

// Bytes a lane stores, from where it begins.  Of even rows all it has: what it shares with a neighbour is the same sum in both.  Of odd
// rows, whose eighth feature comes from the neighbour's first word, the lane in front of the last only what that one does not (4, 8, 12
// or 16 bytes): its neighbour is moved back and does not begin 16 bytes further.
constexpr uint32_t entry_lane_stores(uint32_t lane, uint32_t lane_bytes, uint32_t row_len, bool odd)
{
    if (lane * lane_bytes >= row_len) return 0u;
    if (!odd) return lane_bytes;
    if (entry_lane_last(lane, lane_bytes, row_len)) return 14u;
    const uint32_t in_front = row_len - 14u - lane * 16u;
    return in_front < 16u ? in_front : 16u;
}

// Wave `tile` of a workgroup of the narrow kernels has sums of the features from narrow_tile_first on, 16 of an even N and 15 of an odd
// one, and stores those from narrow_tile_own to narrow_tile_end (less those behind the last one).  The second tile of an odd N begins
// with the first one's last feature, so that it, too, begins on a word.
constexpr uint32_t narrow_tile_first(uint32_t tile, bool odd) { return tile * (odd ? 14u : 16u); }
constexpr uint32_t narrow_tile_own(uint32_t tile, bool odd) { return tile * (odd ? 15u : 16u); }
constexpr uint32_t narrow_tile_end(uint32_t tile, bool odd) { return narrow_tile_first(tile, odd) + (odd ? 15u : 16u); }

}  // namespace hspmm
