// Plain tiles to bitmap tiles on the host (hspmm_pack.cpp).  The header words are those the gather kernels read
// (bitmap_header_from_caller in hspmm_create.hip writes the same from a caller's bitmaps): eight per 8 x 16 tile of
// 16-bit elements (elem = 2), four per 8 x 8 tile of 32-bit elements (elem = 4).
#pragma once
#include <cstddef>
#include <cstdint>

namespace hspmm_host {

// The masks and counts of n tiles; returns their number of stored elements (those whose bit pattern is not +0).
uint64_t tile_masks(const void *tiles, size_t n, uint32_t elem, uint32_t *header);
// The positions of n tiles' stored elements, which begin at `first`, to the header.
void place_tiles(uint32_t *header, size_t n, uint32_t elem, uint64_t first);
// The stored elements of n tiles to stored[first ..].
void pack_tiles(const void *tiles, size_t n, uint32_t elem, const uint32_t *header, uint64_t first, void *stored);

}  // namespace hspmm_host
