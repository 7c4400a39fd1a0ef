// Plain tiles to bitmap tiles on the host (plan creation, hspmm_create.hip): which elements are stored, and the stored
// elements one after the other.  Host code only, compiled without a device pass: the masks are made with the host's
// vector instructions.
#include "hspmm_pack.hpp"
#include <cstring>
#if defined(__AVX2__)
#include <immintrin.h>
#endif

namespace hspmm_host {

namespace {

// bit i of the result: element i of the 32 at v is stored (any bit pattern but +0)
inline uint32_t mask32(const uint16_t *v)
{
#if defined(__AVX2__)
    const __m256i zero = _mm256_setzero_si256();
    const __m256i a = _mm256_cmpeq_epi16(_mm256_loadu_si256(reinterpret_cast<const __m256i *>(v)), zero);
    const __m256i b = _mm256_cmpeq_epi16(_mm256_loadu_si256(reinterpret_cast<const __m256i *>(v + 16)), zero);
    // (the pack works inside 128-bit halves: put its quarters back in order)
    const __m256i p = _mm256_permute4x64_epi64(_mm256_packs_epi16(a, b), 0xD8);
    return ~uint32_t(_mm256_movemask_epi8(p));
#else
    uint32_t m = 0;
    for (uint32_t i = 0; i < 32; ++i) m |= uint32_t(v[i] != 0) << i;
    return m;
#endif
}

inline uint32_t mask32(const uint32_t *v)
{
    uint32_t m = 0;
#if defined(__AVX2__)
    const __m256i zero = _mm256_setzero_si256();
    for (uint32_t q = 0; q < 4; ++q) {
        const __m256i e = _mm256_cmpeq_epi32(_mm256_loadu_si256(reinterpret_cast<const __m256i *>(v + 8 * q)), zero);
        m |= (~uint32_t(_mm256_movemask_ps(_mm256_castsi256_ps(e))) & 0xFFu) << (8 * q);
    }
#else
    for (uint32_t i = 0; i < 32; ++i) m |= uint32_t(v[i] != 0) << i;
#endif
    return m;
}

template <class V>
inline V *take(V *to, const V *tile, uint32_t mask)
{
    for (; mask; mask &= mask - 1) *to++ = tile[__builtin_ctz(mask)];
    return to;
}

}  // namespace

uint64_t tile_masks(const void *tiles, size_t n, uint32_t elem, uint32_t *header)
{
    uint64_t stored = 0;
    if (elem == 2u) {
        const uint16_t *v = static_cast<const uint16_t *>(tiles);
        for (size_t t = 0; t < n; ++t, v += 128, header += 8) {
            uint32_t seen = 0, counts = 0;
            for (uint32_t q = 0; q < 4; ++q) {
                header[q] = mask32(v + 32 * q);
                if (q) counts |= seen << (8 * q);
                seen += uint32_t(__builtin_popcount(header[q]));
            }
            header[4] = counts;
            header[6] = header[7] = 0;
            stored += seen;
        }
    } else {
        const uint32_t *v = static_cast<const uint32_t *>(tiles);
        for (size_t t = 0; t < n; ++t, v += 64, header += 4) {
            header[0] = mask32(v);
            header[1] = mask32(v + 32);
            header[3] = uint32_t(__builtin_popcount(header[0])) + uint32_t(__builtin_popcount(header[1]));
            stored += header[3];
        }
    }
    return stored;
}

void place_tiles(uint32_t *header, size_t n, uint32_t elem, uint64_t first)
{
    uint32_t at = uint32_t(first);
    for (size_t t = 0; t < n; ++t) {
        if (elem == 2u) {
            header[5] = at;
            at += (header[4] >> 24) + uint32_t(__builtin_popcount(header[3]));     // (in front of the last word, in it)
            header += 8;
        } else {
            header[2] = at;
            at += header[3];
            header += 4;
        }
    }
}

void pack_tiles(const void *tiles, size_t n, uint32_t elem, const uint32_t *header, uint64_t first, void *stored)
{
    if (elem == 2u) {
        const uint16_t *v = static_cast<const uint16_t *>(tiles);
        uint16_t *to = static_cast<uint16_t *>(stored) + first;
        for (size_t t = 0; t < n; ++t, v += 128, header += 8)
            for (uint32_t q = 0; q < 4; ++q) to = take(to, v + 32 * q, header[q]);
    } else {
        const uint32_t *v = static_cast<const uint32_t *>(tiles);
        uint32_t *to = static_cast<uint32_t *>(stored) + first;
        for (size_t t = 0; t < n; ++t, v += 64, header += 4) to = take(take(to, v, header[0]), v + 32, header[1]);
    }
}

}  // namespace hspmm_host
