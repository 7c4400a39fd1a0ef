// What the full-tile and the wide-tile kernels share: reading second operands from LDS, and summing rows again where B is
// not finite.
#pragma once
#include "spmm_panel_kernel.hpp"

namespace hspmm {

typedef uint32_t t_u32x2 __attribute__((ext_vector_type(2)));
typedef u32x4 u32x4_any __attribute__((aligned(2)));
typedef t_u32x2 u32x2_any __attribute__((aligned(2)));

typedef tr16x4 __attribute__((address_space(3))) *tile_tr_ptr;
// First column of block b: the last block is moved back to end with the matrix (whose columns are kK at least), so that
// every row of B a chunk reads is there.
__host__ __device__ __forceinline__ uint32_t tile_first_column(uint32_t b, uint32_t kk, uint32_t cols)
{
    return b * kk + kk <= cols ? b * kk : cols - kk;
}

// Second-operand registers of 16 features and 32 rows of B: p addresses the lane's 8 bytes of the first 16 rows.
template <uint32_t PITCH>
__device__ __forceinline__ u32x4 tile_operand(const char *p)
{
    const __attribute__((address_space(3))) char *q = (const __attribute__((address_space(3))) char *)p;
    const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((tile_tr_ptr)q));
    const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((tile_tr_ptr)(q + 16 * PITCH)));
    u32x4 b;
    b[0] = lo[0]; b[1] = lo[1]; b[2] = hi[0]; b[3] = hi[1];
    return b;
}

// Element types as rows are summed again by.
template <bool BF> struct HalfStored {
    static constexpr uint32_t kElem = 2, kPerWord = 2;
    __device__ static __forceinline__ bool not_finite(uint32_t bits) { return (~bits & (BF ? 0x7F80u : 0x7C00u)) == 0u; }
    __device__ static __forceinline__ float value(uint32_t bits) { return (float)__builtin_bit_cast(typename HalfOps<BF>::elem_t, uint16_t(bits)); }
    // element i (of kPerWord) of a word of a tile
    __device__ static __forceinline__ uint32_t bits(uint32_t word, uint32_t i) { return i ? word >> 16 : word & 0xFFFFu; }
    __device__ static __forceinline__ uint32_t load_one(const char *p) { return *reinterpret_cast<const uint16_t *>(p); }
    __device__ static __forceinline__ void store_one(char *p, const float v) { *reinterpret_cast<uint16_t *>(p) = uint16_t(HalfOps<BF>::pack(v, 0.f)); }
};
struct FloatStored {
    static constexpr uint32_t kElem = 4, kPerWord = 1;
    __device__ static __forceinline__ bool not_finite(uint32_t bits) { return (~bits & 0x7F800000u) == 0u; }
    __device__ static __forceinline__ float value(uint32_t bits) { return __builtin_bit_cast(float, bits); }
    __device__ static __forceinline__ uint32_t bits(uint32_t word, uint32_t) { return word; }
    __device__ static __forceinline__ uint32_t load_one(const char *p) { return *reinterpret_cast<const uint32_t *>(p); }
    __device__ static __forceinline__ void store_one(char *p, const float v) { *reinterpret_cast<float *>(p) = v; }
};

// First effective window at or behind `row`.
__device__ __forceinline__ uint32_t first_window(const uint32_t *rowIdx, uint32_t n_windows, uint32_t row)
{
    uint32_t lo = 0, hi = n_windows;
    while (lo < hi) {
        const uint32_t mid = lo + (hi - lo) / 2u;
        if (rowIdx[mid] < row) lo = mid + 1u; else hi = mid;
    }
    return lo;
}

// fn(row in the block, column, element number) for every stored element of row block rb; a thread takes a tile column.
template <class E, class F>
__device__ __forceinline__ void for_entries(const TileSource &src, uint32_t row0, uint32_t rows, F fn)
{
    constexpr uint32_t CW = E::kElem == 4u ? 8u : 16u;
    const uint32_t w0 = first_window(src.rowIdx, src.n_windows, row0), w1 = first_window(src.rowIdx, src.n_windows, row0 + rows);
    for (uint32_t w = w0; w < w1; ++w) {
        const uint32_t m0 = src.rowIdx[w] - row0;
        const size_t c1 = size_t(src.rowOffset[w + 1u]) * CW;
        for (size_t c = size_t(src.rowOffset[w]) * CW + threadIdx.x; c < c1; c += blockDim.x) {
            const uint32_t id = src.a2b[c];
            if (id == kIdxMax) continue;
            const size_t first = (c / CW) * (8u * CW) + c % CW;
#pragma unroll
            for (uint32_t r = 0; r < 8u; ++r) {
                const size_t e = first + r * CW;
                const bool stored = E::kElem == 4u ? static_cast<const uint32_t *>(src.tiles)[e] != 0u : static_cast<const uint16_t *>(src.tiles)[e] != 0u;
                if (stored) fn(m0 + r, id, e);
            }
        }
    }
}

// Sums 16 RF rows x WIDTH features of C again, over the stored entries of the plan's tiles alone, where C is not finite: only
// rows that name a row of B then get what its infinities and NaNs make of them.  Features below `own` and from `end` on belong to other
// waves, which may still be storing them.
// A wave with its lanes on features, 64 / WIDTH tiles of a window at a time, two trips to memory each: slow, and off the path of
// finite data (bf16, 4096 x 11008 at 10 %, N = 16: 1.0 ms with an infinity in B, 17.3 us without, as before the check).
// FEW: fewer registers, a trip more per row of a tile.
template <class E, int RF, uint32_t WIDTH, bool FEW = false, class Args>
__device__ __forceinline__ void tile_sum_again(const Args &ta, const uint32_t row0, const uint32_t f0, const uint32_t own, const uint32_t end, const uint32_t lane)
{
    constexpr uint32_t kShares = 64u / WIDTH, CW = E::kElem == 4u ? 8u : 16u;
    const TileSource src = *ta.src;
    const uint32_t mine = lane % WIDTH, share = lane / WIDTH, f = f0 + mine, f_in = umin32(f, ta.N - 1u);
    const size_t row_bytes = size_t(ta.N) * E::kElem;
    const char *b_lane = static_cast<const char *>(ta.B) + size_t(f_in) * E::kElem;
    char *c_lane = static_cast<char *>(ta.C) + size_t(f_in) * E::kElem;
    wait_stores_acknowledged();
    bool found = false;
    for (uint32_t m = share; m < RF * 16u; m += kShares)
        if (row0 + m < ta.rows) found |= E::not_finite(E::load_one(c_lane + size_t(row0 + m) * row_bytes));
    const uint64_t lanes = __ballot(found && f >= own && f < umin32(end, ta.N));
    if (!lanes) return;
    bool again = false;
    for (uint32_t s = 0; s < kShares; ++s) again |= (lanes >> (s * WIDTH + mine)) & 1u;
    for (uint32_t q = 0; q < RF * 2u; ++q) {
        const uint32_t row = row0 + q * 8u;
        if (row >= ta.rows) return;
        const uint32_t w = first_window(src.rowIdx, src.n_windows, row);
        float sum[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) sum[r] = 0.f;
        const bool there = w < src.n_windows && src.rowIdx[w] == row;
        const uint32_t t1 = there ? src.rowOffset[w + 1u] : 0u;
        for (uint32_t t = there ? src.rowOffset[w] + share : 0u; t < t1; t += kShares) {
            const u32x4 *ids = reinterpret_cast<const u32x4 *>(src.a2b + size_t(t) * CW);
            const u32x4 *tile = reinterpret_cast<const u32x4 *>(static_cast<const char *>(src.tiles) + size_t(t) * 256u);
            u32x4 id[CW / 4u], a[FEW ? 2 : 16];
            uint32_t b[CW];
#pragma unroll
            for (uint32_t k = 0; k < CW / 4u; ++k) id[k] = ids[k];
            if constexpr (!FEW) {
#pragma unroll
                for (uint32_t k = 0; k < 16u; ++k) a[k] = tile[k];
            }
#pragma unroll
            for (uint32_t k = 0; k < CW; ++k) {
                const uint32_t at = id[k / 4u][k % 4u];             // (padding: nothing is stored there)
                b[k] = E::load_one(b_lane + size_t(at == kIdxMax ? id[0][0] : at) * row_bytes);
            }
#pragma unroll
            for (uint32_t r = 0; r < 8u; ++r) {
                if constexpr (FEW) { a[0] = tile[2u * r]; a[1] = tile[2u * r + 1u]; }
#pragma unroll
                for (uint32_t k = 0; k < CW; ++k) {
                    const uint32_t word = k / E::kPerWord, x = E::bits(a[(FEW ? 0u : 2u * r) + word / 4u][word % 4u], k % E::kPerWord);
                    if (x) sum[r] = __builtin_fmaf(E::value(x), E::value(b[k]), sum[r]);
                }
                __builtin_amdgcn_sched_barrier(0);                  // (registers: one row's elements at a time)
            }
        }
#pragma unroll
        for (int r = 0; r < 8; ++r) {
#pragma unroll
            for (uint32_t m = WIDTH; m < 64u; m <<= 1) sum[r] += __shfl_xor(sum[r], int(m));
            if (again && share == 0u && row + uint32_t(r) < ta.rows) E::store_one(c_lane + size_t(row + uint32_t(r)) * row_bytes, sum[r]);
        }
    }
}

}  // namespace hspmm
