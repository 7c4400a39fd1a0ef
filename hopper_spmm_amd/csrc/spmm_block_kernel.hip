// Kernels for few features of weights kept in 16 x 16 blocks: C = A * B by whole blocks, read where a plan's tiles lie (the
// reference's 8-row windows, src/utils/class.h:74-85): two windows with one column list are the halves of a row of blocks.
//
// The gather kernels (spmm_mfma_kernel.hpp), which take any column list, load a row of B at a time, in words: with 16 features a
// quarter of what a compute unit's address path could bring.  The columns of a block are neighbours: its rows of B are one stretch of memory.
#include "spmm_tile_common.hpp"

namespace hspmm {

// A workgroup has a unit (16 rows; 8 where a window is alone), its W waves take the unit's blocks in turn, two at a time: 32 columns are one
// matrix instruction per 16 features.  A lane loads eight columns of a row of A as they lie in the tile; the blocks' 32 rows of B go through
// LDS, a wave's own, without a barrier, and come back transposed.  The waves' sums are added at the end, in LDS and in order.
// What bounds it: bytes that come into a compute unit, 65 to 85 KB a microsecond, and in the largest matrices the tiles' way from memory:
// 4096 x 14336 at 50 %, fp16, N = 16 11.3 us (59 MB of tiles; 15.4 by the gather kernels), 32 12.3 (15.2), 64 17.8 (20.5); 4096^2 at 50 %, N = 16
// 5.5 (8.9), 64 8.1 (11.4); 14336 x 4096, bf16, N = 16 12 (16.2); 16000 x 1111 at 25 %, N = 16 4.9 (8.1); three matrices in turn each.
// 160 matrices of 20 to 60 % of blocks: 1.4 to 2.7 times as fast up to 32 features, 1.2 to 1.7 from 33 on.  Sixteen waves, or four, are
// slower on the mean (0.93); with registers for eight waves a SIMD instead of six a wave asks for less at a time (N <= 16: 0.92).
// Narrow: fewer than eight features; a piece holds what is behind its row, too.
// Odd: rows of B of an odd number of elements, B on a word.  Every other row begins between two words, and loads that are not whole words
// take twice their time: such a row's pieces are loaded from the word before on and shifted by half a word, the element behind a piece
// coming from the next lane's.  The last piece of a row then has seven features.  (N = 9 .. 15 1.67 -> 1.9 times the gather kernels' speed, 17 .. 31
// 1.13 -> 1.56; of three tiles of features on the wide-tile kernels are as fast.)
template <bool BF, int CF, int W, bool Odd, bool Narrow>
__global__ __launch_bounds__(64 * W, CF <= 2 ? 6 : 2) void spmm_block_kernel(const BlockArgs ba)
{
    typedef HalfStored<BF> E;
    constexpr uint32_t kPitch = CF * 32u + (CF % 2 ? 0u : 32u), kImage = 32u * kPitch;      // of a wave
    constexpr int kAhead = 3;
    static_assert(kImage >= CF * 1024u, "a wave's sums take its image's place");
    static_assert(!Odd || 64u % (2u * CF) == 0u, "the pieces of a row in one wave's lanes");
    __shared__ __attribute__((aligned(16))) char smem[W * kImage];
    __shared__ uint32_t not_finite;

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, j = lane & 15u;
    const BlockUnit unit = ba.units[blockIdx.x];
    const uint32_t rows_here = unit.lower != kIdxMax ? 16u : 8u;
    const size_t row_bytes = size_t(ba.N) * 2u;
    if (tid == 0u) not_finite = 0u;

    // this lane's pieces of the rows of B: 16 bytes, features 8 h .. 8 h + 7 (the last piece of a row is moved back to end with it, or one behind)
    constexpr uint32_t kLanes = 2u * CF;      // of a row
    constexpr int kPieces = int(kLanes / 2u);
    const uint32_t n_halves = (ba.N + 7u) / 8u;
    uint32_t row_of[kPieces], feature_of[kPieces], image_off[kPieces];
    bool last_of[kPieces];
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
        const uint32_t n = uint32_t(i) * 64u + lane, h = umin32(n % kLanes, n_halves - 1u);
        row_of[i] = n / kLanes;
        last_of[i] = h + 1u == n_halves;
        feature_of[i] = Odd ? (last_of[i] ? ba.N - 7u : 8u * h) : Narrow ? 0u : umin32(8u * h, ba.N - 8u);
        image_off[i] = row_of[i] * kPitch + h * 16u;
    }
    const uint32_t behind = Odd ? (8u * n_halves - 1u - ba.N) / 2u : 0u;      // word of the last piece that begins with what the piece before needs
    char *const image = smem + wave * kImage;
    const char *const b_lane = image + (8u * g + (j >> 2)) * kPitch + (j & 3u) * 8u;
    const bool upper = j < 8u, a_there = upper || rows_here == 16u;
    const char *const a_lane = static_cast<const char *>(ba.tiles) + size_t(upper || rows_here == 8u ? unit.upper : unit.lower) * 256u + (j & 7u) * 32u + (g & 1u) * 16u;
    const char *const B = static_cast<const char *>(ba.B);

    f32x4 acc[CF];
#pragma unroll
    for (int c = 0; c < CF; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint32_t pairs = (unit.steps + 1u) >> 1;
    for (uint32_t q0 = wave; q0 < pairs; q0 += 64u * W) {           // (64 pairs of column numbers at a time, one a lane)
        const uint32_t n = umin32((pairs - q0 + W - 1u) / W, 64u);
        const u32x2 mine = reinterpret_cast<const u32x2 *>(ba.columns)[unit.pair_begin + umin32(q0 + lane * W, pairs - 1u)];
        u32x4 a[kAhead], b[kAhead][kPieces];
        uint32_t odds[kAhead];
        auto request_a = [&](auto slot, uint32_t i) __attribute__((always_inline)) {
            constexpr int S = decltype(slot)::value;
            const uint32_t step = 2u * (q0 + umin32(i, n - 1u) * W) + (g >> 1);
            a[S] = *reinterpret_cast<const u32x4 *>(a_lane + size_t(umin32(step, unit.steps - 1u)) * 256u);
            if (!a_there || step >= unit.steps) a[S] = u32x4{0u, 0u, 0u, 0u};
        };
        auto request_b = [&](auto slot, uint32_t i) __attribute__((always_inline)) {
            constexpr int S = decltype(slot)::value;
            const int at = int(umin32(i, n - 1u));
            const uint32_t first = __builtin_amdgcn_readlane(mine[0], at), second = __builtin_amdgcn_readlane(mine[1], at);
            odds[S] = 0u;
#pragma unroll
            for (int k = 0; k < kPieces; ++k) {
                // (a block that ends behind the last column: that row of B, which zeros multiply)
                const uint32_t row = umin32((row_of[k] < 16u ? first : second) + (row_of[k] & 15u), ba.cols - 1u);
                // (nothing behind B is read)
                const uint32_t odd = Odd ? (last_of[k] && row == ba.cols - 1u ? 1u : row & 1u) : 0u;
                odds[S] |= odd << k;
                const char *from = B + (row * uint32_t(row_bytes) + (feature_of[k] - odd) * 2u);
                if (Narrow && (ba.cols - row) * ba.N < 8u) {
                    const uint16_t *one = reinterpret_cast<const uint16_t *>(from);
                    u32x4 v{0u, 0u, 0u, 0u};
#pragma unroll
                    for (uint32_t e = 0; e < 7u; ++e)
                        if (e < ba.N) v[e / 2u] |= uint32_t(one[e]) << e % 2u * 16u;
                    b[S][k] = v;
                } else {
                    b[S][k] = *reinterpret_cast<const u32x4_any *>(from);
                }
            }
        };
        auto multiply = [&](auto slot, uint32_t i) __attribute__((always_inline)) {
            constexpr int S = decltype(slot)::value;
#pragma unroll
            for (int k = 0; k < kPieces; ++k) {
                u32x4 v = b[S][k];
                if constexpr (Odd) {
                    const uint32_t mine = !last_of[k] || behind == 0u ? v[0] : behind == 1u ? v[1] : behind == 2u ? v[2] : v[3], by = (odds[S] >> k & 1u) * 16u;
                    const uint32_t next = uint32_t(__builtin_amdgcn_mov_dpp(int(mine), 0x130, 0xF, 0xF, true));     // (the next lane's)
                    v[0] = __builtin_amdgcn_alignbit(v[1], v[0], by);
                    v[1] = __builtin_amdgcn_alignbit(v[2], v[1], by);
                    v[2] = __builtin_amdgcn_alignbit(v[3], v[2], by);
                    v[3] = __builtin_amdgcn_alignbit(next, v[3], by);
                }
                *reinterpret_cast<u32x4 *>(image + image_off[k]) = v;
            }
            request_b(slot, i + kAhead);
            asm volatile("" ::: "memory");
            u32x4 op[CF];
#pragma unroll
            for (int c = 0; c < CF; ++c) {
                const __attribute__((address_space(3))) char *p = (const __attribute__((address_space(3))) char *)(b_lane + c * 32);
                const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((tile_tr_ptr)p));
                const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((tile_tr_ptr)(p + 4 * kPitch)));
                op[c][0] = lo[0]; op[c][1] = lo[1]; op[c][2] = hi[0]; op[c][3] = hi[1];
            }
            asm volatile("" ::: "memory");
#pragma unroll
            for (int c = 0; c < CF; ++c) acc[c] = HalfOps<BF>::mfma(a[S], op[c], acc[c]);
            request_a(slot, i + kAhead);
        };
        typedef std::integral_constant<int, 0> S0;
        typedef std::integral_constant<int, 1> S1;
        typedef std::integral_constant<int, 2> S2;
        request_a(S0{}, 0); request_b(S0{}, 0);
        request_a(S1{}, 1); request_b(S1{}, 1);
        request_a(S2{}, 2); request_b(S2{}, 2);
        uint32_t i = 0;
        for (; i + 3u <= n; i += 3u) { multiply(S0{}, i); multiply(S1{}, i + 1u); multiply(S2{}, i + 2u); }
        if (i < n) multiply(S0{}, i);
        if (i + 1u < n) multiply(S1{}, i + 1u);
    }

    // lane (g, j) has rows 4 g .. 4 g + 3 of feature j
    float *const sums = reinterpret_cast<float *>(image);
#pragma unroll
    for (int c = 0; c < CF; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) sums[(c * 4 + e) * 64 + lane] = acc[c][e];
    __syncthreads();
    char *const C = static_cast<char *>(ba.C);
    for (uint32_t t = tid; t < 128u * CF; t += 64u * W) {
        const uint32_t two = t & 7u, r = t >> 3 & 15u, c = t >> 7, h = 2u * c + (two >> 2);
        const uint32_t begin = Odd && h + 1u == n_halves ? ba.N - 7u : Narrow ? 0u : umin32(8u * h, ba.N - 8u), feature = begin + 2u * (two & 3u), row = unit.row + r;
        const float *in = reinterpret_cast<const float *>(smem) + (c * 4u + (r & 3u)) * 64u + (r >> 2) * 16u + 2u * two;
        float x = 0.f, y = 0.f;
#pragma unroll
        for (int w = 0; w < W; ++w) { x += in[w * (kImage / 4u)]; y += in[w * (kImage / 4u) + 1u]; }
        if (r < rows_here && row < ba.rows && 8u * h < ba.N && feature < ba.N) {
            const uint32_t word = HalfOps<BF>::pack(x, y);
            char *to = C + size_t(row) * row_bytes + feature * 2u;
            typedef uint32_t word_any __attribute__((aligned(2)));
            const bool first = feature >= 8u * h, second = feature + 1u >= 8u * h && feature + 1u < ba.N;
            if (first && second) *reinterpret_cast<word_any *>(to) = word;
            else if (first) *reinterpret_cast<uint16_t *>(to) = uint16_t(word);
            else if (second) *reinterpret_cast<uint16_t *>(to + 2) = uint16_t(word >> 16);
            if ((first && !(x * 0.f == 0.f)) || (second && !(y * 0.f == 0.f))) not_finite = 1u;
        }
    }
    // rows of windows without entries: in front of the first unit, and behind each
    for (uint32_t range = blockIdx.x ? 1u : 0u; range < 2u; ++range) {
        const uint32_t from = range ? unit.row + rows_here : 0u, to = umin32(range ? unit.next_row : unit.row, ba.rows);
        if (from < to)
            for (size_t at = size_t(from) * ba.N + tid; at < size_t(to) * ba.N; at += 64u * W) reinterpret_cast<uint16_t *>(C)[at] = 0u;
    }
    // An infinity or a NaN in B makes the sums of its feature NaN in every row of blocks that holds its row, since blocks hold zeros too: such
    // sums once more, over the stored entries alone (a finite sum has met neither).
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (not_finite) {
        BlockArgs again = ba;
        again.rows = umin32(ba.rows, unit.row + rows_here);
        for (uint32_t f = wave * 16u; f < ba.N; f += W * 16u) tile_sum_again<E, 1, 16, true>(again, unit.row, f, f, umin32(ba.N, f + 16u), lane);
    }
}

// The same of fp32 storage, in fp32 products: a unit's steps are eight columns, two of them four matrix instructions per 16 features.  Their
// second operands are a feature of four rows of B, which lanes load as they lie: lane (g, j) the features V j .. V j + V - 1.
// What bounds it: the tiles' way from memory, and for 64 features the matrix instructions (32 cycles each).  us, three matrices in turn, by the
// gather or LDS-panel kernels / here: 4096 x 14336 at 50 %, N = 8 36.0 / 33.7, 15 47.1 / 33.6, 33 79.7 / 54.3; 4096^2 at 50 %, N = 16 15.1 / 10.2,
// 32 14.9 / 11.6, 47 39.0 / 17.9; 16000 x 1111 at 25 %, N = 16 12.2 / 8.7.
template <int V, int W>
__global__ __launch_bounds__(64 * W, 2) void spmm_block_f32_kernel(const BlockArgs ba)
{
    constexpr int kAhead = 3;
    typedef float floats __attribute__((ext_vector_type(4)));
    __shared__ float smem[W * V * 256];
    __shared__ uint32_t not_finite;

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, j = lane & 15u;
    const BlockUnit unit = ba.units[blockIdx.x];
    const uint32_t rows_here = unit.lower != kIdxMax ? 16u : 8u;
    const size_t row_bytes = size_t(ba.N) * 4u;
    if (tid == 0u) not_finite = 0u;

    const uint32_t features = umin32(uint32_t(V) * j, ba.N - V) * 4u;       // (lanes behind the last feature are moved back to end with the row)
    const bool upper = j < 8u, a_there = upper || rows_here == 16u;
    const char *const a_lane = static_cast<const char *>(ba.tiles) + size_t(upper || rows_here == 8u ? unit.upper : unit.lower) * 256u + (j & 7u) * 32u + (g & 1u) * 16u;
    const char *const B = static_cast<const char *>(ba.B) + features;

    f32x4 acc[V];
#pragma unroll
    for (int c = 0; c < V; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint32_t pairs = (unit.steps + 1u) >> 1;
    for (uint32_t q0 = wave; q0 < pairs; q0 += 64u * W) {
        const uint32_t n = umin32((pairs - q0 + W - 1u) / W, 64u);
        const u32x2 mine = reinterpret_cast<const u32x2 *>(ba.columns)[unit.pair_begin + umin32(q0 + lane * W, pairs - 1u)];
        floats a[kAhead];
        float b[kAhead][4][V];
        auto request = [&](auto slot, uint32_t i) __attribute__((always_inline)) {
            constexpr int S = decltype(slot)::value;
            const uint32_t at = umin32(i, n - 1u), step = 2u * (q0 + at * W) + (g >> 1);
            a[S] = *reinterpret_cast<const floats *>(a_lane + size_t(umin32(step, unit.steps - 1u)) * 256u);
            if (!a_there || step >= unit.steps) a[S] = floats{0.f, 0.f, 0.f, 0.f};
            const uint32_t first = __builtin_amdgcn_readlane(mine[0], int(at)), second = __builtin_amdgcn_readlane(mine[1], int(at));
            const uint32_t column = (g < 2u ? first : second) + (g & 1u) * 4u;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const char *from = B + umin32(column + k, ba.cols - 1u) * uint32_t(row_bytes);      // (behind the last column: zeros multiply it)
                if constexpr (V == 1) {
                    b[S][k][0] = *reinterpret_cast<const float *>(from);
                } else {
                    typedef float some __attribute__((ext_vector_type(V), aligned(4)));
                    const some x = *reinterpret_cast<const some *>(from);
#pragma unroll
                    for (int c = 0; c < V; ++c) b[S][k][c] = x[c];
                }
            }
        };
        auto multiply = [&](auto slot, uint32_t i) __attribute__((always_inline)) {
            constexpr int S = decltype(slot)::value;
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int c = 0; c < V; ++c) acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[S][k], b[S][k][c], acc[c], 0, 0, 0);
            request(slot, i + kAhead);
        };
        typedef std::integral_constant<int, 0> S0;
        typedef std::integral_constant<int, 1> S1;
        typedef std::integral_constant<int, 2> S2;
        request(S0{}, 0); request(S1{}, 1); request(S2{}, 2);
        uint32_t i = 0;
        for (; i + 3u <= n; i += 3u) { multiply(S0{}, i); multiply(S1{}, i + 1u); multiply(S2{}, i + 2u); }
        if (i < n) multiply(S0{}, i);
        if (i + 1u < n) multiply(S1{}, i + 1u);
    }

    // lane (g, j) has rows 4 g .. 4 g + 3 of its features
#pragma unroll
    for (int c = 0; c < V; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) smem[(wave * V + c) * 256 + e * 64 + lane] = acc[c][e];
    __syncthreads();
    float *const C = static_cast<float *>(ba.C);
    for (uint32_t t = tid; t < 256u * V; t += 64u * W) {
        const uint32_t r = t / (16u * V), of = t % (16u * V) / V, c = t % V, feature = umin32(V * of, ba.N - V) + c, row = unit.row + r;
        float x = 0.f;
#pragma unroll
        for (int w = 0; w < W; ++w) x += smem[(w * V + c) * 256 + (r & 3u) * 64 + (r >> 2) * 16 + of];
        if (r < rows_here && row < ba.rows && V * of < ba.N && feature >= V * of) {
            C[size_t(row) * ba.N + feature] = x;
            if (!(x * 0.f == 0.f)) not_finite = 1u;
        }
    }
    for (uint32_t range = blockIdx.x ? 1u : 0u; range < 2u; ++range) {
        const uint32_t from = range ? unit.row + rows_here : 0u, to = umin32(range ? unit.next_row : unit.row, ba.rows);
        if (from < to)
            for (size_t at = size_t(from) * ba.N + tid; at < size_t(to) * ba.N; at += 64u * W) C[at] = 0.f;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (not_finite) {
        BlockArgs again = ba;
        again.rows = umin32(ba.rows, unit.row + rows_here);
        for (uint32_t f = wave * 16u; f < ba.N; f += W * 16u) tile_sum_again<FloatStored, 1, 16, true>(again, unit.row, f, f, umin32(ba.N, f + 16u), lane);
    }
}

hipError_t launch_spmm_block(int dtype, const BlockArgs &ba, uint32_t n_units, hipStream_t s)
{
    if (!n_units || n_units >= (1u << 22) || !ba.N || ba.N > 64u || !ba.cols || uint64_t(ba.cols) * ba.N * (dtype == kDtypeF32 ? 4u : 2u) > (1ull << 32)) return hipErrorInvalidValue;
    const uint32_t blocks = (ba.N + 15u) / 16u;
    const bool odd = ba.N % 2u && ba.N > 8u && reinterpret_cast<uintptr_t>(ba.B) % 4u == 0u;
#define HSPMM_BLOCK(CF, BF, ODD, NARROW) { spmm_block_kernel<BF, CF, 8, ODD, NARROW><<<dim3(n_units), 512, 0, s>>>(ba); return hipGetLastError(); }
#define HSPMM_BLOCKS(CF) \
    if (blocks == CF && dtype == kDtypeF16) HSPMM_BLOCK(CF, false, false, false) \
    if (blocks == CF && dtype == kDtypeBf16) HSPMM_BLOCK(CF, true, false, false)
#define HSPMM_BLOCKS_ODD(CF) \
    if (odd && blocks == CF && dtype == kDtypeF16) HSPMM_BLOCK(CF, false, true, false) \
    if (odd && blocks == CF && dtype == kDtypeBf16) HSPMM_BLOCK(CF, true, true, false)
    if (dtype == kDtypeF32) {
        if (ba.N <= 16u) spmm_block_f32_kernel<1, 8><<<dim3(n_units), 512, 0, s>>>(ba);
        else if (ba.N <= 32u) spmm_block_f32_kernel<2, 8><<<dim3(n_units), 512, 0, s>>>(ba);
        else spmm_block_f32_kernel<4, 8><<<dim3(n_units), 512, 0, s>>>(ba);
        return hipGetLastError();
    }
    if (ba.N < 8u && dtype == kDtypeF16) HSPMM_BLOCK(1, false, false, true)
    if (ba.N < 8u && dtype == kDtypeBf16) HSPMM_BLOCK(1, true, false, true)
    HSPMM_BLOCKS_ODD(1) HSPMM_BLOCKS_ODD(2) HSPMM_BLOCKS(1) HSPMM_BLOCKS(2) HSPMM_BLOCKS(3) HSPMM_BLOCKS(4)
#undef HSPMM_BLOCKS_ODD
#undef HSPMM_BLOCKS
#undef HSPMM_BLOCK
    return hipErrorInvalidValue;
}

}  // namespace hspmm
