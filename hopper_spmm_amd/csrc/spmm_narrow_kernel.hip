// Kernels for up to 32 features of matrices that are sparse in storage but dense to a workgroup (weights pruned to some per cent), 16-bit
// types: C = A * B by full operands of A, which every wave puts together from stored entries, and the kernels that make the stream they
// read from a plan's tiles (the reference's 8-row windows, src/utils/class.h:74-85) on the device.
//
// With few features what counts is that every compute unit starts at once and none waits for another: the full-tile kernels
// (spmm_tile_kernel.hip) share a C tile of 128 rows between workgroups, whose sums then go through memory, and put blocks together behind
// barriers (13 us of every launch); the entry kernels read a row of B for every entry.
#include "spmm_tile_common.hpp"
#include "lane_ranges.hpp"

namespace hspmm {

constexpr uint32_t kNarrowRows = 16, kNarrowImage = 4096;

// A block's image of 4 KB: operand by operand of matrix instructions, 1 KB each, 16 bytes a lane; lane (g, m) holds elements of row m.
// 16-bit types.  A load of B brings eight rows, two features a lane, and lanes of two rows exchange so that each has one feature of both.
// Where N is odd, every other row starts between two words: its lanes take features 2 q - 1 and 2 q instead of 2 q and 2 q + 1 (loads that
// are not whole words cost twice their time: 4096 x 11008 at 10 %, N = 15 14.6 us, 16 9.1), and a tile has 15 features.
template <bool BF, bool ODD> struct NarrowHalf : HalfStored<BF> {
    static constexpr uint32_t kColumns = kNarrowColumns, kStep = 32, kLoads = 4, kLoadRows = 8;     // of an operand: columns, loads of B; rows of one
    static constexpr bool kOdd = ODD;
    __device__ static __forceinline__ uint32_t position(uint32_t m, uint32_t k)
    {
        return k / 32u * 1024u + ((k >> 1 & 3u) * 16u + m) * 16u + ((k >> 3 & 3u) * 2u + (k & 1u)) * 2u;
    }
    __device__ static __forceinline__ uint32_t load_row(uint32_t lane) { return lane >> 3; }
    // (features behind the last one: the last ones)
    __device__ static __forceinline__ int load_feature(uint32_t lane, uint32_t f0, uint32_t N)
    {
        return ODD ? int(umin32(f0 + (lane & 7u) * 2u, N - 1u)) - int(lane >> 3 & 1u) : int(umin32(f0 + (lane & 7u) * 2u, N - 2u));
    }
    __device__ static __forceinline__ uint32_t feature(uint32_t lane)           // of sums (none: far behind the last)
    {
        const uint32_t q = lane & 7u, odd = lane >> 3 & 1u;
        return ODD ? (odd ? (q ? q * 2u - 1u : 1u << 30) : q * 2u) : q * 2u + odd;
    }
    __device__ static __forceinline__ uint32_t selector(uint32_t lane) { return ODD ? (lane & 8u ? 0x01000706u : 0x07060100u) : lane & 8u ? 0x03020706u : 0x05040100u; }
    // whether a load reaches beyond its row, which the last one must not
    static constexpr uint32_t kBeyond = ODD ? 1 : 0;
    __device__ static __forceinline__ uint32_t load_b(const char *p)
    {
        typedef uint32_t word_any __attribute__((aligned(2)));
        return *reinterpret_cast<const word_any *>(p);
    }
    __device__ static __forceinline__ uint32_t load_last(const NarrowArgs &na, uint32_t row, int f)
    {
        // (rows behind the last one, which A's operands multiply by zero: that row)
        const int64_t at = (int64_t(umin32(row, na.cols - 1u)) * na.N + f) * 2, last = int64_t(na.cols) * na.N * 2 - 4;
        if (!ODD) return load_b(static_cast<const char *>(na.B) + at);
        const uint32_t x = load_b(static_cast<const char *>(na.B) + (at < 0 ? 0 : at > last ? last : at));
        return at > last ? x >> 16 : x;
    }
    struct Entries { t_u32x2 e; };                          // two: position | value << 16
    __device__ static __forceinline__ void load(Entries &x, const NarrowArgs &na, size_t first, uint32_t i)
    {
        x.e = *reinterpret_cast<const t_u32x2 *>(na.entries + first * 4u + i);
    }
    __device__ static __forceinline__ void scatter(char *image, const Entries &x)
    {
#pragma unroll
        for (int i = 0; i < 2; ++i) *reinterpret_cast<uint16_t *>(image + (x.e[i] & 0xFFFFu)) = uint16_t(x.e[i] >> 16);
    }
    __device__ static __forceinline__ f32x4 multiply(const u32x4 a, const uint32_t (&b)[kLoads], uint32_t sel, f32x4 acc)
    {
        u32x4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            int other = __builtin_amdgcn_mov_dpp(int(b[i]), 0x128, 0xF, 0xF, true);                             // the lane eight away
            if (ODD) other = __builtin_amdgcn_update_dpp(other, int(b[i]), 0x129, 0xF, 0xC, false);             // upper eight: nine below
            o[i] = __builtin_amdgcn_perm(uint32_t(other), b[i], sel);
        }
        return HalfOps<BF>::mfma(a, o, acc);
    }
};

// A workgroup of W waves multiplies 16 rows of A with CF tiles of features; a wave takes every W-th block of 128 columns by itself, without
// a barrier: it scatters the block's entries (CAP x 128 of them asked for two blocks earlier; more are loaded when their turn comes) into
// its image in LDS, reads the image back as first operands, clears it, and multiplies it with B's rows, which come straight into
// registers, asked for a block earlier.  The waves' sums are added in LDS at the end, always in the same order.  (LDS serves the
// requests of a wave in order.)
// What bounds it: the loads of a block - 16 of B, 2 words a lane CAP times for entries -, which keep the L1's return path busy for 54 %
// of a launch (4096 x 11008 at 10 %, N = 16), and 3 us of launch and first loads.  With B in loads of one 16-bit feature, 32 of
// them a block, that took 11.0 us instead of 9.1, and N = 32 16.2 instead of 12.9; with B in 16-byte pieces, 4 a block, through LDS
// and its transposing reads 11.1.
// Measured, bf16 (this / the full-tile kernels, the entry kernels (e) or the gather kernels (g), us): 4096 x 11008 at 10 %, N = 1 9.3 / 11.7 e,
// 8 8.9 / 15.3 e, 15 9.3 / 18.8, 16 9.1 / 17.1, 32 12.9 / 19.8;  11008 x 4096 at 30 %, N = 7 14.4 / 38.5 e, 16 14.1 / 18.6;  1500 x 9001 at 30 %,
// N = 15 10.6 / 26.9 g, 29 13.0 / 19.1.  1994 launches of N = 1 to 32 with 2.5 to 30 %: 1.23 times the entry kernels' speed on the launches
// taken from them and those left, 1.75 the gather kernels', 1.39 the full-tile kernels'.
template <class E, int CF, int CAP, int W>
__global__ __launch_bounds__(64 * W, 4)
void spmm_narrow_kernel(const NarrowArgs na)
{
    constexpr int kOps = E::kColumns / E::kStep;
    __shared__ __attribute__((aligned(16))) char smem[W * kNarrowImage];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t unit = blockIdx.x, row0 = unit * kNarrowRows, g = lane >> 4;
    const uint32_t row_bytes = na.N * E::kElem;
    char *const image = smem + wave * kNarrowImage;
    f32x4 acc[CF];
#pragma unroll
    for (int p = 0; p < CF; ++p) acc[p] = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint32_t mine = na.n_blocks > wave ? (na.n_blocks - wave + W - 1u) / W : 0u;         // blocks wave, wave + W, ...
    if (mine) {
        // lane i: the first four entries of the wave's block i, and of what comes behind it
        const uint32_t *at = na.blocks + size_t(unit) * na.n_blocks + umin32(wave + lane * W, na.n_blocks - 1u);
        const uint32_t starts = at[0], ends = at[1];
        typename E::Entries x[2][CAP];
        uint32_t b[kOps][CF][E::kLoads];
        auto request = [&](auto set_c, uint32_t i) __attribute__((always_inline)) {
            constexpr int S = decltype(set_c)::value;
            i = umin32(i, mine - 1u);
            const uint32_t first = __builtin_amdgcn_readlane(starts, i), most = (__builtin_amdgcn_readlane(ends, i) - first) * 4u - 2u;
#pragma unroll
            for (int c = 0; c < CAP; ++c) E::load(x[S][c], na, first, umin32(c * 128u + lane * 2u, most));
        };
        const uint32_t sel = E::selector(lane);
        int lane_f[CF];
        uint32_t lane_b[CF];
#pragma unroll
        for (int p = 0; p < CF; ++p) {
            lane_f[p] = E::load_feature(lane, narrow_tile_first(p, E::kOdd), na.N);
            lane_b[p] = E::load_row(lane) * row_bytes + uint32_t(lane_f[p]) * E::kElem;
        }
        auto request_b = [&](auto op_c, uint32_t i) __attribute__((always_inline)) {
            constexpr int O = decltype(op_c)::value;
            const uint32_t k0 = (umin32(i, mine - 1u) * W + wave) * E::kColumns + O * E::kStep;
            if (k0 + E::kStep + E::kBeyond <= na.cols) {
                const char *p = static_cast<const char *>(na.B) + size_t(k0) * row_bytes;
#pragma unroll
                for (uint32_t l = 0; l < E::kLoads; ++l, p += E::kLoadRows * size_t(row_bytes))
#pragma unroll
                    for (int q = 0; q < CF; ++q) b[O][q][l] = E::load_b(p + lane_b[q]);
            } else {
#pragma unroll
                for (uint32_t l = 0; l < E::kLoads; ++l)
#pragma unroll
                    for (int q = 0; q < CF; ++q) b[O][q][l] = E::load_last(na, k0 + E::kLoadRows * l + E::load_row(lane), lane_f[q]);
            }
        };
        typedef std::integral_constant<int, 0> I0;
        typedef std::integral_constant<int, 1> I1;
        typedef std::integral_constant<int, 2> I2;
        typedef std::integral_constant<int, 3> I3;
        request(I0{}, 0u);
        request(I1{}, 1u);
        request_b(I0{}, 0u); request_b(I1{}, 0u); request_b(I2{}, 0u); request_b(I3{}, 0u);
#pragma unroll
        for (int o = 0; o < kOps; ++o) *reinterpret_cast<u32x4 *>(image + o * 1024 + lane * 16u) = u32x4{0u, 0u, 0u, 0u};
        asm volatile("" ::: "memory");
        auto step = [&](auto set_c, uint32_t i) __attribute__((always_inline)) {
            constexpr int S = decltype(set_c)::value;
            const uint32_t first = __builtin_amdgcn_readlane(starts, i), n = (__builtin_amdgcn_readlane(ends, i) - first) * 4u;
#pragma unroll
            for (int c = 0; c < CAP; ++c) E::scatter(image, x[S][c]);
            for (uint32_t c = CAP * 128u; c < n; c += 128u) {
                typename E::Entries more;
                E::load(more, na, first, umin32(c + lane * 2u, n - 2u));
                E::scatter(image, more);
            }
            asm volatile("" ::: "memory");                          // (entries and operands are of different types)
            request(set_c, i + 2u);
            u32x4 a[kOps];
#pragma unroll
            for (int o = 0; o < kOps; ++o) {
                u32x4 *p = reinterpret_cast<u32x4 *>(image + o * 1024 + lane * 16u);
                a[o] = *p;
                *p = u32x4{0u, 0u, 0u, 0u};
            }
            asm volatile("" ::: "memory");
            auto op = [&](auto op_c) __attribute__((always_inline)) {
                constexpr int O = decltype(op_c)::value;
#pragma unroll
                for (int q = 0; q < CF; ++q) acc[q] = E::multiply(a[O], b[O][q], sel, acc[q]);
                request_b(op_c, i + 1u);
            };
            op(I0{}); op(I1{}); op(I2{}); op(I3{});
        };
        uint32_t i = 0;
        for (; i + 1u < mine; i += 2u) {
            step(I0{}, i);
            step(I1{}, i + 1u);
        }
        if (i < mine) step(I0{}, i);
    }

    // the waves' sums, always in the same order
#pragma unroll
    for (int p = 0; p < CF; ++p) *reinterpret_cast<f32x4 *>(image + p * 1024 + lane * 16u) = acc[p];
    __syncthreads();
    if (wave >= uint32_t(CF)) return;
    f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < W; ++w) v += *reinterpret_cast<const f32x4 *>(smem + w * kNarrowImage + wave * 1024u + lane * 16u);
    const uint32_t f0 = narrow_tile_first(wave, E::kOdd), own = narrow_tile_own(wave, E::kOdd), f = f0 + E::feature(lane);
    char *c = static_cast<char *>(na.C) + size_t(row0 + 4u * g) * row_bytes + size_t(f) * E::kElem;
    float met = 0.f;
#pragma unroll
    for (uint32_t e = 0; e < 4u; ++e) {
        if (f >= own && f < na.N && row0 + 4u * g + e < na.rows) {
            E::store_one(c + size_t(e) * row_bytes, v[e]);
            met = __builtin_fmaf(v[e], 0.f, met);
        }
    }
    if (__ballot(met != 0.f)) tile_sum_again<E, 1, 16, true>(na, row0, f0, own, narrow_tile_end(wave, E::kOdd), lane);
}

template <class E, int CF, int W>
static hipError_t launch_narrow(const NarrowArgs &na, uint32_t loads, uint32_t groups, hipStream_t s)
{
    switch (loads) {
    case 1: spmm_narrow_kernel<E, CF, 1, W><<<dim3(groups), 64 * W, 0, s>>>(na); break;
    case 2: spmm_narrow_kernel<E, CF, 2, W><<<dim3(groups), 64 * W, 0, s>>>(na); break;
    case 3: spmm_narrow_kernel<E, CF, 3, W><<<dim3(groups), 64 * W, 0, s>>>(na); break;
    case 4: spmm_narrow_kernel<E, CF, 4, W><<<dim3(groups), 64 * W, 0, s>>>(na); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <class E>
static hipError_t launch_narrow_e(const NarrowArgs &na, uint32_t waves, uint32_t loads, hipStream_t s)
{
    const uint64_t groups = (uint64_t(na.rows) + kNarrowRows - 1u) / kNarrowRows;
    // (a load of B reads two elements, and a lane has the first entries of each of its wave's blocks)
    if (!na.rows || !na.N || uint64_t(na.N) * na.cols < 2u || na.N > narrow_tile_end(1, E::kOdd) || groups >= (1u << 21) ||
        uint64_t(na.n_blocks) * E::kColumns < na.cols || na.n_blocks > kNarrowMostBlocks || na.n_blocks > 64u * waves)
        return hipErrorInvalidValue;
    constexpr uint32_t kOne = narrow_tile_end(0, E::kOdd);          // features of one tile
    if (waves == 4u) return na.N <= kOne ? launch_narrow<E, 1, 4>(na, loads, uint32_t(groups), s) : launch_narrow<E, 2, 4>(na, loads, uint32_t(groups), s);
    if (waves == 8u) return na.N <= kOne ? launch_narrow<E, 1, 8>(na, loads, uint32_t(groups), s) : launch_narrow<E, 2, 8>(na, loads, uint32_t(groups), s);
    if (waves == 16u) return na.N <= kOne ? launch_narrow<E, 1, 16>(na, loads, uint32_t(groups), s) : launch_narrow<E, 2, 16>(na, loads, uint32_t(groups), s);
    return hipErrorInvalidValue;
}

hipError_t launch_spmm_narrow(int dtype, const NarrowArgs &na, uint32_t waves, uint32_t loads, hipStream_t s)
{
    const bool odd = na.N & 1u;
    if (dtype == kDtypeF16) return odd ? launch_narrow_e<NarrowHalf<false, true>>(na, waves, loads, s) : launch_narrow_e<NarrowHalf<false, false>>(na, waves, loads, s);
    if (dtype == kDtypeBf16) return odd ? launch_narrow_e<NarrowHalf<true, true>>(na, waves, loads, s) : launch_narrow_e<NarrowHalf<true, false>>(na, waves, loads, s);
    return hipErrorInvalidValue;
}

// ---------------------------------------------------------------------------
// The stream, from the plan's tiles: a workgroup per 16 rows.  Blocks without entries have some of value zero.
// ---------------------------------------------------------------------------

typedef NarrowHalf<false, false> NarrowLayout;              // (of every one of them)

__global__ __launch_bounds__(256) void narrow_count_kernel(const TileSource src, uint32_t n_blocks, uint32_t *__restrict__ counts)
{
    __shared__ uint32_t seen[kNarrowMostBlocks];
    for (uint32_t i = threadIdx.x; i < n_blocks; i += 256u) seen[i] = 0u;
    __syncthreads();
    for_entries<NarrowLayout>(src, blockIdx.x * kNarrowRows, kNarrowRows, [&](uint32_t, uint32_t id, size_t) { atomicAdd(&seen[id / kNarrowColumns], 1u); });
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < n_blocks; i += 256u) counts[size_t(blockIdx.x) * n_blocks + i] = seen[i] ? seen[i] : 1u;
}

// Entries in any order inside a block; the last four are filled up with the last one.
__global__ __launch_bounds__(256) void narrow_fill_kernel(const TileSource src, uint32_t n_blocks, const uint32_t *__restrict__ counts,
                                                          const uint32_t *__restrict__ blocks, uint32_t *__restrict__ entries)
{
    __shared__ uint32_t next[kNarrowMostBlocks];
    for (uint32_t i = threadIdx.x; i < n_blocks; i += 256u) next[i] = 0u;
    __syncthreads();
    const size_t base = size_t(blockIdx.x) * n_blocks;
    for_entries<NarrowLayout>(src, blockIdx.x * kNarrowRows, kNarrowRows, [&](uint32_t m, uint32_t id, size_t e) {
        const uint32_t b = id / kNarrowColumns, p = atomicAdd(&next[b], 1u), n = counts[base + b];
        const uint32_t x = NarrowLayout::position(m, id % kNarrowColumns) | uint32_t(static_cast<const uint16_t *>(src.tiles)[e]) << 16;
        uint32_t *at = entries + size_t(blocks[base + b]) * 4u;
        for (uint32_t i = p; i < (p + 1u == n ? (n + 3u) & ~3u : p + 1u); ++i) at[i] = x;
    });
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < n_blocks * 4u; i += 256u)
        if (!next[i / 4u]) entries[size_t(blocks[base + i / 4u]) * 4u + i % 4u] = 0u;
}

static bool narrow_fits(uint32_t n_units, uint32_t n_blocks)
{
    return n_units && n_blocks && n_blocks <= kNarrowMostBlocks && uint64_t(n_units) * n_blocks < (1u << 30);
}

hipError_t launch_narrow_count(const TileSource &src, uint32_t n_units, uint32_t n_blocks, uint32_t *counts, uint32_t *blocks, hipStream_t s)
{
    if (!narrow_fits(n_units, n_blocks)) return hipErrorInvalidValue;
    narrow_count_kernel<<<dim3(n_units), 256, 0, s>>>(src, n_blocks, counts);
    if (hipError_t e = hipGetLastError()) return e;
    return launch_tile_scan(counts, n_units * n_blocks, blocks, s);
}

hipError_t launch_narrow_fill(const TileSource &src, uint32_t n_units, uint32_t n_blocks, const uint32_t *counts, const uint32_t *blocks, uint32_t *entries, hipStream_t s)
{
    if (!narrow_fits(n_units, n_blocks)) return hipErrorInvalidValue;
    narrow_fill_kernel<<<dim3(n_units), 256, 0, s>>>(src, n_blocks, counts, blocks, entries);
    return hipGetLastError();
}

}  // namespace hspmm
