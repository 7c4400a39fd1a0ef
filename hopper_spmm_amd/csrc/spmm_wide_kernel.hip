// Kernels for feature dimensions from 32 on of matrices that are sparse in storage but dense to a workgroup (weights pruned to some
// per cent), 16-bit types: C = A * B by full operands of A, and the kernel that makes the stream they read from a plan's tiles (the
// reference's 8-row windows, src/utils/class.h:74-85) on the device.
//
// At 10 % density and more a 16-row unit touches 81 % of all columns and more: the LDS-panel kernels (spmm_panel_kernel.hpp), which
// condense columns, read a second operand from LDS for every matrix instruction and stream tiles that are mostly zeros all the same.
// Here A is kept as first operands, 16 rows x 64 columns each, no columns condensed: a wave loads an operand straight into the
// registers of its matrix instructions, and a second operand serves the one to three units of a wave.
#include "spmm_tile_common.hpp"

namespace hspmm {

typedef uint32_t u32x8 __attribute__((ext_vector_type(8)));

constexpr uint32_t kWideRows = 16;

// Second-operand registers of 16 features and 64 rows of B.
template <uint32_t PITCH>
__device__ __forceinline__ u32x8 wide_operand(const char *p)
{
    const u32x4 a = tile_operand<PITCH>(p), b = tile_operand<PITCH>(p + 32 * PITCH);
    u32x8 o;
    o[0] = a[0]; o[1] = a[1]; o[2] = a[2]; o[3] = a[3]; o[4] = b[0]; o[5] = b[1]; o[6] = b[2]; o[7] = b[3];
    return o;
}

// Element types.
template <bool BF> struct WideHalf : HalfStored<BF> {
    struct A { u32x4 f[2]; };                               // 16 rows x 64 columns
    __device__ static __forceinline__ void load_a(A &a, const char *src, uint32_t lane)
    {
        a.f[0] = *reinterpret_cast<const u32x4 *>(src + lane * 16u);
        a.f[1] = *reinterpret_cast<const u32x4 *>(src + (lane * 16u + 1024u));
    }
    template <int RF> __device__ static __forceinline__ void multiply(const A (&a)[RF], const u32x8 b, f32x4 *const (&acc)[RF])
    {
        const u32x4 lo = {b[0], b[1], b[2], b[3]}, hi = {b[4], b[5], b[6], b[7]};
#pragma unroll
        for (int u = 0; u < RF; ++u) *acc[u] = HalfOps<BF>::mfma(a[u].f[0], lo, *acc[u]);
#pragma unroll
        for (int u = 0; u < RF; ++u) *acc[u] = HalfOps<BF>::mfma(a[u].f[1], hi, *acc[u]);
    }
    // A block of 16 x 16 sums, of which lane (g, j) has rows 4 g .. 4 g + 3 of feature j: two lanes exchange what makes two features of a
    // row each.  Features below `skip` are another tile's.
    __device__ static __forceinline__ void store(char *c, size_t row_bytes, uint32_t rows_left, uint32_t skip, const f32x4 v, uint32_t lane)
    {
        const bool odd = lane & 1u;
#pragma unroll
        for (uint32_t e = 0; e < 4u; e += 2u) {
            const float mine = odd ? v[e + 1u] : v[e], other = odd ? v[e] : v[e + 1u];
            const float got = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, other), 0xB1, 0xF, 0xF, true));
            const uint32_t row = (lane >> 4) * 4u + e + (odd ? 1u : 0u), f = lane & 14u, word = HalfOps<BF>::pack(odd ? got : mine, odd ? mine : got);
            if (row >= rows_left) continue;
            char *at = c + size_t(row) * row_bytes + f * 2u;
            typedef uint32_t word_any __attribute__((aligned(2)));
            if (f >= skip) *reinterpret_cast<word_any *>(at) = word;
            else if (f + 1u >= skip) *reinterpret_cast<uint16_t *>(at + 2) = uint16_t(word >> 16);
        }
    }
};

// A workgroup multiplies WR RF x 16 rows of A with 16 CF features of B: WK sets of WR waves, a wave RF units of 16 rows and all the
// features, a set every WK-th chunk of 64 columns.  The sets' sums are added at the end, in LDS and always in the same order.
// A chunk of a set: its rows of B, asked for a chunk earlier, go to LDS, what comes behind them is asked for, a barrier, the
// multiplication - RF matrix instructions for every second operand read -, a barrier.  Neighbouring sets are a step apart, so that
// of the two waves of a SIMD one multiplies while the other moves data.
// What bounds it: bytes that come into a compute unit, 2 KB a unit and chunk and 128 a feature; they arrive at 38 to 48 a cycle
// whatever the shape (WR, RF, CF = 4, 2, 4: 0.27 us for 24 KB; 4, 3, 8: 0.55 us for 40 KB, where the matrix instructions take 0.37).  A
// second workgroup on a compute unit doubles the time, more loads in flight (two sets of B, four of A) change nothing, nor do sets
// that run in step with two LDS buffers each.  Start and end are 4 us for the smallest tiles and 10 for the largest.
// Fewer C tiles than compute units are cut: each workgroup takes a part of the chunks and leaves its sums in memory, and a second kernel adds
// them (4096 x 14336, N = 64 45 -> 26 us, 512 x 11008, N = 256 24.8 -> 13.0).  Operands are laid out chunk by chunk, since the
// workgroups walk the chunks side by side: unit by unit, 4096 x 14336 took 57.8 instead of 54.2 us at N = 128 and 39.3 instead of 35.8 at 32.
// Measured, bf16 (this / the LDS-panel or full-tile kernels, us): 5003 x 3001 at 20 %, N = 64 10.5 / 15.7, 128 12.1 / 15.6, 333
// 21.0 / 28.1; 4096^2 at 10 %, N = 256 15.7 / 20.7, 512 21.7 / 28.5; 3840 x 1155 at 29 %, N = 208 8.3 / 13.9; 14080 x 2815 at 26 %,
// N = 101 19.8 / 42.3.  2531 launches of 508 matrices at 3 to 30 %: 1.37 times as fast on the 63 % of them where it is faster.
template <class E, int RF, int CF, int WR, int WK>
__global__ __launch_bounds__(64 * WR * WK, WR * WK / 4)
void spmm_wide_kernel(const WideArgs wa)
{
    constexpr uint32_t kSet = 64u * WR, NT = uint32_t(CF) * 16u;
    constexpr uint32_t kLine = NT * 2u, kPitch = kLine + ((kLine / 32u) % 2u ? 0u : 32u), kB = 64u * kPitch;       // of a chunk of B in LDS
    constexpr uint32_t kPieces = NT / 8u, kPer = 64u * kPieces / kSet;                      // 16-byte pieces of a row of B; that a thread takes
    static_assert(64u * kPieces % kSet == 0u, "the pieces of a chunk must divide among the threads of a set of waves");
    constexpr uint32_t kSums = RF * CF * 1024u, kAll = WK / 2 * WR * kSums, kRoom = kAll > WK * kB ? kAll : WK * kB;
    __shared__ __attribute__((aligned(16))) char smem[kRoom];

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wr = wave % WR, set = wave / WR;
    // consecutive tiles on one XCD (workgroups are dealt out to the eight in turn): the feature tiles of a row block share its
    // operands, neighbours their rows of B
    const uint32_t n_groups = gridDim.x, xcd = blockIdx.x & 7u;
    const uint32_t tile = xcd * (n_groups >> 3) + umin32(xcd, n_groups & 7u) + (blockIdx.x >> 3);
    const uint32_t rbc = tile / wa.n_feat_tiles, ft = tile - rbc * wa.n_feat_tiles, rb = rbc / wa.n_cuts, cut = rbc - rb * wa.n_cuts;
    const uint32_t all_stages = wa.n_chunks / WK, stage0 = cut * all_stages / wa.n_cuts, n_stages = (cut + 1u) * all_stages / wa.n_cuts - stage0;
    const uint32_t unit0 = (rb * WR + wr) * RF, row0 = unit0 * kWideRows;
    const size_t row_bytes = size_t(wa.N) * E::kElem;
    const uint32_t own = ft * NT, f0 = umin32(own, wa.N - NT);      // the last tile is moved back to end with the row; it stores from `own` on

    const char *src_b = static_cast<const char *>(wa.B) + size_t(f0) * E::kElem;
    uint32_t piece_row[kPer], piece_col[kPer];
#pragma unroll
    for (uint32_t i = 0; i < kPer; ++i) { const uint32_t n = i * kSet + tid % kSet; piece_row[i] = n / kPieces; piece_col[i] = n % kPieces * 16u; }
    const char *src_a[RF];                                          // (units behind the last one: that unit, not stored)
#pragma unroll
    for (int u = 0; u < RF; ++u) src_a[u] = static_cast<const char *>(wa.frags) + (size_t(set) * wa.n_units + umin32(unit0 + u, wa.n_units - 1u)) * kWideUnitBytes;
    u32x4 piece[kPer];
    typename E::A a[2][RF];
    uint32_t ask_a = 0, ask_b = 0;
    auto request_b = [&]() __attribute__((always_inline)) {
        // (rows behind the last one: that row, which the operands multiply by zero)
        const uint32_t first = umin32(((stage0 + umin32(ask_b, n_stages - 1u)) * WK + set) * 64u, wa.cols - 1u), last = wa.cols - 1u - first;
        const char *p = src_b + size_t(first) * row_bytes;
#pragma unroll
        for (uint32_t i = 0; i < kPer; ++i) piece[i] = *reinterpret_cast<const u32x4_any *>(p + (umin32(piece_row[i], last) * uint32_t(row_bytes) + piece_col[i]));
        ++ask_b;
    };
    auto request_a = [&](auto set_c) __attribute__((always_inline)) {
        constexpr int S = decltype(set_c)::value;
        const size_t off = size_t(stage0 + umin32(ask_a, n_stages - 1u)) * wa.n_units * (WK * kWideUnitBytes);
#pragma unroll
        for (int u = 0; u < RF; ++u) E::load_a(a[S][u], src_a[u] + off, lane);
        ++ask_a;
    };
    typedef std::integral_constant<int, 0> Set0;
    typedef std::integral_constant<int, 1> Set1;
    f32x4 acc[RF][CF];
#pragma unroll
    for (int u = 0; u < RF; ++u)
#pragma unroll
        for (int p = 0; p < CF; ++p) acc[u][p] = f32x4{0.f, 0.f, 0.f, 0.f};
    request_b();
    request_a(Set0{});
    char *const mine = smem + set * kB;
    const char *b_lane = mine + (4u * (lane >> 4) + ((lane & 15u) >> 2)) * kPitch + (lane & 3u) * 8u;
    // a chunk, whose first operands are (or will be) in set S of the two
    auto stage = [&](auto set_c) __attribute__((always_inline)) {
        constexpr int S = decltype(set_c)::value;
#pragma unroll
        for (uint32_t i = 0; i < kPer; ++i) *reinterpret_cast<u32x4 *>(mine + piece_row[i] * kPitch + piece_col[i]) = piece[i];
        request_b();
        request_a(std::integral_constant<int, S ^ 1>{});
        panel_barrier();
        __builtin_amdgcn_sched_barrier(0);
        u32x8 op[2];
        op[0] = wide_operand<kPitch>(b_lane);
#pragma unroll
        for (int p = 0; p < CF; ++p) {
            if (p + 1 < CF) op[(p + 1) & 1] = wide_operand<kPitch>(b_lane + (p + 1) * 32);
            __builtin_amdgcn_sched_barrier(0);                      // (the next operand is on its way while this one is multiplied)
            f32x4 *to[RF];
#pragma unroll
            for (int u = 0; u < RF; ++u) to[u] = &acc[u][p];
            E::template multiply<RF>(a[S], op[p & 1], to);
            __builtin_amdgcn_sched_barrier(0);
        }
        panel_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    if (set & 1u) panel_barrier();
    uint32_t s = 0;
    for (; s + 1u < n_stages; s += 2u) {
        stage(Set0{});
        stage(Set1{});
    }
    if (s < n_stages) stage(Set0{});
    if (!(set & 1u)) panel_barrier();                               // (every wave has passed as many)

    // the upper half of the sets to the lower half, until one is left
#pragma unroll
    for (uint32_t w = WK / 2; w; w /= 2) {
        f32x4 *slot = reinterpret_cast<f32x4 *>(smem + (set % w * WR + wr) * kSums + lane * 16u);
        panel_barrier();
        if (set >= w && set < 2u * w) {
#pragma unroll
            for (int i = 0; i < RF * CF; ++i) slot[i * 64] = acc[i / CF][i % CF];
        }
        panel_barrier();
        if (set < w) {
#pragma unroll
            for (int i = 0; i < RF * CF; ++i) acc[i / CF][i % CF] += slot[i * 64];
        }
    }
    if (set != 0u) return;
    if (wa.n_cuts > 1u) {
        f32x4 *out = reinterpret_cast<f32x4 *>(wa.sums) + ((size_t(cut) * (n_groups / wa.n_cuts) + rb * wa.n_feat_tiles + ft) * WR + wr) * (RF * CF * 64u) + lane;
#pragma unroll
        for (int i = 0; i < RF * CF; ++i) out[i * 64] = acc[i / CF][i % CF];
        return;
    }
    float met = 0.f;
#pragma unroll
    for (int u = 0; u < RF; ++u) {
        const uint32_t row = row0 + uint32_t(u) * kWideRows;
        if (row >= wa.rows) break;
        char *c = static_cast<char *>(wa.C) + size_t(row) * row_bytes + size_t(f0) * E::kElem;
#pragma unroll
        for (int p = 0; p < CF; ++p) {
            const uint32_t at = uint32_t(p) * 16u;
            E::store(c + at * E::kElem, row_bytes, wa.rows - row, own - f0 > at ? own - f0 - at : 0u, acc[u][p], lane);
#pragma unroll
            for (int e = 0; e < 4; ++e) met = __builtin_fmaf(acc[u][p][e], 0.f, met);
        }
    }
    // An infinity or a NaN in B makes every sum of its feature NaN - the operands hold a zero wherever no entry is - and a sum that is
    // finite has met none (0 times a finite sum is 0).  What is not finite is summed again, over the stored entries alone.
    if (__ballot(met != 0.f)) {
        constexpr uint32_t kOnce = NT < 64u ? NT : 64u;
#pragma unroll 1
        for (uint32_t f = 0; f < NT; f += kOnce) tile_sum_again<E, RF, kOnce>(wa, row0, f0 + f, own, wa.N, lane);
    }
}

// The sums of the cuts of a C tile, in order: a wave per 16 rows x 16 features.
template <class E>
__global__ __launch_bounds__(256) void wide_sum_kernel(const WideArgs wa, const WideShape sh, uint32_t n_blocks)
{
    const uint32_t lane = threadIdx.x & 63u, i = __builtin_amdgcn_readfirstlane(blockIdx.x * 4u + (threadIdx.x >> 6));
    if (i >= n_blocks) return;
    const uint32_t block = i % sh.blocks, unit_of = i / sh.blocks % (sh.units * sh.rows), tile = i / sh.blocks / (sh.units * sh.rows);
    const uint32_t rb = tile / wa.n_feat_tiles, ft = tile - rb * wa.n_feat_tiles, nt = sh.blocks * 16u;
    const uint32_t row0 = (rb * sh.rows * sh.units + unit_of) * kWideRows, own = ft * nt, f0 = umin32(own, wa.N - nt) + block * 16u;
    if (row0 >= wa.rows || f0 + 16u <= own) return;
    const f32x4 *in = reinterpret_cast<const f32x4 *>(wa.sums) + size_t(i) * 64u + lane;
    f32x4 v = in[0];
#pragma unroll 4
    for (uint32_t c = 1; c < wa.n_cuts; ++c) v += in[size_t(c) * n_blocks * 64u];
    const size_t row_bytes = size_t(wa.N) * E::kElem;
    E::store(static_cast<char *>(wa.C) + size_t(row0) * row_bytes + size_t(f0) * E::kElem, row_bytes, wa.rows - row0, own > f0 ? own - f0 : 0u, v, lane);
    float met = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) met = __builtin_fmaf(v[e], 0.f, met);
    if (__ballot(met != 0.f)) tile_sum_again<E, 1, 16, true>(wa, row0, f0, own, wa.N, lane);
}

template <class E>
static hipError_t launch_wide_sums(const WideArgs &wa, const WideShape &sh, uint32_t groups, hipStream_t s, hipEvent_t mid)
{
    if (hipError_t e = hipGetLastError()) return e;
    if (wa.n_cuts == 1u) return hipSuccess;
    if (mid) { if (hipError_t e = hipEventRecord(mid, s)) return e; }
    const uint32_t n_blocks = groups * sh.blocks * sh.units * sh.rows;
    wide_sum_kernel<E><<<dim3((n_blocks + 3u) / 4u), 256, 0, s>>>(wa, sh, n_blocks);
    return hipGetLastError();
}

template <class E>
static hipError_t launch_wide_e(const WideArgs &wa, const WideShape &sh, uint32_t groups, hipStream_t s, hipEvent_t mid)
{
#define HSPMM_WIDE(RF, CF, WR, WK) \
    if (sh.units == RF && sh.blocks == CF && sh.rows == WR && sh.splits == WK) { spmm_wide_kernel<E, RF, CF, WR, WK><<<dim3(groups * wa.n_cuts), 64 * WR * WK, 0, s>>>(wa); return launch_wide_sums<E>(wa, sh, groups, s, mid); }
    HSPMM_WIDE(1, 2, 2, 4) HSPMM_WIDE(1, 2, 4, 2) HSPMM_WIDE(1, 4, 4, 2) HSPMM_WIDE(2, 2, 4, 2) HSPMM_WIDE(2, 4, 4, 2) HSPMM_WIDE(3, 4, 2, 4)
    HSPMM_WIDE(3, 4, 4, 2) HSPMM_WIDE(2, 8, 4, 2) HSPMM_WIDE(3, 8, 4, 2)
#undef HSPMM_WIDE
    return hipErrorInvalidValue;
}

hipError_t launch_spmm_wide(int dtype, const WideArgs &wa, const WideShape &sh, hipStream_t s, hipEvent_t mid)
{
    const uint64_t rows = uint64_t(sh.units) * sh.rows * kWideRows, nt = uint64_t(sh.blocks) * 16u;
    // (a row of B holds a tile, offsets inside a chunk of it fit 32 bits, and the chunks and units are all there)
    if (!rows || !nt || !sh.splits || wa.N < nt || wa.N >= (1u << 21) || !wa.rows || !wa.cols || wa.n_chunks % sh.splits || uint64_t(wa.n_chunks) * 64u < wa.cols ||
        uint64_t(wa.n_units) * kWideRows < wa.rows || wa.n_feat_tiles != (wa.N + nt - 1u) / nt)
        return hipErrorInvalidValue;
    const uint64_t groups = (wa.rows + rows - 1u) / rows * wa.n_feat_tiles;
    if (!wa.n_cuts || groups * wa.n_cuts >= (1u << 22) || wa.n_cuts > wa.n_chunks / sh.splits || (wa.n_cuts > 1u && !wa.sums)) return hipErrorInvalidValue;
    if (dtype == kDtypeBf16) return launch_wide_e<WideHalf<true>>(wa, sh, uint32_t(groups), s, mid);
    if (dtype == kDtypeF16) return launch_wide_e<WideHalf<false>>(wa, sh, uint32_t(groups), s, mid);
    return hipErrorInvalidValue;
}

// ---------------------------------------------------------------------------
// The operands from the plan's tiles: a workgroup per window, a thread a tile column.  Memory is cleared in front of it.
// ---------------------------------------------------------------------------

// Lane (g, j) of an instruction has row j and the columns 4 g .. 4 g + 3 and 16 + 4 g .. 16 + 4 g + 3 of 32: the rows of B that the
// transposing LDS reads bring it.
__global__ __launch_bounds__(256) void wide_fill_kernel(const TileSource src, uint32_t n_units, char *__restrict__ frags)
{
    const uint32_t w = blockIdx.x, row0 = src.rowIdx[w];
    char *unit = frags + size_t(row0 / kWideRows) * kWideUnitBytes;
    const size_t c1 = size_t(src.rowOffset[w + 1u]) * 16u;
    for (size_t c = size_t(src.rowOffset[w]) * 16u + threadIdx.x; c < c1; c += blockDim.x) {
        const uint32_t id = src.a2b[c];
        if (id == kIdxMax) continue;
        const uint16_t *tile = static_cast<const uint16_t *>(src.tiles) + (c / 16u) * 128u + c % 16u;
        const uint32_t k = id & 31u;
        uint16_t *to = reinterpret_cast<uint16_t *>(unit + size_t(id >> 6) * n_units * kWideUnitBytes + (id & 32u) * 32u) +
                       (((k & 15u) >> 2) * 16u + (row0 & 15u)) * 8u + (k & 3u) + 4u * (k >> 4);
#pragma unroll
        for (uint32_t r = 0; r < 8u; ++r) {
            const uint16_t v = tile[r * 16u];
            if (v) to[r * 8u] = v;
        }
    }
}

hipError_t launch_wide_fill(const TileSource &src, uint32_t rows, uint32_t n_chunks, void *frags, hipStream_t s)
{
    if (!src.n_windows || src.n_windows >= (1u << 23)) return hipErrorInvalidValue;
    const uint32_t n_units = (rows + kWideRows - 1u) / kWideRows;
    if (hipError_t e = launch_fill_zero(frags, size_t(n_units) * n_chunks * kWideUnitBytes, s)) return e;
    wide_fill_kernel<<<dim3(src.n_windows), 256, 0, s>>>(src, n_units, static_cast<char *>(frags));
    return hipGetLastError();
}

}  // namespace hspmm
