// Kernels for narrow feature dimensions: C = A * B entry by entry, and the kernels that make the entry stream they
// walk from a plan's tiles (the reference's 8-row windows, src/utils/class.h:74-85) on the device.
//
// The MFMA gather kernels (spmm_mfma_kernel.hpp) multiply 16 columns by 8 rows by at least 32 features in one
// instruction and spend a quarter-wave on every gathered row of B.  With a few features that is mostly idle lanes,
// and the tiles of a sparse matrix are mostly zeros (a graph stores 16 of 128 elements).  Here a row of B is one load of
// a few lanes, and only stored entries are read: 4 bytes of column id and one value each.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <algorithm>
#include "hspmm_device.h"
#include "lane_ranges.hpp"

namespace hspmm {

typedef uint32_t e_u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t e_u32x3 __attribute__((ext_vector_type(3)));
typedef uint32_t e_u32x4 __attribute__((ext_vector_type(4)));

// Element types: how four stored values are read, how a word of a row of B is multiplied in, how sums are rounded.
struct EntryF16 {
    static constexpr uint32_t kElem = 2;
    typedef e_u32x2 Vals;
    __device__ static __forceinline__ bool stored(const Vals v, int i) { return (v[i >> 1] & ((i & 1) ? 0xFFFF0000u : 0xFFFFu)) != 0u; }
    __device__ static __forceinline__ float value(const Vals v, int i)
    {
        const uint32_t w = v[i >> 1];
        return (float)__builtin_bit_cast(_Float16, uint16_t((i & 1) ? w >> 16 : w));
    }
    __device__ static __forceinline__ float low(uint32_t w) { return (float)__builtin_bit_cast(_Float16, uint16_t(w)); }
    __device__ static __forceinline__ float high(uint32_t w) { return (float)__builtin_bit_cast(_Float16, uint16_t(w >> 16)); }
    __device__ static __forceinline__ uint16_t round(float f) { return __builtin_bit_cast(uint16_t, (_Float16)f); }
};
struct EntryBf16 {
    static constexpr uint32_t kElem = 2;
    typedef e_u32x2 Vals;
    __device__ static __forceinline__ bool stored(const Vals v, int i) { return (v[i >> 1] & ((i & 1) ? 0xFFFF0000u : 0xFFFFu)) != 0u; }
    __device__ static __forceinline__ float value(const Vals v, int i)
    {
        const uint32_t w = v[i >> 1];
        return __builtin_bit_cast(float, (i & 1) ? w & 0xFFFF0000u : w << 16);
    }
    __device__ static __forceinline__ float low(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
    __device__ static __forceinline__ float high(uint32_t w) { return __builtin_bit_cast(float, w & 0xFFFF0000u); }
    __device__ static __forceinline__ uint16_t round(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
};
struct EntryF32 {
    static constexpr uint32_t kElem = 4;
    typedef e_u32x4 Vals;
    __device__ static __forceinline__ bool stored(const Vals v, int i) { return v[i] != 0u; }
    __device__ static __forceinline__ float value(const Vals v, int i)
    {
        const uint32_t w = v[i];
        return __builtin_bit_cast(float, w);
    }
};

// VB bytes of a row of B or C, wherever they lie (rows of an odd feature dimension start anywhere).
template <int VB> struct Piece;
template <> struct Piece<2> { typedef uint16_t mem __attribute__((aligned(2))); uint32_t w[1];
    __device__ __forceinline__ void load(const char *p) { w[0] = *reinterpret_cast<const mem *>(p); }
    __device__ __forceinline__ void store(char *p) const { *reinterpret_cast<mem *>(p) = uint16_t(w[0]); } };
template <> struct Piece<4> { typedef uint32_t mem __attribute__((aligned(2))); uint32_t w[1];
    __device__ __forceinline__ void load(const char *p) { w[0] = *reinterpret_cast<const mem *>(p); }
    __device__ __forceinline__ void store(char *p) const { *reinterpret_cast<mem *>(p) = w[0]; } };
template <> struct Piece<8> { typedef e_u32x2 mem __attribute__((aligned(2))); uint32_t w[2];
    __device__ __forceinline__ void load(const char *p) { const e_u32x2 x = *reinterpret_cast<const mem *>(p); w[0] = x[0]; w[1] = x[1]; }
    __device__ __forceinline__ void store(char *p) const { e_u32x2 x; x[0] = w[0]; x[1] = w[1]; *reinterpret_cast<mem *>(p) = x; } };
template <> struct Piece<16> { typedef e_u32x4 mem __attribute__((aligned(2))); uint32_t w[4];
    __device__ __forceinline__ void load(const char *p) { const e_u32x4 x = *reinterpret_cast<const mem *>(p); w[0] = x[0]; w[1] = x[1]; w[2] = x[2]; w[3] = x[3]; }
    __device__ __forceinline__ void store(char *p) const { e_u32x4 x; x[0] = w[0]; x[1] = w[1]; x[2] = w[2]; x[3] = w[3]; *reinterpret_cast<mem *>(p) = x; } };

__device__ __forceinline__ uint32_t umin_e(uint32_t a, uint32_t b) { return a < b ? a : b; }

template <class E, int VB, int NF>
__device__ __forceinline__ void multiply_in(float (&acc)[NF], const Piece<VB> &b, const float a)
{
    if constexpr (E::kElem == 4) {
#pragma unroll
        for (int i = 0; i < NF; ++i) acc[i] = __builtin_fmaf(a, __builtin_bit_cast(float, b.w[i]), acc[i]);
    } else if constexpr (NF == 1) {
        acc[0] = __builtin_fmaf(a, E::low(b.w[0]), acc[0]);
    } else {
#pragma unroll
        for (int i = 0; i < NF / 2; ++i) {
            acc[2 * i] = __builtin_fmaf(a, E::low(b.w[i]), acc[2 * i]);
            acc[2 * i + 1] = __builtin_fmaf(a, E::high(b.w[i]), acc[2 * i + 1]);
        }
    }
}

template <class E, int VB, int NF>
__device__ __forceinline__ Piece<VB> round_sums(const float (&acc)[NF])
{
    Piece<VB> out;
    if constexpr (E::kElem == 4) {
#pragma unroll
        for (int i = 0; i < NF; ++i) out.w[i] = __builtin_bit_cast(uint32_t, acc[i]);
    } else if constexpr (NF == 1) {
        out.w[0] = E::round(acc[0]);
    } else {
#pragma unroll
        for (int i = 0; i < NF / 2; ++i) out.w[i] = uint32_t(E::round(acc[2 * i])) | uint32_t(E::round(acc[2 * i + 1])) << 16;
    }
    return out;
}

// One row of C per group of g = 2^log2g subgroups; a subgroup is L lanes of VB bytes each, which together cover a
// row of B (where the row does not divide, the last lanes are moved back to end with it and compute what they share
// with their neighbour a second time).  The subgroups of a group take the row's units - four entries, one load of
// ids and one of values - in turn and their sums are added at the end, in a fixed order.  Rows are sorted by length,
// so that the subgroups of a wave run alike; the classes of EntryArgs say how many subgroups a row gets.
// What bounds it: the rows of B.  A wave keeps four of them per subgroup in flight and has no other loads to wait for than the next
// unit's, and with up to eight waves per SIMD (64 registers) a compute unit has 72 to 85 requests to its L2 under way all the time
// and its L1's return path busy for 25 to 62 % of it and waiting for the L2 for most of the rest; what a request takes - 250 to 580
// cycles - goes by how many hit the L2 (counted, us / requests under way / L2 hits: graph of 2^18, bf16, N = 16 26.4 / 79 / 82 %; of 150001, fp32, N = 100 91 / 72 /
// 59 %; of 500000, fp16, N = 1 23.7 / 74 / 89 %; uniform 65536^2, N = 128 28.5 / 85 / 41 %, 6.3 TB/s past the L2s).  A launch as
// short as 4096^2 at 1 %, N = 64 - 4.5 us, 22 under way - is its chain of descriptor, ids, rows and sums.
// Odd: 16-bit types with an odd number of elements in a row of B, whose every other row starts between two words, and loads that
// are not whole words take twice their time (graph of 2^18, fp16, N = 65 / 66: 109 / 73 us).  Such a row is loaded from the word before on and
// shifted by half a word, the word behind a lane's last one being its neighbour's first; the last lane of a block has seven features,
// which the load holds either way, and is moved back, so that the last feature of the lane in front of it is another one's sum: that lane
// stores what lies in front of the last lane's alone (entry_lane_stores).  Before / with it, us: that graph, N = 33 59.4 / 50.6, 65 109 / 75.5, 129 225 / 174; of 40001, N = 33 12.1 /
// 10.3; uniform 16384^2, 64 per row, N = 17 13.9 / 10.7, 65 28.4 / 21.0, 129 50.1 / 31.5.
template <class E, int VB, int L, int U, bool Cut, bool Odd>
__global__ __launch_bounds__(256)
void spmm_entries_kernel(const EntryArgs ea)
{
    constexpr uint32_t S = 64u / L;                         // subgroups of a wave
    constexpr int NF = VB / int(E::kElem);                  // features of a lane
    uint32_t group = blockIdx.x, fb = 0;
    if (ea.xcd_split) {
        // Feature blocks with XCDs of their own (see spmm_mfma_kernel.hpp): block f of F runs on XCDs 8f/F .. 8(f+1)/F - 1.
        const uint32_t per_fb = 8u / ea.n_feat_blocks, xcd = blockIdx.x & 7u;
        fb = xcd / per_fb;
        group = (blockIdx.x >> 3) * per_fb + (xcd - fb * per_fb);
        if (group >= ea.n_groups) return;
    } else if (ea.n_feat_blocks > 1u) {
        fb = blockIdx.x / ea.n_groups;
        group = blockIdx.x - fb * ea.n_groups;
    }
    uint32_t c = 0;
    while (c + 1u < ea.n_classes && group >= ea.cls[c + 1u].group_begin) ++c;
    const uint32_t logs = ea.cls[c].logs, log2g = logs & 0xFFu, log2parts = Cut ? logs >> 8 : 0u, g = 1u << log2g;
    const uint32_t sub = threadIdx.x / L, lane = threadIdx.x % L;
    // (Cut: a class may cut its rows into 2^log2parts parts, each a subgroup group of its own.  An instance of its own: where
    // no class does, the arithmetic for it is 1 - 3 % of a launch)
    const uint32_t nth = (group - ea.cls[c].group_begin) * ((4u * S) >> log2g) + (sub >> log2g);
    const uint32_t slot = ea.cls[c].slot_begin + (nth >> log2parts);
    const bool exists = slot < ea.cls[c].slot_end;
    const uint32_t member = sub & (g - 1u);
    const uint32_t *d = ea.desc + size_t(exists ? slot : ea.cls[c].slot_begin) * 3u;
    uint32_t first = d[0], units = exists ? d[1] : 0u, part = 0;
    const uint32_t row = d[2];
    if (Cut && log2parts) {
        part = nth & ((1u << log2parts) - 1u);
        const uint32_t of_part = (units + (1u << log2parts) - 1u) >> log2parts, skip = part * of_part;
        first += skip;
        units = units > skip ? umin_e(of_part, units - skip) : 0u;
    }

    // bytes of a row this block covers, and where: a last block that would reach past the row is moved back to end with it
    const uint32_t row_len = ea.block_bytes;
    static_assert(!Odd || (VB == 16 && E::kElem == 2), "16 bytes of 16-bit elements");
    const bool last = entry_lane_last(lane, VB, row_len);
    const uint32_t off = entry_lane_begin(lane, VB, row_len, Odd);
    const size_t pitch = size_t(ea.ld) * E::kElem;
    const size_t block = umin_e(fb * row_len, uint32_t(pitch) - row_len);
    const char *B = reinterpret_cast<const char *>(ea.B) + block + off;
    const uint32_t *ids = ea.ids + size_t(first) * 4u;
    const typename E::Vals *vals = reinterpret_cast<const typename E::Vals *>(ea.vals) + first;

    // A row's piece, and whether it begins half a word into what is loaded.  (The last row of B always does, so that nothing behind
    // B is read: where that row does begin on a word, the load is the one that does not.)
    const uint32_t flip = uint32_t(block) >> 1;
    auto load = [&](Piece<VB> &b, uint32_t id) __attribute__((always_inline)) {
        const uint32_t odd = Odd ? ((id + (id == ea.last_row ? 1u - (id & 1u) : 0u)) ^ flip) & 1u : 0u;
        b.load(B + size_t(id) * pitch - odd * 2u);
        return odd;
    };
    auto shift = [&](Piece<VB> &b, uint32_t odd) __attribute__((always_inline)) {
        if constexpr (Odd) {
            const uint32_t next = uint32_t(__builtin_amdgcn_mov_dpp(int(b.w[0]), 0x130, 0xF, 0xF, true)), by = odd * 16u;      // (the next lane's)
#pragma unroll
            for (int i = 0; i < 3; ++i) b.w[i] = __builtin_amdgcn_alignbit(b.w[i + 1], b.w[i], by);
            b.w[3] = __builtin_amdgcn_alignbit(next, b.w[3], by);
        }
    };
    float acc[NF];
#pragma unroll
    for (int i = 0; i < NF; ++i) acc[i] = 0.f;
    // U units of a subgroup in flight - 4 U rows of B - and the ids and values of the units behind them.
    uint32_t u = member;
    if (u < units) {
        e_u32x4 id[U];
        typename E::Vals v[U];
        auto request = [&](uint32_t from) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < U; ++k) {
                const uint32_t ask = umin_e(from + uint32_t(k) * g, units - 1u);      // (past the end: not used)
                id[k] = *reinterpret_cast<const e_u32x4 *>(ids + size_t(ask) * 4u);
                v[k] = vals[ask];
            }
        };
        request(u);
        for (;;) {
            Piece<VB> b[4 * U];
            typename E::Vals now[U];
            uint32_t odds = 0;                              // a bit a row
#pragma unroll
            for (int k = 0; k < U; ++k) {
                now[k] = v[k];
                if (k == 0 || u + uint32_t(k) * g < units) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) odds |= load(b[4 * k + i], id[k][i]) << (4 * k + i);
                }
            }
            const uint32_t next = u + uint32_t(U) * g;
            if (next < units) request(next);
#pragma unroll
            for (int k = 0; k < U; ++k)
                if (k == 0 || u + uint32_t(k) * g < units) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        shift(b[4 * k + i], odds >> (4 * k + i) & 1u);
                        multiply_in<E, VB, NF>(acc, b[4 * k + i], E::value(now[k], i));
                    }
                }
            if (next >= units) break;
            u = next;
        }
        // What fills a row's last unit up (+0, which no stored value is, at the row's last column) counts for nothing, unless that
        // row of B is not finite there: then once more, the stored entries alone, in the same order.
        float met = 0.f;
        if (Odd && last) acc[NF - 1] = 0.f;                 // (no feature)
#pragma unroll
        for (int i = 0; i < NF; ++i) met = __builtin_fmaf(acc[i], 0.f, met);
        bool again = met != 0.f;
        if constexpr (Odd) again = (__ballot(again) >> ((threadIdx.x & 63u) - lane)) & ((uint64_t(1) << L) - 1u);    // (lanes need their neighbours)
        if (again) {
#pragma unroll
            for (int i = 0; i < NF; ++i) acc[i] = 0.f;
            for (u = member; u < units; u += g) {
                const e_u32x4 at = *reinterpret_cast<const e_u32x4 *>(ids + size_t(u) * 4u);
                const typename E::Vals a = vals[u];
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (E::stored(a, i)) {
                        Piece<VB> b;
                        const uint32_t odd = load(b, at[i]);
                        shift(b, odd);
                        multiply_in<E, VB, NF>(acc, b, E::value(a, i));
                    }
            }
        }
    }
    // the subgroups of one wave, then those of the waves of the workgroup
#pragma unroll
    for (uint32_t m = 1u; m < S; m <<= 1)
        if (m < g) {
#pragma unroll
            for (int i = 0; i < NF; ++i) acc[i] += __shfl_xor(acc[i], int(m * L));
        }
    if (g > S) {
        __shared__ float sums[4][L * NF];
        const uint32_t wave = threadIdx.x >> 6;
        if ((threadIdx.x & 63u) < L) {
#pragma unroll
            for (int i = 0; i < NF; ++i) sums[wave][i * L + lane] = acc[i];
        }
        __syncthreads();
        if (member == 0u) {
            for (uint32_t w = 1; w < g / S; ++w) {
#pragma unroll
                for (int i = 0; i < NF; ++i) acc[i] += sums[wave + w][i * L + lane];
            }
        }
    }
    if (!exists || member != 0u) return;
    uint32_t row_out = row;
    const bool piece = c == 0u && ea.n_pieces;
    if (piece || (Cut && log2parts)) {
        // A piece of a row longer than kEntryPieceUnits, or a part of either: its sums go to memory, and the subgroup that
        // brings the row's last part adds all of them, in order.  They cross the L2s of different XCDs: device-scope accesses,
        // and the writes are acknowledged before the arrival is counted (lanes of one subgroup are in one wave).
        uint32_t mine = ea.part_begin[c] + nth, head = ea.part_begin[c] + (nth - part), count = 1u << log2parts;
        if (piece) {
            const uint32_t *pc = ea.pieces + size_t(row) * 3u;
            mine = (row << log2parts) + part; head = pc[1] << log2parts; count = pc[2] << log2parts;
            row_out = pc[0];
        }
        float *out = ea.scratch + ((size_t(mine) * ea.n_feat_blocks + fb) * L + lane) * NF;
#pragma unroll
        for (int i = 0; i < NF; ++i) __hip_atomic_store(out + i, acc[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        uint32_t old = 0;
        if (lane == 0u) old = __hip_atomic_fetch_add(ea.arrive + size_t(head) * ea.n_feat_blocks + fb, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        old = __shfl(old, int((threadIdx.x & 63u) - lane));
        asm volatile("" ::: "memory");
        if (old + 1u != count) return;
#pragma unroll
        for (int i = 0; i < NF; ++i) acc[i] = 0.f;
        for (uint32_t k = 0; k < count; ++k) {
            const float *in = ea.scratch + ((size_t(head + k) * ea.n_feat_blocks + fb) * L + lane) * NF;
#pragma unroll
            for (int i = 0; i < NF; ++i) acc[i] += __hip_atomic_load(in + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (lane == 0u) __hip_atomic_store(ea.arrive + size_t(head) * ea.n_feat_blocks + fb, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const uint32_t stores = entry_lane_stores(lane, VB, row_len, Odd);
    if (!stores) return;                                    // (a lane behind the row's end: its neighbour's copy)
    const Piece<VB> out = round_sums<E, VB, NF>(acc);
    char *c_row = reinterpret_cast<char *>(ea.C) + size_t(row_out) * pitch + block + off;
    if constexpr (Odd) {
        if (stores < 16u) {                                 // (4, 8, 12 or 14 bytes)
            Piece<8> front;
            Piece<4> behind;
            Piece<2> end;
            front.w[0] = out.w[0]; front.w[1] = out.w[1]; behind.w[0] = stores & 8u ? out.w[2] : out.w[0]; end.w[0] = out.w[3];
            if (stores & 8u) front.store(c_row);
            if (stores & 4u) behind.store(c_row + (stores & 8u));
            if (stores & 2u) end.store(c_row + 12);
            return;
        }
    }
    out.store(c_row);
}

template <class E, bool Cut>
static hipError_t launch_entries_e(const EntryArgs &ea, uint32_t lane_bytes, uint32_t lanes, hipStream_t s)
{
    const uint32_t sets = ea.xcd_split ? 8u / ea.n_feat_blocks : 1u;      // workgroups of one feature block in a round over the XCDs
    const uint32_t grid = ea.xcd_split ? 8u * ((ea.n_groups + sets - 1u) / sets) : ea.n_groups * ea.n_feat_blocks;
#define HSPMM_ENTRIES(VB, L) \
    if (lane_bytes == VB && lanes == L) { spmm_entries_kernel<E, VB, L, (E::kElem == 2 && VB * L <= 128) ? 2 : 1, Cut, false><<<dim3(grid), 256, 0, s>>>(ea); return hipGetLastError(); }
#define HSPMM_ENTRIES_ODD(L) \
    if (ea.odd && lane_bytes == 16u && lanes == L) { spmm_entries_kernel<E, 16, L, L <= 8 ? 2 : 1, Cut, true><<<dim3(grid), 256, 0, s>>>(ea); return hipGetLastError(); }
    if constexpr (E::kElem == 2) { HSPMM_ENTRIES_ODD(2) HSPMM_ENTRIES_ODD(4) HSPMM_ENTRIES_ODD(8) HSPMM_ENTRIES_ODD(16) HSPMM_ENTRIES_ODD(32) HSPMM_ENTRIES(2, 1) }
#undef HSPMM_ENTRIES_ODD
    HSPMM_ENTRIES(4, 1) HSPMM_ENTRIES(4, 2) HSPMM_ENTRIES(8, 1) HSPMM_ENTRIES(8, 2)
    HSPMM_ENTRIES(16, 1) HSPMM_ENTRIES(16, 2) HSPMM_ENTRIES(16, 4) HSPMM_ENTRIES(16, 8) HSPMM_ENTRIES(16, 16) HSPMM_ENTRIES(16, 32)
#undef HSPMM_ENTRIES
    return hipErrorInvalidValue;
}

hipError_t launch_spmm_entries(int dtype, const EntryArgs &ea, uint32_t lane_bytes, uint32_t lanes, hipStream_t s)
{
    if (!ea.n_groups) return hipSuccess;
    if (ea.xcd_split && ea.n_feat_blocks != 2u && ea.n_feat_blocks != 4u && ea.n_feat_blocks != 8u) return hipErrorInvalidValue;
    // (a lane's load stays inside its block, a block inside the row, and the lanes reach over the block)
    if (ea.block_bytes < lane_bytes || ea.block_bytes > lane_bytes * lanes || ea.n_feat_blocks < 1u ||
        uint64_t(ea.ld) * (dtype == kDtypeF32 ? 4u : 2u) < ea.block_bytes || uint64_t(ea.n_groups) * ea.n_feat_blocks >= kEntryMostGroups)
        return hipErrorInvalidValue;
    // (rows of an odd number of 16-bit elements, B on a word, two of its rows at least, a block's last lane seven features)
    if (ea.odd && (dtype == kDtypeF32 || ea.ld % 2u == 0u || ea.block_bytes % 4u != 2u || ea.block_bytes < 18u || reinterpret_cast<uintptr_t>(ea.B) % 4u || !ea.last_row ||
                   (ea.n_feat_blocks > 1u && ea.block_bytes % 16u != 14u)))
        return hipErrorInvalidValue;
    bool cut = false;
    for (uint32_t c = 0; c < ea.n_classes; ++c) cut |= (ea.cls[c].logs >> 8) != 0u;
#define HSPMM_ENTRIES_OF(E) (cut ? launch_entries_e<E, true>(ea, lane_bytes, lanes, s) : launch_entries_e<E, false>(ea, lane_bytes, lanes, s))
    if (dtype == kDtypeF32) return HSPMM_ENTRIES_OF(EntryF32);
    if (dtype == kDtypeBf16) return HSPMM_ENTRIES_OF(EntryBf16);
    return HSPMM_ENTRIES_OF(EntryF16);
#undef HSPMM_ENTRIES_OF
}

// ---------------------------------------------------------------------------
// The entry stream from the plan's tiles.  Chunks of up to kEntryChunkTiles tiles of one window, a wave each; a lane
// is a row of a tile (eight tiles at a time).
// ---------------------------------------------------------------------------

// Which elements of row r of tile t are stored (any bit pattern but +0), lowest column first: 32 bytes either way.
template <int ELEM>
__device__ __forceinline__ uint32_t tile_row_mask(const void *tiles, size_t t, uint32_t r)
{
    const e_u32x4 *src = reinterpret_cast<const e_u32x4 *>(static_cast<const char *>(tiles) + t * 256u + r * 32u);
    uint32_t mask = 0;
#pragma unroll
    for (uint32_t q = 0; q < 2; ++q) {
        const e_u32x4 v = src[q];
#pragma unroll
        for (uint32_t e = 0; e < 4; ++e) {
            if constexpr (ELEM == 4) {
                mask |= (v[e] ? 1u : 0u) << (q * 4u + e);
            } else {
                mask |= ((v[e] & 0xFFFFu) ? 1u : 0u) << (q * 8u + 2u * e);
                mask |= ((v[e] >> 16) ? 1u : 0u) << (q * 8u + 2u * e + 1u);
            }
        }
    }
    return mask;
}

// first_chunk[w]: chunks in front of window w (n_windows + 1 of them); chunk_window[chunk]: its window; totals and cursors cleared.
// One workgroup.
__global__ __launch_bounds__(1024) void entry_chunks_kernel(const uint32_t *__restrict__ rowOffset, uint32_t n_windows,
                                                            uint32_t *__restrict__ first_chunk, uint32_t *__restrict__ chunk_window,
                                                            uint32_t *__restrict__ totals)
{
    __shared__ uint32_t sums[1024];
    if (threadIdx.x < 2u * (kEntryBins + 1u)) totals[threadIdx.x] = 0u;
    const uint32_t per = (n_windows + 1023u) / 1024u, b = umin_e(threadIdx.x * per, n_windows), e = umin_e(b + per, n_windows);
    uint32_t sum = 0;
    for (uint32_t w = b; w < e; ++w) sum += (rowOffset[w + 1u] - rowOffset[w] + kEntryChunkTiles - 1u) / kEntryChunkTiles;
    sums[threadIdx.x] = sum;
    __syncthreads();
    for (uint32_t m = 1u; m < 1024u; m <<= 1) {
        const uint32_t x = threadIdx.x >= m ? sums[threadIdx.x - m] : 0u;
        __syncthreads();
        sums[threadIdx.x] += x;
        __syncthreads();
    }
    uint32_t at = threadIdx.x ? sums[threadIdx.x - 1u] : 0u;
    for (uint32_t w = b; w < e; ++w) {
        first_chunk[w] = at;
        for (uint32_t n = (rowOffset[w + 1u] - rowOffset[w] + kEntryChunkTiles - 1u) / kEntryChunkTiles; n; --n) chunk_window[at++] = w;
    }
    if (threadIdx.x == 1023u) first_chunk[n_windows] = sums[1023];
}

// Tiles t0 .. t0 + n - 1 of a chunk.
struct ChunkTiles { uint32_t window, t0, n; };
__device__ __forceinline__ ChunkTiles chunk_tiles(const EntrySource &src, uint32_t chunk)
{
    const uint32_t w = src.chunk_window[chunk], t0 = src.rowOffset[w] + (chunk - src.first_chunk[w]) * kEntryChunkTiles;
    return {w, t0, umin_e(kEntryChunkTiles, src.rowOffset[w + 1u] - t0)};
}

// counts[chunk][8]: stored entries per row of the chunk's window.
template <int ELEM>
__global__ __launch_bounds__(256) void entry_count_kernel(const EntrySource src, uint32_t *__restrict__ counts)
{
    const uint32_t chunk = blockIdx.x * 4u + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
    if (chunk >= src.first_chunk[src.n_windows]) return;
    const ChunkTiles c = chunk_tiles(src, chunk);
    uint32_t count = 0;
    for (uint32_t i = lane >> 3; i < c.n; i += 8u)
        count += uint32_t(__builtin_popcount(tile_row_mask<ELEM>(src.tiles, size_t(c.t0) + i, lane & 7u)));
    for (uint32_t m = 8; m < 64u; m <<= 1) count += __shfl_xor(count, int(m));
    if (lane < 8u) counts[size_t(chunk) * 8u + lane] = count;
}

// Bin of a row of `units` units of four entries: 0 = pieces of rows above kEntryPieceUnits, then the classes from the
// longest to the shortest in four steps each, kEntryBins - 1 = rows without entries.
__device__ __forceinline__ uint32_t entry_bin(uint32_t units)
{
    if (units == 0u) return kEntryBins - 1u;
    if (units > kEntryPieceUnits) return 0u;
    uint32_t c = 0, step = units - 1u;
    if (units > 4u) {
        c = 30u - uint32_t(__builtin_clz(units - 1u));      // units in (2^(c+1), 2^(c+2)]
        step = (units - 1u - (2u << c)) >> (c - 1u);
    }
    return 1u + (kEntryClassesByLength - 1u - c) * 4u + (3u - step);
}

// One thread per matrix row: its length (all chunks of its window; their counts become positions inside the row) and
// the number of rows per bin.  totals: kEntryBins counts (bin 0: pieces), then the units of the rows cut into pieces.
__global__ __launch_bounds__(256) void entry_rows_kernel(const EntrySource src, uint32_t rows, uint32_t *__restrict__ counts,
                                                         uint32_t *__restrict__ row_len, uint32_t *__restrict__ totals)
{
    const uint32_t *rowIdx = src.rowIdx, *first_chunk = src.first_chunk;
    const uint32_t n_windows = src.n_windows;
    __shared__ uint32_t bins[kEntryBins + 1u];
    if (threadIdx.x < kEntryBins + 1u) bins[threadIdx.x] = 0u;
    __syncthreads();
    const uint32_t row = blockIdx.x * 256u + threadIdx.x;
    if (row < rows) {
        const uint32_t start = row & ~(kRowWindow - 1u);
        uint32_t lo = 0, hi = n_windows;                    // first effective window at or behind the row's window
        while (lo < hi) {
            const uint32_t mid = lo + (hi - lo) / 2u;
            if (rowIdx[mid] < start) lo = mid + 1u; else hi = mid;
        }
        uint32_t len = 0;
        if (lo < n_windows && rowIdx[lo] == start)
            for (uint32_t ch = first_chunk[lo], e = first_chunk[lo + 1u]; ch < e; ++ch) {
                const uint32_t n = counts[size_t(ch) * 8u + (row & 7u)];
                counts[size_t(ch) * 8u + (row & 7u)] = len;
                len += n;
            }
        row_len[row] = len;
        const uint32_t units = len / 4u + ((len & 3u) != 0u), bin = entry_bin(units);
        atomicAdd(&bins[bin], bin == 0u ? (units + kEntryPieceUnits - 1u) / kEntryPieceUnits : 1u);
        if (bin == 0u) atomicAdd(&bins[kEntryBins], units);
    }
    __syncthreads();
    if (threadIdx.x < kEntryBins + 1u && bins[threadIdx.x]) atomicAdd(&totals[threadIdx.x], bins[threadIdx.x]);
}

// One thread per matrix row: its slot in its bin and its place in the stream.  cursors: as totals, cleared.
__global__ __launch_bounds__(256) void entry_place_kernel(const uint32_t *__restrict__ row_len, uint32_t rows,
                                                          const EntryPlaces at, uint32_t *__restrict__ cursors,
                                                          uint32_t *__restrict__ desc, uint32_t *__restrict__ pieces,
                                                          uint32_t *__restrict__ row_first)
{
    __shared__ uint32_t bins[kEntryBins], base[kEntryBins], places[3u * kEntryBins];
    if (threadIdx.x < kEntryBins) bins[threadIdx.x] = 0u;
    if (threadIdx.x < 3u * kEntryBins) places[threadIdx.x] = at.places[threadIdx.x];
    __syncthreads();
    const uint32_t row = blockIdx.x * 256u + threadIdx.x;
    const uint32_t len = row < rows ? row_len[row] : 0u, units = len / 4u + ((len & 3u) != 0u), bin = entry_bin(units);
    uint32_t rank = 0;
    if (row < rows && bin) rank = atomicAdd(&bins[bin], 1u);
    __syncthreads();
    if (threadIdx.x < kEntryBins && bins[threadIdx.x]) base[threadIdx.x] = atomicAdd(&cursors[threadIdx.x], bins[threadIdx.x]);
    __syncthreads();
    if (row >= rows) return;
    if (bin == 0u) {
        const uint32_t n = (units + kEntryPieceUnits - 1u) / kEntryPieceUnits;
        const uint32_t head = atomicAdd(&cursors[0], n), first = places[1] + atomicAdd(&cursors[kEntryBins], units);
        for (uint32_t i = 0; i < n; ++i) {
            uint32_t *d = desc + size_t(places[0] + head + i) * 3u, *pc = pieces + size_t(head + i) * 3u;
            const uint32_t left = units - i * kEntryPieceUnits;
            d[0] = first + i * kEntryPieceUnits; d[1] = left < kEntryPieceUnits ? left : kEntryPieceUnits; d[2] = head + i;
            pc[0] = row; pc[1] = head; pc[2] = n;
        }
        row_first[row] = first;
        return;
    }
    rank += base[bin];
    const uint32_t slot = places[bin * 3u] + rank, first = places[bin * 3u + 1u] + rank * places[bin * 3u + 2u];
    uint32_t *d = desc + size_t(slot) * 3u;
    d[0] = units ? first : 0u; d[1] = units; d[2] = row;
    row_first[row] = first;
}

// Ids and values to their places; the last unit of a row is filled up with its last column and zeros.
template <int ELEM>
__global__ __launch_bounds__(256) void entry_fill_kernel(const EntrySource src, const uint32_t *__restrict__ positions,
                                                         const uint32_t *__restrict__ row_len,
                                                         const uint32_t *__restrict__ row_first, uint32_t rows,
                                                         uint32_t *__restrict__ ids, void *__restrict__ vals)
{
    constexpr uint32_t CW = ELEM == 4 ? 8u : 16u;
    const uint32_t chunk = blockIdx.x * 4u + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
    if (chunk >= src.first_chunk[src.n_windows]) return;
    const void *tiles = src.tiles;
    const uint32_t *a2b = src.a2b;
    const ChunkTiles c = chunk_tiles(src, chunk);
    const uint32_t t0 = c.t0, n = c.n, r = lane & 7u, row = src.rowIdx[c.window] + r;
    const bool inside = row < rows;
    const uint32_t len = inside ? row_len[row] : 0u;
    const size_t first = inside ? size_t(row_first[row]) * 4u : 0u;
    uint32_t at = positions[size_t(chunk) * 8u + r];
    for (uint32_t i0 = 0; i0 < n; i0 += 8u) {
        const uint32_t i = i0 + (lane >> 3);
        const size_t t = size_t(t0) + i;
        uint32_t mask = i < n && inside ? tile_row_mask<ELEM>(tiles, t, r) : 0u;
        const uint32_t mine = uint32_t(__builtin_popcount(mask));
        uint32_t upto = mine;                               // of this row's entries in this lane's tile and those in front of it
        for (uint32_t m = 8; m < 64u; m <<= 1) {
            const uint32_t x = __shfl_up(upto, m);
            if (lane >= m) upto += x;
        }
        const uint32_t all = __shfl(upto, int(56u + r));
        uint32_t pos = at + upto - mine;
        at += all;
        uint32_t id = 0;
        const bool wrote = mask != 0u;
        while (mask) {
            const uint32_t k = uint32_t(__builtin_ctz(mask));
            mask &= mask - 1u;
            id = a2b[t * CW + k];
            ids[first + pos] = id;
            const size_t e = t * (8u * CW) + r * CW + k;
            if constexpr (ELEM == 4) static_cast<uint32_t *>(vals)[first + pos] = static_cast<const uint32_t *>(tiles)[e];
            else static_cast<uint16_t *>(vals)[first + pos] = static_cast<const uint16_t *>(tiles)[e];
            ++pos;
        }
        if (wrote && pos == len)
            for (; pos & 3u; ++pos) {
                ids[first + pos] = id;
                if constexpr (ELEM == 4) static_cast<uint32_t *>(vals)[first + pos] = 0u;
                else static_cast<uint16_t *>(vals)[first + pos] = 0u;
            }
    }
}

hipError_t launch_entry_count(int elem, const EntrySource &src, uint32_t most_chunks, uint32_t rows, uint32_t *first_chunk, uint32_t *chunk_window,
                              uint32_t *counts, uint32_t *row_len, uint32_t *totals, hipStream_t s)
{
    entry_chunks_kernel<<<dim3(1), 1024, 0, s>>>(src.rowOffset, src.n_windows, first_chunk, chunk_window, totals);
    const dim3 grid((most_chunks + 3u) / 4u);
    if (elem == 4) entry_count_kernel<4><<<grid, 256, 0, s>>>(src, counts);
    else entry_count_kernel<2><<<grid, 256, 0, s>>>(src, counts);
    entry_rows_kernel<<<dim3((rows + 255u) / 256u), 256, 0, s>>>(src, rows, counts, row_len, totals);
    return hipGetLastError();
}

hipError_t launch_entry_fill(int elem, const EntrySource &src, uint32_t most_chunks, const uint32_t *positions, const uint32_t *row_len,
                             uint32_t rows, const EntryPlaces &places, uint32_t *cursors, uint32_t *desc, uint32_t *pieces,
                             uint32_t *row_first, uint32_t *ids, void *vals, hipStream_t s)
{
    entry_place_kernel<<<dim3((rows + 255u) / 256u), 256, 0, s>>>(row_len, rows, places, cursors, desc, pieces, row_first);
    const dim3 grid((most_chunks + 3u) / 4u);
    if (elem == 4) entry_fill_kernel<4><<<grid, 256, 0, s>>>(src, positions, row_len, row_first, rows, ids, vals);
    else entry_fill_kernel<2><<<grid, 256, 0, s>>>(src, positions, row_len, row_first, rows, ids, vals);
    return hipGetLastError();
}

}  // namespace hspmm
