// Kernels for matrices that are sparse in storage but dense to a workgroup (pruned weights, random matrices from a few per
// cent on): C = A * B by full 128 x 64 blocks of A that are put together in LDS from their stored entries, and the kernels
// that make the entry stream they read from a plan's tiles (the reference's 8-row windows, src/utils/class.h:74-85) on the
// device.
//
// At 10 % density a window of 8 rows touches 57 % of all columns and two of them 81 %: condensing columns saves little,
// costs a row gather per window and streams tiles that are mostly zeros.  Here a stored entry is two bytes of position
// and its value, a row of B is read by 128 rows of A at a time, and every operand of a matrix instruction is shared by
// several of them.
#include "spmm_tile_common.hpp"

namespace hspmm {

constexpr uint32_t kTileRows = 128, kTileImage = 16384;

// Where element (row m, column k) of a block lies in its image of 16 KB, in bytes.  An image is the first operands of the
// matrix instructions, 1 KB each, 16 bytes per lane: rows 16 f .. 16 f + 15, 32 columns.  Lane (g, j) holds row j and the
// columns 4 g .. 4 g + 3 and 16 + 4 g .. 16 + 4 g + 3: with that order the eight rows of B which the transposing LDS
// read takes at a time are consecutive and lie in different banks.
__device__ __forceinline__ uint32_t tile_position(uint32_t m, uint32_t k)
{
    const uint32_t kf = k >> 5, kk = k & 31u, lane = ((kk & 15u) >> 2) * 16u + (m & 15u), i = (kk & 3u) + 4u * (kk >> 4);
    return ((kf * 8u + (m >> 4)) * 512u + lane * 8u + i) * 2u;
}

// Element types.  A block is kK columns; kParts operands of 16 bits per element (fp32 storage: bf16 hi and lo parts, whose
// images follow one another, see Fp32Split in spmm_panel_kernel.hpp).
template <bool BF> struct TileHalf : HalfStored<BF> {
    static constexpr uint32_t kK = 64, kParts = 1;
    typedef t_u32x2 Vals;                                   // four values
    typedef uint16_t Stored;
    __device__ static __forceinline__ Stored stored(const void *tiles, size_t i) { return static_cast<const uint16_t *>(tiles)[i]; }
    __device__ static __forceinline__ void scatter(char *img, const uint32_t (&at)[4], const Vals v)
    {
        *reinterpret_cast<uint16_t *>(img + at[0]) = uint16_t(v[0]);
        *reinterpret_cast<uint16_t *>(img + at[1]) = uint16_t(v[0] >> 16);
        *reinterpret_cast<uint16_t *>(img + at[2]) = uint16_t(v[1]);
        *reinterpret_cast<uint16_t *>(img + at[3]) = uint16_t(v[1] >> 16);
    }
    template <int NT>
    __device__ static __forceinline__ void write_piece(char *row, uint32_t c, const u32x4 x) { *reinterpret_cast<u32x4 *>(row + c * 16u) = x; }
    struct A { u32x4 h; };
    struct B { u32x4 h; };
    __device__ static __forceinline__ A read_a(const char *p) { return {*reinterpret_cast<const u32x4 *>(p)}; }
    template <int NT, uint32_t PITCH>
    __device__ static __forceinline__ B read_b(const char *p);
    __device__ static __forceinline__ f32x4 mma(const A &a, const B &b, f32x4 c) { return HalfOps<BF>::mfma(b.h, a.h, c); }
    // four features of a row of C
    __device__ static __forceinline__ void store(char *p, const f32x4 v)
    {
        t_u32x2 o;
        o[0] = HalfOps<BF>::pack(v[0], v[1]);
        o[1] = HalfOps<BF>::pack(v[2], v[3]);
        *reinterpret_cast<u32x2_any *>(p) = o;
    }
    __device__ static __forceinline__ void store_one(char *p, const float v)
    {
        *reinterpret_cast<uint16_t *>(p) = uint16_t(HalfOps<BF>::pack(v, 0.f));
    }
};

template <bool BF> template <int NT, uint32_t PITCH>
__device__ __forceinline__ typename TileHalf<BF>::B TileHalf<BF>::read_b(const char *p) { return {tile_operand<PITCH>(p)}; }

struct TileSplit : FloatStored {
    static constexpr uint32_t kK = 32, kParts = 2;
    typedef u32x4 Vals;                                     // four values: hi half | lo half << 16
    typedef uint32_t Stored;
    __device__ static __forceinline__ Stored stored(const void *tiles, size_t i)
    {
        const uint32_t v = static_cast<const uint32_t *>(tiles)[i];
        return v >> 16 | pack_bf16_rn(split_rest(v), 0.f) << 16;
    }
    __device__ static __forceinline__ void scatter(char *img, const uint32_t (&at)[4], const Vals v)
    {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            *reinterpret_cast<uint16_t *>(img + at[i]) = uint16_t(v[i]);
            *reinterpret_cast<uint16_t *>(img + at[i] + kTileImage / 2u) = uint16_t(v[i] >> 16);
        }
    }
    template <int NT>
    __device__ static __forceinline__ void write_piece(char *row, uint32_t c, const u32x4 x)
    {
        u32x2 hi, lo;
        hi[0] = __builtin_amdgcn_perm(x[1], x[0], 0x07060302u);
        hi[1] = __builtin_amdgcn_perm(x[3], x[2], 0x07060302u);
        lo[0] = pack_bf16_rn(split_rest(x[0]), split_rest(x[1]));
        lo[1] = pack_bf16_rn(split_rest(x[2]), split_rest(x[3]));
        *reinterpret_cast<u32x2 *>(row + c * 8u) = hi;
        *reinterpret_cast<u32x2 *>(row + NT * 2u + c * 8u) = lo;
    }
    struct A { u32x4 hi, lo; };
    struct B { u32x4 hi, lo; };
    __device__ static __forceinline__ A read_a(const char *p)
    {
        return {*reinterpret_cast<const u32x4 *>(p), *reinterpret_cast<const u32x4 *>(p + kTileImage / 2u)};
    }
    template <int NT, uint32_t PITCH>
    __device__ static __forceinline__ B read_b(const char *p) { return {tile_operand<PITCH>(p), tile_operand<PITCH>(p + NT * 2)}; }
    __device__ static __forceinline__ f32x4 mma(const A &a, const B &b, f32x4 c)
    {
        // small terms first, as in PanelOps<Fp32Split>
        c = HalfOps<true>::mfma(b.hi, a.lo, c);
        c = HalfOps<true>::mfma(b.lo, a.hi, c);
        return HalfOps<true>::mfma(b.hi, a.hi, c);
    }
    __device__ static __forceinline__ void store(char *p, const f32x4 v)
    {
        typedef f32x4 f32x4_any __attribute__((aligned(4)));
        *reinterpret_cast<f32x4_any *>(p) = v;
    }
};

// 16 bytes from `back` (< 16) bytes further on in the 16 loaded, zeros behind them.
__device__ __forceinline__ u32x4 shift_down(u32x4 v, uint32_t back)
{
    if (back & 8u) { v[0] = v[2]; v[1] = v[3]; v[2] = 0u; v[3] = 0u; }
    if (back & 4u) { v[0] = v[1]; v[1] = v[2]; v[2] = v[3]; v[3] = 0u; }
    const uint32_t b = back & 3u;
    u32x4 o;
    o[0] = __builtin_amdgcn_alignbyte(v[1], v[0], b);
    o[1] = __builtin_amdgcn_alignbyte(v[2], v[1], b);
    o[2] = __builtin_amdgcn_alignbyte(v[3], v[2], b);
    o[3] = __builtin_amdgcn_alignbyte(0u, v[3], b);
    return o;
}

// A workgroup of four waves multiplies blocks of 128 rows x K columns with K rows x NT features of B: WR waves share out
// the rows and 4 / WR the features.  The chunks of all C tiles (row block slowest, then features, then columns) are one
// row of n_tiles x n_chunks items that the workgroups divide evenly; where a C tile is cut, its parts leave their sums in
// memory and the workgroup that brings the last part adds them in order.
// Two LDS buffers.  While one is multiplied, the other is cleared, B is written to it and - a barrier later, between the
// two halves of the multiplication - the stored entries; what they come from was requested a chunk earlier.
// What bounds it: the chain of a chunk - clear, write, barrier, operands, multiply, twice - which three or four waves per
// SIMD cover in part (0.55 us per 128 x 64 x 64 chunk and compute unit, 0.35 with 16 features; matrix instructions 0.1), and
// 6 to 8 us of launch, first loads and sums of parts: pruned to 20 %, 11008 x 4096, bf16, N = 32: 16.4 us where the gather
// kernels took 34.5.  Counted, 4096 x 11008 at 10 %, bf16, N = 16, 17.1 us: matrix instructions busy for 4 % of the time, the L1s'
// return path for 28 %, 14 requests under way per compute unit.  Tiles of 128 features and fp32 storage from N = 48 on measured slower than the LDS-panel kernels.
template <class E, int NT, int WR, int OCC, bool RAGGED>
__global__ __launch_bounds__(256, OCC)
void spmm_tile_kernel(const TileArgs ta)
{
    constexpr int WC = 4 / WR, RF = 8 / WR, CF = NT / 16 / WC;
    constexpr uint32_t K = E::kK, kLine = NT * 2u * E::kParts, kPitch = kLine + ((kLine / 32u) % 2u ? 0u : 32u);
    constexpr uint32_t kPieces = NT * E::kElem / 16u;               // 16-byte pieces of a row of B
    constexpr int kPer = K * kPieces < 256u ? 1 : int(K * kPieces / 256u), kUnits = 2;   // pieces and (at least) units of entries a thread takes
    constexpr uint32_t kA = kTileImage, kB = K * kPitch;
    static_assert(uint32_t(kPer) * 256u % (K * kPieces) == 0u, "the pieces of a chunk must divide among the threads");
    __shared__ __attribute__((aligned(16))) char smem[2u * (kA + kB)];
    __shared__ uint32_t last_part;

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wr = wave / WC, wc = wave % WC;
    // consecutive items on one XCD (workgroups are dealt out to the eight in turn): the feature tiles of a row block
    // share its entries, neighbours their rows of B
    const uint32_t n_groups = gridDim.x, xcd = blockIdx.x & 7u;
    const uint32_t group = xcd * (n_groups >> 3) + umin32(xcd, n_groups & 7u) + (blockIdx.x >> 3);
    const uint32_t begin = group * ta.share + umin32(group, ta.rest), end = begin + ta.share + (group < ta.rest ? 1u : 0u);
    const uint32_t n_chunks = ta.n_chunks;
    const const_u32_ptr blocks = as_const(ta.blocks);

    struct Cursor { uint32_t tile, k, rb, ft; };
    auto advance = [&](Cursor &c) __attribute__((always_inline)) {
        if (++c.k == n_chunks) { c.k = 0; ++c.tile; if (++c.ft == ta.n_feat_tiles) { c.ft = 0; ++c.rb; } }
    };
    Cursor now;
    now.tile = begin / n_chunks; now.k = begin - now.tile * n_chunks;
    now.rb = now.tile / ta.n_feat_tiles; now.ft = now.tile - now.rb * ta.n_feat_tiles;
    Cursor ahead = now;                                             // what is requested next

    const uint32_t row_bytes = ta.N * E::kElem;
    const uint32_t piece_row = tid % (K * kPieces) / kPieces, piece_col = tid % kPieces;      // (16 features: every piece twice)
    // a feature dimension that ends inside its only tile: a piece that reaches past the row is read from where it ends there
    const uint32_t col_bytes = RAGGED ? umin32(piece_col * 16u, row_bytes - 16u) : piece_col * 16u;
    const uint32_t shift = RAGGED ? umin32(piece_col * 16u - col_bytes, 15u) : 0u;
    auto first_feature = [&](uint32_t ft) __attribute__((always_inline)) -> uint32_t {
        return RAGGED ? 0u : umin32(ft * NT, ta.N - NT);            // (the last tile is moved back to end with the row)
    };

    uint32_t piece_off[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) piece_off[i] = (piece_row + uint32_t(i) * (256u / kPieces)) * row_bytes + col_bytes;
    // Two sets of what is on its way: chunk j is in set (j - begin) % 2, requested three chunks in front of its use.
    u32x4 piece[2][kPer];
    t_u32x2 pos[2][kUnits];
    typename E::Vals val[2][kUnits];
    uint32_t unit0[2], units[2];                                    // units of entries of the chunk in a set
    uint32_t next_unit0 = 0, next_units = 0;                        // of the chunk `ahead` (looked up a chunk in front of its request)
    auto look_up = [&]() __attribute__((always_inline)) {
        const uint32_t b = ahead.rb * n_chunks + ahead.k;
        next_unit0 = blocks[b];
        next_units = blocks[b + 1u] - next_unit0;
    };
    auto request = [&](auto set_c) __attribute__((always_inline)) {
        constexpr int S = decltype(set_c)::value;
        // uniform bases and offsets that stay the same from chunk to chunk: no address arithmetic in the vector units
        const char *src = reinterpret_cast<const char *>(ta.B) + size_t(tile_first_column(ahead.k, K, ta.cols)) * row_bytes +
                          first_feature(ahead.ft) * E::kElem;
#pragma unroll
        for (int i = 0; i < kPer; ++i) piece[S][i] = *reinterpret_cast<const u32x4_any *>(src + piece_off[i]);
        unit0[S] = next_unit0; units[S] = next_units;
        // (a thread whose unit lies behind the block's last one reads what follows: not used, and the arrays end with
        // kTileSpareUnits spare units)
        const char *src_pos = static_cast<const char *>(ta.pos) + size_t(next_unit0) * 8u;
        const char *src_val = static_cast<const char *>(ta.vals) + size_t(next_unit0) * sizeof(typename E::Vals);
#pragma unroll
        for (int j = 0; j < kUnits; ++j) {
            pos[S][j] = *reinterpret_cast<const t_u32x2 *>(src_pos + (tid * 8u + uint32_t(j) * 2048u));
            val[S][j] = *reinterpret_cast<const typename E::Vals *>(src_val + (tid * uint32_t(sizeof(typename E::Vals)) + uint32_t(j) * 256u * uint32_t(sizeof(typename E::Vals))));
        }
    };
    auto write_b = [&](const uint32_t buf, auto set_c) __attribute__((always_inline)) {
        constexpr int S = decltype(set_c)::value;
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            u32x4 x = piece[S][i];
            if constexpr (RAGGED) x = shift_down(x, shift);
            E::template write_piece<NT>(smem + buf + (piece_row + uint32_t(i) * (256u / kPieces)) * kPitch, piece_col, x);
        }
    };
    auto clear_a = [&](const uint32_t buf) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t i = 0; i < kA / 4096u; ++i) *reinterpret_cast<u32x4 *>(smem + buf + i * 4096u + tid * 16u) = u32x4{0u, 0u, 0u, 0u};
    };
    auto put = [&](const uint32_t buf, const t_u32x2 p, const typename E::Vals v) __attribute__((always_inline)) {
        const uint32_t at[4] = {p[0] & 0xFFFFu, p[0] >> 16, p[1] & 0xFFFFu, p[1] >> 16};
        E::scatter(smem + buf, at, v);
    };
    auto scatter = [&](const uint32_t buf, auto set_c) __attribute__((always_inline)) {
        constexpr int S = decltype(set_c)::value;
#pragma unroll
        for (int j = 0; j < kUnits; ++j)
            if (tid + uint32_t(j) * 256u < units[S]) put(buf, pos[S][j], val[S][j]);
        for (uint32_t u = tid + kUnits * 256u; u < units[S]; u += 256u)      // (blocks over a quarter full)
            put(buf, reinterpret_cast<const t_u32x2 *>(ta.pos)[unit0[S] + u], reinterpret_cast<const typename E::Vals *>(ta.vals)[unit0[S] + u]);
    };

    f32x4 acc[RF][CF];
#pragma unroll
    for (int r = 0; r < RF; ++r)
#pragma unroll
        for (int p = 0; p < CF; ++p) acc[r][p] = f32x4{0.f, 0.f, 0.f, 0.f};
    // rows r0 .. r1 - 1 of the wave's RF times 32 columns
    const uint32_t a_lane = wr * RF * 1024u + lane * 16u;
    const uint32_t b_lane = (4u * (lane >> 4) + ((lane & 15u) >> 2)) * kPitch + (lane & 3u) * 8u + wc * CF * 32u;
    auto multiply = [&](const uint32_t a, const uint32_t b, auto kf_c, auto r0_c, auto r1_c) __attribute__((always_inline)) {
        constexpr int kf = decltype(kf_c)::value, r0 = decltype(r0_c)::value, r1 = decltype(r1_c)::value;
        constexpr uint32_t kFrag = uint32_t(kf) * 8192u;
        typename E::A fa[r1 - r0];
        typename E::B fb[CF];
#pragma unroll
        for (int r = r0; r < r1; ++r) fa[r - r0] = E::read_a(smem + a + a_lane + kFrag + uint32_t(r) * 1024u);
#pragma unroll
        for (int p = 0; p < CF; ++p) fb[p] = E::template read_b<NT, kPitch>(smem + b + b_lane + uint32_t(kf) * 32u * kPitch + uint32_t(p) * 32u);
#pragma unroll
        for (int r = r0; r < r1; ++r)
#pragma unroll
            for (int p = 0; p < CF; ++p) acc[r][p] = E::mma(fa[r - r0], fb[p], acc[r][p]);
    };
    auto half = [&](const uint32_t a, const uint32_t b, auto h_c) __attribute__((always_inline)) {
        constexpr int h = decltype(h_c)::value, frags = int(K / 32u);
        if constexpr (frags == 1) {
            multiply(a, b, std::integral_constant<int, 0>{}, std::integral_constant<int, h * RF / 2>{}, std::integral_constant<int, (h + 1) * RF / 2>{});
        } else {
            multiply(a, b, std::integral_constant<int, h>{}, std::integral_constant<int, 0>{}, std::integral_constant<int, RF>{});
        }
    };

    auto store_tile = [&]() __attribute__((always_inline)) {
        const uint32_t f0 = first_feature(now.ft), own = now.ft * NT;    // features below `own` belong to the tile in front
#pragma unroll
        for (int r = 0; r < RF; ++r) {
            const uint32_t row = now.rb * kTileRows + (wr * RF + uint32_t(r)) * 16u + (lane & 15u);
            if (row >= ta.rows) continue;
            char *c_row = reinterpret_cast<char *>(ta.C) + size_t(row) * row_bytes;
#pragma unroll
            for (int p = 0; p < CF; ++p) {
                const uint32_t f = f0 + (wc * CF + uint32_t(p)) * 16u + (lane >> 4) * 4u;
                if (f >= own && f + 4u <= ta.N) E::store(c_row + size_t(f) * E::kElem, acc[r][p]);
                else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (f + e >= own && f + e < ta.N) { const float v = acc[r][p][e]; E::store_one(c_row + size_t(f + e) * E::kElem, v); }
                }
            }
        }
    };
    // The workgroup that has item i, as `begin` above deals them out.
    auto owner = [&](uint32_t i) __attribute__((always_inline)) -> uint32_t {
        const uint32_t longer = ta.rest * (ta.share + 1u);
        return i < longer ? i / (ta.share + 1u) : ta.rest + (i - longer) / ta.share;
    };
    // Where the sums of workgroup g's part of tile t go (see tile_parts).
    auto part = [&](uint32_t g, uint32_t t) __attribute__((always_inline)) -> uint32_t {
        if (ta.n_row_blocks * ta.n_feat_tiles <= n_groups) return g + t;
        return 2u * g + (g * ta.share + umin32(g, ta.rest) < t * n_chunks ? 1u : 0u);
    };
    // The first to the last C tile whose sums this wave has found not finite (it has finished all between them: only the first
    // and the last tile of a workgroup may be another's to finish).
    uint32_t again_begin = 0, again_end = 0;
    auto finish = [&](uint32_t k_first, uint32_t k_last) __attribute__((always_inline)) {
        if (k_first != 0u || k_last + 1u != n_chunks) {
            constexpr uint32_t kSums = RF * CF * 4096u;             // bytes of a part
            const uint32_t first = owner(now.tile * n_chunks), count = owner((now.tile + 1u) * n_chunks - 1u) - first + 1u;
            {
                const __amdgpu_buffer_rsrc_t out = device_scope_buffer(reinterpret_cast<char *>(ta.scratch) + size_t(part(group, now.tile)) * kSums);
#pragma unroll
                for (int i = 0; i < RF * CF; ++i) store_device_scope(out, uint32_t(i) * 4096u + tid * 16u, acc[i / CF][i % CF]);
            }
            wait_stores_acknowledged();
            __syncthreads();
            if (tid == 0u) {
                const uint32_t old = __hip_atomic_fetch_add(ta.arrive + first, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                last_part = old + 1u == count;
                if (old + 1u == count) __hip_atomic_store(ta.arrive + first, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            __syncthreads();
            asm volatile("" ::: "memory");
            if (!__builtin_amdgcn_readfirstlane(last_part)) return;
#pragma unroll
            for (int i = 0; i < RF * CF; ++i) acc[i / CF][i % CF] = f32x4{0.f, 0.f, 0.f, 0.f};
            for (uint32_t s = 0; s < count; ++s) {
                const __amdgpu_buffer_rsrc_t in = device_scope_buffer(reinterpret_cast<const char *>(ta.scratch) + size_t(part(first + s, now.tile)) * kSums);
#pragma unroll
                for (int i = 0; i < RF * CF; ++i) acc[i / CF][i % CF] += load_device_scope(in, uint32_t(i) * 4096u + tid * 16u);
            }
        }
        store_tile();
        // An infinity or a NaN in B makes every sum of its feature NaN - the images hold a zero wherever no entry is - and a sum
        // that is finite has met none (0 times a finite sum is 0).  What is not finite is summed again at the end.
        float met = 0.f;
#pragma unroll
        for (int i = 0; i < RF * CF * 4; ++i) met = __builtin_fmaf(acc[i / (4 * CF)][i / 4 % CF][i % 4], 0.f, met);
        if (__ballot(met != 0.f)) { if (again_end == 0u) again_begin = now.tile; again_end = now.tile + 1u; }
    };

    if (begin >= end) return;
    typedef std::integral_constant<int, 0> Set0;
    typedef std::integral_constant<int, 1> Set1;
    uint32_t left = end - begin;                                    // chunks behind `ahead`'s, itself included
    // past the last chunk: that chunk again (its loads hit, and nothing uses them)
    auto step_ahead = [&]() __attribute__((always_inline)) { if (left > 1u) { --left; advance(ahead); } look_up(); };
    look_up();
    request(Set0{});
    step_ahead();
    request(Set1{});
    clear_a(0u);
    step_ahead();
    panel_barrier();
    scatter(0u, Set0{});
    write_b(2u * kA, Set0{});
    request(Set0{});
    step_ahead();
    uint32_t k_first = now.k;
    // chunk i, which is in LDS buffers S; the chunk behind it is in set S ^ 1, the one behind that on its way to set S
    auto chunk = [&](const uint32_t i, auto set_c) __attribute__((always_inline)) {
        constexpr uint32_t S = decltype(set_c)::value;
        typedef std::integral_constant<int, int(S ^ 1u)> Other;
        constexpr uint32_t a = S * kA, b = 2u * kA + S * kB, a_next = kA - a, b_next = 4u * kA + kB - b;
        panel_barrier();                                            // this chunk is in its buffers, the other ones are free
        clear_a(a_next);
        half(a, b, Set0{});
        write_b(b_next, Other{});
        panel_barrier();                                            // cleared
        scatter(a_next, Other{});
        request(Other{});
        step_ahead();
        half(a, b, Set1{});
        if (now.k + 1u == n_chunks || i + 1u == end) {
            finish(k_first, now.k);
#pragma unroll
            for (int r = 0; r < RF; ++r)
#pragma unroll
                for (int p = 0; p < CF; ++p) acc[r][p] = f32x4{0.f, 0.f, 0.f, 0.f};
            k_first = 0u;
        }
        advance(now);
    };
    // (pairs of chunks, the odd one behind the loop: the compiler counts outstanding loads per path, and a path from a first
    // chunk to the next first chunk would have every wait in the loop wait for everything)
    uint32_t i = begin;
    for (; i + 1u < end; i += 2u) {
        chunk(i, Set0{});
        chunk(i + 1u, Set1{});
    }
    if (i < end) chunk(i, Set0{});
    for (uint32_t t = again_begin; t < again_end; ++t) {
        const uint32_t rb = t / ta.n_feat_tiles, ft = t - rb * ta.n_feat_tiles;
        tile_sum_again<E, RF, CF * 16u>(ta, rb * kTileRows + wr * RF * 16u, first_feature(ft) + wc * CF * 16u, ft * NT, ta.N, lane);
    }
}

template <class E>
static hipError_t launch_tile_e(const TileArgs &ta, uint32_t nt, uint32_t groups, hipStream_t s)
{
    const bool ragged = ta.N < nt;
#define HSPMM_TILE(NT, WR, OCC) \
    if (nt == NT) { \
        if (ragged) spmm_tile_kernel<E, NT, WR, OCC, true><<<dim3(groups), 256, 0, s>>>(ta); \
        else spmm_tile_kernel<E, NT, WR, OCC, false><<<dim3(groups), 256, 0, s>>>(ta); \
        return hipGetLastError(); \
    }
    HSPMM_TILE(16, 4, 4) HSPMM_TILE(32, 4, 3) HSPMM_TILE(64, 2, 3)
#undef HSPMM_TILE
    return hipErrorInvalidValue;
}

uint32_t tile_block_columns(int dtype) { return dtype == kDtypeF32 ? TileSplit::kK : TileHalf<false>::kK; }

hipError_t launch_spmm_tile(int dtype, const TileArgs &ta, uint32_t nt, uint32_t groups, hipStream_t s)
{
    const uint64_t items = uint64_t(groups) * ta.share + ta.rest, elem = dtype == kDtypeF32 ? 4u : 2u;
    // (a piece of B stays inside the row, the items are all there, every group has one)
    if (ta.N * elem < 16u || ta.cols < tile_block_columns(dtype) || !groups || ta.rest >= groups || !ta.share || items != uint64_t(ta.n_chunks) * ta.n_feat_tiles * ta.n_row_blocks ||
        uint64_t(ta.n_feat_tiles) * nt < ta.N || uint64_t(ta.n_row_blocks) * kTileRows < ta.rows)
        return hipErrorInvalidValue;
    if (dtype == kDtypeF32) return launch_tile_e<TileSplit>(ta, nt, groups, s);
    if (dtype == kDtypeBf16) return launch_tile_e<TileHalf<true>>(ta, nt, groups, s);
    return launch_tile_e<TileHalf<false>>(ta, nt, groups, s);
}

// ---------------------------------------------------------------------------
// The entry stream from the plan's tiles: a workgroup per row block, whose tiles follow one another.
// ---------------------------------------------------------------------------

// counts[row block][block]: stored entries
template <class E>
__global__ __launch_bounds__(256) void tile_count_kernel(const TileSource src, uint32_t n_blocks, uint32_t *__restrict__ counts)
{
    __shared__ uint32_t seen[kTileMaxBlocks];
    for (uint32_t i = threadIdx.x; i < n_blocks; i += 256u) seen[i] = 0u;
    __syncthreads();
    for_entries<E>(src, blockIdx.x * kTileRows, kTileRows, [&](uint32_t, uint32_t id, size_t) { atomicAdd(&seen[id / E::kK], 1u); });
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < n_blocks; i += 256u) counts[size_t(blockIdx.x) * n_blocks + i] = seen[i];
}

// blocks[i]: units of four entries in front of block i (n + 1 of them).  One workgroup.
__global__ __launch_bounds__(1024) void tile_scan_kernel(const uint32_t *__restrict__ counts, uint32_t n, uint32_t *__restrict__ blocks)
{
    __shared__ uint32_t sums[1024];
    const uint32_t per = (n + 1023u) / 1024u, b = umin32(threadIdx.x * per, n), e = umin32(b + per, n);
    uint32_t sum = 0;
    for (uint32_t i = b; i < e; ++i) sum += (counts[i] + 3u) / 4u;
    sums[threadIdx.x] = sum;
    __syncthreads();
    for (uint32_t m = 1u; m < 1024u; m <<= 1) {
        const uint32_t x = threadIdx.x >= m ? sums[threadIdx.x - m] : 0u;
        __syncthreads();
        sums[threadIdx.x] += x;
        __syncthreads();
    }
    uint32_t at = threadIdx.x ? sums[threadIdx.x - 1u] : 0u;
    for (uint32_t i = b; i < e; ++i) { blocks[i] = at; at += (counts[i] + 3u) / 4u; }
    if (threadIdx.x == 1023u) blocks[n] = sums[1023];
}

// Positions and values to their places (in any order inside a block: they go to different places of its image); the last
// unit of a block is filled up with its last entry.
template <class E>
__global__ __launch_bounds__(256) void tile_fill_kernel(const TileSource src, uint32_t n_blocks, const uint32_t *__restrict__ counts,
                                                        const uint32_t *__restrict__ blocks, uint16_t *__restrict__ pos, void *__restrict__ vals)
{
    __shared__ uint32_t next[kTileMaxBlocks];
    for (uint32_t i = threadIdx.x; i < n_blocks; i += 256u) next[i] = 0u;
    __syncthreads();
    const size_t base = size_t(blockIdx.x) * n_blocks;
    for_entries<E>(src, blockIdx.x * kTileRows, kTileRows, [&](uint32_t m, uint32_t id, size_t e) {
        const uint32_t b = id / E::kK, p = atomicAdd(&next[b], 1u), n = counts[base + b];
        const uint16_t where = uint16_t(tile_position(m, id - tile_first_column(b, E::kK, src.cols)));
        const typename E::Stored v = E::stored(src.tiles, e);
        const size_t at = size_t(blocks[base + b]) * 4u;
        for (uint32_t i = p; i < (p + 1u == n ? (n + 3u) & ~3u : p + 1u); ++i) {
            pos[at + i] = where;
            static_cast<typename E::Stored *>(vals)[at + i] = v;
        }
    });
}

hipError_t launch_tile_scan(const uint32_t *counts, uint32_t n, uint32_t *blocks, hipStream_t s)
{
    tile_scan_kernel<<<dim3(1), 1024, 0, s>>>(counts, n, blocks);
    return hipGetLastError();
}

hipError_t launch_tile_count(int dtype, const TileSource &src, uint32_t n_row_blocks, uint32_t n_blocks, uint32_t *counts, uint32_t *blocks, hipStream_t s)
{
    if (n_blocks > kTileMaxBlocks || !n_row_blocks) return hipErrorInvalidValue;
    if (dtype == kDtypeF32) tile_count_kernel<TileSplit><<<dim3(n_row_blocks), 256, 0, s>>>(src, n_blocks, counts);
    else tile_count_kernel<TileHalf<false>><<<dim3(n_row_blocks), 256, 0, s>>>(src, n_blocks, counts);
    if (hipError_t e = hipGetLastError()) return e;
    return launch_tile_scan(counts, n_row_blocks * n_blocks, blocks, s);
}

hipError_t launch_tile_fill(int dtype, const TileSource &src, uint32_t n_row_blocks, uint32_t n_blocks, const uint32_t *counts,
                            const uint32_t *blocks, void *pos, void *vals, hipStream_t s)
{
    if (dtype == kDtypeF32) tile_fill_kernel<TileSplit><<<dim3(n_row_blocks), 256, 0, s>>>(src, n_blocks, counts, blocks, static_cast<uint16_t *>(pos), vals);
    else tile_fill_kernel<TileHalf<false>><<<dim3(n_row_blocks), 256, 0, s>>>(src, n_blocks, counts, blocks, static_cast<uint16_t *>(pos), vals);
    return hipGetLastError();
}

}  // namespace hspmm
