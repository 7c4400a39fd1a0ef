// Host side of the full-tile kernels (spmm_tile_kernel.hip): which plans carry their stream, which launches they take, the
// launch.
#include "hspmm_plan.hpp"

using namespace hspmm_host;

namespace {

// Features of a C tile: the narrowest that covers N, else 64.
uint32_t tile_features(uint32_t N) { return N <= 16u ? 16u : N <= 32u ? 32u : 64u; }

struct TileShape {
    uint32_t nt, n_feat_tiles, n_chunks, n_tiles, groups, share, rest;
    bool cut;                           // C tiles shared by workgroups
    size_t sums_bytes;                  // of their parts
};

TileShape choose_tile_shape(const hspmm_plan *p, uint32_t N)
{
    const hspmm_plan::Tile &t = p->tile;
    TileShape sh;
    sh.nt = tile_features(N);
    sh.n_feat_tiles = (N + sh.nt - 1u) / sh.nt;
    sh.n_chunks = t.n_blocks;
    sh.n_tiles = t.n_row_blocks * sh.n_feat_tiles;
    // Workgroups: one per compute unit while they are short - a workgroup more is a part more to add up, through memory -
    // and from about 9 chunks each (20 of the longer ones of 64 features) more, up to what is resident at a time
    // (pruned to 20 %, 11008 x 4096, N = 16: 256 / 512 / 688 workgroups 16.8 / 14.5 / 14.9 us; 4096 x 4096: 10.9 / 13.6).
    const uint64_t items = uint64_t(sh.n_tiles) * sh.n_chunks, cu = uint64_t(p->compute_units), most = 3u;
    const uint64_t per_cu = std::min<uint64_t>(most, std::max<uint64_t>(1u, items / (cu * (sh.nt >= 64u ? 20u : 9u))));
    sh.groups = uint32_t(std::max<uint64_t>(1u, std::min(cu * per_cu, items / 4u)));
    // Every mode of launching has the same shape, and its parts and counters fit what hspmm_run_static has: the limit is met
    // from 16257 rows on at N = 65 .. 127 (767 workgroups instead of 768) and stays at 511, two per compute unit, for any more.
    const size_t part_bytes = size_t(sh.nt) * hspmm::kTileBlockRows * 4u;
    for (;;) {
        sh.share = uint32_t(items / sh.groups);
        sh.rest = uint32_t(items % sh.groups);
        sh.cut = sh.rest || sh.share % sh.n_chunks;
        sh.sums_bytes = sh.cut ? size_t(hspmm::tile_parts(sh.groups, sh.n_tiles)) * part_bytes : 0u;
        if (sh.sums_bytes + size_t(sh.groups) * 4u <= HSPMM_STATIC_SCRATCH_BYTES) break;
        const size_t any = HSPMM_STATIC_SCRATCH_BYTES / (2u * part_bytes + 4u), few = HSPMM_STATIC_SCRATCH_BYTES / (part_bytes + 4u);
        sh.groups = uint32_t(std::max(any, few > sh.n_tiles ? few - sh.n_tiles : size_t(0)));
    }
    return sh;
}

// Stored entries, as estimated from a sample.
double entries_estimated(const hspmm_plan *p) { return double(p->T) * p->cw * p->per_column; }

// Whether a stream can be made of this matrix, and - unless they are asked for wherever they can - whether it is of the kind they are for.
// Block-clustered weights (over four of a column's eight elements stored) stay with kernels that read whole tiles.
bool tile_suits(const hspmm_plan *p)
{
    using namespace hspmm;
    const uint32_t kk = tile_block_columns(p->dtype), n_blocks = (p->cols + kk - 1u) / kk, n_row_blocks = (p->rows + kTileBlockRows - 1u) / kTileBlockRows;
    if (p->cfg.tile == 0 || !p->canonical || p->cfg.kernel_mode != 0) return false;
    if (p->cols < kk || n_blocks > kTileMaxBlocks || uint64_t(n_blocks) * n_row_blocks >= (1u << 26) || n_row_blocks >= (1u << 23)) return false;
    return p->cfg.tile > 0 || (p->G == 1 && p->per_column <= 4.0 && entries_estimated(p) >= 0.04 * double(p->rows) * p->cols &&
                               (p->elem != 4u || (p->panel.built && p->panel.split)));
}

constexpr uint32_t kMostFloats = 32, kMostHalves = 127;       // features

// Stored entries x features that a launch has at least.
double fewest_products(const hspmm_plan *p) { return p->elem == 4u ? 75e6 : 65e6; }

}  // namespace

namespace hspmm_host {

// Made where some feature dimension would take it (tile_serves) by the stored entries as estimated from a sample.
int build_tile_stream(hspmm_plan *p)
{
    using namespace hspmm;
    hspmm_plan::Tile &t = p->tile;
    // (fp32 storage: an estimate that is off by a twentieth loses no launch)
    const double most = entries_estimated(p) * (p->elem == 4u ? kMostFloats / 0.95 : kMostHalves);
    if (!tile_suits(p) || (p->cfg.tile < 0 && most < fewest_products(p))) return HSPMM_OK;
    const uint32_t kk = tile_block_columns(p->dtype), n_blocks = (p->cols + kk - 1u) / kk, n_row_blocks = (p->rows + kTileBlockRows - 1u) / kTileBlockRows;
    const uint64_t cells = uint64_t(n_blocks) * n_row_blocks;
    const TileSource src{p->d_rowOffset, p->d_rowIdx, p->d_a2b_raw, p->d_data, p->W, p->cols};
    void *room = nullptr;
    if (int rc = plan_alloc(p, (size_t(cells) + 1u) * 4u, &room)) return rc;
    uint32_t *blocks = static_cast<uint32_t *>(room);
    struct Temporary { void *p = nullptr; ~Temporary() { (void)hipFree(p); } } counts;
    HSPMM_HIP(hipMalloc(&counts.p, size_t(cells) * 4u));
    HSPMM_HIP(launch_tile_count(p->dtype, src, n_row_blocks, n_blocks, static_cast<uint32_t *>(counts.p), blocks, nullptr));
    uint32_t units = 0;
    HSPMM_HIP(hipMemcpy(&units, blocks + cells, 4, hipMemcpyDeviceToHost));
    if (units >= (1u << 30)) return HSPMM_OK;
    void *pos = nullptr, *vals = nullptr;
    if (int rc = plan_alloc(p, (size_t(units) + kTileSpareUnits) * 8u, &pos)) return rc;
    if (int rc = plan_alloc(p, (size_t(units) + kTileSpareUnits) * 4u * p->elem, &vals)) return rc;
    HSPMM_HIP(launch_tile_fill(p->dtype, src, n_row_blocks, n_blocks, static_cast<uint32_t *>(counts.p), blocks, pos, vals, nullptr));
    if (int rc = upload(p, &t.d_source, &src, 1)) return rc;
    HSPMM_HIP(hipStreamSynchronize(nullptr));
    t.d_blocks = blocks; t.d_pos = pos; t.d_vals = vals;
    t.entries = uint64_t(units) * 4u;
    t.n_blocks = n_blocks; t.n_row_blocks = n_row_blocks;
    t.built = true;
    return HSPMM_OK;
}

// Narrower than what the LDS-panel kernels take, wider than what the entry kernels are best at.  A chunk costs the same
// whatever it stores, an entry of the other kernels a row of B, so the line goes by entries x N, and by the density for
// large matrices.  Measured (this / the kernels otherwise chosen, us):
//   bf16, 11008 x 4096 at 20 %: N = 8 15 / 18, 16 14.5 / 29, 32 16 / 34, 64 23 / 53;  4096 x 11008 at 10 %: N = 8 18 / 13,
//   16 17 / 21, 32 19.5 / 27, 64 24 / 36;  5003 x 3001 at 20 %: N = 16 10.5 / 10.6, 32 11.7 / 15.2, 64 14.2 / 22;  4096^2 at 10 %:
//   N = 32 12.4 / 8.8, 64 14.5 / 15.4;  fp32, 11008 x 4096 at 20 %: N = 16 24 / 42, 32 28 / 35, 64 36 / 35;
//   4096 x 11008 at 10 %: N = 16 25.7 / 26.6, 32 29 / 34 - but 36 67 / 39, 6000^2 at 15 % 49 / 35: from 33 features on, which leave a C
//   tile ragged, not for fp32.  N = 256 and more: the LDS-panel kernels by a fifth.
// fp32 storage is multiplied in bf16 parts here: only where the LDS-panel kernels would do the same (panel.split; N from 16 on,
// in rows of whole 16-byte pieces).  Other N keep the fp32 products of the entry and gather kernels.
static bool tile_pays(const hspmm_plan *p, double entries, uint32_t N, uint32_t most)
{
    const double fill = entries / (double(p->rows) * p->cols);
    if (p->elem == 4u && !(p->panel.split && panel_serves(p, N))) return false;
    return N >= 8u && N <= most && entries * N >= fewest_products(p) && fill >= 0.04 && fill * N >= 1.5;
}

static bool other_settings(const Config &c) { return c.kernel_mode != 0 || c.buffer_stage || c.consumer_warp_num || c.producer_warp_group_num || c.fused_fixup >= 0; }

bool tile_serves(const hspmm_plan *p, uint32_t N)
{
    if (!p->tile.built || other_settings(p->cfg) || uint64_t(N) * p->elem < 16u) return false;
    const TileShape sh = choose_tile_shape(p, N);
    if (uint64_t(sh.n_tiles) * sh.n_chunks >= (1u << 31) || uint64_t(N) * p->elem >= (1u << 24)) return false;
    return p->cfg.tile > 0 || tile_pays(p, double(p->tile.entries), N, p->elem == 4u ? kMostFloats : kMostHalves);
}

// 33 to 47 features of fp32 storage that would be theirs, by what has been said so far, and are left to the LDS-panel kernels, whose
// arithmetic is the same (or, see entries_serve, to the entry kernels).  A plan need not have their stream for that.
bool tile_leaves(const hspmm_plan *p, uint32_t N)
{
    if (p->elem != 4u || p->cfg.tile > 0 || N <= kMostFloats || other_settings(p->cfg) || !tile_suits(p)) return false;
    return tile_pays(p, p->tile.built ? double(p->tile.entries) : entries_estimated(p), N, 47u);
}

// 16-bit types, from 32 features on: a fit to 1233 launches (standard deviation 10 to 18 %).  33 to 63 features, which leave a C tile of 64
// ragged, take one and a half times as long.
double tile_expected(const hspmm_plan *p, uint32_t N)
{
    const double ragged = N > 32u && N < 64u ? 1.5 : 1.0;
    const double chunks = double(p->tile.n_row_blocks) * p->tile.n_blocks / p->compute_units, tiles = double((N + 63u) / 64u);
    return ragged * (13.3 + (N <= 32u ? 0.14 : 0.49) * chunks * tiles + 0.29e-6 * double(p->tile.entries) * tiles);
}

int run_tile(hspmm_plan *p, const void *dB, void *dC, uint32_t N, hipStream_t s, RunMode mode)
{
    const hspmm_plan::Tile &t = p->tile;
    const TileShape sh = choose_tile_shape(p, N);
    hspmm::TileArgs ta{};
    ta.share = sh.share; ta.rest = sh.rest;
    if (sh.cut) {
        const size_t counters = size_t(sh.groups) * 4u;
        std::lock_guard<std::mutex> lk(p->mu);
        if (mode == RunMode::kStatic) {
            if (const int rc = scratch_for(p, s, sh.sums_bytes + counters, mode, &ta.scratch)) return rc;
            ta.arrive = reinterpret_cast<uint32_t *>(reinterpret_cast<char *>(ta.scratch) + sh.sums_bytes);
            HSPMM_HIP(hspmm::launch_fill_zero(ta.arrive, counters, s));
        } else {
            if (const int rc = scratch_for(p, s, sh.sums_bytes, mode, &ta.scratch)) return rc;
            if (const int rc = ensure_arrive(p, s, sh.groups, mode, &ta.arrive)) return rc;
        }
    }
    if (mode == RunMode::kPrepare) return HSPMM_OK;
    ta.blocks = t.d_blocks; ta.pos = t.d_pos; ta.vals = t.d_vals;
    ta.B = dB; ta.C = dC; ta.rows = p->rows; ta.cols = p->cols; ta.N = N;
    ta.src = t.d_source;
    ta.n_row_blocks = t.n_row_blocks; ta.n_chunks = sh.n_chunks; ta.n_feat_tiles = sh.n_feat_tiles;
    const uint32_t kind = p->dtype == HSPMM_FP16 ? 1u : 2u;
    p->note_launch("spmm_tile_kernel", 3, kind, uint64_t(sh.n_tiles) * sh.n_chunks * (sh.nt / 16u) * 8u * (p->dtype == HSPMM_TF32 ? 3u : 2u));
    HSPMM_HIP(hspmm::launch_spmm_tile(p->dtype, ta, sh.nt, sh.groups, s));
    return HSPMM_OK;
}

}  // namespace hspmm_host
