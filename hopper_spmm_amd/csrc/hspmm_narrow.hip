// Host side of the narrow kernels (spmm_narrow_kernel.hip): which plans carry their stream, which launches they take and in which
// shape, the launch.
#include "hspmm_plan.hpp"

using namespace hspmm_host;

namespace {

// A launch takes `start` us, `round` us for every round of workgroups (16 waves are resident on a compute unit), `chain` us for every block of
// a wave in these rounds, and `block` + 1e-4 x (entries of a block) us for every block of the busiest compute unit; odd N a twentieth
// more.  A fit to 2075 launches of 460 pruned matrices at 2.5 to 30 %, N = 1 to 32, each with 4, 8 and 16 waves: standard deviations of 7 to
// 10 %, and the number of waves it picks is 0.3 % behind the fastest on average, 2 % at the 95th percentile.
struct Cost { uint32_t waves; double start, round, chain, block; };
const Cost kCosts[2][3] = {
    {{4, 2.6, 0.0, 0.364, 0.029}, {8, 2.0, 0.8, 0.239, 0.035}, {16, 1.9, 0.84, 0.0, 0.049}},
    {{4, 2.75, 0.0, 0.441, 0.050}, {8, 2.2, 0.77, 0.241, 0.063}, {16, 1.5, 1.22, 0.0, 0.077}},
};
constexpr double kFewestEntries = 0.028, kMostEntries = 0.31;         // of all
constexpr uint32_t kMostRowsTwoTiles = 16384;                         // see narrow_serves

uint32_t one_tile(uint32_t N) { return N % 2u ? 15u : 16u; }
uint32_t most_features(uint32_t N) { return N % 2u ? 29u : 32u; }

double per_block(const hspmm_plan::Narrow &n) { return double(n.entries) / (double(n.n_units) * n.n_blocks); }

// The waves of a workgroup, a function of the plan and N alone, and the time that a launch is expected to take; 0: none will do.
uint32_t choose_waves(const hspmm_plan *p, uint32_t N, double *expected)
{
    const hspmm_plan::Narrow &n = p->narrow;
    const double cu = double(p->compute_units), units = double(n.n_units), entries = per_block(n);
    uint32_t best = 0;
    for (const Cost &c : kCosts[N > one_tile(N)]) {
        if (n.n_blocks > 64u * c.waves || (p->cfg.narrow_waves > 0 && uint32_t(p->cfg.narrow_waves) != c.waves)) continue;
        const double of_wave = double((n.n_blocks + c.waves - 1u) / c.waves), rounds = std::ceil(units * c.waves / (16.0 * cu));
        const double t = (c.start + rounds * (c.round + of_wave * c.chain) + of_wave * c.waves * std::ceil(units / cu) * (c.block + 1e-4 * entries)) *
                         (N % 2u ? 1.05 : 1.0);
        if (!best || t < *expected) { best = c.waves; *expected = t; }
    }
    return best;
}

}  // namespace

namespace hspmm_host {

// Made where some feature dimension would take it by the stored entries as estimated from a sample.  Block-clustered weights (over four
// of a column's eight elements stored) stay with kernels that read whole tiles, and plans that keep the caller's cuts of windows with
// kernels that walk windows.
int build_narrow_stream(hspmm_plan *p)
{
    using namespace hspmm;
    hspmm_plan::Narrow &n = p->narrow;
    if (p->elem != 2u || p->cfg.narrow == 0 || !p->canonical || p->cfg.kernel_mode != 0 || !p->T || p->W >= (1u << 23) || p->cols < 2u || !p->caller_cuts.empty()) return HSPMM_OK;
    const double fill = double(p->T) * p->cw * p->per_column / (double(p->rows) * p->cols);
    if (p->cfg.narrow < 0 && (p->G != 1 || p->per_column > 4.0 || fill < kFewestEntries || fill > 1.1 * kMostEntries)) return HSPMM_OK;
    const uint32_t n_units = (p->rows + 15u) / 16u, n_blocks = (p->cols + kNarrowColumns - 1u) / kNarrowColumns;
    if (n_blocks > kNarrowMostBlocks || uint64_t(n_units) * n_blocks >= (1u << 28) || n_units >= (1u << 21)) return HSPMM_OK;
    const uint32_t all = n_units * n_blocks;
    const TileSource src{p->d_rowOffset, p->d_rowIdx, p->d_a2b_raw, p->d_data, p->W, p->cols};
    // (a plan whose device memory does not hold the stream, or what it takes to make it, is made without)
    const size_t blocks_bytes = (size_t(all) + 1u) * 4u;
    void *blocks = nullptr, *entries = nullptr, *source = nullptr;
    struct Temporary { void *p = nullptr; ~Temporary() { (void)hipFree(p); } } counts;
    auto without = [&]() {
        (void)hipGetLastError();
        plan_release(p, blocks, blocks_bytes);
        plan_release(p, source, sizeof src);
        return HSPMM_OK;
    };
    if (plan_alloc(p, blocks_bytes, &blocks) || plan_alloc(p, sizeof src, &source) || hipMalloc(&counts.p, size_t(all) * 4u) != hipSuccess) return without();
    HSPMM_HIP(launch_narrow_count(src, n_units, n_blocks, static_cast<uint32_t *>(counts.p), static_cast<uint32_t *>(blocks), nullptr));
    uint32_t fours = 0;
    HSPMM_HIP(hipMemcpy(&fours, static_cast<uint32_t *>(blocks) + all, 4, hipMemcpyDeviceToHost));
    if (fours >= (1u << 30) || plan_alloc(p, size_t(fours) * 16u, &entries)) return without();
    HSPMM_HIP(launch_narrow_fill(src, n_units, n_blocks, static_cast<uint32_t *>(counts.p), static_cast<uint32_t *>(blocks), static_cast<uint32_t *>(entries), nullptr));
    HSPMM_HIP(hipMemcpy(source, &src, sizeof src, hipMemcpyHostToDevice));
    HSPMM_HIP(hipStreamSynchronize(nullptr));
    n.d_blocks = static_cast<uint32_t *>(blocks); n.d_entries = static_cast<uint32_t *>(entries); n.d_source = static_cast<TileSource *>(source);
    n.entries = uint64_t(fours) * 4u;
    n.n_units = n_units; n.n_blocks = n_blocks;
    n.built = true;
    return HSPMM_OK;
}

// Where they are expected to be faster than the kernels that would take the launch: by 10 % than the wide-tile and the entry
// kernels, and by 0.3 us more than these (whose short launches are faster than the fit says); the full-tile and the gather kernels lose every
// launch but 2 of 249 (by 2 %).  Over 2075 launches the rule gives 1.22 times the speed of the entry kernels (1.27 if every launch took the
// faster one; 5 % of those taken lose, 5 % on average).  Up to 31 % of entries, as far as times are known.
// 480 launches taken, six to 48 matrices of 800 MB together in turn, whose streams come from memory / one matrix over and over, old time
// over new: entry kernels 1.65 / 1.48, full-tile 1.21 / 1.34, gather 2.2 / 2.0; 7 / 23 lose more than 3 %, up to 20 %, most of them of less than 10 us.
// Matrices of more rows than those of the fit take many rounds of workgroups, and with more than one tile of features the full-tile kernels, which
// put a block of A together once for 128 rows, are ahead (39040 x 5440 at 15 %, N = 32 52.1 / 41.6 us, 21888 x 5952 at 11 % 34.4 / 29.4,
// but N = 16 25.0 / 26.1).
// B that begins between two words makes these kernels half as slow again, and with two tiles of features 1.7 times; the full-tile and wide-tile
// kernels take as long as ever, the entry kernels 1.5 times, but not at up to eight features (8704 x 5120 at 5 %, N = 32 34 us, full tiles
// 17.9; 12800 x 1963 at 9 %, N = 2 12.5, entries 6.8, N = 16 12.6, entries 16.8).
bool narrow_serves(const hspmm_plan *p, uint32_t N, bool on_word)
{
    const Config &c = p->cfg;
    if (!p->narrow.built || c.kernel_mode != 0 || !N || N > most_features(N)) return false;
    double expected = 0.0;
    if (!choose_waves(p, N, &expected)) return false;
    if (c.narrow > 0) return true;
    // (settings of other kernels)
    if (c.buffer_stage || c.consumer_warp_num || c.producer_warp_group_num || c.fused_fixup >= 0 || c.panel_chunks || c.panel_max_windows ||
        c.panel_units_per_group || c.aligned_small >= 0 || c.xcd_split >= 0 || c.gather_bitmap >= 0 || c.tile > 0 || c.entries > 0 || c.wide > 0)
        return false;
    if (double(p->narrow.entries) > kMostEntries * p->rows * p->cols) return false;
    if (!on_word && (wide_serves(p, N) || tile_serves(p, N) || (N <= 8u && entries_serve(p, N)))) return false;
    if (wide_serves(p, N)) return expected < 0.9 * p->wide.expected_fewest;     // (N = 32)
    if (tile_serves(p, N)) return N <= one_tile(N) || p->rows <= kMostRowsTwoTiles;
    if (entries_serve(p, N)) return expected < 0.9 * entries_expected(p, N) - 0.3;
    return !panel_serves(p, N);
}

int run_narrow(hspmm_plan *p, const void *dB, void *dC, uint32_t N, hipStream_t s, RunMode mode)
{
    if (mode == RunMode::kPrepare) return HSPMM_OK;
    const hspmm_plan::Narrow &n = p->narrow;
    double expected = 0.0;
    const uint32_t waves = choose_waves(p, N, &expected);
    hspmm::NarrowArgs na{};
    na.blocks = n.d_blocks; na.entries = n.d_entries;
    na.B = dB; na.C = dC; na.rows = p->rows; na.cols = p->cols; na.N = N;
    na.n_blocks = n.n_blocks; na.src = n.d_source;
    // As many entries asked for ahead as most blocks have (4096 x 11008, N = 16, one to four loads, us: at 8 % 11.6 / 10.7 / 11.3 / 11.9, at 20 %
    // 14.4 / 13.3 / 12.8 / 12.6, before B came in words)
    const uint32_t loads = uint32_t(std::min(4.0, std::max(1.0, std::ceil((per_block(n) + 8.0) / 128.0))));
    p->note_launch("spmm_narrow_kernel", 3, p->dtype == HSPMM_FP16 ? 1u : 2u, uint64_t(n.n_units) * n.n_blocks * (N > one_tile(N) ? 8u : 4u));
    HSPMM_HIP(hspmm::launch_spmm_narrow(p->dtype, na, waves, loads, s));
    return HSPMM_OK;
}

}  // namespace hspmm_host
