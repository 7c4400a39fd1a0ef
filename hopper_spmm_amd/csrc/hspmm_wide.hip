// Host side of the wide-tile kernels (spmm_wide_kernel.hip): which plans carry their stream, which launches they take and in which
// shape, the launch.
#include "hspmm_plan.hpp"
#include <cmath>

using namespace hspmm_host;

namespace {

// A launch takes `start` us and `chunk[i]` us for every chunk of 64 columns of a workgroup and round of workgroups, one of them per
// compute unit and round - a second one on a compute unit takes its time on top -; i: rows of B of whole 128-byte lines, of whole
// 16-byte pieces, of whole words, any.  Where C tiles are cut, `cut` us and what is below, too.  A fit to 50153 launches of 395 matrices of
// 64 to 16384 rows and 1024 to 16384 columns, N = 32 to 1024, every shape with one to 16 cuts: standard deviations of 5 to 9 %, and the
// launch it picks is 1.3 % behind the fastest on average, 8 % at the 95th percentile.  Seven more shapes were measured and are
// the fastest of no launch, or by little.
struct ShapeCost { hspmm::WideShape shape; double start, chunk[4], cut; };
const ShapeCost kShapes[] = {
    {{1, 2, 2, 4}, 3.5, {0.112, 0.115, 0.122, 0.135}, 2.2},       //  32 rows x  32 features
    {{1, 2, 4, 2}, 3.7, {0.158, 0.162, 0.168, 0.178}, 1.8},       //  64 x  32
    {{1, 4, 4, 2}, 4.2, {0.201, 0.212, 0.223, 0.247}, 1.6},       //  64 x  64
    {{2, 2, 4, 2}, 4.2, {0.236, 0.237, 0.248, 0.257}, 1.4},       // 128 x  32
    {{2, 4, 4, 2}, 5.0, {0.284, 0.305, 0.316, 0.343}, 1.0},       // 128 x  64
    {{3, 4, 2, 4}, 6.7, {0.253, 0.273, 0.286, 0.308}, 0.6},       //  96 x  64
    {{3, 4, 4, 2}, 6.1, {0.369, 0.391, 0.408, 0.432}, 0.1},       // 192 x  64
    {{2, 8, 4, 2}, 6.6, {0.462, 0.459, 0.461, 0.518}, 0.0},       // 128 x 128
    {{3, 8, 4, 2}, 6.9, {0.605, 0.598, 0.600, 0.638}, 0.0},       // 192 x 128
};
constexpr double kPerCut = 0.1, kPerSumsByte = 0.34e-6;           // us
// Times are of three matrices in turn, whose streams share the memory-side cache of 256 MB; from 75 MB on they no longer do, which is what
// this adds (100 MB: 8 us more).  See wide_serves for streams of any size that come from memory.
constexpr double kLargeStream = 75e6;
constexpr uint32_t kShapeCount = sizeof kShapes / sizeof kShapes[0], kFewestFeatures = 32u, kMostCuts = 16u;
constexpr size_t kMostBytes = size_t(8) << 30;             // 64k x 64k
constexpr double kMostEntries = 0.31;

uint64_t workgroups(const hspmm_plan *p, uint32_t N, const hspmm::WideShape &s)
{
    const uint64_t rows = uint64_t(s.units) * s.rows * 16u, features = uint64_t(s.blocks) * 16u;
    return (p->rows + rows - 1u) / rows * ((N + features - 1u) / features);
}

// fp32 sums of a C tile
uint64_t tile_sums_bytes(const hspmm::WideShape &s) { return uint64_t(s.units) * s.rows * s.blocks * 1024u; }

// The shape of a launch and the workgroups of a C tile, a function of the plan and N alone, and the time it is expected to take.
struct WideChoice { const ShapeCost *cost = nullptr; uint32_t cuts = 1; double expected = 0.0; };        // (cuts: below 256)
WideChoice choose_wide_shape(const hspmm_plan *p, uint32_t N)
{
    const uint64_t row_bytes = uint64_t(N) * p->elem, cu = uint64_t(p->compute_units);
    const int i = row_bytes % 128u == 0 ? 0 : row_bytes % 16u == 0 ? 1 : row_bytes % 4u == 0 ? 2 : 3;
    const double stream = 2.0 * p->rows * p->cols, large = std::min(std::max((stream - kLargeStream) / 25e6, 0.0), 1.5) * 0.085e-6 * stream;
    WideChoice best;
    for (const ShapeCost &c : kShapes) {
        if (N < c.shape.blocks * 16u || (p->cfg.wide_shape >= 0 && uint32_t(p->cfg.wide_shape) % kShapeCount != uint32_t(&c - kShapes))) continue;
        const uint64_t groups = workgroups(p, N, c.shape), sums = groups * tile_sums_bytes(c.shape);
        const uint32_t stages = p->wide.n_chunks / c.shape.splits;
        uint32_t tried = 0;
        // as many cuts as there are compute units for, once and twice; two stages each at least, and sums that hspmm_run_static has room for
        for (uint64_t round = 0; round <= 2u; ++round) {
            const uint64_t most = std::min<uint64_t>(std::min<uint64_t>(kMostCuts, stages / 2u), HSPMM_STATIC_SCRATCH_BYTES / sums);
            uint32_t cuts = uint32_t(std::max<uint64_t>(1u, std::min(round * cu / groups, most)));
            if (p->cfg.wide_cuts > 0) cuts = uint32_t(std::max<uint64_t>(1u, std::min<uint64_t>(uint64_t(p->cfg.wide_cuts), most)));
            if (cuts == tried) continue;
            tried = cuts;
            const double all = double(groups * cuts), rounds = all <= double(cu) ? 0.87 + 0.13 * all / double(cu) : 1.04 * std::ceil(all / double(cu));
            double t = c.start + c.chunk[i] * double((stages + cuts - 1u) / cuts * c.shape.splits) * rounds + large;
            if (cuts > 1u) t += c.cut + kPerCut * cuts + kPerSumsByte * double(sums) * cuts;
            if (!best.cost || t < best.expected) { best.cost = &c; best.cuts = cuts; best.expected = t; }
        }
    }
    return best;
}

// What the gather kernels take for matrices of 16 x 16 blocks, us: a fit to 1834 launches of 20 to 60 % (standard deviation 17 to 34 %).  Up
// to 64 features in whole 16-byte pieces are one pass over the tiles, others one per 32.
double blocks_gather_expected(const hspmm_plan *p, uint32_t N)
{
    const double tiles = 1e-3 * p->T, passes = double((N + 31u) / 32u);
    if (N % 8u == 0u) return N <= 32u ? 4.7 + 0.077 * tiles : N <= 64u ? 5.3 + 0.112 * tiles : 12.5 + 0.162 * tiles;
    return (N % 2u ? 10.3 + 0.25 * tiles : 6.3 + 0.18 * tiles) * (1.0 + 0.36 * (passes - 2.0));
}

bool of_blocks(const hspmm_plan *p) { return p->G == 2 && p->per_column > 4.0; }

bool worth_taking(const hspmm_plan *p, uint32_t N)
{
    const double expected = choose_wide_shape(p, N).expected;
    if (of_blocks(p)) {
        if (panel_serves(p, N)) return expected < 0.9 * (6.2 + 0.9 * panel_expected(p, N));
        return expected < (N % 8u == 0u ? 0.75 : 0.9) * blocks_gather_expected(p, N);
    }
    if (tile_serves(p, N)) return double(p->tile.entries) <= kMostEntries * p->rows * p->cols && expected < 0.95 * tile_expected(p, N);
    if (entries_serve(p, N)) return N < 256u && expected < 0.9 * entries_expected(p, N);
    if (panel_serves(p, N)) return expected < 0.95 * (5.56 + 1.07 * panel_expected(p, N));
    return true;
}

// Index of the shape, cuts, whether the launch is taken.
uint32_t kept_choice(const hspmm_plan *p, uint32_t N)
{
    return p->wide.choices.get(N, [&]() -> uint32_t {
        const WideChoice choice = choose_wide_shape(p, N);
        const bool taken = choice.cost && workgroups(p, N, choice.cost->shape) * choice.cuts < (1u << 22) && (p->cfg.wide > 0 || worth_taking(p, N));
        return (choice.cost ? uint32_t(choice.cost - kShapes) << 16 : 0u) | choice.cuts << 8 | (taken ? 1u : 0u);
    });
}

}  // namespace

namespace hspmm_host {

// Made where some feature dimension would take it by the stored entries as estimated from a sample: from 4 % on (at 3 to 4 % the
// launches it would take gain 2 % of the time of all, at 4 to 6 % 12 %, above 10 % 31 %, for 2 bytes per element of the matrix), of weights in
// 16 x 16 blocks (units of two windows, over four of a column's eight elements stored) from 15 % on.  Plans that keep the caller's cuts
// of windows stay with kernels that walk windows.
int build_wide_stream(hspmm_plan *p)
{
    using namespace hspmm;
    hspmm_plan::Wide &w = p->wide;
    if (p->elem != 2u || p->cfg.wide == 0 || !p->canonical || p->cfg.kernel_mode != 0 || !p->T || p->W >= (1u << 23) || !p->caller_cuts.empty()) return HSPMM_OK;
    const double fill = double(p->T) * p->cw * p->per_column / (double(p->rows) * p->cols);
    if (p->cfg.wide < 0 && (of_blocks(p) ? fill < 0.15 : p->G != 1 || p->per_column > 4.0 || fill < 0.04)) return HSPMM_OK;
    const uint32_t n_units = (p->rows + 15u) / 16u, n_chunks = ((p->cols + 63u) / 64u + 3u) & ~3u;
    const TileSource src{p->d_rowOffset, p->d_rowIdx, p->d_a2b_raw, p->d_data, p->W, p->cols};
    // (a plan whose device memory does not hold the stream is made without)
    const size_t bytes = size_t(n_units) * n_chunks * kWideUnitBytes;
    void *frags = nullptr, *source = nullptr;
    if (bytes > kMostBytes) return HSPMM_OK;
    if (plan_alloc(p, bytes, &frags) || plan_alloc(p, sizeof src, &source)) {
        (void)hipGetLastError();
        plan_release(p, frags, bytes);
        return HSPMM_OK;
    }
    HSPMM_HIP(launch_wide_fill(src, p->rows, n_chunks, frags, nullptr));
    HSPMM_HIP(hipMemcpy(source, &src, sizeof src, hipMemcpyHostToDevice));
    HSPMM_HIP(hipStreamSynchronize(nullptr));
    w.d_frags = frags; w.d_source = static_cast<TileSource *>(source);
    w.n_units = n_units; w.n_chunks = n_chunks;
    w.expected_fewest = choose_wide_shape(p, kFewestFeatures).expected;
    w.built = true;
    return HSPMM_OK;
}

// Where they are expected to be faster, by 5 or 10 % - or by a quarter, where the time to beat is known least: the gather kernels' in
// whole 16-byte pieces -, than the kernels that would take the launch; the gather kernels lose every launch but one in a hundred of
// pruned weights.  Times by the kernels that otherwise take a launch over the time that these are expected
// to take, with the launches taken by this rule and those left: LDS-panel 1.22 (4385 launches, 1.23 if every one took the faster kernel),
// full-tile 1.67 (1233, whose times are known up to kMostEntries: denser launches stay), gather 1.69 (475); of blocks of 16 x 16
// LDS-panel 1.08 (1832), gather 1.75 (1834).
// Without cut C tiles rows x columns with few workgroups left compute units idle, us (uncut / cut / other kernels): 512 x 11008 at 10 %,
// N = 64 20.5 / 9.9 / 17, 256 24.8 / 13.0 / 19, 4096 x 14336, N = 64 45 / 26.
// In a model of many layers every stream comes from memory, and this one is the largest: 678 launches taken by the rule, six to 48 matrices
// of 800 MB together in turn / one matrix over and over, old time over new: LDS-panel 1.14 / 1.27, full-tile 1.54 / 2.0, gather 1.9 / 2.2;
// of blocks LDS-panel 1.11 / 1.29, gather 2.3 / 2.5.  35 / 4 of them lose more than 3 %, 25 of the former by less than 6 % or below 6 % of entries.
// The launches from the LDS-panel kernels take 0.9 / 0.1 % longer than if each took the faster one.  Of 177 launches beyond 75 MB the rule
// leaves the LDS-panel kernels 126, which would be 7 / 10 % faster if each took the faster one.
bool wide_serves(const hspmm_plan *p, uint32_t N)
{
    const Config &c = p->cfg;
    if (!p->wide.built || c.kernel_mode != 0 || N < kFewestFeatures || N >= (1u << 20)) return false;
    // (settings of other kernels)
    if (c.wide < 0 && (c.buffer_stage || c.consumer_warp_num || c.producer_warp_group_num || c.fused_fixup >= 0 || c.panel_chunks || c.panel_max_windows ||
                       c.panel_units_per_group || c.aligned_small >= 0 || c.xcd_split >= 0 || c.gather_bitmap >= 0 || c.tile > 0 || c.entries > 0))
        return false;
    return kept_choice(p, N) & 1u;
}

double blocks_expected(const hspmm_plan *p, uint32_t N) { return wide_serves(p, N) ? choose_wide_shape(p, N).expected : blocks_gather_expected(p, N); }

int run_wide(hspmm_plan *p, const void *dB, void *dC, uint32_t N, hipStream_t s, hipEvent_t mid, RunMode mode)
{
    const hspmm_plan::Wide &w = p->wide;
    const uint32_t choice = kept_choice(p, N);
    const hspmm::WideShape &sh = kShapes[choice >> 16 & 0xFFu].shape;
    const uint64_t groups = workgroups(p, N, sh);
    hspmm::WideArgs wa{};
    wa.n_cuts = choice >> 8 & 0xFFu;
    if (wa.n_cuts > 1u) {
        std::lock_guard<std::mutex> lk(p->mu);
        if (const int rc = scratch_for(p, s, size_t(groups * wa.n_cuts * tile_sums_bytes(sh)), mode, &wa.sums)) return rc;
    }
    if (mode == RunMode::kPrepare) return HSPMM_OK;
    wa.frags = w.d_frags; wa.B = dB; wa.C = dC;
    wa.rows = p->rows; wa.cols = p->cols; wa.N = N;
    wa.n_units = w.n_units; wa.n_chunks = w.n_chunks; wa.n_feat_tiles = (N + sh.blocks * 16u - 1u) / (sh.blocks * 16u);
    wa.src = w.d_source;
    p->note_launch("spmm_wide_kernel", 3, p->dtype == HSPMM_FP16 ? 1u : 2u, groups * w.n_chunks * sh.units * sh.rows * sh.blocks * 2u);
    HSPMM_HIP(hspmm::launch_spmm_wide(p->dtype, wa, sh, s, mid));
    return HSPMM_OK;
}

}  // namespace hspmm_host
