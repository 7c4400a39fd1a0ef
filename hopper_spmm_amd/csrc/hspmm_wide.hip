// Host side of the wide-tile kernels (spmm_wide_kernel.hip): which plans carry their stream, which launches they take and in which
// shape, the launch.
#include "hspmm_plan.hpp"

using namespace hspmm_host;

namespace {

// A launch takes `start` us and `chunk[i]` us for every chunk of 64 columns and round of workgroups, one of them per compute unit and
// round - a second one on a compute unit takes its time on top -; i: rows of B of whole 128-byte lines, of whole 16-byte pieces, of
// whole words, any.  A fit to 3078 launches of 560 pruned matrices of 1024 to 16384 rows and columns at 2 to 31 %, N = 32 to 1024, every
// shape measured: standard deviations of 3 to 7 % (the first: 12 %), and the shape it picks is 0.3 % behind the fastest on
// average, 2.5 % at the 95th percentile.  Seven more shapes were measured and are the fastest of no launch, or by little.
struct ShapeCost { hspmm::WideShape shape; double start, chunk[4]; };
const ShapeCost kShapes[] = {
    {{1, 2, 2, 4}, 3.9, {0.118, 0.123, 0.135, 0.143}},       //  32 rows x  32 features
    {{1, 2, 4, 2}, 3.9, {0.159, 0.163, 0.172, 0.178}},       //  64 x  32
    {{1, 4, 4, 2}, 4.2, {0.191, 0.205, 0.214, 0.239}},       //  64 x  64
    {{2, 2, 4, 2}, 3.7, {0.241, 0.244, 0.261, 0.271}},       // 128 x  32
    {{2, 4, 4, 2}, 4.7, {0.273, 0.305, 0.315, 0.350}},       // 128 x  64
    {{3, 4, 2, 4}, 6.6, {0.237, 0.261, 0.273, 0.298}},       //  96 x  64
    {{3, 4, 4, 2}, 6.1, {0.355, 0.386, 0.396, 0.433}},       // 192 x  64
    {{2, 8, 4, 2}, 7.7, {0.431, 0.434, 0.439, 0.529}},       // 128 x 128
    {{3, 8, 4, 2}, 9.9, {0.550, 0.552, 0.555, 0.619}},       // 192 x 128
};
constexpr uint32_t kShapeCount = sizeof kShapes / sizeof kShapes[0], kFewestFeatures = 32u;
constexpr size_t kMostBytes = size_t(8) << 30;             // 64k x 64k
constexpr double kMostEntries = 0.31, kShort = 11.0;        // us
constexpr uint32_t kFewRows = 1024u;

uint64_t workgroups(const hspmm_plan *p, uint32_t N, const hspmm::WideShape &s)
{
    const uint64_t rows = uint64_t(s.units) * s.rows * 16u, features = uint64_t(s.blocks) * 16u;
    return (p->rows + rows - 1u) / rows * ((N + features - 1u) / features);
}

// The shape of a launch, a function of the plan and N alone, and the time it is expected to take.
const ShapeCost *choose_wide_shape(const hspmm_plan *p, uint32_t N, double *expected)
{
    const uint64_t row_bytes = uint64_t(N) * p->elem, cu = uint64_t(p->compute_units);
    const int i = row_bytes % 128u == 0 ? 0 : row_bytes % 16u == 0 ? 1 : row_bytes % 4u == 0 ? 2 : 3;
    const ShapeCost *best = nullptr;
    for (const ShapeCost &c : kShapes) {
        if (N < c.shape.blocks * 16u || (p->cfg.wide_shape >= 0 && uint32_t(p->cfg.wide_shape) % kShapeCount != uint32_t(&c - kShapes))) continue;
        const uint64_t groups = workgroups(p, N, c.shape);
        const double rounds = groups <= cu ? 0.87 + 0.13 * double(groups) / double(cu) : 1.04 * double((groups + cu - 1u) / cu);
        const double t = c.start + c.chunk[i] * p->wide.n_chunks * rounds;
        if (!best || t < *expected) { best = &c; *expected = t; }
    }
    return best;
}

}  // namespace

namespace hspmm_host {

// Made where some feature dimension would take it by the stored entries as estimated from a sample: from 4 % on (at 3 to 4 % the
// launches it would take gain 2 % of the time of all, at 4 to 6 % 12 %, above 10 % 31 %, for 2 bytes per element of the matrix).
// Block-clustered weights (over four of a column's eight elements stored) stay with kernels that read whole tiles.
int build_wide_stream(hspmm_plan *p)
{
    using namespace hspmm;
    hspmm_plan::Wide &w = p->wide;
    if (p->elem != 2u || p->cfg.wide == 0 || !p->canonical || p->cfg.kernel_mode != 0 || !p->T || p->W >= (1u << 23)) return HSPMM_OK;
    const double cells = double(p->rows) * p->cols;
    if (p->cfg.wide < 0 && (p->G != 1 || p->per_column > 4.0 || double(p->T) * p->cw * p->per_column < 0.04 * cells)) return HSPMM_OK;
    const uint32_t n_units = (p->rows + 15u) / 16u, n_chunks = ((p->cols + 63u) / 64u + 3u) & ~3u;
    const TileSource src{p->d_rowOffset, p->d_rowIdx, p->d_a2b_raw, p->d_data, p->W, p->cols};
    // (a plan whose device memory holds no such stream is made without)
    const size_t bytes = size_t(n_units) * n_chunks * kWideUnitBytes;
    void *frags = nullptr;
    if (bytes > kMostBytes) return HSPMM_OK;
    if (plan_alloc(p, bytes, &frags)) { (void)hipGetLastError(); return HSPMM_OK; }
    HSPMM_HIP(launch_wide_fill(src, p->rows, n_chunks, frags, nullptr));
    if (int rc = upload(p, &w.d_source, &src, 1)) return rc;
    HSPMM_HIP(hipStreamSynchronize(nullptr));
    w.d_frags = frags;
    w.n_units = n_units; w.n_chunks = n_chunks;
    w.built = true;
    return HSPMM_OK;
}

double wide_expected(const hspmm_plan *p, uint32_t N)
{
    double expected = 0.0;
    return choose_wide_shape(p, N, &expected) ? expected : 0.0;
}

// Where they are expected to be faster, by 5 % at least, than the kernels that would take the launch.  Launches of the entry kernels stay
// theirs (at the few features they take from such matrices 1 in 20 would gain), and those of the gather kernels from 32 features on are
// all taken (of 184, one in eight lost, 13 % at most; 1.35 times as fast on average).  Over 3078 launches the rule gives
// 1.16 times the speed of the LDS-panel kernels (1.175 if every launch took the faster one; 3 % of those taken lose, 4 % on average),
// 1.44 of the full-tile ones (1.52; none loses), whose times are known up to kMostEntries: denser launches of theirs stay.
// With fewer than kFewRows rows a long chain of chunks leaves compute units idle, where the other kernels cut the columns: 512 rows x
// 11008 at 10 %, N = 64 / 128 / 512 / 1024 21 / 22 / 31 / 41 us by these kernels, 17 / 17 / 21 / 27 by the others, 512 x 4096 8 / 10 / 13 / 17
// and 9 / 13 / 15 / 16, 512 x 1024 7.0 for each and 7.0 / 9.0 / 9.8 / 10.7: only launches expected to be short are taken.
bool wide_serves(const hspmm_plan *p, uint32_t N)
{
    const Config &c = p->cfg;
    if (!p->wide.built || c.kernel_mode != 0 || N < kFewestFeatures || N >= (1u << 21)) return false;
    double expected = 0.0;
    const ShapeCost *shape = choose_wide_shape(p, N, &expected);
    if (!shape || workgroups(p, N, shape->shape) >= (1u << 22)) return false;
    if (c.wide > 0) return true;
    // (settings of other kernels)
    if (c.buffer_stage || c.consumer_warp_num || c.producer_warp_group_num || c.fused_fixup >= 0 || c.panel_chunks || c.panel_max_windows ||
        c.panel_units_per_group || c.aligned_small >= 0 || c.xcd_split >= 0 || c.gather_bitmap >= 0 || c.tile > 0 || c.entries > 0)
        return false;
    if (tile_serves(p, N)) return double(p->tile.entries) <= kMostEntries * p->rows * p->cols && expected < 0.95 * tile_expected(p, N);
    if (entries_serve(p, N)) return false;
    if (p->rows < kFewRows && expected > kShort) return false;
    if (panel_serves(p, N)) return expected < 0.95 * (5.56 + 1.07 * panel_expected(p, N));
    return true;
}

int run_wide(hspmm_plan *p, const void *dB, void *dC, uint32_t N, hipStream_t s, RunMode mode)
{
    if (mode == RunMode::kPrepare) return HSPMM_OK;
    const hspmm_plan::Wide &w = p->wide;
    double expected = 0.0;
    const hspmm::WideShape &sh = choose_wide_shape(p, N, &expected)->shape;
    hspmm::WideArgs wa{};
    wa.frags = w.d_frags; wa.B = dB; wa.C = dC;
    wa.rows = p->rows; wa.cols = p->cols; wa.N = N;
    wa.n_units = w.n_units; wa.n_chunks = w.n_chunks; wa.n_feat_tiles = (N + sh.blocks * 16u - 1u) / (sh.blocks * 16u);
    wa.src = w.d_source;
    p->note_launch("spmm_wide_kernel", 3, p->dtype == HSPMM_FP16 ? 1u : 2u, workgroups(p, N, sh) * w.n_chunks * sh.units * sh.rows * sh.blocks * 2u);
    HSPMM_HIP(hspmm::launch_spmm_wide(p->dtype, wa, sh, s));
    return HSPMM_OK;
}

}  // namespace hspmm_host
