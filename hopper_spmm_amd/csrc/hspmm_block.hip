// Host side of the block kernels (spmm_block_kernel.hip): which plans carry their units, which launches they take, the launch.
#include "hspmm_plan.hpp"

using namespace hspmm_host;

namespace {

constexpr uint32_t kMostFeatures = 64u, kAlwaysFeatures = 32u;

// us, from 33 features on, an even number: a fit to 140 launches of 160 matrices of 1024 to 16384 rows, 20 to 60 % of blocks kept, three matrices
// in turn (standard deviation 11 to 14 %).
double expected(const hspmm_plan *p, uint32_t N)
{
    const double steps = double(p->n_steps);
    return 3.5 + (N <= 48u ? 0.13e-3 : 0.15e-3) * steps + 0.008 * steps / double(p->n_units);
}

// us, fp32 storage up to 32 features: the tiles' way from memory, or the walk of a wave over its share of a unit's blocks.
double expected_f32(const hspmm_plan *p)
{
    return 3.5 + std::max(256.0 * p->T / 4.0e6, 0.02 * double(p->n_steps) / double(p->n_units));
}

}  // namespace

namespace hspmm_host {

// Made where every step's columns are neighbours (16 x 16 blocks anywhere in a row of blocks; the last block may end inside): for a pair of
// windows a record of 32 bytes, for a step four bytes.  The tiles are read where the plan has them.
int build_block_units(hspmm_plan *p, const StepStream &st, const uint32_t *rowOffset, const uint32_t *tcA2B)
{
    using namespace hspmm;
    if (p->cfg.block == 0 || !p->canonical || p->cfg.kernel_mode != 0 || p->G != 2 || !p->caller_cuts.empty() || p->n_units >= (1u << 22)) return HSPMM_OK;
    if (p->cfg.block < 0 && p->per_column <= 4.0) return HSPMM_OK;
    const size_t n = st.unitRow.size(), cw = p->cw;
    std::vector<uint32_t> pairs(n + 1);
    for (size_t u = 0; u < n; ++u) pairs[u + 1] = pairs[u] + (st.unitOffset[u + 1] - st.unitOffset[u] + 1u) / 2u;
    // one upload: where the tiles are, the units, the first columns
    static_assert(sizeof(TileSource) <= 64u && sizeof(BlockUnit) == 32u, "");
    const size_t columns_at = 64u + n * sizeof(BlockUnit);
    std::vector<char> image(columns_at + size_t(pairs[n]) * 8u);
    const TileSource src{p->d_rowOffset, p->d_rowIdx, p->d_a2b_raw, p->d_data, p->W, p->cols};
    std::memcpy(image.data(), &src, sizeof src);
    BlockUnit *units = reinterpret_cast<BlockUnit *>(image.data() + 64u);
    uint32_t *columns = reinterpret_cast<uint32_t *>(image.data() + columns_at);
    std::atomic<bool> neighbours{true};
    parallel_blocks(n, 32, [&](size_t ub, size_t ue) {
        for (size_t u = ub; u < ue && neighbours.load(std::memory_order_relaxed); ++u) {
            const uint32_t w = st.unitWindow[u], steps = st.unitOffset[u + 1] - st.unitOffset[u];
            units[u] = BlockUnit{rowOffset[w], (st.unitRow[u] & 1u) ? rowOffset[w + 1u] : HSPMM_IDX_MAX, steps, st.unitRow[u] & ~7u,
                                 u + 1 < n ? st.unitRow[u + 1] & ~7u : p->rows, pairs[u], {0u, 0u}};
            const uint32_t *ids = tcA2B + size_t(rowOffset[w]) * cw;
            uint32_t *to = columns + size_t(pairs[u]) * 2u;
            for (uint32_t s = 0; s < steps; ++s) {
                const uint32_t *id = ids + s * cw;
                for (uint32_t k = 1; k < cw; ++k)
                    if (id[k] != id[0] + k && id[k] != HSPMM_IDX_MAX) neighbours.store(false, std::memory_order_relaxed);
                to[s] = id[0];
            }
            if (steps & 1u) to[steps] = to[steps - 1u];
        }
    });
    if (!neighbours.load()) return HSPMM_OK;
    char *device = nullptr;
    if (upload(p, &device, image.data(), image.size())) {           // (a plan whose device memory does not hold it is made without)
        (void)hipGetLastError();
        return HSPMM_OK;
    }
    hspmm_plan::Block &b = p->block_units;
    b.d_source = reinterpret_cast<const TileSource *>(device);
    b.d_units = reinterpret_cast<const BlockUnit *>(device + 64u);
    b.d_columns = reinterpret_cast<const uint32_t *>(device + columns_at);
    b.n_units = uint32_t(n);
    b.built = true;
    return HSPMM_OK;
}

// Up to 32 features always: of 700 launches of 260 matrices (1024 to 16384 rows, 20 to 60 % of blocks kept, all N) three were slower than by
// the gather kernels, by 1 to 11 %.  From 33 on, even numbers, by expected time: of 450 launches taken 11 are slower by more than 3 % (16 % at
// most), 1.45 times as fast on the mean.  Odd ones stay with the wide-tile kernels (0.9 to 1.2 there), and from 65 on all (0.7 to 1.2).  fp32 storage: every launch
// of the gather kernels (207 of 60 matrices: 1.07 to 3.5 times as fast); those of the LDS-panel kernels, which are faster from 33 features on
// and for the largest matrices, by expected time (134 taken: 1.49 on the mean, 0.88 at least; 26 up to 32 features left).
bool block_serves(const hspmm_plan *p, uint32_t N)
{
    const Config &c = p->cfg;
    if (!p->block_units.built || N > kMostFeatures || uint64_t(p->cols) * N * p->elem > (uint64_t(1) << 32)) return false;
    // (settings of other kernels)
    if (c.block < 0 && (c.buffer_stage || c.consumer_warp_num || c.producer_warp_group_num || c.fused_fixup >= 0 || c.panel_chunks || c.panel_max_windows ||
                        c.panel_units_per_group || c.aligned_small >= 0 || c.xcd_split >= 0 || c.gather_bitmap >= 0 || c.tile > 0 || c.entries > 0 || c.wide > 0))
        return false;
    if (p->elem == 4u) {
        if (c.block > 0 || N < 16u || N % 4u || !panel_serves(p, N)) return true;
        return N <= kAlwaysFeatures && p->block_units.taken.get(N, [&]() -> uint32_t { return expected_f32(p) < 0.95 * (6.2 + 0.9 * panel_expected(p, N)); });
    }
    if (N <= kAlwaysFeatures) return true;
    if (N % 2u) return false;
    if (c.block > 0) return true;
    return p->block_units.taken.get(N, [&]() -> uint32_t { return expected(p, N) < blocks_expected(p, N); });
}

int run_block(hspmm_plan *p, const void *dB, void *dC, uint32_t N, hipStream_t s, RunMode mode)
{
    if (mode == RunMode::kPrepare) return HSPMM_OK;
    const hspmm_plan::Block &b = p->block_units;
    hspmm::BlockArgs ba{};
    ba.units = b.d_units; ba.columns = b.d_columns; ba.tiles = p->d_data; ba.B = dB; ba.C = dC;
    ba.rows = p->rows; ba.cols = p->cols; ba.N = N;
    ba.src = b.d_source;
    p->note_launch("spmm_block_kernel", 2, p->dtype == HSPMM_FP16 ? 1u : p->dtype == HSPMM_BF16 ? 2u : 3u, uint64_t(p->n_steps + 1u) / 2u * (p->elem == 4u ? N <= 16u ? 4u : N <= 32u ? 8u : 16u : (N + 15u) / 16u));
    HSPMM_HIP(hspmm::launch_spmm_block(p->dtype, ba, b.n_units, s));
    return HSPMM_OK;
}

}  // namespace hspmm_host
