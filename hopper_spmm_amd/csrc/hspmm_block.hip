// Host side of the block kernels (spmm_block_kernel.hip): which plans carry their units, which launches they take, the launch.
#include "hspmm_plan.hpp"

using namespace hspmm_host;

namespace {

constexpr uint32_t kMostFeatures = 64u, kAlwaysFeatures = 32u;

// us, from 33 features on, an even number: a fit to 140 launches of 160 matrices of 1024 to 16384 rows, 20 to 60 % of blocks kept, three matrices
// in turn (standard deviation 11 to 14 %), or the longest unit's walk (50 units of 200 steps, one of 401: N = 44 9.7, 62 11.2; one of 1024 30.5).
double expected(const hspmm_plan *p, uint32_t N)
{
    const double steps = double(p->n_steps);
    return 3.5 + std::max((N <= 48u ? 0.13e-3 : 0.15e-3) * steps + 0.008 * steps / double(p->n_units), (N <= 48u ? 0.0165 : 0.025) * double(p->block_units.longest));
}

// us, fp32 storage up to 32 features: the tiles' way from memory, or the walk of a wave over its share of the longest unit's blocks (one unit of 2048
// steps: N = 16 46.7, 32 58.3).
double expected_f32(const hspmm_plan *p, uint32_t N)
{
    return 3.5 + std::max(256.0 * p->T / 4.0e6, (N <= 16u ? 0.02 : 0.025) * double(p->block_units.longest));
}

// A workgroup has a unit: a launch takes as long as the longest unit, and every unit costs a workgroup however short it is.  us, by the kernels that
// take them otherwise / here.  Many short units, N = 16 / 64, 16 bits: 2048 of 6 blocks 8.4 / 5.5, 10.0 / 10.6; 3072 of 6 9.1 / 7.9, 10.2 / 15.1; 4096
// of 10 10.4 / 11.6, 12.3 / 20.8; 8192 of 6 10.9 / 18.7, 12.9 / 34.6; fp32 2048 of 6 10.4 / 7.9, 29.6 / 15.7, 8192 of 6 18.4 / 23.6: up to eight a
// compute unit (from 33 features on, 16 bits, four: block_serves).
// Uneven ones: where the gather kernels give every unit a workgroup's waves, too (aligned_group), units of up to six times the mean were ahead on all
// launches (64 to 1024 units of 6 to 200 blocks, one of 1.5 to 6 times as many).  Where their waves have even shares they do not wait for the longest
// unit (1024 units of 55 blocks, one of 1024, N = 16 / 64: 17.4 / 34.3, 21.9 / 55.9; 256 of 20 blocks, eight of 1024, fp32, N = 32: 21.3 / 59.1;
// lengths drawn between 1 and 400, 64 units, fp32, N = 8: 14.1 / 19.2): twice the mean and 16 blocks, 256 blocks or 160 of fp32 storage.
// Workgroups go to the eight XCDs in turn: units of which every other one is short leave half of them with little (1600 units of 1 and 44 blocks in
// turn, N = 23: 11.4 / 12.7, 808 of 1 and 64, N = 52: 10.5 / 12.6).
// 900 matrices of 16 to 6000 units, even ones and uneven, five N each: of 3300 launches taken 14 slower by more than 3 % (21 % at most), twice as fast
// on the mean.
bool units_suit(const hspmm_plan *p, const StepStream &st, uint32_t longest)
{
    const uint64_t units = p->n_units, steps = p->n_steps, all = uint64_t(longest) * units, block = 16u / p->cw;
    if (units > uint64_t(p->compute_units) * 8u) return false;
    uint64_t of_xcd[8] = {};
    for (size_t u = 0; u < units; ++u) of_xcd[u % 8u] += st.unitOffset[u + 1] - st.unitOffset[u];
    if (units > uint32_t(p->compute_units) && *std::max_element(of_xcd, of_xcd + 8) * 32u > steps * 5u) return false;
    if (p->aligned_group) return all <= 6u * steps;
    return all <= 2u * steps + 16u * block * units && longest <= (p->elem == 4u ? 160u : 256u) * block;
}

}  // namespace

namespace hspmm_host {

// Made where every step's columns are neighbours (16 x 16 blocks anywhere in a row of blocks; the last block may end inside): for a pair of
// windows a record of 32 bytes, for a step four bytes.  The tiles are read where the plan has them.
int build_block_units(hspmm_plan *p, const StepStream &st, const uint32_t *rowOffset, const uint32_t *tcA2B)
{
    using namespace hspmm;
    if (p->cfg.block == 0 || !p->canonical || p->cfg.kernel_mode != 0 || p->G != 2 || !p->caller_cuts.empty() || p->n_units >= (1u << 22)) return HSPMM_OK;
    const size_t n = st.unitRow.size(), cw = p->cw;
    uint32_t longest = 0;
    for (size_t u = 0; u < n; ++u) longest = std::max(longest, st.unitOffset[u + 1] - st.unitOffset[u]);
    if (p->cfg.block < 0 && (p->per_column <= 4.0 || !units_suit(p, st, longest))) return HSPMM_OK;
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
    b.longest = longest;
    b.built = true;
    return HSPMM_OK;
}

// Of the rows of blocks that units_suit takes, up to 32 features: of 700 launches of 260 matrices (1024 to 16384 rows, 20 to 60 % of blocks kept, all N) three were slower than by
// the gather kernels, by 1 to 11 %.  From 33 on, even numbers, by expected time: of 450 launches taken 11 are slower by more than 3 % (16 % at
// most), 1.45 times as fast on the mean.  Odd ones stay with the wide-tile kernels (0.9 to 1.2 there), and from 65 on all (0.7 to 1.2).  fp32 storage: every launch
// of the gather kernels (207 of 60 matrices: 1.07 to 3.5 times as fast); those of the LDS-panel kernels, which are faster from 33 features on
// and for the largest matrices, by expected time (134 taken: 1.49 on the mean, 0.88 at least; 26 up to 32 features left).
// Not at N = 32 on more than 65 % of all blocks, where the wide-tile kernels take it (11 of 14 launches were 2 to 20 % slower here, of 20 below none), and
// not above 32 features on rows of over 512 blocks of fp32 storage (nine with B off its alignment: 0.9).  A B that begins between two words has loads of
// twice the time: the wide-tile kernels keep theirs (224 launches: 0.87 times as fast here), and above 32 features units of over 128 blocks stay (91:
// 1.1, 26 behind, by up to 34 %); the others were 1.28 (up to 32 features) and 1.48 times as fast.
bool block_serves(const hspmm_plan *p, uint32_t N, bool on_word)
{
    const Config &c = p->cfg;
    if (!p->block_units.built || N > kMostFeatures || uint64_t(p->cols) * N * p->elem > (uint64_t(1) << 32)) return false;
    // (settings of other kernels)
    if (c.block < 0 && (c.buffer_stage || c.consumer_warp_num || c.producer_warp_group_num || c.fused_fixup >= 0 || c.panel_chunks || c.panel_max_windows ||
                        c.panel_units_per_group || c.aligned_small >= 0 || c.xcd_split >= 0 || c.gather_bitmap >= 0 || c.tile > 0 || c.entries > 0 || c.wide > 0))
        return false;
    if (p->elem == 4u) {
        if (c.block <= 0 && N > kAlwaysFeatures && p->block_units.longest > 1024u) return false;
        if (c.block > 0 || N < 16u || N % 4u || !panel_serves(p, N)) return true;
        return N <= kAlwaysFeatures && p->block_units.taken.get(N, [&]() -> uint32_t { return expected_f32(p, N) < 0.95 * (6.2 + 0.9 * panel_expected(p, N)); });
    }
    if (c.block > 0) return N <= kAlwaysFeatures || N % 2u == 0u;
    if (!on_word && (wide_serves(p, N) || (N > kAlwaysFeatures && p->block_units.longest > 128u))) return false;
    if (N < kAlwaysFeatures) return true;
    if (N == kAlwaysFeatures) return uint64_t(p->n_steps) * 320u <= uint64_t(p->n_units) * p->cols * 13u || !wide_serves(p, N);
    if (N % 2u) return false;
    if (p->n_units > uint32_t(p->compute_units) * 4u) return false;
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
