// C ABI of the SpMM operator (include/hspmm.h), part 2 of 3: plan creation - validation of the caller's
// arrays (reference src/utils/class.h:55-108), upload, the step streams of the two kernel families, the
// work partition.  Everything the reference's fp16_spmm does before its first launch (reference
// src/fp16.cu:221-254), done once per matrix.
#include "hspmm_plan.hpp"
#include "hspmm_pack.hpp"

using namespace hspmm_host;

namespace hspmm_host {

// The windows: what says how long the arrays of the tiles are.
static int validate_windows(uint32_t rows, uint32_t cols, uint32_t W, uint32_t T, const uint32_t *rowOffset, const uint32_t *tcA2B,
                            const void *data, const uint32_t *rowIdx)
{
    if (W == 0) {
        if (T != 0) return fail(HSPMM_ERR_INVALID, "total_tiles = %u with no effective row window", T);
        return HSPMM_OK;
    }
    if (!rowOffset || !tcA2B || !data || !rowIdx) return fail(HSPMM_ERR_INVALID, "null format array");
    if (rows == 0 || cols == 0) return fail(HSPMM_ERR_INVALID, "empty matrix with %u effective windows", W);
    if (uint64_t(W) > (uint64_t(rows) + 7u) / 8u)
        return fail(HSPMM_ERR_INVALID, "eff_row_windows = %u exceeds the %u windows of %u rows", W, (rows + 7u) / 8u, rows);
    if (rowOffset[0] != 0) return fail(HSPMM_ERR_INVALID, "rowOffset[0] = %u, expected 0", rowOffset[0]);
    for (uint32_t w = 0; w < W; ++w) {
        if (rowOffset[w + 1] <= rowOffset[w])
            return fail(HSPMM_ERR_INVALID, "rowOffset not strictly increasing at window %u", w);
        if (rowIdx[w] % HSPMM_ROW_WINDOW != 0 || rowIdx[w] >= rows)
            return fail(HSPMM_ERR_INVALID, "rowIdx[%u] = %u is not a window start inside %u rows", w, rowIdx[w], rows);
        if (w && rowIdx[w] <= rowIdx[w - 1])
            return fail(HSPMM_ERR_INVALID, "rowIdx not strictly increasing at window %u", w);
    }
    if (rowOffset[W] != T)
        return fail(HSPMM_ERR_INVALID, "rowOffset[%u] = %u differs from total_tiles = %u", W, rowOffset[W], T);
    return HSPMM_OK;
}

// The tiles of windows found good.  canonical (optional): whether every window's real column ids ascend strictly with padding only behind
// the window's last column, as the reference's converter writes them (src/utils/convert.h:166-181).
static int validate_tiles(uint32_t cols, uint32_t W, uint32_t T, uint32_t cw, const uint32_t *rowOffset, const uint32_t *tcA2B, const void *data,
                          bool *canonical, uint32_t *header, uint32_t *window_stored)
{
    if (canonical) *canonical = true;
    if (W == 0) return HSPMM_OK;
    // every tile's ids: real columns below `cols`, padding only behind them.  Checked on all cores; the message
    // names the first tile that fails.
    auto tile_error = [&](uint32_t t, bool report) -> bool {
        const uint32_t *ids = tcA2B + size_t(t) * cw;
        if (ids[0] == HSPMM_IDX_MAX) { if (report) fail(HSPMM_ERR_INVALID, "tile %u starts with a padding column", t); return true; }
        bool pad = false;
        for (uint32_t k = 0; k < cw; ++k) {
            if (ids[k] == HSPMM_IDX_MAX) { pad = true; continue; }
            if (pad) { if (report) fail(HSPMM_ERR_INVALID, "tile %u: column id after padding", t); return true; }
            if (ids[k] >= cols) { if (report) fail(HSPMM_ERR_INVALID, "tile %u: column id %u >= cols %u", t, ids[k], cols); return true; }
        }
        return false;
    };
    // (one pass on all cores for the ids, their order and, where asked for, what the tiles store)
    std::atomic<uint32_t> first_bad{T};
    std::atomic<bool> ordered{true};
    hspmm_host::parallel_weighted(W, size_t(1) << 13, [=](size_t w) { return rowOffset[w]; }, [&](size_t wb, size_t we) {
        for (size_t t = rowOffset[wb], e = rowOffset[we]; t < e; ++t)
            if (tile_error(uint32_t(t), false)) {
                uint32_t seen = first_bad.load(std::memory_order_relaxed);
                while (uint32_t(t) < seen && !first_bad.compare_exchange_weak(seen, uint32_t(t), std::memory_order_relaxed)) {}
                return;
            }
        for (size_t w = wb; canonical && w < we && ordered.load(std::memory_order_relaxed); ++w) {
            const uint32_t *c = tcA2B + size_t(rowOffset[w]) * cw;
            const size_t n = size_t(rowOffset[w + 1] - rowOffset[w]) * cw;
            size_t real = n;
            while (real && c[real - 1] == HSPMM_IDX_MAX) --real;
            bool good = n - real < cw;                      // padding only in the window's last tile
            for (size_t i = 1; i < real && good; ++i) good = c[i] != HSPMM_IDX_MAX && c[i] > c[i - 1];
            if (!good) ordered.store(false, std::memory_order_relaxed);
        }
        for (size_t w = wb; header && w < we; ++w)
            window_stored[w] = uint32_t(hspmm_host::tile_masks(static_cast<const char *>(data) + size_t(rowOffset[w]) * 256u,
                                                               rowOffset[w + 1] - rowOffset[w], cw == 16u ? 2u : 4u,
                                                               header + size_t(rowOffset[w]) * (cw == 16u ? 8u : 4u)));
    });
    if (first_bad.load() < T) { tile_error(first_bad.load(), true); return HSPMM_ERR_INVALID; }
    if (canonical) *canonical = ordered.load();
    return HSPMM_OK;
}

int validate_format(uint32_t rows, uint32_t cols, uint32_t W, uint32_t T, uint32_t cw,
                    const uint32_t *rowOffset, const uint32_t *tcA2B, const void *data, const uint32_t *rowIdx, bool *canonical)
{
    if (int rc = validate_windows(rows, cols, W, T, rowOffset, tcA2B, data, rowIdx)) return rc;
    return validate_tiles(cols, W, T, cw, rowOffset, tcA2B, data, canonical, nullptr, nullptr);
}

int plan_reserve(hspmm_plan *p, size_t bytes)
{
    void *fresh = nullptr;
    HSPMM_HIP(hipMalloc(&fresh, bytes));
    p->owned.push_back(fresh);
    p->block = static_cast<char *>(fresh);
    p->block_left = bytes;
    p->fixed_bytes += bytes;
    return HSPMM_OK;
}

int plan_alloc(hspmm_plan *p, size_t bytes, void **out)
{
    const size_t rounded = (bytes + 255u) & ~size_t(255);
    if (rounded <= p->block_left) {
        *out = p->block;
        p->block += rounded;
        p->block_left -= rounded;
    } else {
        HSPMM_HIP(hipMalloc(out, bytes));
        p->owned.push_back(*out);
        p->fixed_bytes += bytes;
    }
    return HSPMM_OK;
}

void plan_release(hspmm_plan *p, const void *ptr, size_t bytes)
{
    const auto it = std::find(p->owned.begin(), p->owned.end(), ptr);
    if (it == p->owned.end()) return;           // (part of the reserved block)
    (void)hipFree(*it);
    p->owned.erase(it);
    p->fixed_bytes -= bytes;
}

int choose_ranges(const hspmm_plan *p)
{
    const int waves_per_simd = p->cfg.producer_warp_group_num > 0 ? p->cfg.producer_warp_group_num : 4;
    uint64_t g = uint64_t(p->compute_units) * 4u * uint64_t(waves_per_simd);
    const uint64_t cap = (uint64_t(p->n_steps) + kMinTilesPerRange - 1) / kMinTilesPerRange;
    if (g > cap) g = cap;
    if (g < 1) g = 1;
    return int(g);
}

int build_and_upload_partition(hspmm_plan *p, int level, uint32_t group, bool aligned)
{
    hspmm_plan::DevPartition &dp = p->parts[aligned ? 4 : group > 1 ? 3 : level];
    if (dp.built || p->W == 0) return HSPMM_OK;
    const double window_cost = kWindowCost, slack = kSlack, margin = kWholeWindowMargin;
    uint32_t target = uint32_t(choose_ranges(p)) >> level;
    const uint32_t floor_ranges = uint32_t(p->compute_units) * 4u;       // at least one range per SIMD
    if (target < floor_ranges) target = std::min<uint32_t>(floor_ranges, uint32_t(choose_ranges(p)));
    dp.part = aligned ? hspmm::build_aligned_partition(p->n_units, p->h_unitOffset.data(), group)
                      : hspmm::build_partition(p->n_units, p->h_unitOffset.data(), target, window_cost, slack, margin, group,
                                               p->caller_cuts.empty() ? nullptr : &p->caller_cuts);
    const auto &part = dp.part;
    std::vector<uint32_t> rw(part.ranges.size() * hspmm::kRangeWords, 0u);
    for (size_t i = 0; i < part.ranges.size(); ++i) {
        uint32_t *d = rw.data() + i * hspmm::kRangeWords;
        d[0] = part.ranges[i].tile_begin; d[1] = part.ranges[i].tile_end; d[2] = part.ranges[i].first_window;
        d[3] = part.ranges[i].head_slot; d[4] = part.ranges[i].tail_slot;
        d[5] = part.ranges[i].head_split; d[6] = part.ranges[i].tail_split;
        d[7] = part.ranges[i].combine;
    }
    std::vector<uint32_t> sw(part.split.size() * hspmm::kFixWords, 0u);
    for (size_t i = 0; i < part.split.size(); ++i) {
        uint32_t *d = sw.data() + i * hspmm::kFixWords;
        d[0] = part.split[i].window; d[1] = part.split[i].slot_begin; d[2] = part.split[i].slot_count;
    }
    int rc;
    if ((rc = upload(p, &dp.d_ranges, rw.data(), rw.size()))) return rc;
    if ((rc = upload(p, &dp.d_split, sw.data(), sw.size()))) return rc;
    if ((rc = upload(p, &dp.d_fix_slots, part.fix_slots.data(), part.fix_slots.size()))) return rc;
    dp.built = true;
    return HSPMM_OK;
}

}  // namespace hspmm_host

namespace {

// Re-tiles the matrix panel by panel for the LDS-panel kernels (spmm_panel_kernel.hpp):
// inside every window the columns of one panel of kPanelRows columns get tiles of
// their own.  Every step carries the number of panels it lies behind the step in
// front of it (4 bits; a longer run of panels without a step gets an all-zero step
// every 15 panels).  Returns false when the kernels would not pay (criteria inside).
bool build_panel_stream(hspmm_plan *p, const StepStream &gather_st, const uint32_t *rowOffset, const uint32_t *tcA2B,
                        const void *data, const uint32_t *rowIdx, bool forced, int *rc_out)
{
    *rc_out = HSPMM_OK;
    PhaseTimer timer;
    const uint32_t cw = p->cw, W = p->W;
    // fp32: products of bf16 hi / lo parts (Fp32Split) unless the caller asked for fp32 products
    const bool split = p->dtype == HSPMM_TF32 && p->cfg.kernel_mode != 5;
    const uint32_t KP = (cw == 16 || split) ? hspmm::kPanelRowsWide : hspmm::kPanelRowsFp32;
    const uint32_t NP = (p->cols + KP - 1) / KP;
    constexpr uint32_t kMaxJump = 15;
    if (gather_st.unitRow.empty() || NP == 0) return false;
    // worth it when a unit has a few steps in every 128 columns it meets: the panel image is
    // then read from LDS several times per load from the L2.  Measured break-even against the gather
    // kernels on uniformly random matrices: 1.2 tiles per 128 columns for the kernels built on the
    // 16-bit MFMA (8192 x 8192 at 2 %, fp16: 31 against 34 us at N = 128, 56 against 110 at N = 512; at
    // 1 %: 29 against 16 and 48 against 42), about 2 for the fp32 MFMA forms.
    const double density = double(gather_st.n_steps) / (double(gather_st.unitRow.size()) * double((p->cols + 127u) / 128u));
    if (!forced && density < ((cw == 16 || split) ? 1.2 : 2.0)) return false;
    if (uint64_t(gather_st.unitRow.size()) * (NP + 1) > (1ull << 28)) return false;
    // columns per re-tiled step: the kernels built on 16-bit MFMAs contract 32 columns per step, the fp32
    // MFMA kernels a tile's 8
    const uint32_t rw = (cw == 16 || split) ? 32u : cw;
    // The units of this stream.  The kernels built on the 16-bit MFMA run groups of up to four adjacent
    // windows with one column list as one unit, and give neighbours the union of their lists wherever
    // that saves work (merge_groups); the fp32 MFMA forms walk the units of the gather kernels.
    Unioned un;
    StepStream st = gather_st;
    if (rw == 32 && p->cfg.pairing != 1 && W > 1) {
        // Units of three and four windows halve the LDS reads per row but leave half as many, twice as
        // long waves: measured on pruned and block-clustered 16-bit matrices they pay once the units
        // still fill the compute units at small N (16384 rows: 1.0 - 1.2 x, 28672 rows: 1.2 - 1.3 x;
        // 8192 and 11008 rows: 0.93 - 1.1 x up to N = 512, 1.2 - 1.3 x only from N = 2048 on), and for
        // fp32 storage in bf16 parts, with twice the MFMAs per LDS read, they gain nothing (0.82 - 1.2 x).
        // Pairing mode 2 takes them wherever windows qualify.
        const double wide_cost = kPanelWideCost;
        uint32_t max_windows = (p->cfg.pairing == 2 || cw == 16) ? 4u : 2u;
#ifndef HSPMM_EXPERIMENTAL
        if (split) max_windows = 2u;            // (units of four windows in bf16 parts measured 0.82 - 1.2 x: not built)
#endif
        size_t min_wide_units = p->cfg.pairing == 2 ? 0u : size_t(p->compute_units) * 3u / 2u;
        if (p->cfg.panel_max_windows) {                                                           // tuning override
            max_windows = uint32_t(p->cfg.panel_max_windows);
            min_wide_units = 0;
#ifndef HSPMM_EXPERIMENTAL
            if (split) max_windows = 2u;
#endif
        }
        std::vector<uint32_t> first, count;
        group_windows(W, cw, uint32_t(p->elem), KP, rw, max_windows, wide_cost, min_wide_units, rowOffset, tcA2B, data,
                      rowIdx, un, first, count);
        st = StepStream();
        st.unitOffset.push_back(0);
        uint32_t widest = 1;
        for (size_t g = 0; g < first.size(); ++g) {
            const uint32_t w = first[g];
            st.unitWindow.push_back(w);
            st.unitRow.push_back(rowIdx[w] | (count[g] - 1u));
            st.unitOffset.push_back(st.unitOffset.back() + (rowOffset[w + 1] - rowOffset[w]));
            st.n_paired += count[g] >= 2u;
            st.n_wide += count[g] >= 3u;
            widest = std::max(widest, count[g]);
        }
        st.n_steps = st.unitOffset.back();
        st.G = widest >= 3u ? 4 : int(widest);
    }
    timer.mark("  panel: units of windows");
    const uint32_t U = uint32_t(st.unitRow.size());
    const uint32_t T = rowOffset[W];
    // Two units per consumer wave (merge_unit_pairs below): the second unit's first step follows whatever step of
    // the first unit lies in front of it, so it, too, may be at most kMaxJump panels from its predecessor - every
    // unit of such a stream gets its all-zero steps from panel 0 on, not only behind its first step.
    const bool tall_stream = rw == 32 && st.G <= 2 && U >= 2 && (p->cfg.panel_tall > 0 || p->cfg.panel_packed > 0);
    const size_t es = p->elem, src_tile_bytes = size_t(8) * cw * es, tile_bytes = size_t(8) * rw * es;
    // Two passes over the windows, both on all cores: the steps every window gets, then the steps.
    std::vector<uint32_t> rt_rowOffset(size_t(W) + 1, 0u), rt_panel;
    const uint8_t *src_data = static_cast<const uint8_t *>(data);
    auto real_columns = [&](uint32_t w) {
        const uint32_t *col = tcA2B + size_t(rowOffset[w]) * cw;
        uint32_t nreal = (rowOffset[w + 1] - rowOffset[w]) * cw;
        while (nreal && col[nreal - 1] == HSPMM_IDX_MAX) --nreal;
        return nreal;
    };
    const size_t windows_per_worker = std::max<size_t>(1, (size_t(1) << 14) / std::max<uint32_t>(1u, T / W));
    hspmm_host::parallel_blocks(W, windows_per_worker, [&](size_t wb, size_t we) {
        for (size_t w = wb; w < we; ++w) {
            const uint32_t *col = tcA2B + size_t(rowOffset[w]) * cw;
            const uint32_t nreal = real_columns(uint32_t(w));
            uint32_t i = 0, tiles = 0, last_pn = 0;
            while (i < nreal) {
                const uint32_t pn = col[i] / KP, a = i;
                while (i < nreal && col[i] / KP == pn) ++i;
                while ((tiles || tall_stream) && pn - last_pn > kMaxJump) { last_pn += kMaxJump; ++tiles; }
                tiles += (i - a + rw - 1) / rw;
                last_pn = pn;
            }
            rt_rowOffset[w + 1] = tiles;
        }
    });
    for (uint32_t w = 0; w < W; ++w) rt_rowOffset[w + 1] += rt_rowOffset[w];
    const size_t RT = rt_rowOffset[W];
    hspmm_host::ZeroedBuffer<uint32_t> rt_ids(RT * rw);
    rt_panel.assign(RT, 0u);
    hspmm_host::ZeroedBuffer<uint8_t> rt_data(RT * tile_bytes);
    hspmm_host::parallel_blocks(W, windows_per_worker, [&](size_t wb, size_t we) {
        for (size_t w = wb; w < we; ++w) {
            const uint32_t t0 = rowOffset[w];
            const uint32_t *col = tcA2B + size_t(t0) * cw;
            const uint32_t nreal = real_columns(uint32_t(w));
            uint32_t i = 0, last_pn = 0;
            size_t at = rt_rowOffset[w];                             // next step of the window
            while (i < nreal) {
                const uint32_t pn = col[i] / KP, a = i;
                while (i < nreal && col[i] / KP == pn) ++i;
                while ((at > rt_rowOffset[w] || tall_stream) && pn - last_pn > kMaxJump) {   // all-zero step that only carries the jump
                    last_pn += kMaxJump;
                    rt_panel[at++] = last_pn;
                }
                const uint32_t cnt = i - a, nt = (cnt + rw - 1) / rw;
                // The columns of every step.  16-bit MFMA forms: one LDS instruction reads, in each block of 16
                // lanes, the rows of four columns of the step (block g, instruction h: columns 8g + 4h .. + 3), the
                // LDS serves two blocks (g = 0, 1 or g = 2, 3) at a time, and rows whose numbers differ mod 8 lie
                // in different banks.  So a step should hold every remainder mod 8 at most four times, dealt out over
                // the four sets of eight columns that are read together.  Any choice of columns makes a step: the
                // window's columns in this panel, ordered by remainder (stable), are dealt out over the panel's
                // steps in turn - a step then holds floor or ceil of every remainder's share (pruned weights at 10 %:
                // about 26 of 32 rows per remainder and 7 steps; consecutive columns per step gave five or six of one
                // remainder in most steps, one conflict cycle per LDS read) and the steps are equally full.
                uint32_t perm[hspmm::kPanelRowsWide];
                if (rw == 32) {
                    uint32_t m = 0;
                    for (uint32_t res = 0; res < 8; ++res)
                        for (uint32_t k = a; k < i; ++k)
                            if (((col[k] - pn * KP) & 7u) == res) perm[m++] = k;
                }
                for (uint32_t tl = 0; tl < nt; ++tl, ++at) {
                    rt_panel[at] = pn;
                    // n columns: rw == 32: perm[tl], perm[tl + nt], ... (in remainder order); else consecutive ones
                    const uint32_t n = rw == 32 ? (cnt - tl + nt - 1) / nt : std::min(rw, cnt - tl * rw);
                    auto source = [&](uint32_t k) { return rw == 32 ? perm[tl + k * nt] : a + tl * rw + k; };
                    uint32_t order[32];
                    if (rw == 32) {
                        for (uint32_t k = 0; k < rw; ++k) {
                            const uint32_t set = k % 4, e = k / 4;          // set = 2 * (g / 2) + h
                            const uint32_t g = 2 * (set / 2) + e / 4, h = set % 2;
                            order[8 * g + 4 * h + e % 4] = k;
                        }
                    } else {
                        for (uint32_t k = 0; k < rw; ++k) order[k] = k;
                    }
                    uint8_t *dt_tile = rt_data.data() + at * tile_bytes;
                    for (uint32_t k = 0; k < rw; ++k) {
                        const uint32_t from = order[k];
                        // Padding (its tile column stays zero) takes the row of a real column that is read together
                        // with it - entries four apart are in one set - so that it asks for no bank of its own: lanes
                        // that read one address are served together.
                        uint32_t real = from;
                        while (real >= n && real >= 4u) real -= 4u;
                        if (real >= n) real = n - 1;
                        const uint32_t srci = source(real);
                        rt_ids[at * rw + k] = col[srci] - pn * KP;      // row inside the panel
                        if (from >= n) continue;
                        const uint8_t *st_tile = src_data + size_t(t0 + srci / cw) * src_tile_bytes;
                        for (uint32_t r = 0; r < 8; ++r)
                            std::memcpy(dt_tile + (size_t(r) * rw + k) * es, st_tile + (size_t(r) * cw + srci % cw) * es, es);
                    }
                }
                last_pn = pn;
            }
        }
    });
    timer.mark("  panel: steps per panel");
    // the units with the re-tiled step counts
    StepStream ps;
    ps.G = st.G; ps.unitRow = st.unitRow; ps.unitWindow = st.unitWindow; ps.n_paired = st.n_paired; ps.n_wide = st.n_wide;
    ps.unitOffset.assign(1, 0u);
    for (uint32_t u = 0; u < U; ++u) {
        const uint32_t w = st.unitWindow[u];
        ps.unitOffset.push_back(ps.unitOffset.back() + (rt_rowOffset[w + 1] - rt_rowOffset[w]));
    }
    ps.n_steps = ps.unitOffset.back();
    // padding inside every panel must not eat the gain
    // (fp32 MFMA forms only: the measurements above include the padding of the 32-column steps)
    if (!forced && rw == cw && double(ps.n_steps) > 1.35 * double(gather_st.n_steps)) return false;
    // poff[u][pn]: first step of unit u at or behind panel pn; step_panel[s]: panel of step s
    std::vector<uint32_t> poff(size_t(U) * (NP + 1)), step_panel(ps.n_steps ? ps.n_steps : 1, 0u);
    // fp32, per step four words: word g packs the panel rows quarter-wave g reads (ids g and g + 4, 7 bits
    // each) and in bits 28..31 the panels the step lies behind its predecessor.
    // 16-bit types, per step one word per four lanes (word q = l / 4, g = q / 4): 9 x the panel rows of
    // columns 8g + q % 4 (bits 4..15) and 8g + 4 + q % 4 (bits 16..27); bits 0..3: the panel count.
    const uint32_t id_words = rw == 32 ? 16u : 4u;
    std::vector<uint32_t> ids(size_t(ps.n_steps) * id_words);
    // fp32 single windows run through the 4x4x1 instruction, which wants row offsets (see Fp32Quad)
    const bool quad = p->dtype == HSPMM_TF32 && !split && st.G == 1;
    hspmm_host::parallel_blocks(U, 16, [&](size_t ub, size_t ue) {
        for (size_t u = ub; u < ue; ++u) {
            const uint32_t t0 = rt_rowOffset[st.unitWindow[u]], n = ps.unitOffset[u + 1] - ps.unitOffset[u];
            uint32_t *po = poff.data() + size_t(u) * (NP + 1);
            uint32_t at = 0;
            for (uint32_t pn = 0; pn <= NP; ++pn) {
                while (at < n && rt_panel[t0 + at] < pn) ++at;
                po[pn] = ps.unitOffset[u] + at;
            }
            for (uint32_t i = 0; i < n; ++i) {
                const uint32_t *src = rt_ids.data() + size_t(t0 + i) * rw;
                uint32_t *dst = ids.data() + size_t(ps.unitOffset[u] + i) * id_words;
                const uint32_t jump = i ? rt_panel[t0 + i] - rt_panel[t0 + i - 1] : 0u;     // <= kMaxJump by construction
                step_panel[ps.unitOffset[u] + i] = rt_panel[t0 + i];
                if (rw == 32) {
                    for (uint32_t q = 0; q < 16; ++q) {
                        const uint32_t c0 = 8u * (q >> 2) + (q & 3u);
                        dst[q] = jump | (src[c0] * 9u) << 4 | (src[c0 + 4] * 9u) << 16;
                    }
                    continue;
                }
                for (uint32_t g = 0; g < 4; ++g) {
                    if (quad)   // byte offsets of rows g and g + 4 inside the panel image; the jump in bits 0..3 of word 0
                        dst[g] = (src[g] << 8 | (g == 0 ? jump : 0u)) | (src[g + 4] << 8) << 16;
                    else
                        dst[g] = (src[g] | src[g + 4] << 7) | jump << 28;
                }
            }
        }
    });
    timer.mark("  panel: ids, offsets");
    hspmm_plan::Panel &pl = p->panel;
    int rc;
    hspmm_host::ZeroedBuffer<uint32_t> tiles = split      ? lane_order_split_steps(ps, rt_rowOffset.data(), rt_data.data())
                                  : cw == 16 ? lane_order_wide_steps(ps, rt_rowOffset.data(), rt_data.data())
                                             : lane_order_tiles(ps, p->dtype, rt_rowOffset.data(), rt_data.data());
    // Two units per consumer wave, and tiles without their zeros (kernels built on the 16-bit MFMA, units of one
    // or two windows): fewer 128-byte lines through the compute units' L1s (one copy of a panel in LDS serves
    // twice the rows; a packed step is its stored values and 64 bytes of masks).  Measured, the lines go down
    // by a third and by 60 % and the time does not: what binds these kernels is the LDS reads and MFMAs of a
    // step, which a SIMD runs one after the other.  Both are therefore taken on request only
    // (hspmm_set_panel_stream, libraries built with EXPERIMENTAL=1).
    timer.mark("  panel: tiles in lane order");
    bool tall = false, packed = false;
    if (tall_stream) {
        tall = true;
        const size_t tile_words = split ? 512u : 256u;
        merge_unit_pairs(U, NP, tile_words, ps.unitOffset, poff, step_panel, ids, tiles);
        packed = p->cfg.panel_packed > 0;
    }
    if ((rc = upload(p, &pl.d_poff, poff.data(), poff.size()))) { *rc_out = rc; return false; }
    if ((rc = upload(p, &pl.d_step_panel, step_panel.data(), step_panel.size()))) { *rc_out = rc; return false; }
    if ((rc = upload(p, &pl.d_ids, ids.data(), ids.size()))) { *rc_out = rc; return false; }
    if (packed) {
        std::vector<uint64_t> masks;
        std::vector<uint8_t> vals;
        std::vector<uint32_t> step_voff;
        pack_steps(ps.n_steps, split, tiles, masks, vals, step_voff);
        if (vals.size() >= (size_t(1) << 32)) packed = false;        // positions are 32-bit byte offsets in the kernel
        else {
            uint8_t *dv = nullptr;
            if ((rc = upload(p, &pl.d_masks, masks.data(), masks.size()))) { *rc_out = rc; return false; }
            if ((rc = upload(p, &dv, vals.data(), vals.size()))) { *rc_out = rc; return false; }
            pl.d_vals = dv;
            if ((rc = upload(p, &pl.d_step_voff, step_voff.data(), step_voff.size()))) { *rc_out = rc; return false; }
        }
    }
    if (!packed) {
        uint32_t *dt = nullptr;
        if ((rc = upload(p, &dt, tiles.data(), tiles.size()))) { *rc_out = rc; return false; }
        pl.d_tiles = dt;
    }
    pl.tall = tall; pl.packed = packed;
    if (tall) {
        size_t stored = 0;
        const uint16_t *hv = reinterpret_cast<const uint16_t *>(tiles.data());
        if (packed) for (size_t i = 0, n = tiles.size() * 2; i < n; ++i) stored += hv[i] != 0;
        const double step_bytes = 64.0 + (packed ? 64.0 + 2.0 * double(stored) / double(std::max<uint32_t>(ps.n_steps, 1u))
                                                 : double(tiles.size()) * 4.0 / double(std::max<uint32_t>(ps.n_steps, 1u)));
        pl.unit_lines = step_bytes * double(ps.n_steps) / (double(U) * double(NP)) / 128.0;
    }
    if ((rc = upload(p, &pl.d_unitRow, st.unitRow.data(), st.unitRow.size()))) { *rc_out = rc; return false; }
    pl.n_units = U; pl.G = st.G; pl.n_paired = st.n_paired; pl.n_wide = st.n_wide;
    pl.n_panels = NP; pl.n_steps = ps.n_steps; pl.quad = quad; pl.split = split; pl.density = density; pl.built = true;
    timer.mark("  panel: upload");
    return true;
}

// The caller's bitmap tiles (HSPMM_BITS_PER_TILE words: two per 8 x 16 tile, one per 8 x 8 tile of fp32 storage):
// reference BTCF_MTX, src/utils/class.h:55-67.
struct BitmapSource { const uint32_t *nnzOffset; const uint64_t *tcBit; const void *data; };
// The ends of the caller's groups (groupOffset of the reference's GBTCF_MTX, src/utils/class.h:93-108), n + 1 of them.
struct GroupCuts { const uint32_t *offsets; uint32_t n_groups; };
constexpr int kNeedsPlainTiles = -1000;     // create_plan with a BitmapSource: this matrix needs the tiles on the host

// Header of the gather kernels' bitmap stream straight from the caller's arrays; returns the first tile whose bit
// count differs from its nnzOffset span (HSPMM_IDX_MAX: none).
uint32_t bitmap_header_from_caller(uint32_t T, uint32_t elem, const BitmapSource &src, hspmm_host::ZeroedBuffer<uint32_t> &header)
{
    header = hspmm_host::ZeroedBuffer<uint32_t>(size_t(T) * (elem == 2u ? 8u : 4u));
    std::atomic<uint32_t> first_bad{HSPMM_IDX_MAX};
    hspmm_host::parallel_blocks(T, 4096, [&](size_t tb, size_t te) {
        for (size_t t = tb; t < te; ++t) {
            if (elem == 4u) {
                // 8 x 8 tiles of 32-bit elements: one 64-bit word per tile; header = rows 0..3, rows 4..7, position, count
                uint32_t *hd = header.data() + t * 4u;
                hd[0] = uint32_t(src.tcBit[t]); hd[1] = uint32_t(src.tcBit[t] >> 32);
                hd[2] = src.nnzOffset[t];
                hd[3] = uint32_t(__builtin_popcount(hd[0])) + uint32_t(__builtin_popcount(hd[1]));
                if (src.nnzOffset[t + 1] < src.nnzOffset[t] || src.nnzOffset[t + 1] - src.nnzOffset[t] != hd[3]) {
                    uint32_t seen = first_bad.load();
                    while (uint32_t(t) < seen && !first_bad.compare_exchange_weak(seen, uint32_t(t))) {}
                }
                continue;
            }
            uint32_t *hd = header.data() + t * 8u;
            hd[0] = uint32_t(src.tcBit[2 * t]); hd[1] = uint32_t(src.tcBit[2 * t] >> 32);
            hd[2] = uint32_t(src.tcBit[2 * t + 1]); hd[3] = uint32_t(src.tcBit[2 * t + 1] >> 32);
            const uint32_t c0 = uint32_t(__builtin_popcount(hd[0])), c1 = c0 + uint32_t(__builtin_popcount(hd[1])),
                           c2 = c1 + uint32_t(__builtin_popcount(hd[2])), c3 = c2 + uint32_t(__builtin_popcount(hd[3]));
            hd[4] = c0 << 8 | c1 << 16 | c2 << 24;
            hd[5] = src.nnzOffset[t];
            if (src.nnzOffset[t + 1] < src.nnzOffset[t] || src.nnzOffset[t + 1] - src.nnzOffset[t] != c3) {
                uint32_t seen = first_bad.load();
                while (uint32_t(t) < seen && !first_bad.compare_exchange_weak(seen, uint32_t(t))) {}
            }
        }
    });
    return first_bad.load();
}

// Stored entries per real tile column, from 256 groups of 64 tiles spread over the matrix (every tile of a small one).
// header: their masks, where they are known.
double entries_per_column(uint32_t T, uint32_t cw, uint32_t elem, const uint32_t *tcA2B, const void *data, const BitmapSource *bitmap,
                          const uint32_t *header)
{
    const uint32_t group = 64u, groups = std::min(256u, (T + group - 1u) / group);
    uint64_t stored = 0, columns = 0;
    for (uint32_t g = 0; g < groups; ++g) {
        const uint32_t t0 = uint32_t(uint64_t(T) * g / groups), t1 = std::min(T, t0 + group);
        for (size_t i = size_t(t0) * cw; i < size_t(t1) * cw; ++i) columns += tcA2B[i] != HSPMM_IDX_MAX;
        if (bitmap) {
            stored += bitmap->nnzOffset[t1] - bitmap->nnzOffset[t0];
        } else if (header) {
            const uint32_t words = elem == 2u ? 8u : 4u, masks = words / 2u;
            for (size_t t = t0; t < t1; ++t)
                for (uint32_t q = 0; q < masks; ++q) stored += uint32_t(__builtin_popcount(header[t * words + q]));
        } else if (elem == 2u) {
            const uint16_t *v = static_cast<const uint16_t *>(data);
            for (size_t i = size_t(t0) * 8u * cw; i < size_t(t1) * 8u * cw; ++i) stored += v[i] != 0;
        } else {
            const uint32_t *v = static_cast<const uint32_t *>(data);
            for (size_t i = size_t(t0) * 8u * cw; i < size_t(t1) * 8u * cw; ++i) stored += v[i] != 0;
        }
    }
    return columns ? double(stored) / double(columns) : 8.0;
}

// Whether the gather kernels of a plan would read these plain tiles (single windows) as bitmap + stored elements:
// 32 + 2 e bytes against 256 per tile with e stored elements (16 + 4 e for fp32) - worth it below about a third full, and
// where the tile stream is large enough to be traffic at all (a matrix whose tiles sit in the L2s only pays the longer
// dependent chain: 4096 x 4096 at 1 %, 2.7 MB of tiles: 6.8 -> 7.5 us).  From 64 groups of 64 tiles spread over the matrix.
// share: the part of their elements that the sample stores (0: not looked at), whatever the answer.
bool tiles_look_sparse(const Config &cfg, uint32_t T, uint32_t elem, const void *data, double *share)
{
    *share = 0.0;
    if (cfg.gather_bitmap >= 0) return cfg.gather_bitmap > 0;
    if (size_t(T) * 256u < (size_t(8) << 20)) return false;
    std::vector<uint32_t> header(64u * 8u);
    uint64_t stored = 0, seen = 0;
    for (uint32_t g = 0; g < 64u; ++g) {
        const size_t t0 = size_t(uint64_t(T) * g / 64u), n = std::min<size_t>(64u, T - t0);
        stored += hspmm_host::tile_masks(static_cast<const char *>(data) + t0 * 256u, n, elem, header.data());
        seen += n * (256u / elem);
    }
    *share = double(stored) / double(seen);
    return stored * 3u < seen;
}

// What a step of a plan's creation that may run on another thread came to: its code, and its message, which belongs to that thread.
struct Outcome {
    int rc = HSPMM_OK;
    std::string text;
    static Outcome of(int rc) { return {rc, rc ? hspmm_last_error() : ""}; }
};

// The device the plan is for.
int find_device(hspmm_plan *p)
{
    hipError_t e = hipGetDevice(&p->device);
    if (e != hipSuccess) return fail(HSPMM_ERR_DEVICE, "hipGetDevice failed: %s", hipGetErrorString(e));
    hipDeviceProp_t prop;
    e = hipGetDeviceProperties(&prop, p->device);
    if (e != hipSuccess) return fail(HSPMM_ERR_DEVICE, "hipGetDeviceProperties failed: %s", hipGetErrorString(e));
    if (strncmp(prop.gcnArchName, "gfx950", 6) != 0)
        return fail(HSPMM_ERR_UNSUPPORTED, "device %d is %s; this library is built for gfx950 only", p->device, prop.gcnArchName);
    p->compute_units = p->cfg.sm_num > 0 ? p->cfg.sm_num : prop.multiProcessorCount;
    // the address of this device's fixed scratch array, for hspmm_run_static (which then looks nothing up)
    float *unused = nullptr;
    return static_scratch_address(p->device, &unused);
}

// (worker threads start on the first device)
int copy_up(const hspmm_plan *p, void *to, const void *from, size_t bytes)
{
    HSPMM_HIP(hipSetDevice(p->device));
    HSPMM_HIP(hipMemcpy(to, from, bytes, hipMemcpyHostToDevice));
    return HSPMM_OK;
}

// One block of device memory for everything whose size is known early and, where there is as much, for `likely` bytes that a sample speaks of, and
// the arrays that are checked already or lie inside checked bounds.
int upload_windows(hspmm_plan *p, const uint32_t *rowOffset, const uint32_t *rowIdx, const uint32_t *tcA2B, size_t block, size_t likely)
{
    HSPMM_HIP(hipSetDevice(p->device));
    int rc = plan_reserve(p, block + likely);
    if (rc && likely) { (void)hipGetLastError(); rc = plan_reserve(p, block); }
    if (rc) return rc;
    if (int rc = upload(p, &p->d_rowOffset, rowOffset, size_t(p->W) + 1)) return rc;
    if (int rc = upload(p, &p->d_rowIdx, rowIdx, size_t(p->W))) return rc;
    return upload(p, &p->d_a2b_raw, tcA2B, size_t(p->T) * p->cw);
}

int upload_units(hspmm_plan *p, const StepStream &st)
{
    HSPMM_HIP(hipSetDevice(p->device));
    if (int rc = upload(p, &p->d_unitOffset, st.unitOffset.data(), st.unitOffset.size())) return rc;
    return upload(p, &p->d_unitRow, st.unitRow.data(), st.unitRow.size());
}

// What the kernels walk of a schedule, in host memory.
struct ScheduleTables {
    enum { kOffset, kInfo, kItems, kRanges, kSplit, kFix, kCount };
    std::vector<uint32_t> words;
    size_t at[kCount] = {};
    uint32_t n_units = 0, n_ranges = 0, n_split = 0, n_slots = 0;
    bool wanted() const { return n_units != 0; }
};

// (from the caller's windows: what they say is checked already, their tiles may not be)
ScheduleTables schedule_tables(const hspmm_plan *p, const uint32_t *rowOffset, const uint32_t *rowIdx)
{
    ScheduleTables out;
    const uint32_t T = p->T, W = p->W;
    if (p->cfg.schedule == 0 || p->elem != 2u || (p->cfg.kernel_mode != 0 && p->cfg.kernel_mode != 3) || p->cfg.gather_bitmap == 0 || p->cfg.consumer_warp_num ||
        p->cfg.producer_warp_group_num || p->cfg.buffer_stage)
        return out;
    if (p->cfg.schedule < 0 && p->cols < kScheduledColumns) return out;
    uint32_t longest = 0, shortest = HSPMM_IDX_MAX;
    for (uint32_t w = 0; w < W; ++w) {
        longest = std::max(longest, rowOffset[w + 1] - rowOffset[w]);
        shortest = std::min(shortest, rowOffset[w + 1] - rowOffset[w]);
    }
    if (!shortest || (p->cfg.schedule < 0 && windows_are_even(longest, W, T))) return out;
    const uint32_t most = (T + kMinTilesPerRange - 1u) / kMinTilesPerRange;
    const uint32_t n_waves = std::max(1u, std::min(p->cfg.schedule > 1 ? uint32_t(p->cfg.schedule) : uint32_t(p->compute_units) * 8u, most));
    if (p->cfg.schedule < 0 && uint64_t(longest) * n_waves > uint64_t(T) * kScheduledLongest) return out;
    const hspmm::Schedule s = hspmm::build_schedule(W, rowOffset, n_waves);
    const uint32_t n = uint32_t(s.items.size()), n_ranges = std::min(n_waves, n);   // (the first waves are the ones that have items)
    // cut windows: their parts have neighbouring slots
    std::vector<uint32_t> entry_of(W, HSPMM_IDX_MAX), split;
    uint32_t n_slots = 0;
    for (uint32_t i = 0; i < n; ++i) {
        const hspmm::ScheduleItem &it = s.items[i];
        if (it.parts == 1u || entry_of[it.window] != HSPMM_IDX_MAX) continue;
        entry_of[it.window] = uint32_t(split.size() / hspmm::kFixWords);
        split.insert(split.end(), {i, n_slots, it.parts, 0u});
        n_slots += it.parts;
    }
    const size_t sizes[ScheduleTables::kCount] = {size_t(n) + 1u, size_t(n) * 4u, size_t(n) * 4u, size_t(n_ranges) * hspmm::kRangeWords, split.size(),
                                                  size_t(n_slots) * 2u};
    size_t total = 0;
    for (size_t k = 0; k < ScheduleTables::kCount; ++k) { out.at[k] = total; total += (sizes[k] + 63u) & ~size_t(63); }
    out.words.assign(total, 0u);
    auto table = [&](int k) { return out.words.data() + out.at[k]; };
    uint32_t *offset = table(ScheduleTables::kOffset), *info = table(ScheduleTables::kInfo), *items = table(ScheduleTables::kItems),
             *ranges = table(ScheduleTables::kRanges), *fix = table(ScheduleTables::kFix);
    for (uint32_t i = 0; i < n; ++i, info += 4, items += 4) {
        const hspmm::ScheduleItem &it = s.items[i];
        const bool cut = it.parts > 1u, last = it.part + 1u == it.parts;
        const uint32_t slot = cut ? split[size_t(entry_of[it.window]) * hspmm::kFixWords + 1u] + it.part : HSPMM_IDX_MAX;
        offset[i + 1u] = offset[i] + it.steps;
        info[0] = (rowIdx[it.window] & ~7u) | (it.window == 0u && it.part == 0u ? 1u : 0u);
        info[1] = !last ? 0u : it.window + 1u < W ? rowIdx[it.window + 1u] & ~7u : p->rows;
        info[2] = slot;
        info[3] = entry_of[it.window];
        if (cut) { fix[slot] = slot; fix[size_t(n_slots) + slot] = i; }
        items[0] = it.first; items[1] = it.stride; items[2] = offset[i]; items[3] = it.steps;
    }
    for (uint32_t w = 0; w < n_ranges; ++w, ranges += hspmm::kRangeWords) {
        std::fill(ranges, ranges + hspmm::kRangeWords, HSPMM_IDX_MAX);
        ranges[0] = offset[s.waves[w]]; ranges[1] = offset[s.waves[w + 1u]]; ranges[2] = s.waves[w]; ranges[7] = 0u;
    }
    for (size_t k = 0; k < split.size(); k += hspmm::kFixWords) split[k + 3u] = n_slots + split[k + 1u];
    std::copy(split.begin(), split.end(), table(ScheduleTables::kSplit));
    out.n_units = n; out.n_ranges = n_ranges; out.n_split = uint32_t(split.size() / hspmm::kFixWords); out.n_slots = n_slots;
    return out;
}

// Device memory of the schedule: ids, headers and tables in one piece; null where there is none for it (the plan is made without).
uint32_t *schedule_room(hspmm_plan *p, const ScheduleTables &t)
{
    void *room = nullptr;
    if (plan_alloc(p, (size_t(p->T) * 24u + t.words.size()) * 4u, &room)) { (void)hipGetLastError(); return nullptr; }
    return static_cast<uint32_t *>(room);
}

// Behind its tables (copied) and the plan's ids and headers.
int fill_schedule(hspmm_plan *p, const ScheduleTables &t, uint32_t *room)
{
    hspmm_plan::Scheduled &sc = p->scheduled;
    uint32_t *ids = room, *header = room + size_t(p->T) * 16u, *tables = header + size_t(p->T) * 8u;
    HSPMM_HIP(hspmm::launch_schedule_fill(tables + t.at[ScheduleTables::kItems], t.n_units, p->d_ids, p->bm.d_header, ids, header, nullptr));
    sc.d_ids = ids; sc.d_header = header;
    sc.d_unitOffset = tables + t.at[ScheduleTables::kOffset]; sc.d_info = tables + t.at[ScheduleTables::kInfo];
    sc.d_ranges = tables + t.at[ScheduleTables::kRanges]; sc.d_split = tables + t.at[ScheduleTables::kSplit]; sc.d_fix_slots = tables + t.at[ScheduleTables::kFix];
    sc.n_units = t.n_units; sc.n_ranges = t.n_ranges; sc.n_split = t.n_split; sc.n_slots = t.n_slots;
    sc.built = true;
    return HSPMM_OK;
}

// hspmm_create; with `bitmap` (data == nullptr) the tiles come as the caller's bitmap arrays,
// which are uploaded as they are, kept as the gather kernels' bitmap stream and expanded on the device for the
// kernels that read plain tiles.  Returns kNeedsPlainTiles when the plan would need the tiles on the host
// (windows paired through equal column lists; the caller then expands them).
int create_plan(hspmm_plan **out, int dtype, uint32_t rows, uint32_t cols, uint32_t eff_row_windows,
                uint32_t total_tiles, const uint32_t *rowOffset, const uint32_t *tcA2B, const void *data,
                const uint32_t *rowIdx, const BitmapSource *bitmap, const GroupCuts *cuts = nullptr)
{
    if (!out) return fail(HSPMM_ERR_INVALID, "null plan pointer");
    *out = nullptr;
    if (dtype != HSPMM_FP16 && dtype != HSPMM_TF32 && dtype != HSPMM_BF16)
        return fail(HSPMM_ERR_INVALID, "unknown dtype %d", dtype);
    const uint32_t cw = dtype == HSPMM_TF32 ? 8u : 16u;
    const uint32_t elem = dtype == HSPMM_TF32 ? 4u : 2u;
    PhaseTimer timer;
    Config cfg;
    { std::lock_guard<std::mutex> lk(g_cfg_mutex); cfg = g_cfg; }
    cfg.read_environment();                         // tuning overrides, once per plan
    bool canonical = true;
    // Tiles that are mostly zeros go to the device as bitmap + stored elements and are expanded there: the gather kernels
    // read that stream, and a graph of 2^18 vertices is 24 MB to send instead of 77.
    hspmm_host::ZeroedBuffer<uint32_t> header;
    std::vector<uint32_t> window_stored;
    double likely_stored = 0.0;
    bool sparse_tiles = !bitmap && data && eff_row_windows && total_tiles && tiles_look_sparse(cfg, total_tiles, elem, data, &likely_stored);
    try {
        if (sparse_tiles) {
            header = hspmm_host::ZeroedBuffer<uint32_t>(size_t(total_tiles) * (elem == 2u ? 8u : 4u));
            window_stored.assign(size_t(eff_row_windows) + 1u, 0u);
        }
    } catch (const std::bad_alloc &) { return fail(HSPMM_ERR_ALLOC, "out of host memory"); }
    const void *tile_values = bitmap ? bitmap->data : data;
    int rc = validate_windows(rows, cols, eff_row_windows, total_tiles, rowOffset, tcA2B, tile_values, rowIdx);
    if (rc) return rc;

    hspmm_plan *p = new (std::nothrow) hspmm_plan;
    if (!p) return fail(HSPMM_ERR_ALLOC, "out of host memory");
    p->dtype = dtype; p->rows = rows; p->cols = cols; p->W = eff_row_windows; p->T = total_tiles;
    p->cw = cw; p->elem = elem;
    p->cfg = cfg;

    auto bail = [&](int code) { hspmm_destroy(p); return code; };
    // (arrays that are not good are told of before a device that is not there)
    Outcome device;
    StepStream st;
    ScheduleTables schedule;
    const size_t n_ids = size_t(total_tiles) * cw, tile_bytes = size_t(total_tiles) * 256u;
    const size_t spare = 8u / elem;                                     // a lane may read 8 bytes from the last element on
    try {
        device = Outcome::of(find_device(p));
        // Side by side: the tiles' checks and masks on all cores, the units, device memory and the arrays whose sizes are known.
        Outcome tiles, arrays;
        std::atomic<int> next{0};
        parallel_workers(p->W ? 4u : 1u, [&](unsigned) {
            for (int task = next++; task < 4; task = next++) {
                if (task == 0) {
                    tiles = Outcome::of(validate_tiles(cols, eff_row_windows, total_tiles, cw, rowOffset, tcA2B, tile_values, &canonical,
                                                       sparse_tiles ? header.data() : nullptr, window_stored.data()));
                } else if (task == 1 && !device.rc && p->W) {
                    arrays = Outcome::of(upload_windows(p, rowOffset, rowIdx, tcA2B,
                                                        entries_count_bytes(p) + (size_t(p->W) * 4u + 2u) * 4u + n_ids * 8u + tile_bytes + header.size() * 4u + (size_t(1) << 20),
                                                        sparse_tiles ? size_t(likely_stored * 1.1 * double(tile_bytes)) : 0u));
                } else if (task == 2 && p->W) {
                    st = build_units(p->W, cw, rowOffset, rowIdx, tcA2B, p->cfg.pairing);
                } else if (task == 3 && !device.rc && p->W) {
                    schedule = schedule_tables(p, rowOffset, rowIdx);
                }
            }
        });
        for (const Outcome *o : {&tiles, &device, &arrays})
            if (o->rc) return bail(fail(o->rc, "%s", o->text.c_str()));
    } catch (const std::bad_alloc &) { return bail(fail(HSPMM_ERR_ALLOC, "out of host memory")); }
    p->canonical = canonical;
    timer.mark("checks, masks, units, ids");

    // (a host allocation that fails anywhere below ends the call with HSPMM_ERR_ALLOC)
    if (p->W) try {
        if (bitmap && st.G != 1) return bail(kNeedsPlainTiles);         // paired windows: their tiles are re-laid out on the host
        p->G = st.G;
        p->n_units = uint32_t(st.unitRow.size());
        p->n_paired = st.n_paired;
        p->n_steps = st.n_steps;
        p->h_unitOffset = st.unitOffset;
        p->h_unitRow = st.unitRow;
        // single windows walked tile by tile: the caller's tile numbers are the stream's, its cuts can be kept
        if (cuts && p->cfg.group_cuts && st.G == 1) p->caller_cuts.assign(cuts->offsets, cuts->offsets + size_t(cuts->n_groups) + 1u);
        uint64_t stored = 0;
        for (uint32_t w = 0; sparse_tiles && w < p->W; ++w) stored += window_stored[w];
        sparse_tiles = sparse_tiles && st.G == 1 && stored + spare < (uint64_t(1) << 31) &&
                       (p->cfg.gather_bitmap > 0 || stored * 3u < uint64_t(total_tiles) * 8u * cw);
        p->per_column = entries_per_column(total_tiles, cw, elem, tcA2B, data, bitmap, sparse_tiles ? header.data() : nullptr);
        const bool scheduled = schedule.wanted() && p->canonical && p->caller_cuts.empty() && (p->cfg.schedule > 0 || p->per_column > kScheduledColumnsShared);
        void *room = nullptr;
        uint32_t *schedule_at = nullptr;
        auto copy_schedule = [&] { return copy_up(p, schedule_at + size_t(total_tiles) * 24u, schedule.words.data(), schedule.words.size() * 4u); };
        if (sparse_tiles) {
            // Side by side: the stored elements one after the other, and what else the launches need of the host.
            std::vector<uint64_t> first(p->W);
            for (uint64_t w = 0, at = 0; w < p->W; ++w) { first[w] = at; at += window_stored[w]; }
            const size_t vals_bytes = (size_t(stored) + spare) * elem, header_bytes = header.size() * 4u;
            hspmm_host::ZeroedBuffer<uint8_t> vals(vals_bytes);
            if ((rc = plan_alloc(p, header_bytes, &room))) return bail(rc);
            p->bm.d_header = static_cast<uint32_t *>(room);
            if ((rc = plan_alloc(p, vals_bytes, &room))) return bail(rc);
            p->bm.d_vals = room;
            if ((rc = plan_alloc(p, tile_bytes, &room))) return bail(rc);
            p->d_data = room;
            if (scheduled) schedule_at = schedule_room(p, schedule);
            const uint32_t header_words = elem == 2u ? 8u : 4u;
            auto by_windows = [&](auto fn) {
                hspmm_host::parallel_weighted(p->W, size_t(1) << 13, [=](size_t w) { return rowOffset[w]; }, fn);
            };
            Outcome elements, rest, walk;
            std::atomic<int> next{0};
            parallel_workers(schedule_at ? 3u : 2u, [&](unsigned) {
                for (int task = next++; task < 3; task = next++) {
                    if (task == 0) {
                        by_windows([&](size_t wb, size_t we) {
                            const uint32_t t0 = rowOffset[wb];
                            hspmm_host::pack_tiles(static_cast<const char *>(data) + size_t(t0) * 256u, rowOffset[we] - t0, elem,
                                                   header.data() + size_t(t0) * header_words, first[wb], vals.data());
                        });
                        elements = Outcome::of(copy_up(p, const_cast<void *>(p->bm.d_vals), vals.data(), vals_bytes));
                    } else if (task == 2) {
                        if (schedule_at) walk = Outcome::of(copy_schedule());
                    } else {
                        rest = Outcome::of(upload_units(p, st));
                        if (!rest.rc) rest = Outcome::of(build_and_upload_partition(p, 0));
                        by_windows([&](size_t wb, size_t we) {
                            const uint32_t t0 = rowOffset[wb];
                            hspmm_host::place_tiles(header.data() + size_t(t0) * header_words, rowOffset[we] - t0, elem, first[wb]);
                        });
                        if (!rest.rc) rest = Outcome::of(copy_up(p, p->bm.d_header, header.data(), header_bytes));
                    }
                }
            });
            for (const Outcome *o : {&elements, &rest, &walk})
                if (o->rc) return bail(fail(o->rc, "%s", o->text.c_str()));
            p->bm.stored = stored; p->bm.built = true;
            HSPMM_HIP_OR(hspmm::launch_expand_bitmap(int(elem), p->bm.d_header, p->bm.d_vals, p->d_data, total_tiles, nullptr), bail);
            timer.mark("bitmap tiles, partition");
        } else if (!bitmap) {
            uint8_t *dd = nullptr;
            if ((rc = upload(p, &dd, static_cast<const uint8_t *>(data), tile_bytes))) return bail(rc);
            p->d_data = dd;
        } else {
            // the caller's bitmap tiles: header from tcBit / nnzOffset, the stored elements as they are (and four
            // more: a lane of the gather kernels reads 8 bytes from its first element), plain tiles by a kernel
            const uint32_t bad = bitmap_header_from_caller(total_tiles, elem, *bitmap, header);
            if (bad != HSPMM_IDX_MAX)
                return bail(fail(HSPMM_ERR_INVALID, "tile %u: %s", bad, "the bit count of tcBit differs from the nnzOffset span"));
            stored = bitmap->nnzOffset[total_tiles];
            if (stored + spare >= (uint64_t(1) << 31)) return bail(kNeedsPlainTiles);    // positions are 32-bit
            if ((rc = plan_alloc(p, tile_bytes, &room))) return bail(rc);
            p->d_data = room;
            if ((rc = upload(p, &p->bm.d_header, header.data(), header.size()))) return bail(rc);
            const size_t vals_bytes = (size_t(stored) + spare) * elem;
            if ((rc = plan_alloc(p, vals_bytes, &room))) return bail(rc);
            char *dv = static_cast<char *>(room);
            p->bm.d_vals = dv; p->bm.stored = stored;
            if (stored) HSPMM_HIP_OR(hipMemcpy(dv, bitmap->data, size_t(stored) * elem, hipMemcpyHostToDevice), bail);
            HSPMM_HIP_OR(hipMemset(dv + size_t(stored) * elem, 0, 8), bail);
            HSPMM_HIP_OR(hspmm::launch_expand_bitmap(int(elem), p->bm.d_header, dv, p->d_data, total_tiles, nullptr), bail);
            HSPMM_HIP_OR(hipStreamSynchronize(nullptr), bail);
            p->bm.from_caller = true;
        }
        timer.mark("upload format arrays");
        if (!sparse_tiles && (rc = upload_units(p, st))) return bail(rc);
        // padding ids -> the real id in front of them (the tile column is all zero; no tile starts with padding)
        if (st.G == 1) {
            // single windows: the steps are the caller's tiles in the caller's order
            if ((rc = plan_alloc(p, n_ids * 4u, &room))) return bail(rc);
            p->d_ids = static_cast<uint32_t *>(room);
            HSPMM_HIP_OR(hspmm::launch_step_ids(int(elem), p->d_a2b_raw, p->d_ids, total_tiles, nullptr), bail);
        } else {
            hspmm_host::ZeroedBuffer<uint32_t> clean_ids(n_ids);
            uint32_t *clean = clean_ids.data();
            hspmm_host::parallel_blocks(p->W, 1024, [&](size_t wb, size_t we) {
                for (size_t i = size_t(rowOffset[wb]) * cw, e = size_t(rowOffset[we]) * cw; i < e; ++i)
                    clean[i] = (tcA2B[i] == HSPMM_IDX_MAX && i) ? clean[i - 1] : tcA2B[i];
            });
            const hspmm_host::ZeroedBuffer<uint32_t> ids = lane_order_ids(st, dtype, rowOffset, clean);
            if ((rc = upload(p, &p->d_ids, ids.data(), ids.size()))) return bail(rc);
        }
        // (single fp32 windows: decided below, once it is known whether the gather kernels of this plan read
        // bitmap tiles - then nothing reads tiles in lane order)
        const bool lane_tiles_later = dtype == HSPMM_TF32 && st.G == 1;
        if (dtype != HSPMM_TF32 && st.G == 1) {
            p->d_tiles = p->d_data;                 // the caller's tile layout already is the lane order
        } else if (!lane_tiles_later) {
            const hspmm_host::ZeroedBuffer<uint32_t> tiles = lane_order_tiles(st, dtype, rowOffset, data);
            uint32_t *dt = nullptr;
            if ((rc = upload(p, &dt, tiles.data(), tiles.size()))) return bail(rc);
            p->d_tiles = dt;
        }
        timer.mark("step stream (ids, tiles)");
        // Single windows with few stored elements per tile (graphs: 16 of 128): the gather kernels read the tiles as
        // bitmap + stored elements, 32 + 2 x 16 bytes per tile instead of 256 (power-law graph 2^20 at N = 128, where
        // the stream is read once per XCD half: 0.64 -> 0.19 GB per launch).
        if (bitmap) {
            // (the rule of tiles_look_sparse, with the exact number of stored elements)
            p->bm.built = total_tiles && p->cfg.gather_bitmap != 0 &&
                          (p->cfg.gather_bitmap > 0 ||
                           (stored * 3u < uint64_t(total_tiles) * 8u * cw && tile_bytes >= (size_t(8) << 20)));
            if (!p->bm.built) {
                plan_release(p, p->bm.d_header, header.size() * 4u);
                plan_release(p, p->bm.d_vals, (size_t(stored) + spare) * elem);
                p->bm.d_header = nullptr; p->bm.d_vals = nullptr;
            }
        }
        if (lane_tiles_later && total_tiles && !(p->bm.built && (p->cfg.kernel_mode == 0 || p->cfg.kernel_mode == 3))) {
            // single fp32 windows: steps are the caller's tiles in the caller's order; a kernel re-orders each for the lanes
            if ((rc = plan_alloc(p, tile_bytes, &room))) return bail(rc);
            p->d_tiles = room;
            HSPMM_HIP_OR(hspmm::launch_lane_order32(p->d_data, room, total_tiles, nullptr), bail);
        }
        {
            uint32_t longest = 0;
            for (size_t u = 0; u + 1 < st.unitOffset.size(); ++u) longest = std::max(longest, st.unitOffset[u + 1] - st.unitOffset[u]);
            p->even_windows = windows_are_even(longest, p->n_units, p->n_steps);
        }
        if (st.G != 1) {
            p->h_winOffset.assign(rowOffset, rowOffset + size_t(p->W) + 1u);
            p->h_winRow.assign(rowIdx, rowIdx + size_t(p->W));
        }
        if ((rc = build_and_upload_partition(p, 0))) return bail(rc);
        if ((rc = count_entries(p))) return bail(rc);                   // (behind the last of the small uploads, which would wait for it)
        timer.mark("partition");
        if (!schedule_at && scheduled && p->G == 1 && p->bm.built && (schedule_at = schedule_room(p, schedule)) && (rc = copy_schedule())) return bail(rc);
        if (schedule_at && (rc = fill_schedule(p, schedule, schedule_at))) return bail(rc);
        timer.mark("schedule");
        {
            // all units long, and so long that the balanced partition cuts each of them several ways:
            // eight ranges per unit where it would cut eight ways or more, four from `four_from` ways on
            uint32_t shortest = 0xFFFFFFFFu;
            for (size_t u = 0; u + 1 < st.unitOffset.size(); ++u)
                shortest = std::min(shortest, st.unitOffset[u + 1] - st.unitOffset[u]);
            const double steps_per_range = double(p->n_steps) / double(p->parts[0].part.ranges.size());
            const double ways = double(p->n_steps) / double(p->n_units) / steps_per_range;
            const double four_from = kAlignedFourFrom;
            const int group = ways >= 8.0 ? hspmm::kAlignedGroupWaves : ways >= four_from ? hspmm::kMaxWavesPerGroup : 0;
            if (group && shortest >= 8u * uint32_t(group) && uint64_t(p->n_units) * group <= (1u << 24)) p->aligned_group = group;
            // A matrix too small to fill the waves of the GPU with ranges of useful length: what its launch takes
            // is one wave walking its range step by step (4096 x 4096 at 1 %: 434 waves of 24 dependent steps).
            // One workgroup per unit, its waves a quarter (an eighth) of the unit's steps each, shortens that walk.
            const uint64_t wave_slots = uint64_t(p->compute_units) * 16u;
            int small_group = 0;
            if (p->cfg.aligned_small < 0) {
                if (!p->aligned_group && p->parts[0].part.ranges.size() * 4u <= wave_slots && uint64_t(p->n_units) * 4u <= wave_slots)
                    small_group = hspmm::kMaxWavesPerGroup;      // (eight waves per unit measured no faster: 7.2 against 6.8 us)
            } else {
                small_group = p->cfg.aligned_small;
            }
            if (small_group && shortest >= 2u * uint32_t(small_group)) p->aligned_group = small_group;
            if (!p->caller_cuts.empty()) p->aligned_group = 0;       // (those partitions cut every unit into equal parts)
        }
        // (the LDS-panel stream re-tiles ascending column lists; a caller's lists in another order stay
        // with the gather and all-shapes kernels)
        if (!bitmap && (p->cfg.kernel_mode == 0 || p->cfg.kernel_mode >= 4) && p->canonical) {
            int prc = HSPMM_OK;
            try { (void)build_panel_stream(p, st, rowOffset, tcA2B, data, rowIdx, p->cfg.kernel_mode >= 4, &prc); }
            catch (const std::bad_alloc &) { return bail(fail(HSPMM_ERR_ALLOC, "out of host memory")); }
            if (prc) return bail(prc);
            timer.mark("LDS-panel stream");
        }
        if ((rc = build_tile_stream(p))) return bail(rc);
        timer.mark("full-tile stream");
        if ((rc = build_narrow_stream(p))) return bail(rc);
        timer.mark("narrow stream");
        if ((rc = build_wide_stream(p))) return bail(rc);
        timer.mark("wide-tile stream");
        if ((rc = build_block_units(p, st, rowOffset, tcA2B))) return bail(rc);
        timer.mark("block units");
        if ((rc = entries_counted(p))) return bail(rc);                 // (any stream may launch now)
    } catch (const std::bad_alloc &) {
        return bail(fail(HSPMM_ERR_ALLOC, "out of host memory"));
    }
    *out = p;
    return HSPMM_OK;
}

}  // namespace

extern "C" {

int hspmm_create(hspmm_plan **out, int dtype, uint32_t rows, uint32_t cols, uint32_t eff_row_windows,
                 uint32_t total_tiles, const uint32_t *rowOffset, const uint32_t *tcA2B, const void *data,
                 const uint32_t *rowIdx)
{
    return create_plan(out, dtype, rows, cols, eff_row_windows, total_tiles, rowOffset, tcA2B, data, rowIdx, nullptr);
}

namespace {
// Widths a tile layout may have for an element type: the default one, and 4 for fp32 storage.
int layout_widths(int dtype, uint32_t col_window, uint32_t &cw, uint32_t &cw_default, uint32_t &elem)
{
    if (dtype != HSPMM_FP16 && dtype != HSPMM_TF32 && dtype != HSPMM_BF16)
        return fail(HSPMM_ERR_INVALID, "unknown dtype %d", dtype);
    cw_default = dtype == HSPMM_TF32 ? 8u : 16u;
    elem = dtype == HSPMM_TF32 ? 4u : 2u;
    cw = col_window ? col_window : cw_default;
    if (cw != cw_default && !(dtype == HSPMM_TF32 && cw == 4u))
        return fail(HSPMM_ERR_INVALID, "col_window %u: %u, or 4 for HSPMM_TF32", col_window, cw_default);
    return HSPMM_OK;
}
}  // namespace

int hspmm_btcf_relayout_sizes(int dtype, uint32_t col_window, uint32_t eff_row_windows, const uint32_t *rowOffset,
                              const uint32_t *tcA2B, uint32_t *total_tiles)
{
    uint32_t cw, cw_default, elem;
    if (int rc = layout_widths(dtype, col_window, cw, cw_default, elem)) return rc;
    if (!total_tiles) return fail(HSPMM_ERR_INVALID, "null output");
    const uint32_t W = eff_row_windows;
    if (W && (!rowOffset || !tcA2B)) return fail(HSPMM_ERR_INVALID, "null format array");
    if (W && rowOffset[0] != 0) return fail(HSPMM_ERR_INVALID, "rowOffset[0] = %u, expected 0", rowOffset[0]);
    uint64_t tiles = 0;
    for (uint32_t w = 0; w < W; ++w) {
        if (rowOffset[w + 1] <= rowOffset[w])
            return fail(HSPMM_ERR_INVALID, "rowOffset not strictly increasing at window %u", w);
        const uint32_t *ids = tcA2B + size_t(rowOffset[w]) * cw;
        uint32_t real = 0;
        for (size_t i = 0, n = size_t(rowOffset[w + 1] - rowOffset[w]) * cw; i < n; ++i) real += ids[i] != HSPMM_IDX_MAX;
        if (!real) return fail(HSPMM_ERR_INVALID, "window %u has no column", w);
        tiles += (real + cw_default - 1u) / cw_default;
    }
    if (tiles > 0xffffffffull) return fail(HSPMM_ERR_INVALID, "more than 2^32 - 1 tiles");
    *total_tiles = uint32_t(tiles);
    return HSPMM_OK;
}

int hspmm_btcf_relayout_fill(int dtype, uint32_t col_window, int transposed, uint32_t eff_row_windows,
                             const uint32_t *rowOffset, const uint32_t *tcA2B, const void *data,
                             uint32_t *out_rowOffset, uint32_t *out_tcA2B, void *out_data)
{
    uint32_t cw, cw_default, elem, NT = 0;
    if (int rc = hspmm_btcf_relayout_sizes(dtype, col_window, eff_row_windows, rowOffset, tcA2B, &NT)) return rc;
    layout_widths(dtype, col_window, cw, cw_default, elem);
    const uint32_t W = eff_row_windows;
    if (!out_rowOffset || (NT && (!data || !out_tcA2B || !out_data))) return fail(HSPMM_ERR_INVALID, "null array");
    out_rowOffset[0] = 0;
    for (uint32_t w = 0; w < W; ++w) {
        const uint32_t *ids = tcA2B + size_t(rowOffset[w]) * cw;
        uint32_t real = 0;
        for (size_t i = 0, n = size_t(rowOffset[w + 1] - rowOffset[w]) * cw; i < n; ++i) real += ids[i] != HSPMM_IDX_MAX;
        out_rowOffset[w + 1] = out_rowOffset[w] + (real + cw_default - 1u) / cw_default;
    }
    std::fill(out_tcA2B, out_tcA2B + size_t(NT) * cw_default, HSPMM_IDX_MAX);
    std::memset(out_data, 0, size_t(NT) * 8u * cw_default * elem);
    const uint8_t *src = static_cast<const uint8_t *>(data);
    uint8_t *dst = static_cast<uint8_t *>(out_data);
    hspmm_host::parallel_blocks(W, 1024, [&](size_t wb, size_t we) {
        for (size_t w = wb; w < we; ++w) {
            size_t at = size_t(out_rowOffset[w]) * cw_default;                // next column slot of the window
            for (uint32_t t = rowOffset[w]; t < rowOffset[w + 1]; ++t)
                for (uint32_t k = 0; k < cw; ++k) {
                    const uint32_t id = tcA2B[size_t(t) * cw + k];
                    if (id == HSPMM_IDX_MAX) continue;                        // the real columns keep their order
                    const size_t nt = at / cw_default, nk = at % cw_default;
                    out_tcA2B[at] = id;
                    for (uint32_t r = 0; r < 8u; ++r) {
                        const size_t from = size_t(t) * 8u * cw + (transposed ? size_t(k) * 8u + r : size_t(r) * cw + k);
                        std::memcpy(dst + ((nt * 8u + r) * cw_default + nk) * elem, src + from * elem, elem);
                    }
                    ++at;
                }
        }
    });
    return HSPMM_OK;
}

int hspmm_create_layout(hspmm_plan **out, int dtype, uint32_t col_window, int transposed, uint32_t rows, uint32_t cols,
                        uint32_t eff_row_windows, uint32_t total_tiles, const uint32_t *rowOffset, const uint32_t *tcA2B,
                        const void *data, const uint32_t *rowIdx)
{
    if (!out) return fail(HSPMM_ERR_INVALID, "null plan pointer");
    *out = nullptr;
    uint32_t cw, cw_default, elem;
    if (int rc = layout_widths(dtype, col_window, cw, cw_default, elem)) return rc;
    if (cw == cw_default && !transposed)
        return hspmm_create(out, dtype, rows, cols, eff_row_windows, total_tiles, rowOffset, tcA2B, data, rowIdx);
    const uint32_t W = eff_row_windows;
    if (W && (!rowOffset || !tcA2B || !data || !rowIdx)) return fail(HSPMM_ERR_INVALID, "null format array");
    for (uint32_t w = 0; w < W; ++w)
        if (rowOffset[w + 1] > total_tiles)
            return fail(HSPMM_ERR_INVALID, "rowOffset[%u] = %u beyond total_tiles = %u", w + 1, rowOffset[w + 1], total_tiles);
    if (W && rowOffset[W] != total_tiles)
        return fail(HSPMM_ERR_INVALID, "rowOffset[%u] = %u differs from total_tiles = %u", W, rowOffset[W], total_tiles);
    // the same matrix in the layout hspmm_create reads: tiles of the default width, element (r, k) at r * width + k
    try {
        uint32_t NT = 0;
        if (int rc = hspmm_btcf_relayout_sizes(dtype, col_window, W, rowOffset, tcA2B, &NT)) return rc;
        std::vector<uint32_t> n_rowOffset(size_t(W) + 1), n_ids(size_t(NT) * cw_default);
        std::vector<uint8_t> n_data(size_t(NT) * 8u * cw_default * elem);
        if (int rc = hspmm_btcf_relayout_fill(dtype, col_window, transposed, W, rowOffset, tcA2B, data, n_rowOffset.data(),
                                              n_ids.data(), n_data.data()))
            return rc;
        return hspmm_create(out, dtype, rows, cols, W, NT, n_rowOffset.data(), n_ids.data(), n_data.data(), rowIdx);
    } catch (const std::bad_alloc &) { return fail(HSPMM_ERR_ALLOC, "out of host memory"); }
}

static int create_from_bitmap(hspmm_plan **out, int dtype, uint32_t rows, uint32_t cols, uint32_t eff_row_windows,
                              uint32_t total_tiles, const uint32_t *rowOffset, const uint32_t *nnzOffset,
                              const uint32_t *tcA2B, const uint64_t *tcBit, const void *data, const uint32_t *rowIdx,
                              const GroupCuts *cuts)
{
    if (!out) return fail(HSPMM_ERR_INVALID, "null plan pointer");
    *out = nullptr;
    if (dtype != HSPMM_FP16 && dtype != HSPMM_TF32 && dtype != HSPMM_BF16)
        return fail(HSPMM_ERR_INVALID, "unknown dtype %d", dtype);
    if (total_tiles && (!nnzOffset || !tcBit)) return fail(HSPMM_ERR_INVALID, "null nnzOffset or tcBit");
    // Sparse windows (graphs) never need their tiles on the host: the bitmap arrays go to the device as they are -
    // the gather kernels read them (spmm_mfma_kernel.hpp, Fp16TileDWB and Fp32TileB) - and kernels expand them
    // for the kernels that read plain tiles.  Dense windows (the LDS-panel stream re-tiles them on the host) and
    // paired windows are expanded here first.
    if (eff_row_windows && total_tiles && rowOffset && nnzOffset[0] == 0 && (!nnzOffset[total_tiles] || data)) {
        int mode;
        { std::lock_guard<std::mutex> lk(g_cfg_mutex); mode = g_cfg.kernel_mode; }
        const double density = double(total_tiles) / (double(eff_row_windows) * double((uint64_t(cols) + 127u) / 128u));
        if (mode < 4 && density < 1.2) {
            const BitmapSource src{nnzOffset, tcBit, data};
            const int rc = create_plan(out, dtype, rows, cols, eff_row_windows, total_tiles, rowOffset, tcA2B, nullptr, rowIdx, &src,
                                       cuts);
            if (rc != kNeedsPlainTiles) return rc;
        }
    }
    const size_t tile_bytes = size_t(HSPMM_ROW_WINDOW) * (dtype == HSPMM_TF32 ? 8u * 4u : 16u * 2u);
    std::vector<uint8_t> dense;
    try { dense.resize(size_t(total_tiles) * tile_bytes); }
    catch (const std::bad_alloc &) { return fail(HSPMM_ERR_ALLOC, "out of host memory"); }
    // hspmm_bitmap_expand leaves its own message behind on failure
    const int rc = hspmm_bitmap_expand(dtype, total_tiles, nnzOffset, tcBit, data, dense.data());
    if (rc) return rc;
    return create_plan(out, dtype, rows, cols, eff_row_windows, total_tiles, rowOffset, tcA2B, dense.data(), rowIdx, nullptr, cuts);
}

int hspmm_create_bitmap(hspmm_plan **out, int dtype, uint32_t rows, uint32_t cols, uint32_t eff_row_windows,
                        uint32_t total_tiles, const uint32_t *rowOffset, const uint32_t *nnzOffset,
                        const uint32_t *tcA2B, const uint64_t *tcBit, const void *data, const uint32_t *rowIdx)
{
    return create_from_bitmap(out, dtype, rows, cols, eff_row_windows, total_tiles, rowOffset, nnzOffset, tcA2B, tcBit, data,
                              rowIdx, nullptr);
}

int hspmm_create_grouped(hspmm_plan **out, int dtype, uint32_t rows, uint32_t cols, uint32_t total_groups,
                         const uint32_t *groupOffset, const uint32_t *nnzOffset, const uint32_t *tcA2B,
                         const uint64_t *tcBit, const void *data, const uint32_t *groupRowIdx,
                         const uint8_t *atomic)
{
    if (!out) return fail(HSPMM_ERR_INVALID, "null plan pointer");
    *out = nullptr;
    if (total_groups && (!groupOffset || !groupRowIdx || !atomic))
        return fail(HSPMM_ERR_INVALID, "null groupOffset, rowIdx or atomic");
    // consecutive groups with one row index are one window again
    std::vector<uint32_t> rowOffset(1, total_groups ? groupOffset[0] : 0u), rowIdx;
    for (uint32_t g = 0; g < total_groups; ++g) {
        if (groupOffset[g + 1] <= groupOffset[g])
            return fail(HSPMM_ERR_INVALID, "groupOffset does not increase at group %u", g);
        const bool first = g == 0 || groupRowIdx[g] != groupRowIdx[g - 1];
        const bool last = g + 1 == total_groups || groupRowIdx[g + 1] != groupRowIdx[g];
        const bool shared = !(first && last);
        if ((atomic[g] != 0) != shared)
            return fail(HSPMM_ERR_INVALID, "atomic[%u] = %u but the group %s its rows with a neighbour", g,
                        unsigned(atomic[g]), shared ? "shares" : "does not share");
        if (first) rowIdx.push_back(groupRowIdx[g]);
        if (last) rowOffset.push_back(groupOffset[g + 1]);
    }
    // groups of one window that are not adjacent show up as a row index that does
    // not increase, which the checks of hspmm_create reject
    const uint32_t W = uint32_t(rowIdx.size());
    const GroupCuts cuts{groupOffset, total_groups};
    return create_from_bitmap(out, dtype, rows, cols, W, rowOffset.back(), rowOffset.data(), nnzOffset, tcA2B, tcBit, data,
                              rowIdx.data(), total_groups && groupOffset[0] == 0 ? &cuts : nullptr);
}

}  // extern "C"
