// Host side of the entry kernels (spmm_entries.hip): which launches they take, the stream they walk, the launch.
#include "hspmm_plan.hpp"
#include <cmath>

using namespace hspmm_host;

namespace {

// How a row of B of `bytes` bytes is shared out over the lanes of a subgroup: the widest load the row can fill.
struct RowShare { uint32_t lane_bytes, lanes; };
RowShare share_row(uint32_t bytes)
{
    if (bytes < 4u) return {2u, 1u};
    if (bytes < 8u) return {4u, bytes > 4u ? 2u : 1u};
    if (bytes < 16u) return {8u, bytes > 8u ? 2u : 1u};
    uint32_t lanes = 1;
    while (lanes * 16u < bytes) lanes <<= 1;
    return {16u, lanes};
}

// Most units of a row of bin b (see entry_bin in spmm_entries.hip).
uint32_t bin_units(uint32_t b)
{
    if (b == 0u || b == hspmm::kEntryBins - 1u) return 0u;
    const uint32_t c = hspmm::kEntryClassesByLength - 1u - (b - 1u) / 4u, step = 3u - (b - 1u) % 4u;
    return c == 0u ? step + 1u : (2u << c) + (step + 1u) * (1u << (c - 1u));
}

hspmm::EntrySource entry_source(const hspmm_plan *p)
{
    const hspmm_plan::Entries &e = p->entries;
    return {p->d_rowOffset, p->d_rowIdx, p->d_a2b_raw, e.d_first_chunk, e.d_chunk_window, p->d_data, p->W};
}

// Makes the entry stream from the uploaded tiles: one allocation, two kernels.  Called with the plan's mutex held; waits for
// the stream, because launches on other streams, and under capture, may follow at once.
int build_entries(hspmm_plan *p, hipStream_t s)
{
    using namespace hspmm;
    hspmm_plan::Entries &e = p->entries;
    EntryPlaces at;
    uint64_t slot = 0, unit = 0;
    for (uint32_t b = 0; b < kEntryBins; ++b) {
        const uint32_t width = bin_units(b);
        at.places[3u * b] = uint32_t(slot); at.places[3u * b + 1u] = uint32_t(unit); at.places[3u * b + 2u] = width;
        slot += e.totals[b];
        unit += b == 0u ? uint64_t(e.totals[kEntryBins]) : uint64_t(e.totals[b]) * width;
    }
    // ids, values, descriptors, pieces
    const size_t units_kept = size_t(unit ? unit : 1u), ids_bytes = units_kept * 16u, vals_bytes = units_kept * 4u * p->elem;
    const size_t desc_bytes = size_t(slot) * 12u, bytes = ids_bytes + vals_bytes + desc_bytes + size_t(e.totals[0]) * 12u;
    void *stream = nullptr;
    if (slot > 0xFFFFFFFFull || unit > 0xFFFFFFFFull || hipMalloc(&stream, bytes) != hipSuccess) {
        (void)hipGetLastError();
        e.unavailable.store(true);              // (for good: a plan's results do not change from call to call)
        return HSPMM_OK;
    }
    e.d_stream = stream;
    p->fixed_bytes += bytes;
    char *base = static_cast<char *>(stream);
    uint32_t *ids = reinterpret_cast<uint32_t *>(base), *desc = reinterpret_cast<uint32_t *>(base + ids_bytes + vals_bytes);
    uint32_t *pieces = reinterpret_cast<uint32_t *>(base + ids_bytes + vals_bytes + desc_bytes);
    // (a failure that uses the cursors up: not tried again either)
    auto failed = [&](int code) { e.unavailable.store(true); return code; };
    HSPMM_HIP_OR(launch_entry_fill(int(p->elem), entry_source(p), e.most_chunks, e.d_positions, e.d_row_len, p->rows, at,
                                   e.d_totals + kEntryBins + 1u, desc, pieces, e.d_row_first, ids, base + ids_bytes, s), failed);
    HSPMM_HIP_OR(hipStreamSynchronize(s), failed);
    e.units = unit;
    e.long_rows = unit >= 64u * uint64_t(slot - e.totals[kEntryBins - 1u]);
    e.d_ids = ids; e.d_vals = base + ids_bytes; e.d_desc = desc; e.d_pieces = pieces;
    e.built = true;
    return HSPMM_OK;
}

// The classes of a launch; returns the number of workgroups.  A subgroup gets at most 4 << shift units where a workgroup has
// subgroups enough; chain: rows that would still leave a subgroup more units than that are cut into parts (0: never).
uint32_t fill_classes(const hspmm_plan *p, uint32_t lanes, int shift, uint32_t chain, hspmm::EntryArgs *ea)
{
    using namespace hspmm;
    const uint32_t subgroups = 256u / lanes;                 // of a workgroup
    uint32_t most = 0;
    while ((2u << most) <= subgroups) ++most;
    const uint32_t *n = p->entries.totals;
    uint32_t group = 0, slot = 0, part = 0;
    ea->n_classes = 0;
    auto add = [&](uint32_t slots, int wanted, uint32_t units) {
        if (!slots) return;
        const uint32_t log2g = std::min(uint32_t(std::max(wanted, 0)), most);
        uint32_t log2parts = 0;
        while (chain && (units >> log2g >> log2parts) > chain) ++log2parts;
        ea->part_begin[ea->n_classes] = part;
        ea->cls[ea->n_classes++] = {group, slot, slot + slots, log2g | log2parts << 8};
        const uint32_t per_group = subgroups >> log2g;
        group += ((slots << log2parts) + per_group - 1u) / per_group;
        slot += slots;
        if (log2parts || (slot == slots && n[0])) part += slots << log2parts;       // (pieces are parts in any case)
    };
    const uint32_t top = kEntryClassesByLength - 1u;
    add(n[0], int(top) - shift, kEntryPieceUnits);
    for (uint32_t c = top;; --c) {
        const uint32_t *bins = n + 1u + (top - c) * 4u;
        add(bins[0] + bins[1] + bins[2] + bins[3], int(c) - shift, 4u << c);
        if (c == 0u) break;
    }
    add(n[kEntryBins - 1u], 0, 0u);
    ea->n_parts = part;
    return group;
}

// Units per subgroup: long chains need few waves and add few sums (all rows long: 4096 x 11008 at 10 %, N = 8: 17.4 -> 13.0 us
// from 4 to 16), but a matrix of few rows then has no workgroups for all compute units: up to 2.5 for each at 4 units it takes these, up to two (one
// and two lanes) or three at 8 units these (bf16, 4 / 8 / 16 units, us: 1274 x 7041 at 4 %, N = 1 3.9 / 5.0 / 7.2, N = 8 4.6 / 6.0 / 9.1, N = 64 6.4 / 7.1 / 8.4;
// 4096^2 at 10 %, N = 8 5.9 / 6.3 / 8.9, N = 16 8.7 / 6.9 / 8.2, N = 32 11.4 / 10.6 / 8.9; fp32, 1551 x 1412 at 19 %, N = 16 4.5 / 5.1 / 6.4).  Not
// rows of over 1024 entries, whose sums are many at 4 units (1100 x 16000 at 10 %, fp32, N = 4 9.0 / 8.3 / 7.3).  And where rows are short a launch takes as long as its longest chain (graph of 2^18, N = 16: 30 us at 8, 26
// at 4) unless it has waves for several rounds.
// A launch of few rounds also cuts rows that a workgroup's subgroups cannot bring down to 8 units each into parts (24894 vertices,
// fp16, N = 88: 20.9 us uncut, 15.2 / 14.5 / 16.7 at 16 / 8 / 4 units; 12288, fp32, N = 128: 20.2 -> 10.2; rows all long, 4096 x
// 11008 at 10 %, N = 8: 12.9 uncut, 19.9 at 8).  The line lies at four rounds of workgroups: graph of 40000, fp16, N = 200 (2.4
// rounds) 37.1 -> 25.4 us, of 73838, N = 128 (2.3) 27.9 -> 29.6, of 100000 (3.1) 24.0 -> 21.0, of 73838, N = 200 (4.6) 50.8 -> 59.9.
void choose_classes(const hspmm_plan *p, uint32_t lanes, bool may_cut, hspmm::EntryArgs *ea)
{
    const uint32_t round = uint32_t(p->compute_units) * 8u;
    int shift = 2;
    if (!p->entries.long_rows) {
        shift = fill_classes(p, lanes, 1, 0, ea) < 2u * round ? 0 : 1;
    } else if (p->entries.units <= 256u * uint64_t(p->rows - p->entries.totals[hspmm::kEntryBins - 1u])) {      // (of the rows that have entries)
        const uint32_t cu = uint32_t(p->compute_units);
        if (fill_classes(p, lanes, 0, 0, ea) * 2u <= 5u * cu) shift = 0;
        else if (fill_classes(p, lanes, 1, 0, ea) <= (lanes <= 2u ? 2u : 3u) * cu) shift = 1;
    }
    ea->n_groups = fill_classes(p, lanes, shift, 0, ea);
    if (may_cut && !p->entries.long_rows && ea->n_groups < 4u * round) ea->n_groups = fill_classes(p, lanes, shift, 8, ea);
}

}  // namespace

namespace hspmm_host {

constexpr uint32_t kEntryMaxBlockBytes = 512, kEntryMostFeatures = 1024;       // 32 lanes of 16 bytes; rows of 2 KB, fp32 storage of 4 KB

// Feature blocks of 128 bytes resp. half a row on XCDs of their own (see spmm_mfma_kernel.hpp), here for rows of 256 bytes
// (fp32 storage: also 512): pays where B is far larger than an L2 and no row of it is hot (uniform 65536^2, 16 per row:
// fp16 N = 128 34 -> 29 us, fp32 N = 64 34 -> 30 us); with the hot rows of a power-law graph it only adds passes over
// the entries (2^20 vertices, N = 128: 474 -> 510 us).
static bool entries_by_xcd(const hspmm_plan *p, uint64_t row_bytes)
{
    return p->even_windows && (row_bytes == 256u || (row_bytes == 512u && p->elem == 4u)) &&
           uint64_t(p->cols) * row_bytes >= (uint64_t(8) << 20);
}

// Bytes of a block: whole 16-byte pieces, or, where rows are loaded from the word before on (EntryArgs::odd), pieces and 14 bytes (the
// last block is moved back to end with the row).
static uint32_t entry_block_bytes(uint32_t row_bytes, uint32_t blocks, bool odd)
{
    if (blocks == 1u) return row_bytes;
    const uint32_t bytes = (row_bytes + blocks - 1u) / blocks;
    return odd ? ((bytes + 1u) & ~15u) + 14u : (bytes + 15u) & ~15u;
}

// Lines of 128 bytes that `bytes` bytes from byte `off` of a row touch: the mean over rows that begin on multiples of `step`.
static double lines_touched(uint32_t off, uint32_t bytes, uint32_t step)
{
    if (step <= 16u) return 1.0 + double((bytes - 1u) / step * step) / 128.0;         // (off, too, is a multiple of step)
    uint32_t lines = 0;
    for (uint32_t at = off; at < off + 128u; at += step) lines += (at + bytes - 1u) / 128u - at / 128u + 1u;
    return double(lines) * step / 128.0;
}

// Blocks a row of B is cut into, passes over the entries one after the other: the cheapest by what an entry takes - the lines of B
// it touches, its lanes (16 bytes each, used or not) as lines, and half a line for every pass - with a tenth more for every time
// a block's part of B doubles beyond half an L2.  A row of 640 bytes that begins on a line is five blocks of eight lanes (5 lines
// + 5 of lanes + 2.5) and not two of 32 (6 + 8 + 1): fp32, graph of 57344, N = 160, 48 against 72 us.  One of 300 bytes that
// begins anywhere is one block of 32 lanes (3.3 + 4 + 0.5) and not three of eight (5.6 + 3 + 1.5): graph of 905216, N = 75, 576
// against 861 us.  The two weights are a fit to 745 graphs and uniform matrices, all types and N, with any number of blocks: the
// choice is 1.6 % behind the fastest on average and 12 % at the 95th percentile, and weights half or twice as large 0.3 % more.
static uint32_t row_blocks(const hspmm_plan *p, uint32_t row_bytes, bool odd)
{
    const uint32_t step = row_bytes % 128u ? row_bytes & (0u - row_bytes) : 128u;
    uint32_t best = 0;
    double least = 0.0;
    for (uint32_t b = (row_bytes + kEntryMaxBlockBytes - 1u) / kEntryMaxBlockBytes; b == 1u || row_bytes / b >= 112u; ++b) {
        const uint32_t bytes = entry_block_bytes(row_bytes, b, odd);
        if (bytes > kEntryMaxBlockBytes || (best && bytes < 128u)) continue;
        double cost = double(b * share_row(bytes).lanes) / 8.0 + 0.5 * double(b);
        if (step <= 16u) cost += double(b) * lines_touched(0u, bytes, step);
        else for (uint32_t i = 0; i < b; ++i) cost += lines_touched(std::min(i * bytes, row_bytes - bytes), bytes, step);
        const double part = double(p->cols) * bytes / double(2u << 20);
        if (part > 1.0) cost *= 1.0 + 0.1 * std::log2(part);
        if (!best || cost < least) { least = cost; best = b; }
    }
    return best;
}

// The blocks of a row, and whether rows are loaded from the word before on: 16-bit types, an odd number of them, B on a word and two of
// its rows at least.  Not where the blocks fill all of their lanes (N = 383, 511, 767, 1023): there is no place for a last lane of seven
// features then, and more blocks, or lanes twice as many, cost what the whole words gain (uniform 26880 x 120320, 25 per row, N = 511
// 116 / 148 us, graph of 65536, N = 383 58 / 73, 6779 launches at odd N: 195 of the 258 that lost by more than 3 %, up to 27 %).
struct RowShape { uint32_t blocks, block_bytes; bool odd; };
static RowShape choose_row_shape(const hspmm_plan *p, uint32_t row_bytes, bool on_word)
{
    if (entries_by_xcd(p, row_bytes)) return {2u, entry_block_bytes(row_bytes, 2u, false), false};
    const uint32_t blocks = row_blocks(p, row_bytes, false), bytes = entry_block_bytes(row_bytes, blocks, false);
    if (p->elem != 2u || row_bytes % 4u != 2u || row_bytes < 18u || p->cols < 2u || !on_word || entry_block_bytes(row_bytes, blocks, true) > 16u * share_row(bytes).lanes)
        return {blocks, bytes, false};
    const uint32_t odd_blocks = row_blocks(p, row_bytes, true);
    return {odd_blocks, entry_block_bytes(row_bytes, odd_blocks, true), true};
}

// What an entry costs here is the lines of its row of B, what a tile column costs in the MFMA kernels does not depend
// on how many of its eight elements are stored nor, up to a block of 32 features (16 of fp32 storage), on N.  So the line goes by
// the bytes of a row of B and by the stored entries per tile column (per_column: 1.0 for graphs, 1.4 for weights
// pruned to 10 %, 1.9 to 20 %, 8 for blocks).  Measured (entry / other kernels, us):
//   16 bits, graph 2^18 N = 1 / 16 / 64: 14.5 / 45, 26 / 41, 44 / 58;  11610 vertices N = 128: 7.6 / 14;  40000 N = 128: 16 / 24;
//   73838 N = 128: 31 / 45;  16052 N = 627: 21 / 43;  117373 N = 528: 175 / 218;  uniform 16896 x 20992, 29 per row, N = 657: 90 / 132;
//   2^20 N = 128: 510 / 474;  uniform 8192^2 at 2 %, N = 256: 35 / 51
//   16 bits, 4096^2 pruned to 10 % N = 8 / 16: 5.8 / 10.3, 7 / 10.4; 4096 x 11008 N = 32: 24.6 / 22.5; to 30 % N = 8 / 16:
//   10 / 15.3, 16 / 15.3;  5376 x 3328 pruned to 3 %, N = 126 / 208 / 387: 12 / 18, 18 / 21, 54 / 26 (LDS-panel kernels)
//   fp32, graph of 150001 N = 16 / 64 / 128: 18 / 39, 43 / 68, 88 / 126;  12288 N = 128 / 256 / 500: 10 / 20, 16 / 26, 28 / 38;
//   4096^2 pruned to 10 % N = 8 / 32 / 64: 6 / 19.5, 12 / 19.5, 21 / 19.4; to 30 % N = 12 / 16: 24 / 29.7, 24 / 21;  graph of 691333
//   (B of 354 MB) N = 128: 326 / 300
bool entries_serve(const hspmm_plan *p, uint32_t N)
{
    const Config &c = p->cfg;
    if (!p->entries.counted || p->entries.unavailable.load()) return false;
    const uint64_t row = uint64_t(N) * p->elem, all = uint64_t(p->cols) * row, product = uint64_t(p->rows) * row;
    if (N > kEntryMostFeatures) return false;       // (16-bit rows of more than 2 KB have not been measured here)
    if (c.entries > 0) return true;
    const double per_column = p->per_column, weight = double(row) * (per_column - 0.8);
    // Power-law graphs that are dense in their hot columns count as sparse up to 1.4 (8192 to 16000 vertices, 18 to 32 edges each, 1.26 to 1.35;
    // entry / gather kernels, us: 16 bits N = 45 8.0 / 24.3, 64 7.0 / 11.2, 133 12.3 / 27.5, 200 11.0 / 14.0, 512 17.8 / 19.4; fp32 N = 64 8.6 / 15.6,
    // 94 12.9 / 32.2, 512 29.8 / 44.5; even rows of that density are weights, for which the other kernels have their own streams).
    const bool sparse = per_column <= 1.25 || (!p->even_windows && per_column <= 1.4);
    if (p->elem == 4u) {
        // 33 to 63 features: the LDS-panel kernels multiply bf16 parts, which no launch that has fp32 products here may lose them to; what
        // would be theirs or the full-tile kernels' goes by expected time, fits to 301 and 878 launches (standard deviations 10 and 7 %):
        // 4096 x 11008 at 10 %, N = 40: 54 us here, 39 there, 67 full tiles.
        if (N > 32u && N < 64u && p->panel.split && panel_serves(p, N) && (weight > 100.0 || tile_leaves(p, N)))
            return 3.6 + 12.7e-6 * double(p->T) * p->cw * per_column < 5.7 + 1.2 * panel_expected(p, N);
        if (weight <= 100.0) return true;
        // Rows that are no whole 16-byte pieces, below the 64 features from which the LDS-panel kernels take any: the other fp32
        // products come in blocks of 16 features where N is odd and of 32 where it is even (pruned 4096 x 11008 at 10 %, N = 47:
        // 57.7 / 122; 11008 x 4096 at 20 %, N = 26 / 47: 70 / 94, 107 / 191; 1500 x 9000 at 25 %, N = 30 / 51 / 63: 56 / 41, 81 / 85,
        // 88 / 85)
        if (N < 64u && N % 4u != 0u) return weight <= (N % 2u ? 350.0 : 135.0);
        // Rows of B of more than 512 features: 12544 x 20250, 24 per row, N = 640 / 933 66 / 108, 149 / 198; 60000 x 8000, 9 per row, 91 / 173,
        // 180 / 334; graph of 16000, 32 edges each, 65 / 104, 107 / 175.  Where columns are hot and B is larger than 156 MB the other kernels read
        // less of it (graph of 81984, 5 edges each, N = 640 / 768 / 1024: 148 / 135, 193 / 162, 274 / 200; of 40000, N = 1024, 156 MB: 140 / 163);
        // uniform ones were ahead at all sizes up to 460 MB (27793 x 118016, N = 768 103 / 112, 1024 140 / 142; 2048 x 100000, N = 1024 108 / 140).
        // (Not where rows of a few entries make a large C, which the other kernels write faster: 341404 x 2685, 1.8 per row, N = 1024 362 / 573; 407281 x
        // 5276, 1 per row, 316 / 449; 465282 x 221802, 1 per row, N = 320 197 / 259; graph of 1.3 entries per tile column, 4 per row, N = 400 0.70.  Up to
        // 64 MB of C all of 682 launches with fewer than 6 entries a row but three were ahead, from 6 entries on all of 899 but four, by up to 8 %.)
        const bool extended = row > 2048u || all > (uint64_t(256) << 20) || per_column > 1.25;
        if (extended && product > (uint64_t(64) << 20) && double(p->T) * p->cw * per_column < 6.0 * p->rows) return false;
        const uint64_t most = p->even_windows ? uint64_t(512) << 20 : row <= 2048u ? uint64_t(256) << 20 : uint64_t(160) << 20;
        return sparse && !p->panel.built && (row <= 256u || all <= most);
    }
    if (weight <= 42.0 || (sparse && row <= 128u)) return true;
    if (!sparse || panel_serves(p, N)) return false;
    // Those dense graphs by wide loads or words above 640 features: graph of 12288, 24 edges each, N = 704 / 800 / 832 / 1024 29.6 / 27.7, 39.8 / 34.7,
    // 34.0 / 31.8, 37.2 / 31.9; of 16000, 40 edges, 1024 64.3 / 58.0; 512, 576 and 640 0.96 to 1.18 times as fast here on eight graphs of 8192 to 16000
    // (768 and 896 0.96 to 1.11: left), other N there 0.98 to 1.9 (700 33.5 / 44.1, 1023 54.1 / 58.1).
    // Above 96 features the wide loads keep N a multiple of 8 but not of 64 (0.7 to 1.5 on 126 launches, a third of them behind), and with them a C of
    // more than 16 MB, with others one of more than 32 MB, is the gather kernels' (333 launches left to them: 1.08 on the mean here, 113 behind, by up to 33 %;
    // 752 taken: 1.73 times as fast, 14 behind by more than 3 %, 18 % at most).
    if (per_column > 1.25) {
        if (N % 8u == 0u && (N > 640u || (N > 96u && N % 64u != 0u))) return false;
        if (product > (uint64_t(N % 8u == 0u ? 16u : 32u) << 20)) return false;
    }
    // N a multiple of 64, hot rows and a B that fills half of the 256 MB memory-side cache: there the other kernels, which then load
    // words and read fewer rows of B, are ahead (graph of 920569, N = 128, 236 MB: 363 / 343 us; of 434176, N = 512, 445 MB:
    // 353 / 322; 18 such graphs: 1.02 on average, and 1.13 behind on 16 with other N a multiple of 8).
    return p->even_windows || N % 64u != 0u || all <= (uint64_t(128) << 20);
}

// What an entry takes by the features of a row: a fit to 2974 launches at 2.5 to 30 % (standard deviation 8 to 25 %).  Rows of up to
// eight features that begin between two words take up to twice as long, longer ones a tenth more.
double entries_expected(const hspmm_plan *p, uint32_t N)
{
    const double odd = N % 2u == 0u ? 1.0 : N == 1u ? 0.9 : N <= 8u ? 1.6 : 1.1;
    const double each = N <= 8u ? 1.9 : N <= 16u ? 3.3 : N <= 64u ? 5.3 : N <= 128u ? 11.5 : 25.0;
    return 3.9 + each * odd * 1e-6 * double(p->T) * p->cw * p->per_column;
}

struct CountArrays { size_t most_chunks, words[6]; };
static CountArrays count_arrays(const hspmm_plan *p)
{
    const size_t most = size_t(p->W) + p->T / hspmm::kEntryChunkTiles;
    return {most, {size_t(p->W) + 1u, most, most * 8u, p->rows, p->rows, 2u * (hspmm::kEntryBins + 1u)}};
}

// Whether a plan whose tiles are not counted yet may want the stream.
static bool entries_possible(const hspmm_plan *p)
{
    const Config &c = p->cfg;
    // (the caller's own settings are settings of the gather kernels)
    if (c.kernel_mode != 0 || c.entries == 0 || c.fused_fixup >= 0 || c.buffer_stage || c.consumer_warp_num || c.producer_warp_group_num)
        return false;
    if (!p->caller_cuts.empty() || p->rows >= (1u << 31) || !p->T || count_arrays(p).most_chunks >= hspmm::kEntryMostChunks) return false;
    return c.entries > 0 || (p->G == 1 && p->per_column <= 3.5);
}

size_t entries_count_bytes(const hspmm_plan *p)
{
    size_t bytes = 0;
    if (p->cfg.entries > 0 || p->G == 1)
        for (size_t words : count_arrays(p).words) bytes += words * 4u + 256u;
    return bytes;
}

// Row lengths and the sizes of all there is in the stream: enqueued by hspmm_create behind the tiles, beside its work on the
// host, so that the first product of a plan has nothing to read back (see build_entries).  First product of a plan, counting in
// its launch / here, us: 4096^2 at 1 %, N = 64 96 / 50; uniform 65536^2, 16 per row, N = 128 208 / 114; graph of 150001, fp32,
// N = 100 388 / 213; of 262144, N = 16 477 / 242, N = 128 510 / 272; hspmm_create takes 0.05 ms more.
int count_entries(hspmm_plan *p)
{
    using namespace hspmm;
    hspmm_plan::Entries &e = p->entries;
    if (!entries_possible(p)) return HSPMM_OK;
    const CountArrays arrays = count_arrays(p);
    uint32_t **const at[] = {&e.d_first_chunk, &e.d_chunk_window, &e.d_positions, &e.d_row_len, &e.d_row_first, &e.d_totals};
    for (int i = 0; i < 6; ++i) {
        void *room = nullptr;
        if (int rc = plan_alloc(p, arrays.words[i] * 4u, &room)) return rc;
        *at[i] = static_cast<uint32_t *>(room);
    }
    e.most_chunks = uint32_t(arrays.most_chunks);
    HSPMM_HIP(launch_entry_count(int(p->elem), entry_source(p), e.most_chunks, p->rows, e.d_first_chunk, e.d_chunk_window, e.d_positions,
                                 e.d_row_len, e.d_totals, nullptr));
    e.counted = true;
    return HSPMM_OK;
}

// Waits for what hspmm_create has enqueued.
int entries_counted(hspmm_plan *p)
{
    if (p->entries.counted) HSPMM_HIP(hipMemcpy(p->entries.totals, p->entries.d_totals, sizeof p->entries.totals, hipMemcpyDeviceToHost));
    else HSPMM_HIP(hipStreamSynchronize(nullptr));
    return HSPMM_OK;
}

int run_entries(hspmm_plan *p, const void *dB, void *dC, uint32_t N, hipStream_t s, RunMode mode, bool *taken)
{
    const uint32_t row_bytes = N * p->elem;
    const RowShape row = choose_row_shape(p, row_bytes, reinterpret_cast<uintptr_t>(dB) % 4u == 0u);
    const uint32_t blocks = row.blocks, block_bytes = row.block_bytes;
    const RowShare share = share_row(block_bytes);
    hspmm::EntryArgs ea{};
    hspmm_plan::Entries &e = p->entries;
    *taken = false;
    {
        std::lock_guard<std::mutex> lk(p->mu);
        if (!e.built) {
            if (mode == RunMode::kStatic)
                return fail(HSPMM_ERR_UNSUPPORTED, "hspmm_run_static: the entry stream of narrow feature dimensions is not built yet; "
                            "call hspmm_prepare(plan, N) or hspmm_run once with this N first");
            hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
            if (mode == RunMode::kLaunch && s && (hipStreamIsCapturing(s, &status) != hipSuccess || status != hipStreamCaptureStatusNone))
                return HSPMM_OK;                // (nothing can be built under capture: the gather kernels take it)
            if (const int rc = build_entries(p, s)) return rc;
            if (!e.built) return HSPMM_OK;
        }
        hspmm::EntryArgs &classes = e.classes[__builtin_ctz(share.lanes)];
        if (!classes.n_classes) choose_classes(p, share.lanes, true, &classes);
        ea = classes;
        // Sums of the parts and behind them their counters: what hspmm_run_static has a fixed array for.  The shape is the same
        // however it is launched: where they do not fit, no rows are cut, and where the pieces of long rows alone do not, this is
        // a launch for the other kernels.
        const size_t sums_of_part = size_t(blocks) * share.lanes * share.lane_bytes / p->elem * 4u, counters_of_part = size_t(blocks) * 4u;
        auto fits = [&]() { return size_t(ea.n_parts) * (sums_of_part + counters_of_part) <= HSPMM_STATIC_SCRATCH_BYTES; };
        if (!fits()) choose_classes(p, share.lanes, false, &ea);
        if (!fits() || uint64_t(ea.n_groups) * blocks >= hspmm::kEntryMostGroups) return HSPMM_OK;
        ea.n_pieces = e.totals[0];
        if (ea.n_parts) {
            const size_t sums = ea.n_parts * sums_of_part, counters = ea.n_parts * counters_of_part;
            if (const int rc = scratch_for(p, s, mode == RunMode::kStatic ? sums + counters : sums, mode, &ea.scratch)) return rc;
            if (mode == RunMode::kStatic) {
                ea.arrive = reinterpret_cast<uint32_t *>(reinterpret_cast<char *>(ea.scratch) + sums);
                HSPMM_HIP(hspmm::launch_fill_zero(ea.arrive, counters, s));
            } else if (const int rc = ensure_arrive(p, s, counters / 4u, mode, &ea.arrive)) {
                return rc;
            }
        }
    }
    *taken = true;
    if (mode == RunMode::kPrepare) return HSPMM_OK;
    ea.desc = e.d_desc; ea.ids = e.d_ids; ea.vals = e.d_vals; ea.pieces = e.d_pieces;
    ea.B = dB; ea.C = dC; ea.ld = N; ea.block_bytes = block_bytes; ea.n_feat_blocks = blocks; ea.xcd_split = entries_by_xcd(p, row_bytes);
    ea.last_row = p->cols - 1u;
    ea.odd = row.odd;
    p->note_launch("spmm_entries_kernel", 2, 0, 0);
    HSPMM_HIP(hspmm::launch_spmm_entries(p->dtype, ea, share.lane_bytes, share.lanes, s));
    return HSPMM_OK;
}

}  // namespace hspmm_host
