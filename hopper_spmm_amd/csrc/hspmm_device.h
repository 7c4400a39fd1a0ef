// Shared between the kernels and the C ABI layer: kernel argument block and
// launch entry points.  Internal; the public interface is include/hspmm.h.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stddef.h>

namespace hspmm {

constexpr uint32_t kIdxMax = 0xFFFFFFFFu;      // reference src/common.h:47
constexpr uint32_t kRowWindow = 8u;            // reference src/common.h:17
constexpr uint32_t kRangeWordsDev = 8u;
constexpr uint32_t kRangeWords = kRangeWordsDev;
constexpr uint32_t kFixWords = 4u;
constexpr int kMaxWavesPerGroup = 4;
constexpr int kAlignedGroupWaves = 8;          // waves of a workgroup that walks one whole unit (aligned partition)

struct KernelArgs {
    // the four format arrays exactly as given (device copies), reference
    // src/fp16.cu:38-41: read by the scalar kernel
    const uint32_t *rowOffset;
    const uint32_t *tcA2B;
    const void     *data;
    const uint32_t *rowIdx;
    // the step stream the MFMA kernels walk
    const uint32_t *unitOffset;  // n_units + 1: first step of every unit
    const uint32_t *unitRow;     // n_units: first matrix row of the unit | its windows less one (1: a pair)
                                 // of a schedule four words: first row (| 1: the first window, rows in front of it are to be cleared), end of the
                                 // rows to be cleared behind it (0: none), its slot (kIdxMax: a whole window), its entry in split
    const uint32_t *ids;         // per step, lane order, padding ids renamed
    const void     *tiles;       // per step, lane order; bitmap stream: the stored elements, tile after tile
    const uint32_t *bm_header;   // bitmap stream (kLayoutDWB): per step 8 words - the tile's four bitmap words, the bit
                                 // counts of words 0, 0..1, 0..2 (bytes 1..3), the position of its first stored element
    // partition
    const uint32_t *ranges;      // n_ranges x kRangeWords
    const uint32_t *split;       // n_split x kFixWords {unit, slot_begin, slot_count, 0}
    const uint32_t *fix_slots;   // (of a schedule, behind the slots: the units of a window's parts, from the split entry's fourth word on)
    float          *scratch;     // partial sums: [slot][feature block][acc reg][lane] x 4 floats
    uint32_t       *arrive;      // [split unit][feature block] arrival counters (all zero between launches);
                                 // null: the partial sums are added by a second kernel
    const void     *B;           // cols x N
    void           *C;           // rows x N
    uint32_t n_ranges, n_split, eff_windows, n_units, rows, N, n_feat_blocks;
    uint32_t ld;                 // elements from one row of B (and of C) to the next: N, or more when the launch
                                 // covers a range of the features only (MFMA kernels; the scalar kernel takes whole rows)
    uint32_t xcd_split;          // != 0 (gather kernels; 2, 4 or 8 feature blocks): every feature block has XCDs of its own
    uint32_t uniform_chunks;     // != 0 (LDS-panel kernels): no split table - entry e is unit e, whose partial sums
                                 // are slots e * uniform_chunks .. + uniform_chunks - 1, in that order
};

// dtype: 0 = fp16 tiles 8x16, 1 = fp32 tiles 8x8, 2 = bf16 tiles 8x16.  V = 32-bit words a lane loads
// per B row (1, 2 or 4).
// layout (fp16 only): kLayoutX4 = wide loads, contiguous features per lane, N % (2V) == 0;
// kLayoutDW = word loads, features strided by 32 per lane, N % (32V) == 0.
constexpr int kLayoutX4 = 0, kLayoutDW = 1, kLayoutDWB = 2;   // DWB: word loads, tiles as bitmap + stored elements (16-bit, G = 1)
// element types, numbered as HSPMM_FP16 / HSPMM_TF32 / HSPMM_BF16 of the public header
constexpr int kDtypeF16 = 0, kDtypeF32 = 1, kDtypeBf16 = 2;
// The gather kernels' prefetch depth (steps of loads in flight per wave) when the caller sets none: what fits 128
// registers per lane without spilling.  Workgroups of eight waves and 64-bit gather offsets are built for this depth
// only; depths 2, 3 and 4 exist for the rest (1, 6 and 8 in builds with HSPMM_EXPERIMENTAL).
constexpr int default_prefetch(int elem_bytes, int G, int V)
{
    return elem_bytes == 4 ? (G == 2 && V == 4 ? 3 : 4) : (G == 2 && V == 4 ? 2 : 3);
}
// narrow: B < 4 GiB and cols < 2^24 (32-bit gather offsets).
// mid: optional event recorded between the main kernel and the partial-sum kernel.
// G: windows per unit in the step stream (1, or 2 when the plan paired windows).
hipError_t launch_spmm_mfma(int dtype, int layout, int G, const KernelArgs &ka, int V, int prefetch, bool narrow,
                            int waves_per_group, hipStream_t s, hipEvent_t mid);
hipError_t launch_spmm_scalar(int dtype, const KernelArgs &ka, hipStream_t s);

// 16-bit bitmap tiles in the order of a schedule, words at 64 features a block, 32-bit gather offsets; ids and headers of that order by
// launch_schedule_fill (items: first tile, stride, first step, steps).
hipError_t launch_spmm_scheduled(int dtype, const KernelArgs &ka, int waves_per_group, hipStream_t s, hipEvent_t mid);
hipError_t launch_schedule_fill(const uint32_t *items, uint32_t n_items, const uint32_t *ids, const uint32_t *header, uint32_t *to_ids, uint32_t *to_header,
                                hipStream_t s);

// LDS-panel kernels (spmm_panel_kernel.hpp).
constexpr uint32_t kPanelRowBytes = 256;       // bytes of a B row one workgroup covers (128 halves / 64 floats)
// B rows per panel: 256 for the kernels built on the transposing LDS read (16-bit types, fp32 in bf16
// parts), 128 for the fp32 MFMA forms
constexpr uint32_t kPanelRowsWide = 256, kPanelRowsFp32 = 128;

struct PanelArgs {
    const uint32_t *unitRow;     // n_units: first matrix row of the unit | its windows less one (0..3)
    const uint32_t *poff;        // n_units x (n_panels + 1): first step of the unit at or behind every panel
    const uint32_t *step_panel;  // per step: its panel
    const uint32_t *ids;         // per step: the rows (inside the panel) each quarter-wave reads and the panels
                                 // between the step and the one in front of it; the format depends on the element
                                 // type (PanelOps in spmm_panel_kernel.hpp)
    const void     *tiles;       // per step, lane order (null when the stream is packed)
    // packed streams (tiles without their zeros): per step eight lane masks; the stored values, (mask, lane)
    // order, values[0] = 0; per step the position of its first value
    const uint64_t *masks;
    const void     *vals;
    const uint32_t *step_voff;
    float          *scratch;     // partial sums [unit * n_chunks + chunk][feature block][acc reg][lane]
    uint32_t       *arrive;      // per (unit, feature block): chunks that have left their sums (zero between launches);
                                 // null: a second kernel adds the sums
    const void     *B;
    void           *C;
    uint32_t n_units, n_steps, rows, cols, N, n_feat_blocks, n_panels, n_chunks, panels_per_chunk;
    uint32_t units_per_group;    // consumer waves of a workgroup that get a unit (<= those the kernel has); the
                                 // others only keep the barriers company
};

// units: 12 or 14 units (consumer waves) per workgroup, 2 more waves copy B to LDS; 13 = 12 units and 4 such waves.
// G: windows per unit at most (1, 2, 4); 0 = fp32 single windows with ids in the format of the 4x4x1 tile.  split (fp32): the plan's
// stream is in the bf16 hi / lo form.  ka: arguments of the kernel that adds the chunk sums (split table with one
// entry per unit), used when pa.n_chunks > 1.
// tall: the stream gives every consumer wave two units (poff per pair of units, steps of the second unit marked);
// packed: its tiles are stored without their zeros (tall streams only).
hipError_t launch_spmm_panel(int dtype, int G, bool split, bool tall, bool packed, const PanelArgs &pa, const KernelArgs &ka,
                             int units, hipStream_t s, hipEvent_t mid);

// Entry kernels for narrow feature dimensions (spmm_entries.hip): stored entries in units of four (the last unit of a
// row filled up with zeros), rows sorted by length.  A class is the rows of 2^(c+1) + 1 .. 2^(c+2) units (c = 0: 1 .. 4);
// rows above kEntryPieceUnits are cut into pieces of that many.
constexpr uint32_t kEntryPieceUnits = 512u, kEntryClassesByLength = 8u, kEntryBins = 2u + 4u * kEntryClassesByLength;
constexpr uint32_t kEntryChunkTiles = 64u, kEntryClasses = 2u + kEntryClassesByLength;
// a launch has under 2^32 work-items: workgroups of 256 threads, and chunks of a wave each
constexpr uint32_t kEntryMostGroups = 1u << 23, kEntryMostChunks = 1u << 25;
struct EntryClass { uint32_t group_begin, slot_begin, slot_end, logs; };    // first workgroup; slots; log2 subgroups per row or part | log2 parts of a row << 8
struct EntryArgs {
    const uint32_t *desc;        // per slot three words: first unit, units, matrix row (pieces: number of the piece)
    const uint32_t *ids;         // per unit four column ids
    const void     *vals;        // per unit four values
    const uint32_t *pieces;      // per piece three words: matrix row, the row's first piece, its number of pieces
    float          *scratch;     // sums of pieces and parts [part][lane][features of a lane]
    uint32_t       *arrive;      // [first part of a row]: parts that have left their sums (zero between launches)
    const void     *B;
    void           *C;
    uint32_t ld;                 // elements from one row of B (and of C) to the next
    uint32_t block_bytes, n_feat_blocks, xcd_split;  // bytes of a row one subgroup covers; blocks side by side; != 0: on XCDs of their own
    uint32_t odd, last_row;      // != 0: rows begin between two words, B begins on one (see spmm_entries_kernel); B's last row
    uint32_t n_groups;           // workgroups of one block
    uint32_t n_pieces, n_classes;
    EntryClass cls[kEntryClasses];   // pieces first where there are any, then from the longest rows to the empty ones
    uint32_t part_begin[kEntryClasses], n_parts;     // number of a class's first part
};
// lane_bytes (2, 4, 8, 16) x lanes (1 .. 32): how a row of B is shared out; at least lane_bytes long
hipError_t launch_spmm_entries(int dtype, const EntryArgs &ea, uint32_t lane_bytes, uint32_t lanes, hipStream_t s);
// The stream from the format arrays, in two steps: count (chunks of up to kEntryChunkTiles tiles of a window, at most most_chunks;
// stored entries per chunk and row, which become positions inside the row; row lengths; totals: rows per bin - bin 0:
// pieces - and behind them the units of the rows cut into pieces, then as many cursors) and fill (which uses the cursors up).
struct EntrySource { const uint32_t *rowOffset, *rowIdx, *a2b, *first_chunk, *chunk_window; const void *tiles; uint32_t n_windows; };
struct EntryPlaces { uint32_t places[3u * kEntryBins]; };      // per bin: first slot, first unit, units of a slot's place
hipError_t launch_entry_count(int elem, const EntrySource &src, uint32_t most_chunks, uint32_t rows, uint32_t *first_chunk, uint32_t *chunk_window,
                              uint32_t *counts, uint32_t *row_len, uint32_t *totals, hipStream_t s);
hipError_t launch_entry_fill(int elem, const EntrySource &src, uint32_t most_chunks, const uint32_t *positions, const uint32_t *row_len,
                             uint32_t rows, const EntryPlaces &places, uint32_t *cursors, uint32_t *desc, uint32_t *pieces,
                             uint32_t *row_first, uint32_t *ids, void *vals, hipStream_t s);
// Full-tile kernels (spmm_tile_kernel.hip): stored entries in blocks of 128 rows x tile_block_columns() columns, in units of
// four: positions inside the block's LDS image (16 bits) and values (fp32 storage: hi | lo parts).
constexpr uint32_t kTileBlockRows = 128u, kTileMaxBlocks = 4096u;     // blocks of a row block at most
constexpr uint32_t kTileSpareUnits = 512u;                            // behind the last unit (read and not used)
uint32_t tile_block_columns(int dtype);
struct TileSource { const uint32_t *rowOffset, *rowIdx, *a2b; const void *tiles; uint32_t n_windows, cols; };   // the format arrays
struct TileArgs {
    const uint32_t *blocks;      // per row block and block: its first unit (n_row_blocks x n_blocks + 1)
    const void     *pos, *vals;
    const void     *B;
    void           *C;
    float          *scratch;     // sums of the parts of cut C tiles (tile_parts of them)
    uint32_t       *arrive;      // per workgroup: parts of the cut C tile it has the first part of that have left their sums
                                 // (zero between launches; of no two cut tiles a workgroup has the first part)
    uint32_t rows, cols, N;
    uint32_t n_row_blocks, n_chunks, n_feat_tiles;               // chunks: blocks of columns
    uint32_t share, rest;        // items (chunks of C tiles) of a workgroup; the first `rest` have one more
    const TileSource *src;       // in device memory (read where B is not finite)
};
// Places for the parts of cut C tiles: a workgroup has two at most, of its first and of its last tile (part 2 g + 0 or 1); with
// no more tiles than workgroups a tile's parts overlap the next one's in one place less (part g + t).
inline uint64_t tile_parts(uint32_t groups, uint32_t n_tiles) { return uint64_t(groups) + (groups < n_tiles ? groups : n_tiles); }
// nt: features of a C tile (16, 32, 64)
hipError_t launch_spmm_tile(int dtype, const TileArgs &ta, uint32_t nt, uint32_t groups, hipStream_t s);
hipError_t launch_tile_count(int dtype, const TileSource &src, uint32_t n_row_blocks, uint32_t n_blocks, uint32_t *counts, uint32_t *blocks, hipStream_t s);
hipError_t launch_tile_fill(int dtype, const TileSource &src, uint32_t n_row_blocks, uint32_t n_blocks, const uint32_t *counts,
                            const uint32_t *blocks, void *pos, void *vals, hipStream_t s);
// Wide-tile kernels (spmm_wide_kernel.hip, 16-bit types): A as first operands of matrix instructions, 16 rows x 64 columns each.
constexpr uint32_t kWideUnitBytes = 2048u;
// A workgroup: `splits` sets of `rows` waves with `units` x 16 rows each, `blocks` x 16 features.
struct WideShape { uint32_t units, blocks, rows, splits; };
struct WideArgs {
    const void     *frags;       // per chunk of 64 columns and unit of 16 rows kWideUnitBytes
    const void     *B;
    void           *C;
    uint32_t rows, cols, N;
    uint32_t n_units, n_chunks, n_feat_tiles;                    // chunks: a multiple of four
    uint32_t n_cuts;             // workgroups of a C tile, each with a part of the chunks
    float *sums;                 // of more than one: their sums, a C tile of fp32 each
    const TileSource *src;       // in device memory (read where B is not finite)
};
// mid: as of launch_spmm_mfma, in front of the kernel that adds the sums of cut C tiles
hipError_t launch_spmm_wide(int dtype, const WideArgs &wa, const WideShape &sh, hipStream_t s, hipEvent_t mid);
hipError_t launch_wide_fill(const TileSource &src, uint32_t rows, uint32_t n_chunks, void *frags, hipStream_t s);
// Block kernels (spmm_block_kernel.hip): units of two windows with one column list (lower: kIdxMax where a window is alone),
// in steps of 16 (fp32 storage: 8) neighbouring columns
struct BlockUnit { uint32_t upper, lower, steps, row, next_row, pair_begin, spare[2]; };     // first tiles; steps; first row, that of the unit behind; first pair of steps
struct BlockArgs {
    const BlockUnit *units;
    const uint32_t *columns;     // per pair of steps their first columns
    const void     *tiles;
    const void     *B;
    void           *C;
    uint32_t rows, cols, N;
    const TileSource *src;       // in device memory (read where B is not finite)
};
hipError_t launch_spmm_block(int dtype, const BlockArgs &ba, uint32_t n_units, hipStream_t s);       // up to 64 features
// Narrow kernels (spmm_narrow_kernel.hip, 16-bit types): stored entries by blocks of 16 rows x kNarrowColumns columns
constexpr uint32_t kNarrowColumns = 128u, kNarrowMostBlocks = 1024u;
struct NarrowArgs {
    const uint32_t *blocks;      // per unit of 16 rows and block: its first four entries (n_units x n_blocks + 1)
    const uint32_t *entries;     // place in the block's image | value << 16
    const void     *B;
    void           *C;
    uint32_t rows, cols, N;
    uint32_t n_blocks;
    const TileSource *src;       // in device memory (read where B is not finite)
};
// A workgroup of `waves` (4, 8, 16) takes 16 rows; a wave asks for `loads` (1 .. 4) x 128 entries of a block at a time.
hipError_t launch_spmm_narrow(int dtype, const NarrowArgs &na, uint32_t waves, uint32_t loads, hipStream_t s);
hipError_t launch_narrow_count(const TileSource &src, uint32_t n_units, uint32_t n_blocks, uint32_t *counts, uint32_t *blocks, hipStream_t s);
hipError_t launch_narrow_fill(const TileSource &src, uint32_t n_units, uint32_t n_blocks, const uint32_t *counts, const uint32_t *blocks, uint32_t *entries, hipStream_t s);
// blocks[i]: units of four of counts[0 .. i - 1], every count rounded up (n + 1 of them)
hipError_t launch_tile_scan(const uint32_t *counts, uint32_t n, uint32_t *blocks, hipStream_t s);
hipError_t launch_fill_zero(void *dst, size_t bytes, hipStream_t s);
// bitmap tiles -> plain tiles.  8 x 16 tiles of 16-bit elements: header as KernelArgs::bm_header; 8 x 8 tiles of 32-bit
// elements: 4 header words per tile - rows 0..3, rows 4..7, position of the first stored element, number of stored elements
hipError_t launch_expand_bitmap(int elem_bytes, const uint32_t *header, const void *vals, void *tiles, uint32_t n_tiles,
                                hipStream_t s);
// n 16-bit elements -> n words with the element in the low half (launch_widen_halves), and back (launch_narrow_words):
// a single feature of a 16-bit type runs as two features, the second all zero
hipError_t launch_widen_halves(const void *src, void *dst, size_t n, hipStream_t s);
hipError_t launch_narrow_words(const void *src, void *dst, size_t n, hipStream_t s);
// plain 8 x 8 tiles of 32-bit elements, single windows -> the order the lanes of the fp32 gather kernels read them in
hipError_t launch_lane_order32(const void *tiles, void *out, uint32_t n_tiles, hipStream_t s);
// column ids of single windows -> without padding, in the order the lanes of the gather kernels read them in
hipError_t launch_step_ids(int elem_bytes, const uint32_t *raw, uint32_t *out, uint32_t n_tiles, hipStream_t s);
// Measurement only (gather_rate_kernel in hspmm_kernels.hip): loads part_bytes (128 or 256) of row ids[i] of B for
// every i < n_ids; parts > 1: `parts` parts of part_bytes each, dealt out by XCD, every part walking all ids.
hipError_t launch_gather_rate(const uint32_t *ids, uint64_t n_ids, const void *B, uint32_t row_bytes, uint32_t part_bytes,
                              uint32_t parts, int compute_units, uint32_t *sink, hipStream_t s);

}  // namespace hspmm
