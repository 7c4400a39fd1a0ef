// Internal header of the library's host code: what hspmm_capi.hip (settings, queries), hspmm_create.hip
// (plan creation) and hspmm_run.hip (launches) share - the plan, the process-wide settings, error reporting.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstdarg>
#include <cstring>
#include <string>
#include <vector>
#include <mutex>
#include <atomic>
#include <chrono>
#include <new>
#include <algorithm>

#include "../../include/hspmm.h"
#include "hspmm_device.h"
#include "partition.hpp"
#include "schedule.hpp"
#include "host_parallel.hpp"
#include "step_stream.hpp"

namespace hspmm_host {

// Stores the message hspmm_last_error returns on this thread and returns `code` (hspmm_capi.hip).
int fail(int code, const char *fmt, ...) __attribute__((format(printf, 2, 3)));

#define HSPMM_HIP(call)                                                                      \
    do {                                                                                     \
        hipError_t e_ = (call);                                                              \
        if (e_ != hipSuccess)                                                                \
            return fail(HSPMM_ERR_DEVICE, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), \
                        __FILE__, __LINE__);                                                 \
    } while (0)

// the same where a failure has to release something first: cleanup(code) is called with the error code and its result returned
#define HSPMM_HIP_OR(call, cleanup)                                                          \
    do {                                                                                     \
        hipError_t e_ = (call);                                                              \
        if (e_ != hipSuccess)                                                                \
            return cleanup(fail(HSPMM_ERR_DEVICE, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), \
                                __FILE__, __LINE__));                                        \
    } while (0)

// The knobs of the reference's Scheduler singleton (reference src/scheduler.h:7-10),
// re-read as: prefetch depth, waves per workgroup, waves per SIMD, compute units.
struct Config {
    int buffer_stage = 0;
    int consumer_warp_num = 0;
    int producer_warp_group_num = 0;
    int sm_num = 0;
    int kernel_mode = 0;
    int fused_fixup = -1;               // 1: the last wave of a cut unit adds its partial sums; 0: second kernel;
                                        // -1: the former in the LDS-panel kernels, and in the gather kernels where few units are cut
    int pairing = 0;                    // 0 automatic, 1 never, 2 whenever two windows share a column list
    int group_cuts = 0;                 // 1: plans of hspmm_create_grouped cut a window only where the caller's groups end
    // Tuning overrides from the environment (HSPMM_*), read once by hspmm_create: a plan's behaviour does
    // not change with the environment afterwards and the launch path reads no variable.
    int panel_chunks = 0;               // chunks of panels (0: searched per N)
    int panel_max_windows = 0;          // 2 or 4: windows per unit of the panel stream (0: by matrix size)
    int aligned_small = -1;             // small matrices: waves per unit of the one-workgroup-per-unit partition (-1: by size; 0, 4, 8)
    int gather_bitmap = -1;             // gather kernels read single 16-bit windows as bitmap + stored elements (-1: by fill)
    int entries = -1;                   // entry kernels for narrow feature dimensions (-1: by width, 0 never, 1 wherever they can)
    int tile = -1;                      // full-tile kernels (-1: by density and width, 0 never, 1 wherever they can)
    int narrow = -1;                    // narrow kernels (-1: by density and expected time, 0 never, 1 wherever they can)
    int narrow_waves = -1;              // waves of their workgroups (-1: by expected time)
    int wide = -1;                      // wide-tile kernels (-1: by density and expected time, 0 never, 1 wherever they can)
    int block = -1;                     // block kernels (-1: by expected time, 0 never, 1 wherever they can)
    int wide_cuts = -1;                 // workgroups of a C tile (-1: by expected time)
    int wide_shape = -1;                // their workgroup's shape, an index into the table of hspmm_wide.hip (-1: by expected time)
    int schedule = -1;                  // gather kernels: waves that sweep the columns together (-1: by matrix, 0 never, 1 wherever they can)
    int xcd_split = -1;                 // gather kernels: two feature blocks dealt out by XCD half (-1: by matrix, 0 never, 1 always)
    // (set through hspmm_set_panel_stream; builds with HSPMM_EXPERIMENTAL only)
    int panel_tall = 0;                 // LDS-panel waves with two units each
    int panel_packed = 0;               // ... and their tiles stored without zeros
    int panel_units_per_group = 0;      // consumer waves of a workgroup that get a unit (0: searched per N)
    // (builds with HSPMM_EXPERIMENTAL only)
    int panel_units = 0;                // workgroup shape of the fp32-MFMA LDS-panel kernels: 12, 13, 14 (0: by tile type)

    void read_environment()
    {
        if (const char *e = std::getenv("HSPMM_FUSED_FIXUP")) fused_fixup = std::atoi(e) != 0;
        if (const char *e = std::getenv("HSPMM_PANEL_CHUNKS")) panel_chunks = std::max(1, std::atoi(e));
        if (const char *e = std::getenv("HSPMM_PANEL_MAX_WINDOWS")) panel_max_windows = std::atoi(e) >= 4 ? 4 : 2;
        if (const char *e = std::getenv("HSPMM_XCD_SPLIT")) xcd_split = std::atoi(e) != 0;
        if (const char *e = std::getenv("HSPMM_SCHEDULE")) schedule = std::atoi(e);
        if (const char *e = std::getenv("HSPMM_ENTRIES")) entries = std::atoi(e) != 0;
        if (const char *e = std::getenv("HSPMM_TILE")) tile = std::atoi(e) != 0;
        if (const char *e = std::getenv("HSPMM_NARROW")) narrow = std::atoi(e) != 0;
        if (const char *e = std::getenv("HSPMM_NARROW_WAVES")) narrow_waves = std::atoi(e);
        if (const char *e = std::getenv("HSPMM_BLOCK")) block = std::atoi(e) != 0;
        if (const char *e = std::getenv("HSPMM_WIDE")) wide = std::atoi(e) != 0;
        if (const char *e = std::getenv("HSPMM_WIDE_SHAPE")) wide_shape = std::max(0, std::atoi(e));
        if (const char *e = std::getenv("HSPMM_WIDE_CUTS")) wide_cuts = std::max(0, std::atoi(e));
        if (const char *e = std::getenv("HSPMM_GATHER_BITMAP")) gather_bitmap = std::atoi(e) != 0;
        if (const char *e = std::getenv("HSPMM_ALIGNED_SMALL")) { const int v = std::atoi(e); aligned_small = v == 4 || v == 8 ? v : 0; }
        if (const char *e = std::getenv("HSPMM_PANEL_UNITS_PER_GROUP")) panel_units_per_group = std::max(1, std::atoi(e));
#ifdef HSPMM_EXPERIMENTAL
        if (const char *e = std::getenv("HSPMM_PANEL_UNITS")) panel_units = std::atoi(e) == 14 ? 14 : std::atoi(e) == 13 ? 13 : 12;
#endif
    }
};
// cost model of partition.hpp (a range costs its steps + 1.5 per unit; a cut within 35 % of a mean range of a unit
// boundary snaps onto it; units up to a mean range + 32 steps are never cut)
constexpr double kWindowCost = 1.5, kSlack = 0.35, kWholeWindowMargin = 32.0;
constexpr double kAlignedFourFrom = 2.5;   // ways the balanced partition must cut every unit before one workgroup walks it
constexpr double kPanelWideCost = 1.25;    // a step of three or four windows, in steps of two
extern std::mutex g_cfg_mutex;          // guards g_cfg (hspmm_capi.hip)
extern Config g_cfg;

constexpr uint32_t kMinTilesPerRange = 24;
// Plans that carry a schedule (power-law graphs, 16-bit bitmap tiles): from 2^18 columns on; built beside the packing of the tiles it adds nothing
// that shows to hspmm_create (10.6 / 10.3 ms at 2^20 vertices, 2.4 / 2.5 at 2^18, 3.7 / 4.0 at 600000) and 24 words a tile to its device memory
// (431 -> 527 MB at 2^20).  Against the partition it was ahead on all of 62 launches (12 graphs of 2^18 to 2^20 vertices, 4 to 32 edges each,
// N = 64 to 512) by 2 to 33 %, and at N = 192, 320, .. 1984 on all of 42 (six graphs) by 5 to 23 %; graphs of fewer vertices, with 8 to 32 MB of B for each
// 64 features, are the entry kernels' (entry kernels / schedule, N = 128: 131072 vertices 60 / 63 us, 150001 43 / 47, 200000 58 / 61, 230000 51 / 50,
// 250000 74 / 76; N = 512, where the partition is the other choice, 4 to 7 % ahead on all of these: not worth the memory).
constexpr uint32_t kScheduledColumns = 1u << 18;
// Bytes of B in a block of 64 features from which a single block, or an odd number of them, goes by the schedule rather than to the entry kernels
// (entry kernels / schedule, us, N = 64: 2^20 vertices, 16 edges each, 262 / 203, 900000, 12 edges, 130 / 123, 800000, 8 edges, 87 / 82, 600000 73 / 77,
// 350000 55 / 63, 2^18 42 / 50).  Two, four or eight blocks, each with XCDs of its own, from the first such plan on (N = 128: 2^19, 16 edges, 239 / 175,
// 350000, 10 edges, 84 / 76, 2^18, 16 edges, 94 / 80; N = 256 at 2^18: 195 / 168).
constexpr uint64_t kScheduledSlice = uint64_t(96) << 20;
// What keeps a launch from the order's gain, of 804 launches of matrices of 4000 to 800000 rows and 2^18 to 1.2 million columns (R-MAT, and rows and
// columns drawn by powers), at all these N: windows so long that the sums of many parts are added one after the other (the longest over 32 of a
// wave's shares: 0.94 times as fast on the mean, 0.27 at least); columns that no windows share (1.01 entries per tile column and less: 1.0, 0.88 at
// least, and slower than the entry kernels); launches too short for it, in which few rows name many columns (C below 64 MB: 0.98, 0.51).  195 launches
// are left, 1.12 times as fast on the mean, 5 slower by more than 3 % (8 % at most).  Graphs as tall as they are wide are all among them.
constexpr uint32_t kScheduledLongest = 32;
constexpr double kScheduledColumnsShared = 1.01;
constexpr uint64_t kScheduledProduct = uint64_t(64) << 20;
// No unit has over eight times the average number of steps.
inline bool windows_are_even(uint32_t longest, uint32_t units, uint32_t steps) { return uint64_t(longest) * units <= uint64_t(steps) * 8u; }

// What a plan answers for a feature dimension, kept for the last few asked for, 32 bits each: the answers are the plan's and N's alone, so
// threads may overwrite each other's.  (A search costs a launch 0.5 to 1 us of the host's; 16, 32, .. 1024 have a slot each.)
class KeptAnswers {
    std::atomic<uint64_t> slots_[16] = {};
public:
    template <class F> uint32_t get(uint32_t N, F find)
    {
        std::atomic<uint64_t> &slot = slots_[N * 0x9E3779B1u >> 28];
        uint64_t kept = slot.load(std::memory_order_relaxed);
        if (uint32_t(kept >> 32) != N) slot.store(kept = uint64_t(N) << 32 | find(), std::memory_order_relaxed);
        return uint32_t(kept);
    }
};

}  // namespace hspmm_host

struct hspmm_plan {
    int dtype = 0;
    int device = 0;
    uint32_t rows = 0, cols = 0, W = 0, T = 0;
    uint32_t cw = 16, elem = 2;
    int compute_units = 0;
    hspmm_host::Config cfg;
    // device copies of the format arrays as given: scalar kernel
    uint32_t *d_rowOffset = nullptr, *d_rowIdx = nullptr;
    uint32_t *d_a2b_raw = nullptr;
    void *d_data = nullptr;
    // the step stream of the MFMA kernels
    int G = 1;                          // windows per unit: 2 when windows were paired
    uint32_t n_units = 0, n_paired = 0, n_steps = 0;
    uint32_t *d_unitOffset = nullptr, *d_unitRow = nullptr;
    uint32_t *d_ids = nullptr;          // per step, lane order, padding renamed to the id in front of it
    void *d_tiles = nullptr;            // per step, lane order (== d_data for fp16 without pairs)
    // partition
    // partitions of the step stream: [0] for one feature block per wave range (built by
    // hspmm_create), [1] / [2] with a half / a quarter of the ranges for feature dimensions
    // that need 2-3 / 4 or more blocks, built on first use (more blocks = more waves per range)
    struct DevPartition {
        bool built = false;
        hspmm::Partition part;
        uint32_t *d_ranges = nullptr, *d_split = nullptr, *d_fix_slots = nullptr;
    };
    DevPartition parts[5];              // [0..2]: fewer ranges per level; [3]: level 0 with sums added per workgroup;
                                        // [4]: every unit cut into the ranges of one workgroup (aligned)
    int aligned_group = 0;              // waves of the workgroup that walks one unit in [4]; 0: units too short for it
    std::vector<uint32_t> h_unitOffset;
    std::vector<uint32_t> h_unitRow;       // first row of every unit | its windows less one (for hspmm_partition_as_groups)
    std::vector<uint32_t> h_winOffset, h_winRow;   // plans whose units merge windows: the caller's rowOffset and rowIdx
                                                   // (hspmm_partition_as_groups writes groups of the caller's tiles)
    std::vector<uint32_t> caller_cuts;     // hspmm_create_grouped with hspmm_set_group_cuts(1): the ends of the caller's groups,
                                           // the only places where the gather kernels' partition cuts a window
    // LDS-panel kernels (matrices whose windows touch a large share of the columns):
    // the unit stream re-tiled panel by panel, built by hspmm_create when it pays
    struct Panel {
        bool built = false;
        uint32_t n_panels = 0, n_steps = 0;
        uint32_t *d_poff = nullptr, *d_ids = nullptr, *d_step_panel = nullptr;
        void *d_tiles = nullptr;
        uint32_t *d_unitRow = nullptr;                           // the units of this stream (first row | paired bit)
        uint32_t n_units = 0, n_paired = 0, n_wide = 0;          // units of two or more / three or four windows
        int G = 1;
        bool quad = false;                                       // ids in the format of the 4x4x1 fp32 tile
        bool split = false;                                      // fp32 stream in the bf16 hi / lo form (Fp32Split)
        bool tall = false;                                       // two units per consumer wave: poff per pair of units,
                                                                 // their steps merged panel by panel
        bool packed = false;                                     // tiles without their zeros: masks, values, step_voff
        double unit_lines = 0.0;                                 // 128-byte lines of tiles and ids per unit and panel (tall streams)
        uint64_t *d_masks = nullptr;
        void *d_vals = nullptr;
        uint32_t *d_step_voff = nullptr;
        double density = 0.0;                                    // steps per unit and 128 columns of the gather stream
        mutable hspmm_host::KeptAnswers expected;                // (see panel_expected)
    } panel;
    // Bitmap stream of the gather kernels (single 16-bit windows whose tiles are mostly zeros): per tile 8 words
    // of header (the reference's tcBit words of the tile, bit counts, position of the first stored element) and
    // the stored elements of all tiles in ascending bit order - nnzOffset / tcBit / data of the reference's BTCF_MTX
    struct Bitmap {
        bool built = false;
        uint32_t *d_header = nullptr;
        void *d_vals = nullptr;
        uint64_t stored = 0;
        bool from_caller = false;     // header and elements are the caller's tcBit / nnzOffset / data, uploaded as they came
    } bm;
    // The same tiles in the order of a schedule (schedule.hpp), for a B far larger than the L2s: ids and headers are copies, elements are not
    struct Scheduled {
        bool built = false;
        const uint32_t *d_ids = nullptr, *d_header = nullptr, *d_unitOffset = nullptr, *d_info = nullptr, *d_ranges = nullptr,
                       *d_split = nullptr, *d_fix_slots = nullptr;
        uint32_t n_units = 0, n_ranges = 0, n_split = 0, n_slots = 0;
    } scheduled;
    // Stored entries, rows sorted by length, for narrow feature dimensions (spmm_entries.hip): counted by hspmm_create, made from
    // the tiles on the device by the first launch (or hspmm_prepare) that wants it
    struct Entries {
        bool counted = false;
        std::atomic<bool> unavailable{false};                    // no memory for it: the other kernels serve this plan
        uint32_t most_chunks = 0;
        uint32_t *d_first_chunk = nullptr, *d_chunk_window = nullptr, *d_positions = nullptr, *d_row_len = nullptr, *d_row_first = nullptr;
        uint32_t *d_totals = nullptr;                            // kEntryBins + 1 counts, then as many cursors
        uint32_t totals[hspmm::kEntryBins + 1u] = {};
        bool built = false;
        void *d_stream = nullptr;                                // one allocation for the four below
        const uint32_t *d_desc = nullptr, *d_ids = nullptr, *d_pieces = nullptr;
        const void *d_vals = nullptr;
        uint64_t units = 0;
        bool long_rows = false;                                  // 64 units and more in a row on average
        hspmm::EntryArgs classes[6] = {};                        // by log2 lanes of a row, once a launch has asked for it
    } entries;
    // Stored entries by blocks of 128 rows x 64 (fp32 storage: 32) columns, for matrices that are dense to a workgroup
    // (spmm_tile_kernel.hip): made from the tiles on the device by hspmm_create
    struct Tile {
        bool built = false;
        const uint32_t *d_blocks = nullptr;
        const void *d_pos = nullptr, *d_vals = nullptr;
        hspmm::TileSource *d_source = nullptr;                   // where the tiles are
        uint32_t n_row_blocks = 0, n_blocks = 0;
        uint64_t entries = 0;                                    // stored entries, blocks rounded up to four
    } tile;
    // The same matrices, 16-bit types, their stored entries by blocks of 16 rows, for few features (spmm_narrow_kernel.hip)
    struct Narrow {
        bool built = false;
        const uint32_t *d_blocks = nullptr, *d_entries = nullptr;
        hspmm::TileSource *d_source = nullptr;
        uint32_t n_units = 0, n_blocks = 0;
        uint64_t entries = 0;                                    // blocks rounded up to four
    } narrow;
    // The same matrices, 16-bit types, as operands of matrix instructions, for wider feature dimensions (spmm_wide_kernel.hip)
    struct Wide {
        bool built = false;
        const void *d_frags = nullptr;
        hspmm::TileSource *d_source = nullptr;
        uint32_t n_units = 0, n_chunks = 0;
        double expected_fewest = 0.0;                            // us, of the fewest features they take (see hspmm_wide.hip)
        mutable hspmm_host::KeptAnswers choices;
    } wide;
    // Weights in 16 x 16 blocks, for few features: units of windows whose steps are neighbouring columns (spmm_block_kernel.hip)
    struct Block {
        bool built = false;
        const hspmm::BlockUnit *d_units = nullptr;
        const uint32_t *d_columns = nullptr;
        const hspmm::TileSource *d_source = nullptr;
        uint32_t n_units = 0, longest = 0;                       // (steps of the longest unit)
        mutable hspmm_host::KeptAnswers taken;
    } block_units;
    double per_column = 8.0;            // stored entries per tile column, from a sample of the tiles
    bool even_windows = false;          // no unit has over eight times the average number of steps
    // What launches write besides C, one set per stream that has launched this plan (launches on different
    // streams may overlap in time): the first stream seen gets set 0, every other stream a set of its own at its
    // first launch - except a stream that is being captured (no allocation under capture) and streams beyond
    // kMaxStreamBuffers, which share set 0.
    struct StreamBuffers {
        hipStream_t stream = nullptr;
        bool unowned = false;               // made by hspmm_prepare before any launch: the first stream to launch takes it
        float *d_scratch = nullptr;         // partial sums of cut units
        size_t scratch_bytes = 0;
        uint32_t *d_arrive = nullptr;       // arrival counters of cut units, zero between launches
        size_t arrive_words = 0;
        uint32_t *d_vector = nullptr;       // a single 16-bit feature widened to words: cols words of B, then rows words
                                            // of C (made by the first launch with N = 1, or by hspmm_prepare(plan, 1))
    };
    static constexpr size_t kMaxStreamBuffers = 16;
    std::vector<StreamBuffers> buffers;
    size_t fixed_bytes = 0;
    std::vector<void *> owned;              // allocations of plan_reserve / plan_alloc
    char *block = nullptr;                  // what is left of the reserved block
    size_t block_left = 0;
    // Every real column list strictly ascending and padding only behind a window's last column: what the
    // reference's converters write (reference src/utils/convert.h:166-181).  The gather and all-shapes
    // kernels take any list; merging windows and the LDS-panel stream need this order.
    bool canonical = true;
    // What a launch may still have to build (a partition for a wider N, larger scratch) is built under
    // this mutex; everything else in the plan is immutable after hspmm_create.
    std::mutex mu;
    // Superseded scratch buffers stay allocated until hspmm_destroy: launches recorded earlier (HIP
    // graphs) carry their addresses.
    std::vector<void *> retired;
    size_t retired_bytes = 0;               // partial-sum buffers among them (counters are part of fixed_bytes)
    std::atomic<uint32_t> last_family{0};   // kernel family of the last hspmm_run: 0 none yet, 1 all-shapes, 2 gather, 3 LDS-panel, 4 clear
    // matrix instructions of the last launch's main kernel: kind (hspmm_plan_info::last_mfma_kind) and count
    std::atomic<uint32_t> last_mfma_kind{0};
    std::atomic<uint64_t> last_mfma_count{0};
    std::atomic<const char *> last_kernel{""};  // its name (hspmm_last_kernel)
    // what the waves of the gather kernels walked in it (hspmm_last_walk)
    std::atomic<uint32_t> last_scheduled{0}, last_ranges{0}, last_split{0};
    void note_launch(const char *kernel, uint32_t family, uint32_t kind, uint64_t count, uint32_t scheduled = 0, uint32_t ranges = 0, uint32_t split = 0)
    {
        last_scheduled.store(scheduled, std::memory_order_relaxed);
        last_ranges.store(ranges, std::memory_order_relaxed);
        last_split.store(split, std::memory_order_relaxed);
        last_kernel.store(kernel, std::memory_order_relaxed);
        last_family.store(family, std::memory_order_relaxed);
        last_mfma_kind.store(kind, std::memory_order_relaxed);
        last_mfma_count.store(count, std::memory_order_relaxed);
    }
};

namespace hspmm_host {

// HSPMM_TIMING=1 in the environment: hspmm_create prints what each of its phases took (stderr).
struct PhaseTimer {
    bool on = std::getenv("HSPMM_TIMING") != nullptr;
    std::chrono::steady_clock::time_point last = std::chrono::steady_clock::now();
    void mark(const char *what)
    {
        if (!on) return;
        const auto now = std::chrono::steady_clock::now();
        std::fprintf(stderr, "hspmm_create: %-28s %8.2f ms\n", what, std::chrono::duration<double, std::milli>(now - last).count());
        last = now;
    }
};

// Device memory of a plan, all of it given back by hspmm_destroy (hspmm_create.hip).  plan_reserve allocates one block
// that later plan_alloc calls are served from as long as they fit (an allocation takes 50 to 100 us, and freeing one as
// long again); what does not fit gets an allocation of its own, which plan_release can give back early.
int plan_reserve(hspmm_plan *p, size_t bytes);
int plan_alloc(hspmm_plan *p, size_t bytes, void **out);
void plan_release(hspmm_plan *p, const void *ptr, size_t bytes);

template <typename T>
int upload(hspmm_plan *p, T **dst, const T *src, size_t n)
{
    void *fresh = nullptr;
    if (int rc = plan_alloc(p, (n ? n : 1) * sizeof(T), &fresh)) return rc;
    *dst = static_cast<T *>(fresh);
    if (n) HSPMM_HIP(hipMemcpy(*dst, src, n * sizeof(T), hipMemcpyHostToDevice));
    return HSPMM_OK;
}

// How a launch gets the memory it needs beyond the plan's fixed arrays.
//   kLaunch:  hspmm_run - may build a partition and grow the plan's scratch buffer (under the plan's mutex)
//   kPrepare: hspmm_prepare - builds and grows exactly like kLaunch and launches nothing
//   kStatic:  hspmm_run_static - partial sums go to the library's fixed device array; builds and allocates nothing
enum class RunMode { kLaunch, kPrepare, kStatic };

// hspmm_create.hip
int validate_format(uint32_t rows, uint32_t cols, uint32_t W, uint32_t T, uint32_t cw,
                    const uint32_t *rowOffset, const uint32_t *tcA2B, const void *data, const uint32_t *rowIdx,
                    bool *canonical = nullptr);
int choose_ranges(const hspmm_plan *p);
int build_and_upload_partition(hspmm_plan *p, int level, uint32_t group = 1, bool aligned = false);

// hspmm_run.hip: memory a launch writes besides C (called with the plan's mutex held)
int ensure_arrive(hspmm_plan *p, hipStream_t s, size_t words, RunMode mode, uint32_t **out);
int scratch_for(hspmm_plan *p, hipStream_t s, size_t bytes, RunMode mode, float **out);
// hspmm_entries.hip: counting what the entry kernels' stream holds (enqueued; hspmm_create reads the totals once it has
// waited) and the device memory that takes, whether they take this launch, and the launch
size_t entries_count_bytes(const hspmm_plan *p);
int count_entries(hspmm_plan *p);
int entries_counted(hspmm_plan *p);
bool entries_serve(const hspmm_plan *p, uint32_t N);

// Feature blocks of one 128-byte line, with XCDs of their own where there are two, four or eight (see spmm_mfma_kernel): pays when B is far
// larger than an XCD's 4 MB L2, so that what an L2 can keep of it decides the hit rate of the gathers (power-law graph 2^20, N = 128: 575 -> 535 us;
// uniform 65536^2: 39.7 -> 35.5 us), and costs a second pass over the tile stream.  Requests below a 128-byte line lose (N = 64 as two blocks of
// 32: 280 -> 510 us).
inline bool splits_features(const hspmm_plan *p, uint32_t N)
{
    return p->cfg.xcd_split > 0 || (p->cfg.xcd_split < 0 && uint64_t(p->cols) * N * p->elem >= (uint64_t(8) << 20));
}

// Whether a launch of the gather kernels walks the plan's schedule, given words of B and C (a launch in blocks of 64 features, which N fills, with
// 32-bit offsets into B).
inline bool scheduled_serves(const hspmm_plan *p, uint32_t N)
{
    const hspmm_plan::Scheduled &sc = p->scheduled;
    if (!sc.built || !(N % 128u == 64u || (splits_features(p, N) && (N == 128u || N == 256u || N == 512u)))) return false;
    if (p->cols >= (1u << 24) || uint64_t(p->cols) * N * p->elem > (uint64_t(1) << 32)) return false;
    if (p->cfg.schedule < 0 && uint64_t(p->rows) * N * p->elem < kScheduledProduct) return false;
    return size_t(sc.n_slots) * (N / 64u) * 2048u <= HSPMM_STATIC_SCRATCH_BYTES;     // (however it is launched)
}

// Where the entry kernels would serve as well: graphs whose columns are hot, so that windows share them.  Uneven rows over uniform columns (one
// entry per tile column; graphs of 2^18 to 2^21 vertices with 2 to 30 edges each have 1.02 to 1.14) gain nothing from the order: N = 128, us, by
// schedule / entry kernels: 2^19 columns 207 / 191, 300000 59.7 / 55.2, 2^18 58.6 / 53.7; N = 64, 2^20 columns 101 / 94, 240 / 218, 66 / 58.
inline bool scheduled_before_entries(const hspmm_plan *p, uint32_t N, uintptr_t align)
{
    return p->cfg.entries < 0 && p->per_column > kScheduledColumnsShared && align % 4u == 0u && scheduled_serves(p, N) &&
           (N % 128u == 0u || uint64_t(p->cols) * 128u >= kScheduledSlice);
}

double entries_expected(const hspmm_plan *p, uint32_t N);       // us, pruned weights of 16 bits, fewer than 256 features
int run_entries(hspmm_plan *p, const void *dB, void *dC, uint32_t N, hipStream_t s, RunMode mode, bool *taken);

// hspmm_run.hip: whether the LDS-panel kernels serve feature dimension N
bool panel_serves(const hspmm_plan *p, uint32_t N);
// ... and the time that their launch shape is expected to take, in us beyond what every launch does (0: none to be had)
double panel_expected(const hspmm_plan *p, uint32_t N);
// hspmm_tile.hip: the full-tile kernels' stream, whether they take this launch, and the launch
int build_tile_stream(hspmm_plan *p);
bool tile_serves(const hspmm_plan *p, uint32_t N);
bool tile_leaves(const hspmm_plan *p, uint32_t N);
double tile_expected(const hspmm_plan *p, uint32_t N);          // us
int run_tile(hspmm_plan *p, const void *dB, void *dC, uint32_t N, hipStream_t s, RunMode mode);

// hspmm_narrow.hip: the narrow kernels' stream, whether they take this launch, and the launch
int build_narrow_stream(hspmm_plan *p);
bool narrow_serves(const hspmm_plan *p, uint32_t N, bool on_word);        // on_word: B begins on a word
int run_narrow(hspmm_plan *p, const void *dB, void *dC, uint32_t N, hipStream_t s, RunMode mode);
// hspmm_block.hip: what the block kernels need to know of the units, whether they take this launch, and the launch
int build_block_units(hspmm_plan *p, const StepStream &st, const uint32_t *rowOffset, const uint32_t *tcA2B);
bool block_serves(const hspmm_plan *p, uint32_t N, bool on_word);        // on_word: B begins on a word
int run_block(hspmm_plan *p, const void *dB, void *dC, uint32_t N, hipStream_t s, RunMode mode);
// hspmm_wide.hip: the wide-tile kernels' stream, whether they take this launch, and the launch
int build_wide_stream(hspmm_plan *p);
bool wide_serves(const hspmm_plan *p, uint32_t N);
double blocks_expected(const hspmm_plan *p, uint32_t N);        // us, weights in 16 x 16 blocks, by these or the gather kernels
int run_wide(hspmm_plan *p, const void *dB, void *dC, uint32_t N, hipStream_t s, hipEvent_t mid, RunMode mode);

// hspmm_run.hip: the address of the device's fixed scratch array (hspmm_run_static); `device` must be current
int static_scratch_address(int device, float **out);

}  // namespace hspmm_host
