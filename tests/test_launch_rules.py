"""Which launches a kernel family takes, and in what shape: the host code's rules at their lines, compiled here without kernels and device.  No
GPU needed."""
import subprocess

import pytest

from test_optional_streams import COMMON, ENTRY_DRIVER, build  # noqa: F401

ENTRY_STUBS = ENTRY_DRIVER[:ENTRY_DRIVER.index("int main()")]


def _run(build, driver, *families):
    run = subprocess.run([build(driver, *families)], stdout=subprocess.PIPE, timeout=60)
    assert run.returncode == 0 and run.stdout == b"ok\n", run.stdout.decode()


def _driver(stubs, body):
    return stubs + """
#define EXPECT(x) do { if (!(x)) { std::printf("line %d: %s\\n", __LINE__, #x); return 1; } } while (0)
int main()
{
    using namespace hspmm_host;
#line 1 "body"
""" + body + """
    std::printf("ok\\n");
    return 0;
}
"""


def test_entry_kernels_take_rows_of_up_to_1024_features(build):  # noqa: F811
    _run(build, _driver(ENTRY_STUBS, """
    for (int dtype : {HSPMM_FP16, HSPMM_TF32, HSPMM_BF16})
        for (int forced : {-1, 1})
            for (bool even : {false, true}) {
                hspmm_plan p;
                p.dtype = dtype; p.elem = dtype == HSPMM_TF32 ? 4 : 2; p.cw = dtype == HSPMM_TF32 ? 8 : 16;
                p.rows = p.cols = 10000; p.W = 1250; p.T = 10000; p.compute_units = 256; p.per_column = 1.0; p.even_windows = even;
                p.entries.counted = true; p.cfg.entries = forced;
                for (uint32_t N : {1u, 512u, 1000u, 1023u, 1024u}) EXPECT(entries_serve(&p, N));
                for (uint32_t N : {1025u, 1030u, 1088u, 1536u, 2047u, 2048u, 4096u}) EXPECT(!entries_serve(&p, N));
            }
"""), "entries")


def test_schedules_serve_where_the_gather_kernels_could_walk_them(build):  # noqa: F811
    """Blocks of 64 features, 32-bit offsets into B: launches of other shapes are not kept from the entry kernels."""
    _run(build, _driver(ENTRY_STUBS, """
    hspmm_plan p;
    p.dtype = HSPMM_FP16; p.rows = 1 << 21; p.per_column = 1.05;
    p.scheduled.built = true; p.scheduled.n_slots = 350;
    for (uint32_t cols : {1u << 18, 1u << 20, 1u << 22, (1u << 23) + 8u, (1u << 24) - 1u, 1u << 24, (1u << 24) + 1000u, 1u << 26})
        for (uint32_t N : {32u, 64u, 96u, 128u, 192u, 256u, 320u, 384u, 512u, 1024u}) {
            const bool blocks = N % 128u == 64u || N == 128u || N == 256u || N == 512u;
            const bool reached = cols < (1u << 24) && uint64_t(cols) * N * 2u <= (uint64_t(1) << 32);
            p.cols = cols; p.cfg.xcd_split = -1;
            EXPECT(scheduled_serves(&p, N) == (blocks && reached));
            EXPECT(!scheduled_before_entries(&p, N, 0u) || scheduled_serves(&p, N));
            EXPECT(!scheduled_before_entries(&p, N, 2u));
            p.cfg.xcd_split = 0;                            // (two, four and eight blocks in one wave then)
            EXPECT(scheduled_serves(&p, N) == (blocks && reached && N % 128u == 64u));
        }
"""), "entries")


def test_schedules_come_before_the_entry_kernels_where_columns_are_hot(build):  # noqa: F811
    """Uneven rows over uniform columns have one stored entry per tile column: no order of the windows brings rows of B back sooner."""
    _run(build, _driver(ENTRY_STUBS, """
    hspmm_plan p;
    p.dtype = HSPMM_FP16; p.rows = p.cols = 1 << 20;
    p.scheduled.built = true; p.scheduled.n_slots = 350;
    for (double per_column : {1.0, 1.0003, 1.004, 1.018, 1.03, 1.1}) {
        p.per_column = per_column;
        for (uint32_t N : {64u, 128u, 256u, 512u, 576u}) EXPECT(scheduled_serves(&p, N) && scheduled_before_entries(&p, N, 0u) == (per_column > 1.01));
    }
"""), "entries")


def test_static_launches_do_not_change_kernels_with_what_ran_before(build):  # noqa: F811
    """B between two words on a plan with a schedule: the entry kernels' launch, so refused while their stream is not built."""
    _run(build, _driver(ENTRY_STUBS, """
    hspmm_plan p;
    p.dtype = HSPMM_FP16; p.rows = p.cols = 1 << 20; p.W = 1 << 17; p.T = 1 << 20; p.compute_units = 256; p.per_column = 1.05;
    p.scheduled.built = true; p.scheduled.n_slots = 350; p.entries.counted = true;
    const void *B = reinterpret_cast<const void *>(uintptr_t(4098));
    EXPECT(entries_serve(&p, 64u) && scheduled_before_entries(&p, 64u, 0u) && !scheduled_before_entries(&p, 64u, 4098u));
    bool taken = true;
    EXPECT(run_entries(&p, B, nullptr, 64u, nullptr, RunMode::kStatic, &taken) == HSPMM_ERR_UNSUPPORTED && !taken);
"""), "entries")


def test_rows_without_entries_do_not_change_the_shape_of_long_ones(build):  # noqa: F811
    """300 rows of 1500 entries (places of 384 units of four), or of 500 (128), alone and among ten thousand without entries."""
    _run(build, _driver(ENTRY_STUBS, """
    uint32_t of[2][2];
    for (int len : {0, 1})
        for (int empty : {0, 1}) {
            hspmm_plan p;
            p.dtype = HSPMM_TF32; p.elem = 4; p.cw = 8; p.cols = 4096; p.compute_units = 256; p.per_column = 1.0;
            p.rows = 300u + empty * 10000u; p.W = (p.rows + 7u) / 8u; p.T = 100000;
            p.entries.counted = true;
            p.entries.totals[len ? 3 : 9] = 300; p.entries.totals[hspmm::kEntryBins - 1u] = empty * 10000u;
            left = 100;
            bool taken = false;
            EXPECT(!run_entries(&p, reinterpret_cast<const void *>(uintptr_t(4096)), nullptr, 4u, nullptr, RunMode::kLaunch, &taken) && taken && p.entries.long_rows);
            EXPECT(hspmm::got.cls[0].slot_begin == 0u && hspmm::got.cls[0].slot_end == 300u);
            of[len][empty] = hspmm::got.cls[0].logs;
        }
    EXPECT(of[0][0] == of[0][1]);
    EXPECT(of[1][0] == of[1][1]);
"""), "entries")


# (device memory as large as it is asked for)
BLOCK_STUBS = COMMON.replace("hipMalloc(void **p, size_t) {", "hipMalloc(void **p, size_t n) {").replace("std::malloc(64)", "std::malloc(n)") + """
namespace hspmm { hipError_t launch_spmm_block(int, const BlockArgs &, uint32_t, hipStream_t) { return hipErrorInvalidValue; } }
namespace hspmm_host {
static double panel = 0.0;                          // us the LDS-panel kernels would take (0: not theirs)
bool panel_serves(const hspmm_plan *, uint32_t) { return panel > 0.0; }
double panel_expected(const hspmm_plan *, uint32_t) { return panel; }
double blocks_expected(const hspmm_plan *, uint32_t) { return 1e9; }
static bool wide = false;                           // whether the wide-tile kernels take it
bool wide_serves(const hspmm_plan *, uint32_t N) { return wide && N >= 32u; }
// A plan of rows of blocks with so many blocks each, every block behind the one in front of it; aligned: the gather kernels cut every unit.
static bool built(hspmm_plan *p, int dtype, const std::vector<uint32_t> &blocks, bool aligned)
{
    StepStream st;
    const uint32_t each = dtype == HSPMM_TF32 ? 2u : 1u;
    p->dtype = dtype; p->elem = 2u * each; p->cw = 16u / each; p->G = 2; p->compute_units = 256; p->aligned_group = aligned ? 4 : 0;
    p->rows = uint32_t(blocks.size()) * 16u;
    std::vector<uint32_t> rowOffset(1, 0u), ids;
    st.unitOffset.push_back(0);
    for (size_t u = 0; u < blocks.size(); ++u) {
        st.unitWindow.push_back(uint32_t(2 * u)); st.unitRow.push_back(uint32_t(u) * 16u | 1u);
        st.unitOffset.push_back(st.unitOffset.back() + blocks[u] * each);
        for (int w = 0; w < 2; ++w) {
            rowOffset.push_back(rowOffset.back() + blocks[u] * each);
            for (uint32_t c = 0; c < blocks[u] * 16u; ++c) ids.push_back(c);
        }
        p->cols = std::max(p->cols, blocks[u] * 16u);
    }
    p->W = uint32_t(2 * blocks.size()); p->T = rowOffset.back();
    p->n_units = uint32_t(blocks.size()); p->n_steps = st.unitOffset.back();
    left = 100;
    return build_block_units(p, st, rowOffset.data(), ids.data()) == HSPMM_OK && p->block_units.built;
}
static std::vector<uint32_t> one_long(size_t units, uint32_t mean, uint32_t longest) { std::vector<uint32_t> b(units, mean); b[units / 2] = longest; return b; }
}
"""


def test_block_kernels_take_even_rows_of_blocks(build):  # noqa: F811
    """A workgroup has a row of blocks: not where one is much longer than the others, nor where there are many thousands of short ones."""
    _run(build, _driver(BLOCK_STUBS, """
    for (int dtype : {HSPMM_FP16, HSPMM_BF16, HSPMM_TF32}) {
        const uint32_t most = dtype == HSPMM_TF32 ? 160u : 256u;
        struct { std::vector<uint32_t> blocks; bool aligned, taken; } at[] = {
            {one_long(256, 448, 480), true, true}, {one_long(64, 13, 30), false, true}, {one_long(1024, 40, 64), false, true},
            {one_long(64, 200, 1024), true, true}, {one_long(256, 40, 260), true, false}, {one_long(1024, 55, 1024), false, false},
            {one_long(256, 10, 36), false, true}, {one_long(256, 10, 38), false, false}, {one_long(64, most, most), false, true},
            {one_long(64, most, most + 1u), false, false}, {one_long(1, 4096, 4096), true, true}, {one_long(2048, 5, 12), false, true},
            {one_long(2049, 5, 12), false, false}, {one_long(8192, 10, 20), false, false},
        };
        for (auto &a : at) {
            hspmm_plan p;
            const bool b = built(&p, dtype, a.blocks, a.aligned);
            if (b != a.taken) { std::printf("dtype %d, %zu units, first of %u, longest of %u: %d\\n", dtype, a.blocks.size(), a.blocks[0], a.blocks[a.blocks.size() / 2], int(b)); return 1; }
            EXPECT(block_serves(&p, 16u, true) == a.taken && block_serves(&p, 31u, true) == a.taken);
            hspmm_plan forced;
            forced.cfg.block = 1;
            EXPECT(built(&forced, dtype, a.blocks, a.aligned));         // (as the tests of the kernels ask for)
        }
        // every other, or every eighth, row of blocks is short or long: the XCDs, which take them in turn, have uneven shares
        for (uint32_t units : {256u, 264u, 1600u})
            for (uint32_t nth : {2u, 8u, 7u}) {
                std::vector<uint32_t> blocks(units, 10);
                for (uint32_t u = 0; u < units; u += nth) blocks[u] = 20;
                hspmm_plan p;
                EXPECT(built(&p, dtype, blocks, true) == (units <= 256u || nth == 7u));
            }
        for (uint32_t units : {512u, 1024u, 1025u, 2048u}) {
            hspmm_plan p;
            EXPECT(built(&p, dtype, one_long(units, 5, 5), false) && block_serves(&p, 32u, true) && block_serves(&p, 64u, true) == (dtype == HSPMM_TF32 || units <= 1024u));
        }
    }
    // fp32 where the LDS-panel kernels would serve: by the longest row of blocks
    panel = 13.5;
    for (uint32_t longest : {80u, 320u, 480u}) {
        hspmm_plan p;
        EXPECT(built(&p, HSPMM_TF32, one_long(64, 80, longest), true) && block_serves(&p, 16u, true) == (longest < 480u) && block_serves(&p, 24u, true) == (longest < 320u) && !block_serves(&p, 48u, true));
    }
"""), "block")


def test_graphs_dense_in_their_hot_columns_by_their_loads(build):  # noqa: F811
    """1.25 to 1.4 entries per tile column: the gather kernels' wide loads come first where N is a multiple of 8, and where C is large."""
    _run(build, _driver(ENTRY_STUBS, """
    hspmm_plan p;
    p.dtype = HSPMM_FP16; p.rows = p.cols = 8000; p.W = 1000; p.T = 14000; p.compute_units = 256; p.per_column = 1.3;
    p.entries.counted = true;
    for (uint32_t N = 1; N <= 1024; ++N) EXPECT(entries_serve(&p, N) == (N <= 96u || N % 8u != 0u || (N <= 640u && N % 64u == 0u)));
    p.rows = 40000;
    for (uint32_t N = 65; N <= 1024; ++N) EXPECT(entries_serve(&p, N) == (N % 8u ? N * 80000u <= (32u << 20) : (N <= 96u || N % 64u == 0u) && N * 80000u <= (16u << 20)));
    for (uint32_t N = 1; N <= 64; ++N) EXPECT(entries_serve(&p, N));
    p.per_column = 1.1;
    for (uint32_t N = 1; N <= 1024; ++N) EXPECT(entries_serve(&p, N));
    p.per_column = 1.3; p.even_windows = true;
    EXPECT(!entries_serve(&p, 512u) && !entries_serve(&p, 97u));
"""), "entries")


def test_large_products_of_short_rows_in_fp32(build):  # noqa: F811
    """Rows of B of over 2 KB, or a B of over 256 MB, or dense graphs: not where a few entries a row make a C of over 64 MB."""
    _run(build, _driver(ENTRY_STUBS, """
    for (double per_row : {1.0, 5.0, 7.0, 20.0})
        for (uint32_t rows : {10000u, 16384u, 20000u, 400000u})
            for (bool even : {false, true}) {
                hspmm_plan p;
                p.dtype = HSPMM_TF32; p.elem = 4; p.cw = 8; p.rows = rows; p.cols = 5000; p.W = rows / 8; p.compute_units = 256; p.per_column = 1.0;
                p.T = uint32_t(per_row * rows / 8.0); p.entries.counted = true; p.even_windows = even;
                for (uint32_t N : {513u, 640u, 1024u}) EXPECT(entries_serve(&p, N) == (per_row >= 6.0 || uint64_t(rows) * N * 4u <= (64u << 20)));
                for (uint32_t N : {65u, 128u, 512u}) EXPECT(entries_serve(&p, N));
                p.cols = 200000;
                EXPECT(entries_serve(&p, 320u));                                        // 256 MB
                EXPECT(entries_serve(&p, 512u) == (even && (per_row >= 6.0 || rows <= 20000u)));
                p.cols = 5000; p.per_column = 1.3; p.T = uint32_t(p.T / 1.3);
                if (!even) EXPECT(entries_serve(&p, 256u) == (per_row >= 6.0 || rows <= 20000u));
            }
"""), "entries")


def test_schedules_of_launches_that_gain_from_the_order(build):  # noqa: F811
    _run(build, _driver(ENTRY_STUBS, """
    hspmm_plan p;
    p.dtype = HSPMM_BF16; p.cols = 1 << 18; p.per_column = 1.1;
    p.scheduled.built = true; p.scheduled.n_slots = 350;
    for (uint32_t rows : {1000u, (1u << 17) - 1u, 1u << 17, 1u << 18, 1u << 20})
        for (uint32_t N : {64u, 128u, 256u, 576u}) {
            p.rows = rows; p.cfg.schedule = -1;
            EXPECT(scheduled_serves(&p, N) == (uint64_t(rows) * N * 2u >= (64u << 20)));
            p.cfg.schedule = 1;
            EXPECT(scheduled_serves(&p, N));
        }
"""), "entries")


def test_block_kernels_where_the_wide_tile_kernels_are_or_b_lies_between_two_words(build):  # noqa: F811
    _run(build, _driver(BLOCK_STUBS, """
    for (int dtype : {HSPMM_FP16, HSPMM_BF16})
        for (uint32_t blocks : {60u, 66u, 100u, 129u})
            for (bool wide_too : {false, true}) {
                hspmm_plan p;
                EXPECT(built(&p, dtype, one_long(64, blocks, blocks), true));
                p.cols = 1600;                                              // (60 to 100 of 100 blocks)
                wide = wide_too;
                for (uint32_t N : {1u, 7u, 16u, 31u}) EXPECT(block_serves(&p, N, true) && block_serves(&p, N, false));
                EXPECT(block_serves(&p, 32u, true) == (!wide_too || blocks == 60u) && block_serves(&p, 32u, false) == !wide_too);
                EXPECT(block_serves(&p, 34u, true) && block_serves(&p, 64u, true) && !block_serves(&p, 33u, true));
                EXPECT(block_serves(&p, 34u, false) == (!wide_too && blocks <= 128u) && block_serves(&p, 64u, false) == (!wide_too && blocks <= 128u));
                p.cfg.block = 1;
                for (uint32_t N : {1u, 32u, 34u, 64u}) EXPECT(block_serves(&p, N, false));
            }
    for (uint32_t longest : {512u, 513u}) {
        hspmm_plan p;
        EXPECT(built(&p, HSPMM_TF32, one_long(64, 400, longest), true) && block_serves(&p, 32u, false) && block_serves(&p, 64u, true) == (longest == 512u));
    }
"""), "block")
