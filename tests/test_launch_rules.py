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
    p.dtype = HSPMM_FP16; p.rows = 1 << 20; p.per_column = 1.05;
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
