"""Host code of the kernel families, compiled here without its kernels and with a device memory that runs out at any allocation: streams a
plan can do without (narrow, wide-tile and full-tile kernels), what it answers for feature dimensions in turn, the shape of a row of B in the
entry kernels.  No GPU needed."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hopper_spmm_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
COMMON = r"""
#include "hspmm_plan.hpp"
#include <cstdarg>
#include <set>

static int left;                                    // allocations that succeed
static std::set<void *> held;
extern "C" {
hipError_t hipMalloc(void **p, size_t) { if (left-- <= 0) return hipErrorOutOfMemory; held.insert(*p = std::malloc(64)); return hipSuccess; }
hipError_t hipFree(void *p) { if (p) { held.erase(p); std::free(p); } return hipSuccess; }
hipError_t hipMemcpy(void *to, const void *from, size_t n, hipMemcpyKind kind) { if (kind == hipMemcpyDeviceToHost) std::memset(to, 1, 1), std::memset((char *)to + 1, 0, n - 1); else std::memcpy(to, from, n); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return ""; }
}
namespace hspmm_host {
int fail(int code, const char *, ...) { return code; }
// (as in hspmm_create.hip, without the reserved block)
int plan_alloc(hspmm_plan *p, size_t bytes, void **out) { HSPMM_HIP(hipMalloc(out, bytes)); p->owned.push_back(*out); p->fixed_bytes += bytes; return HSPMM_OK; }
void plan_release(hspmm_plan *p, const void *ptr, size_t bytes)
{
    const auto it = std::find(p->owned.begin(), p->owned.end(), ptr);
    if (it == p->owned.end()) return;
    (void)hipFree(*it); p->owned.erase(it); p->fixed_bytes -= bytes;
}
int scratch_for(hspmm_plan *, hipStream_t, size_t, RunMode, float **) { return HSPMM_ERR_DEVICE; }
}
"""
DRIVER = COMMON + r"""
namespace hspmm {
hipError_t launch_narrow_count(const TileSource &, uint32_t, uint32_t, uint32_t *, uint32_t *, hipStream_t) { return hipSuccess; }
hipError_t launch_narrow_fill(const TileSource &, uint32_t, uint32_t, const uint32_t *, const uint32_t *, uint32_t *, hipStream_t) { return hipSuccess; }
hipError_t launch_spmm_narrow(int, const NarrowArgs &, uint32_t, uint32_t, hipStream_t) { return hipErrorInvalidValue; }
hipError_t launch_spmm_wide(int, const WideArgs &, const WideShape &, hipStream_t, hipEvent_t) { return hipErrorInvalidValue; }
hipError_t launch_wide_fill(const TileSource &, uint32_t, uint32_t, void *, hipStream_t) { return hipSuccess; }
}
namespace hspmm_host {
double entries_expected(const hspmm_plan *, uint32_t) { return 100.0; }
static bool by_entries, by_tile;                    // kernels that would take a launch
bool entries_serve(const hspmm_plan *, uint32_t) { return by_entries; }
double panel_expected(const hspmm_plan *, uint32_t) { return 100.0; }
static int asked;                                   // searches for a feature dimension's kernel
bool panel_serves(const hspmm_plan *, uint32_t) { ++asked; return true; }
double tile_expected(const hspmm_plan *, uint32_t) { return 100.0; }
bool tile_serves(const hspmm_plan *, uint32_t) { return by_tile; }
}

int main()
{
    using namespace hspmm_host;
    for (int which = 0; which < 2; ++which) {
        int needs = -1;
        for (int n = 0; n < 8; ++n) {
            hspmm_plan p;
            // 4096 x 4096 at 10 %, bf16: 32 columns' worth of tiles a window, a sixth of their elements stored
            p.dtype = HSPMM_BF16; p.rows = p.cols = 4096; p.W = 512; p.T = 512 * 146; p.compute_units = 256; p.per_column = 1.4;
            left = n;
            const int rc = which ? build_wide_stream(&p) : build_narrow_stream(&p);
            const bool built = which ? p.wide.built : p.narrow.built;
            if (rc) { std::printf("%d: %d allocations: plan creation fails\n", which, n); return 1; }
            if (built && needs < 0) needs = n;
            if (built != (needs >= 0)) { std::printf("%d: %d allocations: built %d\n", which, n, int(built)); return 1; }
            if (!built && (!held.empty() || !p.owned.empty() || p.fixed_bytes)) { std::printf("%d: %d allocations: %zu not given back\n", which, n, held.size()); return 1; }
            if (built && held.size() != p.owned.size()) { std::printf("%d: %zu left behind\n", which, held.size() - p.owned.size()); return 1; }
            for (void *x : p.owned) (void)hipFree(x);
        }
        {
            hspmm_plan p;
            p.dtype = HSPMM_BF16; p.rows = p.cols = 4096; p.W = 512; p.T = 512 * 146; p.compute_units = 256; p.per_column = 1.4;
            p.caller_cuts = {0, 100, p.T};
            left = 100;
            if ((which ? build_wide_stream(&p) : build_narrow_stream(&p)) || p.wide.built || p.narrow.built || left != 100) { std::printf("%d: built for a plan with its own cuts\n", which); return 1; }
        }
        if (needs < 2) { std::printf("%d: never built\n", which); return 1; }
    }
    hspmm_plan p;
    p.dtype = HSPMM_BF16; p.rows = p.cols = 4096; p.W = 512; p.T = 512 * 146; p.compute_units = 256; p.per_column = 1.4;
    left = 100;
    if (build_wide_stream(&p)) return 1;
    bool first[6], same = true;
    for (int round = 0; round < 10; ++round)
        for (int i = 0; i < 6; ++i) {
            const bool serves = wide_serves(&p, 32u << i);
            if (round == 0) first[i] = serves;
            same &= serves == first[i];
        }
    if (asked != 6 || !same) { std::printf("%d searches for six feature dimensions in turn\n", asked); return 1; }
    // B between two words: launches of the entry kernels are taken from nine features on, those of the full-tile kernels are not
    hspmm_plan q;
    q.dtype = HSPMM_BF16; q.rows = q.cols = 4096; q.W = 512; q.T = 512 * 146; q.compute_units = 256; q.per_column = 1.4;
    left = 100;
    if (build_narrow_stream(&q)) return 1;
    q.narrow.entries = 1677721;
    for (int which = 0; which < 2; ++which) {
        by_entries = which == 0; by_tile = which == 1;
        for (uint32_t N : {1u, 2u, 7u, 8u, 9u, 15u, 16u, 29u, 32u})
            if (!narrow_serves(&q, N, true) || narrow_serves(&q, N, false) != (by_entries && N > 8u)) { std::printf("N = %u: taken %d %d\n", N, int(narrow_serves(&q, N, true)), int(narrow_serves(&q, N, false))); return 1; }
    }
    // many rows and more than a tile of features are the full-tile kernels'
    for (uint32_t rows : {16384u, 20480u}) {
        hspmm_plan m;
        m.dtype = HSPMM_BF16; m.rows = rows; m.cols = 4096; m.W = rows / 8; m.T = rows / 8 * 146; m.compute_units = 256; m.per_column = 1.4;
        left = 100;
        if (build_narrow_stream(&m)) return 1;
        m.narrow.entries = uint64_t(rows) * 410u;
        by_entries = false; by_tile = true;
        for (uint32_t N : {8u, 15u, 16u, 17u, 32u})
            if (narrow_serves(&m, N, true) != (N <= 16u || rows <= 16384u)) { std::printf("%u rows, N = %u: taken %d\n", rows, N, int(narrow_serves(&m, N, true))); return 1; }
    }
    std::printf("ok\n");
    return 0;
}
"""
TILE_DRIVER = COMMON + r"""
namespace hspmm {
uint32_t tile_block_columns(int) { return 64; }
hipError_t launch_tile_count(int, const TileSource &, uint32_t, uint32_t, uint32_t *, uint32_t *, hipStream_t) { return hipSuccess; }
hipError_t launch_tile_fill(int, const TileSource &, uint32_t, uint32_t, const uint32_t *, const uint32_t *, void *, void *, hipStream_t) { return hipSuccess; }
hipError_t launch_spmm_tile(int, const TileArgs &, uint32_t, uint32_t, hipStream_t) { return hipErrorInvalidValue; }
hipError_t launch_fill_zero(void *, size_t, hipStream_t) { return hipErrorInvalidValue; }
}
namespace hspmm_host {
int ensure_arrive(hspmm_plan *, hipStream_t, size_t, RunMode, uint32_t **) { return HSPMM_ERR_DEVICE; }
bool panel_serves(const hspmm_plan *, uint32_t N) { return N >= 16u && N % 4u == 0u; }
}

int main()
{
    using namespace hspmm_host;
    for (uint32_t rows = 1024; rows <= 8192; rows += 256) {
        // fp32, 4096 columns at 12 %, tiles 8 wide, the LDS-panel kernels multiply bf16 parts
        hspmm_plan p;
        p.dtype = HSPMM_TF32; p.elem = 4; p.cw = 8; p.rows = rows; p.cols = 4096; p.W = rows / 8; p.compute_units = 256; p.per_column = 1.5;
        p.panel.built = p.panel.split = true;
        p.T = uint32_t(0.12 * rows * 4096.0 / (8.0 * 1.5));
        const double entries = double(p.T) * 8.0 * 1.5;
        left = 100;
        if (build_tile_stream(&p)) return 1;
        if (entries * 32.0 >= 75e6 && !p.tile.built) { std::printf("%u rows: no stream\n", rows); return 1; }
        if (entries * 32.0 < 0.94 * 75e6 && (p.tile.built || left != 100)) { std::printf("%u rows: a stream that no launch reads\n", rows); return 1; }
        if (p.tile.built) p.tile.entries = uint64_t(entries);
        for (uint32_t N = 4; N <= 64; N += 4) {
            if (tile_serves(&p, N) != (N >= 16 && N <= 32 && entries * N >= 75e6)) { std::printf("%u rows, N = %u: taken %d\n", rows, N, int(tile_serves(&p, N))); return 1; }
            if (tile_leaves(&p, N) != (N > 32 && N < 48 && entries * N >= 75e6)) { std::printf("%u rows, N = %u: left %d\n", rows, N, int(tile_leaves(&p, N))); return 1; }
        }
    }
    std::printf("ok\n");
    return 0;
}
"""
ENTRY_DRIVER = COMMON + r"""
namespace hspmm {
hipError_t launch_entry_count(int, const EntrySource &, uint32_t, uint32_t, uint32_t *, uint32_t *, uint32_t *, uint32_t *, uint32_t *, hipStream_t) { return hipSuccess; }
hipError_t launch_fill_zero(void *, size_t, hipStream_t) { return hipErrorInvalidValue; }
static EntryArgs got;
static uint32_t lane_bytes, lanes;
hipError_t launch_spmm_entries(int, const EntryArgs &ea, uint32_t bytes, uint32_t of, hipStream_t) { got = ea; lane_bytes = bytes; lanes = of; return hipSuccess; }
hipError_t launch_entry_fill(int, const EntrySource &, uint32_t, const uint32_t *, const uint32_t *, uint32_t, const EntryPlaces &, uint32_t *, uint32_t *, uint32_t *,
                             uint32_t *, uint32_t *, void *, hipStream_t) { return hipSuccess; }
}
extern "C" hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *) { return hipErrorInvalidValue; }
namespace hspmm_host {
int ensure_arrive(hspmm_plan *, hipStream_t, size_t, RunMode, uint32_t **) { return HSPMM_ERR_DEVICE; }
bool panel_serves(const hspmm_plan *, uint32_t) { return false; }
double panel_expected(const hspmm_plan *, uint32_t) { return 0.0; }
bool tile_leaves(const hspmm_plan *, uint32_t) { return false; }
}

int main()
{
    using namespace hspmm_host;
    using hspmm::got;
    for (uint32_t cols : {2u, 2048u, 65536u, 1u << 20}) {
        hspmm_plan p;
        p.dtype = HSPMM_BF16; p.rows = 100; p.cols = cols; p.compute_units = 256;
        p.entries.built = p.entries.counted = true;
        for (auto &c : p.entries.classes) { c.n_classes = 1; c.n_groups = 1; }
        for (uint32_t N = 1; N <= 1024; ++N) {
            hspmm::EntryArgs at[2];
            uint32_t loaded[2];
            for (int off : {0, 2}) {
                bool taken = false;
                if (run_entries(&p, reinterpret_cast<const void *>(uintptr_t(4096 + off)), nullptr, N, nullptr, RunMode::kLaunch, &taken) || !taken) { std::printf("N = %u: not run\n", N); return 1; }
                at[off / 2] = got; loaded[off / 2] = got.n_feat_blocks * hspmm::lanes;
                const uint32_t row = 2u * N, bytes = got.block_bytes, blocks = got.n_feat_blocks;
                if (bytes > row || bytes < hspmm::lane_bytes || bytes > hspmm::lane_bytes * hspmm::lanes || bytes * blocks < row) { std::printf("N = %u: %u blocks of %u bytes\n", N, blocks, bytes); return 1; }
                if (blocks > 1u && bytes % 16u != (got.odd ? 14u : 0u)) { std::printf("N = %u, off %d: blocks of %u bytes\n", N, off, bytes); return 1; }
            }
            const bool may = N % 2u && N >= 9u;
            if (at[1].odd || (at[0].odd && !may)) { std::printf("N = %u: whole words %u %u\n", N, at[0].odd, at[1].odd); return 1; }
            // whole words but where a lane of seven features would cost lanes
            const uint32_t bytes = at[1].block_bytes, blocks = at[1].n_feat_blocks, each = (2u * N + blocks - 1u) / blocks;
            const bool full = blocks > 1u && ((each + 1u) & ~15u) + 14u > 16u * (loaded[1] / blocks);
            if (may && (at[0].odd != 0u) != !full) { std::printf("N = %u: whole words %u of %u blocks of %u bytes\n", N, at[0].odd, blocks, bytes); return 1; }
            if (!at[0].odd && (at[0].block_bytes != bytes || at[0].n_feat_blocks != blocks)) { std::printf("N = %u: another shape by the place of B\n", N); return 1; }
            if (cols > 2u && (N == 511u || N == 767u) && at[0].odd) { std::printf("N = %u: %u lanes instead of %u\n", N, loaded[0], loaded[1]); return 1; }
        }
    }
    std::printf("ok\n");
    return 0;
}
"""


@pytest.fixture(scope="module")
def build(tmp_path_factory):
    """Compiles a driver and links it with the host code of kernel families."""
    at = tmp_path_factory.mktemp("streams")
    compile_ = ["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"), "-I", CSRC, "-x", "c++"]

    def make(driver, *families):
        (at / "driver.cpp").write_text(driver)
        sources = [os.path.join(CSRC, "hspmm_%s.hip" % f) for f in families] + [str(at / "driver.cpp")]
        subprocess.run(compile_ + sources + ["-o", str(at / "driver"), "-lpthread"], check=True)
        return str(at / "driver")
    return make


def test_without_memory_without_use_and_asked_in_turn(build):
    run = subprocess.run([build(DRIVER, "narrow", "wide")], stdout=subprocess.PIPE, timeout=60)
    assert run.returncode == 0 and run.stdout == b"ok\n", run.stdout.decode()


def test_full_tile_streams_of_fp32_plans_only_where_a_launch_reads_them(build):
    run = subprocess.run([build(TILE_DRIVER, "tile")], stdout=subprocess.PIPE, timeout=60)
    assert run.returncode == 0 and run.stdout == b"ok\n", run.stdout.decode()


def test_rows_of_the_entry_kernels_by_their_size_and_place(build):
    run = subprocess.run([build(ENTRY_DRIVER, "entries")], stdout=subprocess.PIPE, timeout=60)
    assert run.returncode == 0 and run.stdout == b"ok\n", run.stdout.decode()
