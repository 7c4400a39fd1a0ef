// Which window a wave of the gather kernels walks when (host code): windows dealt out so that waves sweep the columns at about the same time and
// a row of B that one of them brings into an L2 is still there when others ask for it.  A power-law graph's gathers are bound by the L2s' misses:
// walked in the order of the rows a wave is anywhere in the columns at any time, and an L2 keeps what its latest few thousand gathers asked for
// (2^20 vertices, N = 128: 44 % of the reads hit, 0.47 in a model of the L2 alone and 0.69 there with windows of like length side by side).  Tiles of
// a window ascend in their columns and so do its items here.  Gather kernels in the order of the rows / of a schedule, us, one plan over and over: 2^20
// vertices, 16 edges each, fp16, N = 64 252 / 203, 128 480 / 395, 256 949 / 871, 512 2173 / 2078; 2^18, bf16, N = 128 88 / 80.  (Plans of fresh matrices in
// turn, 2^20, N = 128: 482 / 421.)
// Eight waves a compute unit: 4 / 8 / 12 / 16 measured, in a session of their own, 430 / 400 / 400 / 397 us at 2^20, N = 128, 281 / 206 / 204 / 204 at N = 64, 82 / 80 / 88 / 85 at 2^18,
// N = 128, and 354 / 349 / 355 / 359 at N = 512; they have about 350 (2^20) to 540 parts, of 150 to 200 cut windows.
#pragma once
#include <cstdint>
#include <vector>
#include <algorithm>

namespace hspmm {

// A window, or one of the parts that a long one is cut into: tiles first, first + stride, ..
struct ScheduleItem { uint32_t window, first, stride, steps, part, parts; };

struct Schedule {
    std::vector<ScheduleItem> items;          // wave after wave, in the order they are walked
    std::vector<uint32_t> waves;              // first item of every wave (and the end)
};

// rowOffset: first tile of each of W windows, and the end; window_cost: what finishing a window costs, in half tiles.
// A window of more tiles than a wave's share is cut into parts of every so-many-th tile: a part sweeps all of the window's columns.  Items go
// from the longest to the shortest to the wave that has least, which gives every wave its share and has waves walk items of like length
// side by side.
inline Schedule build_schedule(uint32_t W, const uint32_t *rowOffset, uint32_t n_waves, uint32_t window_cost = 3)
{
    Schedule s;
    const uint32_t T = rowOffset[W];
    const uint32_t share = (T + n_waves - 1u) / n_waves;
    // by length, longest first, windows in their order
    std::vector<uint32_t> place(size_t(share) + 2u, 0u);
    auto each = [&](auto fn) {
        for (uint32_t w = 0; w < W; ++w) {
            const uint32_t n = rowOffset[w + 1] - rowOffset[w], parts = (n + share - 1u) / share;
            for (uint32_t k = 0; k < parts; ++k) fn(ScheduleItem{w, rowOffset[w] + k, parts, (n - k + parts - 1u) / parts, k, parts});
        }
    };
    each([&](const ScheduleItem &i) { ++place[share - i.steps + 1u]; });
    for (size_t k = 1; k < place.size(); ++k) place[k] += place[k - 1];
    std::vector<ScheduleItem> sorted(place.back());
    each([&](const ScheduleItem &i) { sorted[place[share - i.steps]++] = i; });
    // waves by what they have: the least only grows
    std::vector<std::vector<uint32_t>> has(1);
    for (uint32_t w = n_waves; w-- > 0;) has[0].push_back(w);
    std::vector<uint32_t> wave_of(sorted.size());
    size_t least = 0;
    s.waves.assign(size_t(n_waves) + 1u, 0u);
    for (size_t i = 0; i < sorted.size(); ++i) {
        while (has[least].empty()) ++least;
        const uint32_t w = has[least].back();
        has[least].pop_back();
        wave_of[i] = w;
        ++s.waves[w + 1u];
        const size_t now = least + 2u * sorted[i].steps + window_cost;
        if (now >= has.size()) has.resize(now + 1u);
        has[now].push_back(w);
    }
    for (uint32_t w = 0; w < n_waves; ++w) s.waves[w + 1u] += s.waves[w];
    std::vector<uint32_t> next(s.waves.begin(), s.waves.end() - 1);
    s.items.resize(sorted.size());
    for (size_t i = 0; i < sorted.size(); ++i) s.items[next[wave_of[i]]++] = sorted[i];
    return s;
}

}  // namespace hspmm
