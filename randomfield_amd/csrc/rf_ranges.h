// rf_ranges.h -- launches over more blocks than one grid holds (host only).
#pragma once

#include <cstdint>

// A grid dimension is a 32-bit count of work-items, blocks times threads per
// block, not of blocks: the most blocks of one launch.
constexpr int64_t rf_max_blocks(int threads) { return 0xffffffffLL / threads; }

// launch(first, count) over consecutive ranges of n blocks, each within one
// grid; ends at the first result that is not zero (hipSuccess) and returns it.
template <typename F>
auto rf_block_ranges(int64_t n, int threads, F launch) -> decltype(launch((int64_t)0, 0u)) {
    const int64_t most = rf_max_blocks(threads);
    for (int64_t first = 0; first < n; first += most) {
        const auto e = launch(first, (unsigned)(n - first < most ? n - first : most));
        if (e) return e;
    }
    return {};
}
