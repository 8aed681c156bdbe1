// Launch sizes that must fit the dispatch's 32-bit work-item count. Plain C++: the host tests
// compile it without a GPU toolchain.
#pragma once

#include <algorithm>

namespace emc {

// fn(first, count, blocks) for spans of `tiles` tiles in order: a launch of `blocks` blocks covers the
// span's tiles rounded up to whole groups of `group` tiles, blocks_per_tile blocks a tile, and its
// work-items (blocks x threads) stay below 2^32. Spans start at multiples of `group`.
template <typename F>
void for_each_tile_span(long tiles, long group, long blocks_per_tile, long threads, F &&fn) {
    const long most = std::max(1L, ((1L << 32) - 1) / threads / (group * blocks_per_tile)) * group;
    for (long first = 0; first < tiles; first += most) {
        const long count = std::min(most, tiles - first);
        fn(first, count, (unsigned)((count + group - 1) / group * group * blocks_per_tile));
    }
}

}  // namespace emc
