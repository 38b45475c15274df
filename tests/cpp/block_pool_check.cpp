// A BlockPool over counted allocations, for the CPU test.
#include <stdint.h>
#include <stdlib.h>

#include <algorithm>

#include "svm_block_pool.h"

using namespace csvm;

namespace {
size_t allocs, live;
BlockPool* pool;
}  // namespace

extern "C" void pool_new(uint64_t bound) {
    pool = new BlockPool(bound);
    allocs = live = 0;
}
extern "C" uint64_t pool_allocs() { return allocs; }
extern "C" uint64_t pool_live() { return live; }
extern "C" uint64_t pool_kept() { return pool->kept(); }
// `n` calls at once of sizes bytes[], given back in the order of `back`;
// returns the smallest of (block size - size wanted), or -1
extern "C" int64_t pool_calls(const uint64_t* bytes, const uint32_t* back, uint32_t n) {
    std::vector<BlockPool::Block> held(n);
    int64_t least = INT64_MAX;
    for (uint32_t i = 0; i < n; ++i) {
        held[i] = pool->take(bytes[i]);
        if (!held[i].ptr) {
            held[i] = {malloc(1), bytes[i]};
            ++allocs, ++live;
        }
        least = std::min<int64_t>(least, (int64_t)held[i].bytes - (int64_t)bytes[i]);
    }
    for (uint32_t i = 0; i < n; ++i)
        for (uint32_t j = i + 1; j < n; ++j)
            if (held[i].ptr == held[j].ptr) least = -1;
    for (uint32_t i = 0; i < n; ++i)
        for (const BlockPool::Block& b : pool->give(held[back[i]])) {
            free(b.ptr);
            --live;
        }
    return least;
}
