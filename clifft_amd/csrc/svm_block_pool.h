// svm_block_pool.h -- idle blocks of memory between the calls that use them.
#pragma once

#include <stddef.h>

#include <mutex>
#include <vector>

namespace csvm {

// Keeps at most `bound` bytes.  A call takes the smallest idle block that is
// large enough, so a large one left behind serves small calls too; beyond the
// bound the blocks that were given back longest ago go first, so that the sizes
// in use stay.  Allocating and freeing is the caller's, outside the lock.
class BlockPool {
  public:
    struct Block {
        void* ptr = nullptr;
        size_t bytes = 0;
    };
    explicit BlockPool(size_t bound) : bound_(bound) {}

    // ptr is null where none is large enough
    Block take(size_t bytes) {
        std::lock_guard<std::mutex> lock(mu_);
        size_t best = idle_.size();
        for (size_t i = 0; i < idle_.size(); ++i)
            if (idle_[i].bytes >= bytes && (best == idle_.size() || idle_[i].bytes < idle_[best].bytes)) best = i;
        if (best == idle_.size()) return Block();
        const Block b = idle_[best];
        idle_.erase(idle_.begin() + (ptrdiff_t)best);
        kept_ -= b.bytes;
        return b;
    }
    // returns the blocks to free
    std::vector<Block> give(Block b) {
        std::lock_guard<std::mutex> lock(mu_);
        idle_.push_back(b);
        kept_ += b.bytes;
        size_t n = 0;
        for (; kept_ > bound_; ++n) kept_ -= idle_[n].bytes;
        std::vector<Block> out(idle_.begin(), idle_.begin() + (ptrdiff_t)n);
        idle_.erase(idle_.begin(), idle_.begin() + (ptrdiff_t)n);
        return out;
    }
    size_t kept() {
        std::lock_guard<std::mutex> lock(mu_);
        return kept_;
    }

  private:
    const size_t bound_;
    std::mutex mu_;
    std::vector<Block> idle_;  // the longest idle first
    size_t kept_ = 0;
};

}  // namespace csvm
