// Blocks of memory between two owners: objects made and dropped once a request find there what the ones before them had (a
// pinned allocation takes longer than ten decode steps). A block belongs to the device it was made on, whichever device is current
// when its owner lets go of it. It goes back to the runtime when the pool holds kMost blocks or kMostBytes. Any thread may call; a
// block's last user has waited for its launches.
#pragma once
#include <cstddef>
#include <mutex>
#include <vector>

namespace whirl::sampling {

struct Block {
    void* at = nullptr;
    std::size_t bytes = 0;
    int dev = 0;  // the device it was made on
};

// where blocks come from and go to; the first two report failure by throwing
struct BlockMemory {
    int (*device)();  // the current device
    void* (*make)(std::size_t bytes);
    void (*drop)(void*);
};

class BlockPool {
public:
    explicit BlockPool(const BlockMemory& memory) : memory_(memory) { blocks_.reserve(kMost); }
    // at least `bytes` of the current device; fresh: newly made, its contents are anything
    Block take(std::size_t bytes, bool& fresh) {
        const int dev = memory_.device();
        {
            const std::lock_guard<std::mutex> lock(mutex_);
            std::size_t best = blocks_.size();
            for (std::size_t i = 0; i < blocks_.size(); ++i)
                if (blocks_[i].dev == dev && blocks_[i].bytes >= bytes && blocks_[i].bytes / 4 <= bytes && (best == blocks_.size() || blocks_[i].bytes < blocks_[best].bytes)) best = i;
            if (best != blocks_.size()) {
                const Block b = blocks_[best];
                blocks_.erase(blocks_.begin() + static_cast<std::ptrdiff_t>(best));
                held_ -= b.bytes;
                fresh = false;
                return b;
            }
        }
        fresh = true;
        return Block{memory_.make(bytes), bytes, dev};
    }
    // the block's owner has no further use for it; `b` is empty afterwards
    void give(Block& b) {
        if (!b.at) return;
        {
            const std::lock_guard<std::mutex> lock(mutex_);
            if (blocks_.size() < kMost && held_ + b.bytes <= kMostBytes) {
                blocks_.push_back(b);
                held_ += b.bytes;
                b = Block{};
                return;
            }
        }
        drop(b);
    }
    // the same for a block nobody else is to have
    void drop(Block& b) {
        if (b.at) memory_.drop(b.at);
        b = Block{};
    }
    static constexpr std::size_t kMost = 16, kMostBytes = std::size_t{8} << 20;

private:
    BlockMemory memory_;
    std::mutex mutex_;
    std::vector<Block> blocks_;
    std::size_t held_ = 0;
};

}  // namespace whirl::sampling
