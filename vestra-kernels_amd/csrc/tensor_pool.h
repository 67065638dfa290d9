// Device blocks of freed tensors, kept for the next tensor of the same size:
// hipMallocAsync and hipFreeAsync cost a call about 10 us of host time between
// them on MI355X (vh_linear_run at 16 x 768 x 768 18.3 us a call, 8.7 with the
// pool), a lookup here none that shows.  A block only ever serves its runtime's
// one stream, whose order makes the reuse safe exactly as hipFreeAsync's would.
// The blocks held are bounded: larger ones are not kept, and past the bound
// the ones that have waited longest go back, so that sizes which do not come
// back make room for those that do.  No HIP calls here: `release` frees a block.
#pragma once

#include <cstddef>
#include <list>
#include <mutex>
#include <unordered_map>
#include <vector>

namespace vh {

class TensorPool {
public:
    static constexpr size_t kMaxBlock = (size_t)128 << 20, kMaxHeld = (size_t)512 << 20, kGrain = 512;
    static size_t rounded(size_t bytes) { return (bytes + kGrain - 1) / kGrain * kGrain; }

    // A kept block of exactly `bytes`, or null.
    void *take(size_t bytes) {
        std::lock_guard<std::mutex> lock(mu_);
        auto it = by_size_.find(bytes);
        if (it == by_size_.end()) return nullptr;
        void *p = it->second.back()->p;
        blocks_.erase(it->second.back());
        it->second.pop_back();
        if (it->second.empty()) by_size_.erase(it);
        held_ -= bytes;
        return p;
    }

    // Whether p was kept; if not, it is still the caller's.
    template <class Release>
    bool keep(void *p, size_t bytes, Release release) noexcept {
        if (bytes > kMaxBlock) return false;
        std::lock_guard<std::mutex> lock(mu_);
        try {
            blocks_.push_back(Block{p, bytes});
            try {
                by_size_[bytes].push_back(std::prev(blocks_.end()));
            } catch (...) {
                blocks_.pop_back();
                auto it = by_size_.find(bytes);
                if (it != by_size_.end() && it->second.empty()) by_size_.erase(it);
                return false;
            }
        } catch (...) {
            return false;
        }
        held_ += bytes;
        while (held_ > kMaxHeld) {  // (the newest block alone is below the bound)
            const Block old = blocks_.front();
            auto it = by_size_.find(old.bytes);
            it->second.erase(it->second.begin());
            if (it->second.empty()) by_size_.erase(it);
            blocks_.pop_front();
            held_ -= old.bytes;
            release(old.p);
        }
        return true;
    }

    // Releases every block, if ready() says so once no more can be taken.
    template <class Ready, class Release>
    void give_back(Ready ready, Release release) {
        std::lock_guard<std::mutex> lock(mu_);
        if (blocks_.empty() || !ready()) return;
        for (const Block &b : blocks_) release(b.p);
        blocks_.clear();
        by_size_.clear();
        held_ = 0;
    }

    size_t held() {
        std::lock_guard<std::mutex> lock(mu_);
        return held_;
    }

private:
    struct Block {
        void *p;
        size_t bytes;
    };
    std::mutex mu_;  // tensors may be freed from any host thread
    std::list<Block> blocks_;  // the one that has waited longest first
    std::unordered_map<size_t, std::vector<std::list<Block>::iterator>> by_size_;
    size_t held_ = 0;
};

}  // namespace vh
