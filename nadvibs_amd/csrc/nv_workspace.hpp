// Device blocks kept between calls.  A program solves the same kind of problem
// again and again, and an allocation of some hundred megabytes costs as much as
// the kernels that use it, so a block given back stays, up to `cap` bytes in
// all; beyond that the blocks that lie idle longest are freed.  A block
// belongs to one taker at a time, so calls from several threads, contexts and
// streams never share one.  Host code only: Alloc brings the allocation,
//     static int get(void **p, size_t bytes);   // 0, or an error code
//     static void put(void *p);
#pragma once
#include <cstddef>
#include <mutex>
#include <vector>

namespace nv {

template <typename Alloc> class BlockPool {
public:
    struct Block {
        void *p = nullptr;
        size_t bytes = 0;
    };
    explicit BlockPool(size_t cap) : cap_(cap) {}

    // The smallest idle block of at least `bytes`, or a new one; the idle blocks make room for it
    // when the memory is short.
    int take(size_t bytes, Block *b) {
        std::lock_guard<std::mutex> lock(mu_);
        size_t best = idle_.size();
        for (size_t k = 0; k < idle_.size(); ++k)
            if (idle_[k].bytes >= bytes && (best == idle_.size() || idle_[k].bytes < idle_[best].bytes)) best = k;
        if (best < idle_.size()) {
            *b = idle_[best];
            kept_ -= b->bytes;
            idle_.erase(idle_.begin() + best);
            return 0;
        }
        int e = Alloc::get(&b->p, bytes);
        if (e != 0 && release()) e = Alloc::get(&b->p, bytes);
        b->bytes = e == 0 ? bytes : 0;
        if (e != 0) b->p = nullptr;
        return e;
    }

    // Gives a block back (nothing may use it any more).
    void give(Block b) {
        if (!b.p) return;
        std::lock_guard<std::mutex> lock(mu_);
        if (b.bytes > cap_) {
            Alloc::put(b.p);
            return;
        }
        idle_.push_back(b);
        kept_ += b.bytes;
        while (kept_ > cap_) {
            kept_ -= idle_.front().bytes;
            Alloc::put(idle_.front().p);
            idle_.erase(idle_.begin());
        }
    }

    // Frees the idle blocks; whether there were any.
    bool trim() {
        std::lock_guard<std::mutex> lock(mu_);
        return release();
    }

private:
    bool release() {
        const bool any = !idle_.empty();
        for (const Block &b : idle_) Alloc::put(b.p);
        idle_.clear();
        kept_ = 0;
        return any;
    }

    std::mutex mu_;
    std::vector<Block> idle_;  // longest idle first
    size_t kept_ = 0;
    const size_t cap_;
};

}  // namespace nv
