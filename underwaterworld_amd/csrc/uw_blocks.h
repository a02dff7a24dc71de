// Memory blocks kept between uses, host logic only (the caller allocates and frees).
//
// Sizes are rounded up to eighths of a power of two, so that batches of about one size find each other's
// blocks, and a kept block serves a request of at least four fifths of its size: what a user of a block
// holds beyond its need is at most 1/8 + 1/4 of it (above 64 KiB). A pool of blocks that were taken at up
// to four times the request held that much of live memory in slack.
#pragma once

#include <stddef.h>

struct uw_block {
    void* p;
    size_t bytes;
};

class uw_block_pool {
  public:
    static constexpr size_t kMaxBytes = size_t(256) << 20;
    static constexpr int kMaxCount = 64;

    static size_t rounded(size_t bytes) {
        size_t step = size_t(8) << 10;  // blocks of 64 KiB and below: multiples of 8 KiB
        while (step * 16 <= bytes) step *= 2;
        return (bytes + step - 1) / step * step;
    }

    // The smallest kept block that serves `need` bytes, if there is one.
    bool take(size_t need, uw_block* out) {
        int best = -1;
        for (int i = 0; i < count_; ++i)
            if (kept_[i].bytes >= need && kept_[i].bytes - kept_[i].bytes / 5 <= need &&
                (best < 0 || kept_[i].bytes < kept_[best].bytes))
                best = i;
        if (best < 0) return false;
        *out = remove(best);
        return true;
    }

    // Keeps b and hands what has no room to `drop`, the longest kept first (those would otherwise stay
    // for good if no request meets their sizes).
    template <class Drop>
    void give(uw_block b, Drop drop) {
        if (b.bytes > kMaxBytes) {
            drop(b);
            return;
        }
        while (count_ > 0 && (count_ == kMaxCount || bytes_ + b.bytes > kMaxBytes)) drop(remove(0));
        kept_[count_++] = b;
        bytes_ += b.bytes;
    }

    // Hands out every kept block; whether there was one.
    template <class Drop>
    bool clear(Drop drop) {
        const bool any = count_ > 0;
        while (count_ > 0) drop(remove(count_ - 1));
        return any;
    }

    int count() const { return count_; }
    size_t bytes() const { return bytes_; }

  private:
    uw_block remove(int i) {
        const uw_block b = kept_[i];
        for (--count_; i < count_; ++i) kept_[i] = kept_[i + 1];
        bytes_ -= b.bytes;
        return b;
    }
    uw_block kept_[kMaxCount] = {};  // in the order given
    int count_ = 0;
    size_t bytes_ = 0;
};
