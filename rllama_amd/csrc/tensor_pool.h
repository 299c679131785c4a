// tensor_pool.h -- device buffers of freed op-level tensors, kept for later tensors.  Bookkeeping only (no HIP call), so it is checked
// on the CPU; api_ops.hip allocates, waits and frees.
//
// An operation's result is a new tensor, and hipMalloc + hipFree (which waits for the device) cost more than the operation: the
// feed-forward block of 77 rows x 4096 x 11008 through the ops takes 640 us with them and 130 without.
//
// A tensor takes the smallest kept buffer that holds it and is at most twice as large, so tensors of other sizes share buffers.  When the
// pool is full the buffers that have waited longest go first: it follows its user to other sizes.  The limits are those of the 13B
// feed-forward block at up to 512 rows (results of 27, 27, 27 and 10 MiB in f32 mode): over row counts drawn from all of 1 .. 512, 4 % of
// its tensors need a new buffer (f16: none), with buffers at most a quarter larger and 128 MiB 69 % (45 %).
#pragma once

#include <cstddef>

namespace rlh {

class TensorPool {
  public:
    static constexpr size_t kMaxBuffer = (size_t)32 << 20, kMaxTotal = (size_t)192 << 20;
    static constexpr int kMaxCount = 64;

    // A buffer for `bytes` (*capacity: what it holds), or null.
    void *take(size_t bytes, size_t *capacity) {
        int best = -1;
        for (int i = 0; i < count_; i++)
            if (item_[i].bytes >= bytes && item_[i].bytes <= 2 * bytes && (best < 0 || item_[i].bytes <= item_[best].bytes)) best = i;
        if (best < 0) return nullptr;
        *capacity = item_[best].bytes;
        return remove(best);
    }
    // Whether a buffer of that size may be kept, and whether it can be without dropping others first.
    static bool keeps(size_t bytes) { return bytes <= kMaxBuffer; }
    bool room(size_t bytes) const { return count_ < kMaxCount && total_ + bytes <= kMaxTotal; }
    void put(void *p, size_t bytes) { // keeps(bytes) and room(bytes)
        item_[count_++] = {p, bytes};
        total_ += bytes;
    }
    // Hands back the buffer that has waited longest (null: none left); the caller frees it after the work on it.
    void *drop() { return count_ > 0 ? remove(0) : nullptr; }
    size_t total() const { return total_; }
    int count() const { return count_; }

  private:
    struct Item {
        void *p;
        size_t bytes;
    };
    Item item_[kMaxCount]; // in the order they were put
    int count_ = 0;
    size_t total_ = 0;
    void *remove(int i) {
        void *p = item_[i].p;
        total_ -= item_[i].bytes;
        for (count_--; i < count_; i++) item_[i] = item_[i + 1];
        return p;
    }
};

} // namespace rlh
