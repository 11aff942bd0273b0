// Scratch of the ids that leave intermediate results in memory for a second launch of the same call and
// that a caller may issue on several streams at once: one block for the eager launches of each stream, and
// one for each (capture, stream) pair, because a recorded launch replays on any stream, beside eager work
// on the one it was recorded on.  Host logic only; no HIP calls.
//
// Blocks are cut from slabs and never given to another owner, since nothing tells when the last launch or
// the last graph that uses a block is gone; a bound holds for them all.  An owner that gets none runs kernels
// that need no scratch.
#pragma once

#include <cstddef>
#include <cstdint>
#include <mutex>

namespace qmm {

struct ScratchBlock {
  uint64_t capture = 0;          // 0: the stream's eager launches
  const void* stream = nullptr;
  void* ptr = nullptr;
  size_t bytes = 0;
  uint32_t next = 0;             // another block (index + 1) whose owner falls on the same place of the table
  std::mutex busy;               // held from a call's first launch to its last: two threads' calls on one
                                 // stream enqueue one after the other
};

// A stream's eager blocks: one of `small` bytes and one of `large` for what does not fit it (no call asks for more).  A
// capture's is what its call needs, a multiple of `grain`.  Slabs: the first, the later ones, all of them together.
struct ScratchLimits {
  size_t small, large, grain, first_slab, slab, most;
};

class StreamScratch {
 public:
  // 16 MB hold all few-row calls.
  static constexpr size_t kSmallBlock = size_t{16} << 20, kBlockBytes = size_t{128} << 20;
  static constexpr size_t kFirstSlab = size_t{256} << 20, kSlab = size_t{128} << 20, kMaxBytes = size_t{2} << 30;
  static constexpr size_t kGrain = size_t{512} << 10;

  explicit StreamScratch(const ScratchLimits& limits = {kSmallBlock, kBlockBytes, kGrain, kFirstSlab, kSlab, kMaxBytes}) : limits_(limits) {}

  // The owner's block of at least `bytes` (at most the limits' `large`), or null.  `grow(n)` returns n more bytes of
  // device memory or null.
  template <class Grow>
  ScratchBlock* find(uint64_t capture, const void* stream, size_t bytes, Grow&& grow) {
    if (bytes > limits_.large) return nullptr;
    std::lock_guard<std::mutex> lock(mutex_);
    uint32_t& place = places_[((reinterpret_cast<uintptr_t>(stream) >> 4) * 0x9E3779B97F4A7C15ull + capture * 0xD1B54A32D192ED03ull) >> 52];
    for (uint32_t i = place; i != 0; i = blocks_[i - 1].next) {
      ScratchBlock& b = blocks_[i - 1];
      if (b.capture == capture && b.stream == stream && b.bytes >= bytes) return &b;
    }
    if (count_ == kMaxBlocks) return nullptr;
    const size_t size = capture != 0 ? (bytes + limits_.grain - 1) / limits_.grain * limits_.grain
                        : bytes <= limits_.small ? limits_.small : limits_.large;
    unsigned char* from = next_;
    if (left_ >= size) {
      next_ += size;
      left_ -= size;
    } else {
      const size_t slab = total_ == 0 ? limits_.first_slab : limits_.slab;
      if (total_ + slab > limits_.most) return nullptr;
      from = static_cast<unsigned char*>(grow(slab));
      if (from == nullptr) return nullptr;
      total_ += slab;
      if (slab - size > left_) next_ = from + size, left_ = slab - size;   // the larger rest serves the next owners
    }
    ScratchBlock& b = blocks_[count_++];
    b.capture = capture, b.stream = stream, b.ptr = from, b.bytes = size, b.next = place;
    place = static_cast<uint32_t>(count_);
    return &b;
  }

  // Gets the first slab before any launch; false where there is no memory for it.
  template <class Grow>
  bool reserve(Grow&& grow) {
    std::lock_guard<std::mutex> lock(mutex_);
    if (total_ != 0) return true;
    void* fresh = grow(limits_.first_slab);
    if (fresh == nullptr) return false;
    next_ = static_cast<unsigned char*>(fresh);
    left_ = total_ = limits_.first_slab;
    return true;
  }

 private:
  static constexpr size_t kMaxBlocks = 4096;
  static_assert(kBlockBytes <= kSlab && kSlab <= kFirstSlab);
  const ScratchLimits limits_;
  std::mutex mutex_;
  ScratchBlock blocks_[kMaxBlocks];
  uint32_t places_[4096] = {};    // the newest block (index + 1) of the owners that fall there
  size_t count_ = 0;
  unsigned char* next_ = nullptr;
  size_t left_ = 0, total_ = 0;
};

}  // namespace qmm
