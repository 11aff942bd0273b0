// Scratch of the ids that leave intermediate results in memory for a second launch of the same call and
// that a caller may issue on several streams at once: one block for the eager launches of each stream, and
// one for each (capture, stream) pair, because a recorded launch replays on any stream, beside eager work
// on the one it was recorded on.  Host logic only; no HIP calls.
//
// Blocks are cut from slabs and never given to another owner, since nothing tells when the last launch or
// the last graph that uses a block is gone; kMaxBytes bounds them all.  An owner that gets none runs kernels
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
  std::mutex busy;               // held from a call's first launch to its last: two threads' calls on one
                                 // stream enqueue one after the other
};

class StreamScratch {
 public:
  // A stream's eager blocks: one of 16 MB, which all few-row calls fit, and one of 128 MB for what does not fit it.
  // No call asks for more.
  static constexpr size_t kSmallBlock = size_t{16} << 20, kBlockBytes = size_t{128} << 20;
  static constexpr size_t kFirstSlab = size_t{256} << 20, kSlab = size_t{128} << 20, kMaxBytes = size_t{2} << 30;
  static constexpr size_t kGrain = size_t{512} << 10;         // a capture's block is a multiple of this

  // The owner's block of at least `bytes` (at most kBlockBytes), or null.  `grow(n)` returns n more bytes of
  // device memory or null.
  template <class Grow>
  ScratchBlock* find(uint64_t capture, const void* stream, size_t bytes, Grow&& grow) {
    if (bytes > kBlockBytes) return nullptr;
    std::lock_guard<std::mutex> lock(mutex_);
    for (size_t i = count_; i-- > 0;) {
      ScratchBlock& b = blocks_[i];
      if (b.capture == capture && b.stream == stream && b.bytes >= bytes) return &b;
    }
    if (count_ == kMaxBlocks) return nullptr;
    const size_t size = capture != 0 ? (bytes + kGrain - 1) / kGrain * kGrain : bytes <= kSmallBlock ? kSmallBlock : kBlockBytes;
    unsigned char* from = next_;
    if (left_ >= size) {
      next_ += size;
      left_ -= size;
    } else {
      const size_t slab = total_ == 0 ? kFirstSlab : kSlab;
      if (total_ + slab > kMaxBytes) return nullptr;
      from = static_cast<unsigned char*>(grow(slab));
      if (from == nullptr) return nullptr;
      total_ += slab;
      if (slab - size > left_) next_ = from + size, left_ = slab - size;   // the larger rest serves the next owners
    }
    ScratchBlock& b = blocks_[count_++];
    b.capture = capture, b.stream = stream, b.ptr = from, b.bytes = size;
    return &b;
  }

  // Gets the first slab before any launch; false where there is no memory for it.
  template <class Grow>
  bool reserve(Grow&& grow) {
    std::lock_guard<std::mutex> lock(mutex_);
    if (total_ != 0) return true;
    void* fresh = grow(kFirstSlab);
    if (fresh == nullptr) return false;
    next_ = static_cast<unsigned char*>(fresh);
    left_ = total_ = kFirstSlab;
    return true;
  }

 private:
  static constexpr size_t kMaxBlocks = 4096;
  static_assert(kBlockBytes <= kSlab && kSlab <= kFirstSlab);
  std::mutex mutex_;
  ScratchBlock blocks_[kMaxBlocks];
  size_t count_ = 0;
  unsigned char* next_ = nullptr;
  size_t left_ = 0, total_ = 0;
};

}  // namespace qmm
