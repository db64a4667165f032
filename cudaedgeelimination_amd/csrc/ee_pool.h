// Freed device and page-locked memory of a context's sessions and fleets,
// kept for the next (host-only: what frees a block is given).
#pragma once

#include <cstddef>
#include <mutex>
#include <vector>

namespace ee {

// Bounded, released with the context, one lock around it.  A block comes back
// only after the streams that used it were synchronised.  Allocating and
// freeing it anew took 110 us of a session's 270 us to create and 95 us to
// close (15,836 edge slots), and 1.1 ms for 64 graphs.
//
// A session holds 26 blocks and a fleet 27, so kMaxBlocks are those of two;
// kMaxDevice holds a fleet of 600,000 edge slots (64 graphs with 435,000 take
// 46 MiB) and kMaxHost its witnesses and commits.  What comes back last stays:
// the oldest blocks go where a bound is reached, so sizes that are no longer
// asked for make room for those that are.
class MemoryPool {
 public:
  static constexpr size_t kMaxBlocks = 64, kMaxDevice = size_t{64} << 20, kMaxHost = size_t{8} << 20;
  using FreeBlock = void (*)(bool host, void* ptr);
  explicit MemoryPool(FreeBlock free_block);
  ~MemoryPool();
  MemoryPool(const MemoryPool&) = delete;
  MemoryPool& operator=(const MemoryPool&) = delete;
  // A kept block of at least `bytes` (its size in *got), or null: the
  // smallest that fits, of at most twice the size asked for or 128 KiB.
  void* Take(bool host, size_t bytes, size_t* got);
  // Whether the pool keeps the block; the caller frees it otherwise.
  bool Give(bool host, void* ptr, size_t bytes);
  void Release();  // frees what is kept
  // Frees what every pool of the process keeps: an allocation found no memory.
  static void ReleaseAll();

 private:
  struct Block {
    void* ptr;
    size_t bytes;
    bool host;
  };
  Block Remove(size_t at);  // under mu_
  const FreeBlock free_block_;
  std::mutex mu_;
  std::vector<Block> blocks_;  // the oldest first
  size_t held_[2] = {0, 0};
};

}  // namespace ee
