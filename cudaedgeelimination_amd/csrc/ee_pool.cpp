#include "ee_pool.h"

#include <algorithm>

namespace ee {
namespace {

// The process's pools, for ReleaseAll.
struct Pools {
  std::mutex mu;
  std::vector<MemoryPool*> all;
};
Pools& AllPools() {
  static Pools* pools = new Pools;  // never destroyed: contexts may outlive exit
  return *pools;
}

}  // namespace

MemoryPool::MemoryPool(FreeBlock free_block) : free_block_(free_block) {
  blocks_.reserve(kMaxBlocks);
  std::lock_guard<std::mutex> lk(AllPools().mu);
  AllPools().all.push_back(this);
}

MemoryPool::~MemoryPool() {
  {
    std::lock_guard<std::mutex> lk(AllPools().mu);
    auto& all = AllPools().all;
    all.erase(std::find(all.begin(), all.end(), this));
  }
  Release();
}

MemoryPool::Block MemoryPool::Remove(size_t at) {
  const Block b = blocks_[at];
  blocks_.erase(blocks_.begin() + static_cast<std::ptrdiff_t>(at));
  held_[b.host] -= b.bytes;
  return b;
}

void* MemoryPool::Take(bool host, size_t bytes, size_t* got) {
  std::lock_guard<std::mutex> lk(mu_);
  size_t best = blocks_.size();
  for (size_t i = 0; i < blocks_.size(); ++i) {
    const Block& b = blocks_[i];
    if (b.host != host || b.bytes < bytes || b.bytes / 2 > std::max<size_t>(bytes, size_t{64} << 10)) continue;
    if (best == blocks_.size() || b.bytes < blocks_[best].bytes) best = i;
  }
  if (best == blocks_.size()) return nullptr;
  const Block b = Remove(best);
  *got = b.bytes;
  return b.ptr;
}

bool MemoryPool::Give(bool host, void* ptr, size_t bytes) {
  const size_t most = host ? kMaxHost : kMaxDevice;
  if (bytes > most) return false;
  Block dropped[kMaxBlocks];
  size_t count = 0;
  {
    std::lock_guard<std::mutex> lk(mu_);
    if (blocks_.size() == kMaxBlocks) dropped[count++] = Remove(0);
    for (size_t i = 0; held_[host] + bytes > most;) {
      if (blocks_[i].host != host) {
        ++i;
      } else {
        dropped[count++] = Remove(i);
      }
    }
    blocks_.push_back({ptr, bytes, host});
    held_[host] += bytes;
  }
  for (size_t i = 0; i < count; ++i) free_block_(dropped[i].host, dropped[i].ptr);
  return true;
}

void MemoryPool::Release() {
  Block dropped[kMaxBlocks];
  size_t count = 0;
  {
    std::lock_guard<std::mutex> lk(mu_);
    for (const Block& b : blocks_) dropped[count++] = b;
    blocks_.clear();
    held_[0] = held_[1] = 0;
  }
  for (size_t i = 0; i < count; ++i) free_block_(dropped[i].host, dropped[i].ptr);
}

void MemoryPool::ReleaseAll() {
  std::lock_guard<std::mutex> lk(AllPools().mu);  // no pool ends meanwhile
  for (MemoryPool* p : AllPools().all) p->Release();
}

}  // namespace ee
