// Device workspace of a handle (a model or a flow), kept from call to call: a
// call's buffers cost a hipMalloc and a hipFree each (tens of microseconds, and
// hipFree waits for the device), more than a small call's kernels.
//
// A block belongs to one call until its work has finished, then it is idle and
// the handle's next call may take it; blocks of a call that ends in an
// exception may have work in flight and are freed at once (hipFree waits for
// it).  Idle bytes are bounded, per handle and over all handles of the process
// (the longest idle blocks of other handles go first), go with their handle, and
// are all given back when an allocation fails.  Mem is the allocator: DevMem
// here, a counted host one in the tests.
#pragma once
#include <stddef.h>
#include <stdint.h>
#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#endif

#include <exception>
#include <mutex>
#include <vector>

namespace nutsgpu {

template <class Mem>
class BlockPool {
 public:
  static constexpr size_t kKeep = (size_t)1 << 30;     // idle bytes of one handle
  static constexpr size_t kKeepAll = (size_t)4 << 30;  // idle bytes of all handles

  BlockPool() {
    std::lock_guard<std::mutex> lock(all().mu);
    all().pools.push_back(this);
  }
  BlockPool(const BlockPool&) = delete;
  BlockPool& operator=(const BlockPool&) = delete;
  ~BlockPool() {
    std::vector<Block> out;
    {
      std::lock_guard<std::mutex> lock(all().mu);
      take_all(out);
      auto& p = all().pools;
      for (size_t i = 0; i < p.size(); ++i)
        if (p[i] == this) { p.erase(p.begin() + i); break; }
    }
    free_blocks(out);
  }

  // a block of at least `bytes`, its size in *got; null when there is no memory
  void* get(size_t bytes, size_t* got) {
    {
      std::lock_guard<std::mutex> lock(all().mu);
      size_t best = idle_.size();
      for (size_t i = 0; i < idle_.size(); ++i)
        if (idle_[i].n >= bytes && idle_[i].n <= 2 * bytes + 65536 &&
            (best == idle_.size() || idle_[i].n < idle_[best].n))
          best = i;
      if (best < idle_.size()) {
        const Block b = take(best);
        *got = b.n;
        return b.p;
      }
    }
    *got = (bytes + 511) & ~size_t(511);
    return alloc(*got);
  }

  // the call is done with a block
  void put(void* p, size_t n) {
    std::vector<Block> out;
    if (n > kKeep || std::uncaught_exceptions() > 0) {
      out.push_back({p, n, 0});
    } else {
      std::lock_guard<std::mutex> lock(all().mu);
      BlockPool* from = nullptr;
      while (held_ + n <= kKeep && all().held + n > kKeepAll && (from = longest_idle()) != nullptr)
        out.push_back(from->take(from->oldest()));
      if (held_ + n <= kKeep && all().held + n <= kKeepAll) {
        idle_.push_back({p, n, ++all().clock});
        held_ += n;
        all().held += n;
      } else {
        out.push_back({p, n, 0});
      }
    }
    free_blocks(out);
  }

  // memory outside the pools, with the idle blocks given back when there is none left
  static void* alloc(size_t bytes) {
    void* p = nullptr;
    if (Mem::alloc(&p, bytes)) return p;
    if (release() == 0) return nullptr;
    return Mem::alloc(&p, bytes) ? p : nullptr;
  }

  // frees every handle's idle blocks; their bytes
  static size_t release() {
    std::vector<Block> out;
    {
      std::lock_guard<std::mutex> lock(all().mu);
      for (BlockPool* b : all().pools) b->take_all(out);
    }
    size_t n = 0;
    for (const Block& b : out) n += b.n;
    free_blocks(out);
    return n;
  }

 private:
  struct Block { void* p; size_t n; uint64_t since; };
  struct All {
    std::mutex mu;  // of this and of every pool's idle blocks
    std::vector<BlockPool*> pools;
    size_t held = 0;
    uint64_t clock = 0;
  };
  static All& all() {
    static All& a = *new All;  // never destroyed: handles may outlive static objects
    return a;
  }
  Block take(size_t i) {
    const Block b = idle_[i];
    idle_.erase(idle_.begin() + i);
    held_ -= b.n;
    all().held -= b.n;
    return b;
  }
  void take_all(std::vector<Block>& out) {
    while (!idle_.empty()) out.push_back(take(idle_.size() - 1));
  }
  size_t oldest() const {
    size_t o = 0;
    for (size_t i = 1; i < idle_.size(); ++i)
      if (idle_[i].since < idle_[o].since) o = i;
    return o;
  }
  // the other pool that holds the longest idle block, or null
  BlockPool* longest_idle() const {
    BlockPool* r = nullptr;
    for (BlockPool* b : all().pools)
      if (b != this && !b->idle_.empty() &&
          (!r || b->idle_[b->oldest()].since < r->idle_[r->oldest()].since))
        r = b;
    return r;
  }
  static void free_blocks(const std::vector<Block>& v) {
    for (const Block& b : v) Mem::free(b.p);
  }
  std::vector<Block> idle_;
  size_t held_ = 0;
};

#ifdef __HIPCC__
struct DevMem {
  static bool alloc(void** p, size_t n) {
    error() = hipMalloc(p, n);
    if (error() == hipSuccess) return true;
    (void)hipGetLastError();
    return false;
  }
  static void free(void* p) { (void)hipFree(p); }
  // of this thread's last alloc
  static hipError_t& error() {
    static thread_local hipError_t e = hipSuccess;
    return e;
  }
};
using DevPool = BlockPool<DevMem>;
#endif

}  // namespace nutsgpu
