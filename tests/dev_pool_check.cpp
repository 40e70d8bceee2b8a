// The workspace pool with a counted host allocator of limited size.
#include "../cmdstan_amd/csrc/dev_pool.h"

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <memory>
#include <set>
#include <stdexcept>
#include <thread>

static std::mutex mu;
static size_t used = 0, limit = (size_t)64 << 30, frees = 0;
static uintptr_t next_address = 4096;
static std::set<std::pair<uintptr_t, size_t>> live;

struct HostMem {  // addresses only: no block is touched
  static bool alloc(void** p, size_t n) {
    std::lock_guard<std::mutex> lock(mu);
    if (used + n > limit) return false;
    used += n;
    live.insert({next_address, n});
    *p = reinterpret_cast<void*>(next_address);
    next_address += n + 4096;
    return true;
  }
  static void free(void* p) {
    std::lock_guard<std::mutex> lock(mu);
    auto it = live.lower_bound({reinterpret_cast<uintptr_t>(p), 0});
    if (it == live.end() || it->first != reinterpret_cast<uintptr_t>(p)) std::abort();  // freed twice
    used -= it->second;
    live.erase(it);
    ++frees;
  }
};
using Pool = nutsgpu::BlockPool<HostMem>;

#define CHECK(x)                                              \
  do {                                                        \
    if (!(x)) {                                               \
      std::printf("line %d: %s is false\n", __LINE__, #x);    \
      std::exit(1);                                           \
    }                                                         \
  } while (0)

static const size_t MiB = (size_t)1 << 20;

int main() {
  size_t n = 0, m = 0;
  {  // a block goes back to its own handle, which gets it again; another handle does not
    Pool a, b;
    void* p = a.get(1000, &n);
    CHECK(p && n >= 1000);
    a.put(p, n);
    void* q = b.get(1000, &m);
    CHECK(q != p);
    CHECK(a.get(900, &n) == p);
    a.put(p, n);
    b.put(q, m);
    CHECK(used == 2 * 1024);
  }
  CHECK(used == 0);  // blocks go with their handles
  {  // idle bytes of one handle
    Pool a;
    void* p[3];
    for (auto& x : p) x = a.get(400 * MiB, &n);
    for (auto& x : p) a.put(x, n);
    CHECK(used <= Pool::kKeep);
    void* big = a.get(2 * Pool::kKeep, &n);
    a.put(big, n);
    CHECK(used <= Pool::kKeep);
  }
  CHECK(used == 0);
  {  // idle bytes of the process: the longest idle blocks of other handles go first
    std::unique_ptr<Pool> pools[10];
    void* first[10];
    for (int i = 0; i < 10; ++i) {
      pools[i] = std::make_unique<Pool>();
      first[i] = pools[i]->get(900 * MiB, &n);
      pools[i]->put(first[i], n);
      CHECK(used <= Pool::kKeepAll);
    }
    CHECK(used >= Pool::kKeepAll - 900 * MiB);
    CHECK(pools[9]->get(900 * MiB, &n) == first[9]);
    pools[9]->put(first[9], n);
    CHECK(pools[0]->get(900 * MiB, &n) != first[0]);
    const size_t before = used;
    CHECK(Pool::release() > 0 && used == n && before > used);
    HostMem::free(reinterpret_cast<void*>(live.begin()->first));
    CHECK(Pool::release() == 0);
  }
  CHECK(used == 0);
  {  // an allocation that fails takes every handle's idle blocks, and only those
    Pool a, b;
    void* idle = a.get(800 * MiB, &n);
    void* busy = a.get(100 * MiB, &m);
    a.put(idle, n);
    limit = 1000 * MiB;
    void* p = b.get(900 * MiB, &n);
    CHECK(p && used == 1000 * MiB);
    size_t k = 0;
    CHECK(b.get(MiB, &k) == nullptr);
    CHECK(Pool::alloc(MiB) == nullptr);
    b.put(p, n);
    p = Pool::alloc(500 * MiB);  // memory outside the pools as well
    CHECK(p && used == 600 * MiB);
    HostMem::free(p);
    a.put(busy, m);
    limit = (size_t)64 << 30;
  }
  CHECK(used == 0);
  {  // blocks of a call that ends in an exception are freed, not kept
    Pool a;
    struct Buf {
      Pool& a; void* p; size_t n;
      ~Buf() { a.put(p, n); }
    };
    const size_t f0 = frees;
    try {
      Buf b{a, nullptr, 0};
      b.p = a.get(5000, &b.n);
      throw std::runtime_error("the call failed");
    } catch (const std::exception&) {
    }
    CHECK(frees == f0 + 1 && used == 0);
  }
  {  // several threads on two handles: no block is handed to two calls at once
    Pool a, b;
    std::atomic<bool> twice{false};
    std::mutex hm;
    std::set<void*> held;
    auto work = [&](unsigned s) {
      for (int i = 0; i < 4000; ++i) {
        s = s * 1664525u + 1013904223u;
        Pool& p = (s >> 20) & 1 ? a : b;
        size_t got = 0;
        void* x = p.get(1 + (s >> 8) % 100000, &got);
        {
          std::lock_guard<std::mutex> lock(hm);
          if (!held.insert(x).second) twice = true;
        }
        if (i % 500 == 499) Pool::release();
        {
          std::lock_guard<std::mutex> lock(hm);
          held.erase(x);
        }
        p.put(x, got);
      }
    };
    std::thread t[4];
    for (unsigned k = 0; k < 4; ++k) t[k] = std::thread(work, k + 1);
    for (auto& x : t) x.join();
    CHECK(!twice);
  }
  CHECK(used == 0 && live.empty());
  std::puts("ok");
  return 0;
}
