// The kept-block pool over a host allocator: what other threads do while one
// of them waits for the device runs inside the stubbed wait.
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "vkv_blockpool.h"

static std::map<void*, size_t> live;  // every block the "device" holds
static std::mutex live_mu;
static std::function<void()> during_wait;
static bool wait_ok = true, stream_idle = true;
static size_t capacity = ~size_t{0};

#define CHECK(x)                                                  \
  do {                                                            \
    if (!(x)) {                                                   \
      std::printf("line %d: %s\n", __LINE__, #x);                 \
      std::exit(1);                                               \
    }                                                             \
  } while (0)

struct Mem {
  static bool alloc(void** p, size_t bytes, bool* full) {
    std::lock_guard<std::mutex> g(live_mu);
    size_t used = 0;
    for (auto& b : live) used += b.second;
    *full = used + bytes > capacity;
    if (*full) return false;
    *p = std::malloc(1);
    live[*p] = bytes;
    return true;
  }
  static void release(void* p) {
    std::lock_guard<std::mutex> g(live_mu);
    CHECK(live.erase(p) == 1);  // a block of the device, freed once
    std::free(p);
  }
  static bool wait() {
    if (during_wait) {
      auto f = std::move(during_wait);
      during_wait = nullptr;
      f();
    }
    return wait_ok;
  }
  static bool idle() { return stream_idle; }
};
using Pool = vkv::BlockPool<Mem>;
constexpr size_t kMb = size_t{1} << 20;

static size_t live_bytes() {
  size_t n = 0;
  for (auto& b : live) n += b.second;
  return n;
}
static void* fresh(Pool& pool, size_t n) {
  void* p = nullptr;
  CHECK(pool.fresh(0, n, &p));
  return p;
}
static void keep(Pool& pool, int n, size_t bytes) {
  std::vector<void*> b;
  for (int i = 0; i < n; i++) b.push_back(fresh(pool, bytes));
  for (void* p : b) pool.give(p, bytes, 0);
}

// a release while another thread waits: its blocks go back, and the counts
// stay those of the blocks
static void release_during_wait() {
  Pool pool({1024 * kMb, 512 * kMb, 16, 4, 256 * kMb});
  keep(pool, 4, 64 * kMb);
  CHECK(pool.kept(0) == 256 * kMb);
  during_wait = [&] { CHECK(pool.flush(0) == 0); };
  size_t cap = 0;
  CHECK(pool.take(0, 64 * kMb, &cap) == nullptr);
  CHECK(pool.kept(0) == 0 && live_bytes() == 0);
  keep(pool, 3, kMb);  // the limit's loop ends with the blocks it has
  CHECK(pool.kept(0) == 3 * kMb && live_bytes() == 3 * kMb);
  CHECK(pool.flush(0) == 3 * kMb && live.empty());
}

// blocks given back, and others taken, during a wait
static void give_and_take_during_wait() {
  Pool pool({1024 * kMb, 512 * kMb, 16, 4, 256 * kMb});
  keep(pool, 4, 64 * kMb);
  during_wait = [&] {
    keep(pool, 2, 8 * kMb);
    size_t cap = 0;
    during_wait = nullptr;
    void* p = pool.take(0, 8 * kMb, &cap);  // another thread's own wait
    CHECK(p && cap == 8 * kMb);
    Mem::release(p);
  };
  size_t cap = 0;
  void* p = pool.take(0, 64 * kMb, &cap);
  CHECK(p && cap == 64 * kMb);
  CHECK(pool.kept(0) == 3 * 64 * kMb + 8 * kMb);
  Mem::release(p);
  CHECK(pool.kept(0) == live_bytes());
  pool.flush(0);
  CHECK(live.empty());
}

// a wait the device refuses puts the blocks back, not to be used
static void refused_wait() {
  Pool pool({1024 * kMb, 512 * kMb, 16, 4, 256 * kMb});
  keep(pool, 4, 64 * kMb);
  wait_ok = false;
  size_t cap = 0;
  CHECK(pool.take(0, 64 * kMb, &cap) == nullptr && pool.kept(0) == 256 * kMb);
  during_wait = [&] { pool.flush(0); };
  CHECK(pool.take(0, 64 * kMb, &cap) == nullptr && pool.kept(0) == 0 && live.empty());
  wait_ok = true;
}

// the limits hold with blocks in a wait, and when those alone reach them
static void limits() {
  Pool pool({256 * kMb, 128 * kMb, 16, 4, 256 * kMb});
  keep(pool, 2, 128 * kMb);
  during_wait = [&] {
    keep(pool, 1, kMb);  // no room beside the blocks in the wait
    CHECK(pool.kept(0) == 256 * kMb);
  };
  size_t cap = 0;
  void* p = pool.take(0, 128 * kMb, &cap);
  CHECK(p && pool.kept(0) == 128 * kMb);
  keep(pool, 40, kMb);  // 16 blocks at most, the oldest going first
  CHECK(pool.kept(0) == 16 * kMb);
  void* big = fresh(pool, 200 * kMb);
  pool.give(big, 200 * kMb, 0);  // too large to keep
  CHECK(pool.kept(0) == 16 * kMb);
  Mem::release(p);
  pool.flush(0);
  CHECK(live.empty());
}

// a full device gets the kept blocks back before an allocation fails
static void full_device() {
  Pool pool({1024 * kMb, 512 * kMb, 16, 4, 256 * kMb});
  capacity = 512 * kMb;
  keep(pool, 4, 64 * kMb);
  void* p = fresh(pool, 400 * kMb);
  CHECK(pool.kept(0) == 0 && live_bytes() == 400 * kMb);
  void* q = nullptr;
  CHECK(!pool.fresh(0, 200 * kMb, &q) && q == nullptr);
  Mem::release(p);
  capacity = ~size_t{0};
}

// threads that allocate, give back and release at once
static void threads() {
  Pool pool({64 * kMb, 32 * kMb, 16, 4, 16 * kMb});
  std::vector<std::thread> ts;
  for (int t = 0; t < 4; t++)
    ts.emplace_back([&, t] {
      for (int i = 0; i < 2000; i++) {
        const size_t want = (1 + (i * 7 + t) % 5) * kMb;
        size_t cap = want;
        void* p = pool.take(0, want, &cap);
        if (!p) {
          cap = want;
          CHECK(pool.fresh(0, want, &p));
        }
        {
          std::lock_guard<std::mutex> g(live_mu);
          CHECK(live.count(p) && live[p] == cap);
        }
        pool.give(p, cap, 0);
        if (t == 0 && i % 3 == 0) pool.flush(0);
      }
    });
  for (auto& t : ts) t.join();
  CHECK(pool.kept(0) == live_bytes() && pool.kept(0) <= 64 * kMb);
  pool.flush(0);
  CHECK(live.empty());
}

int main(int argc, char** argv) {
  const std::map<std::string, void (*)()> cases = {
      {"release_during_wait", release_during_wait},
      {"give_and_take_during_wait", give_and_take_during_wait},
      {"refused_wait", refused_wait},
      {"limits", limits},
      {"full_device", full_device},
      {"threads", threads}};
  const auto it = cases.find(argc > 1 ? argv[1] : "");
  if (it == cases.end()) return 2;
  it->second();
  std::printf("ok\n");
  return 0;
}
