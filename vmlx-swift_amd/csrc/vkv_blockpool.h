// vkv_blockpool.h -- device blocks kept between objects (DevPool in
// vkv_host.cpp): the bookkeeping, over an allocator type so that it also
// builds and runs without a device.
#pragma once

#include <cstddef>
#include <cstdint>
#include <list>
#include <map>
#include <mutex>

namespace vkv {

// Mem: static functions of the current device
//   bool alloc(void** p, size_t bytes, bool* full)  (*full: out of memory)
//   void release(void* p)     waits for the work queued on the block
//   bool wait()               waits for the whole device; false: refused
//   bool idle()               the calling stream has nothing queued
//
// A block is in one of three places, and its bytes are counted where it is:
// `ready` (the device has been waited for since it was given back),
// `waiting`, or `fenced` while the thread that waits for the device holds it
// with the mutex dropped.  flush() takes what is in the two lists and starts a
// new generation: a thread that comes back from its wait to another
// generation frees its blocks instead of keeping them.
struct PoolLimits {
  size_t bytes;        // kept on a device, fenced blocks included
  size_t block_bytes;  // larger blocks are not kept
  size_t blocks;       // kept on a device, fenced blocks included
  int fence_fits;      // waiting blocks that fit, or
  size_t fence_bytes;  // waiting bytes, at which a busy stream waits too
};

template <class Mem>
class BlockPool {
 public:
  explicit BlockPool(const PoolLimits& l) : lim_(l) {}

  // Bytes kept on the device (none of them in use).
  size_t kept(int dev) {
    std::lock_guard<std::mutex> g(mu_);
    const Device& d = dev_[dev];
    return d.ready.bytes + d.waiting.bytes + d.fenced_bytes;
  }

  // A kept block of at least `want` bytes (*cap: its bytes); nullptr: none.
  void* take(int dev, size_t want, size_t* cap) {
    std::unique_lock<std::mutex> g(mu_);
    Device& d = dev_[dev];
    if (void* p = pick(d.ready, want, cap)) return p;
    int fits = 0;
    fit(d.waiting, want, &fits);
    if (fits == 0 || !(fits >= lim_.fence_fits || d.waiting.bytes >= lim_.fence_bytes || Mem::idle()))
      return nullptr;
    // blocks given back during the wait are not covered by it
    List fenced;
    fenced.splice(d.waiting);
    const size_t n = fenced.bytes, count = fenced.l.size();
    const uint64_t gen = d.generation;
    d.fenced_bytes += n;
    d.fenced_blocks += count;
    g.unlock();
    const bool waited = Mem::wait();
    g.lock();
    d.fenced_bytes -= n;
    d.fenced_blocks -= count;
    if (gen == d.generation) {
      if (waited) {
        d.ready.splice(fenced);
        return pick(d.ready, want, cap);
      }
      fenced.splice(d.waiting);  // refused (another thread captures): as before, the oldest first
      d.waiting.splice(fenced);
      return nullptr;
    }
    g.unlock();
    free_all(fenced);
    return nullptr;
  }

  // Keeps p; what then exceeds the limits goes back, the oldest first.
  void give(void* p, size_t cap, int dev) noexcept {
    if (cap > lim_.block_bytes) {
      Mem::release(p);
      return;
    }
    List node, drop;
    try {
      node.push({p, cap, 0});
      std::lock_guard<std::mutex> g(mu_);
      Device& d = dev_[dev];
      node.l.front().age = age_++;
      d.waiting.splice(node);
      while (d.ready.bytes + d.waiting.bytes + d.fenced_bytes > lim_.bytes ||
             d.ready.l.size() + d.waiting.l.size() + d.fenced_blocks > lim_.blocks) {
        if (d.ready.l.empty() && d.waiting.l.empty()) break;  // (the rest is fenced)
        const bool r = !d.ready.l.empty() &&
                       (d.waiting.l.empty() || d.ready.l.front().age < d.waiting.l.front().age);
        drop.take_front(r ? d.ready : d.waiting);
      }
    } catch (...) {  // no host memory for the record: nothing was linked yet
      Mem::release(p);
      return;
    }
    free_all(drop);
  }

  // Frees every kept block of the device; returns their bytes.
  size_t flush(int dev) {
    List all;
    {
      std::lock_guard<std::mutex> g(mu_);
      Device& d = dev_[dev];
      all.splice(d.ready);
      all.splice(d.waiting);
      d.generation++;
    }
    const size_t n = all.bytes;
    free_all(all);
    return n;
  }

  // New memory; a device that is full gets the kept blocks back first.
  bool fresh(int dev, size_t bytes, void** p) {
    bool full = false;
    if (Mem::alloc(p, bytes, &full)) return true;
    if (!full) return false;
    flush(dev);
    return Mem::alloc(p, bytes, &full);
  }

 private:
  struct Block {
    void* p;
    size_t cap;
    uint64_t age;
  };
  // Blocks, oldest first, and their bytes.
  struct List {
    std::list<Block> l;
    size_t bytes = 0;
    void push(const Block& b) {
      l.push_back(b);
      bytes += b.cap;
    }
    void splice(List& o) {
      l.splice(l.end(), o.l);
      bytes += o.bytes;
      o.bytes = 0;
    }
    void take_front(List& o) {
      bytes += o.l.front().cap;
      o.bytes -= o.l.front().cap;
      l.splice(l.end(), o.l, o.l.begin());
    }
  };
  struct Device {
    List ready, waiting;
    size_t fenced_bytes = 0, fenced_blocks = 0;
    uint64_t generation = 0;
  };

  // The smallest block of at least `bytes` and at most an eighth more, and
  // how many such there are.
  typename std::list<Block>::iterator fit(List& s, size_t bytes, int* fits) {
    auto best = s.l.end();
    int n = 0;
    for (auto it = s.l.begin(); it != s.l.end(); ++it) {
      if (it->cap < bytes || it->cap > bytes + bytes / 8 + 4096) continue;
      n++;
      if (best == s.l.end() || it->cap < best->cap) best = it;
    }
    *fits = n;
    return best;
  }
  void* pick(List& s, size_t bytes, size_t* cap) {
    int fits = 0;
    auto it = fit(s, bytes, &fits);
    if (!fits) return nullptr;
    void* p = it->p;
    *cap = it->cap;
    s.bytes -= it->cap;
    s.l.erase(it);
    return p;
  }
  static void free_all(List& s) {
    for (Block& b : s.l) Mem::release(b.p);
    s.l.clear();
    s.bytes = 0;
  }

  const PoolLimits lim_;
  std::mutex mu_;
  std::map<int, Device> dev_;
  uint64_t age_ = 0;
};

}  // namespace vkv
