// Buffers kept between calls and the threads that share a transfer, without HIP: the allocator and the
// worker are template arguments (or_capi.hip's, or the CPU test's).
#pragma once
#include <cstddef>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace orstage {

// Page-locked host buffers (device -1) and device workspaces kept from one call to the next.  A
// taken buffer belongs to one call at a time.  Idle ones of a kind are kept up to kKeep bytes, the oldest
// going first; the kinds do not count together, so that a large workspace pushes out no host buffer, and a
// buffer above the limit is freed when it is given back, before it pushes out anything.  When memory runs out the idle buffers of the kind are
// freed and the allocation is tried again.
//
// Mem: static int alloc(int device, size_t bytes, void **p), 0 for success; static void free(int device, void *p).
template <class Mem> class BufferPool {
 public:
  static constexpr size_t kKeep = (size_t)128 << 20;
  static constexpr size_t kGrain = (size_t)1 << 18;
  struct Buf {
    void *p = nullptr;
    size_t bytes = 0;
    int device = -1; // -1: page-locked host memory
  };

  int take(int device, size_t bytes, Buf &out) {
    {
      std::lock_guard<std::mutex> lock(m_);
      size_t best = idle_.size();
      for (size_t k = 0; k < idle_.size(); ++k)
        if (idle_[k].device == device && idle_[k].bytes >= bytes &&
            (best == idle_.size() || idle_[k].bytes < idle_[best].bytes))
          best = k;
      if (best < idle_.size()) {
        out = idle_[best];
        held(device) -= out.bytes;
        idle_.erase(idle_.begin() + (ptrdiff_t)best);
        return 0;
      }
    }
    out.device = device;
    out.bytes = (bytes + kGrain - 1) / kGrain * kGrain;
    int e = Mem::alloc(device, out.bytes, &out.p);
    if (e && drop(device, 0)) e = Mem::alloc(device, out.bytes, &out.p);
    if (e) out.p = nullptr;
    return e;
  }

  void give(const Buf &b) noexcept {
    if (!b.p) return;
    bool kept = false;
    if (b.bytes <= kKeep) {
      std::lock_guard<std::mutex> lock(m_);
      try {
        idle_.push_back(b);
        held(b.device) += b.bytes;
        kept = true;
      } catch (...) { // no memory to remember it
      }
    }
    if (kept) drop(b.device, kKeep);
    else Mem::free(b.device, b.p);
  }

  // Frees idle buffers of a kind, the oldest first, until at most `keep` bytes of the kind are idle (keep 0, a
  // device: that device's only).  True if any was freed.
  bool drop(int device, size_t keep) noexcept {
    bool any = false;
    for (;;) {
      Buf b;
      {
        std::lock_guard<std::mutex> lock(m_);
        if (held(device) <= keep) return any;
        size_t k = 0;
        while (k < idle_.size() && (idle_[k].device < 0) != (device < 0)) ++k;
        if (keep == 0)
          while (k < idle_.size() && idle_[k].device != device) ++k;
        if (k == idle_.size()) return any;
        b = idle_[k];
        held(device) -= b.bytes;
        idle_.erase(idle_.begin() + (ptrdiff_t)k);
      }
      Mem::free(b.device, b.p);
      any = true;
    }
  }

  void clear() noexcept {
    std::vector<Buf> all;
    {
      std::lock_guard<std::mutex> lock(m_);
      all.swap(idle_);
      held_[0] = held_[1] = 0;
    }
    for (const Buf &b : all) Mem::free(b.device, b.p);
  }

 private:
  size_t &held(int device) { return held_[device < 0 ? 0 : 1]; }
  std::mutex m_;
  std::vector<Buf> idle_; // oldest first
  size_t held_[2] = {0, 0};
};

// Items 0..n-1, taken in turn by the calling thread and up to nt - 1 helpers, each with a worker of its own
// from make(): begin() and end(error) around its items, 0 for success.  A helper that cannot be
// started or cannot begin (no buffer to be had) leaves its share to the others; only the caller's
// begin, an item or an end that fails ends the whole with its error.
template <class Make> int run_team(int nt, size_t n, const Make &make) {
  std::mutex m;
  size_t next = 0;
  int err = 0;
  auto work = [&](bool helper) {
    auto w = make();
    int e = w.begin();
    if (e && helper) return;
    while (!e) {
      size_t k;
      {
        std::lock_guard<std::mutex> lock(m);
        if (err || next >= n) break;
        k = next++;
      }
      e = w.item(k);
    }
    e = w.end(e);
    if (e) {
      std::lock_guard<std::mutex> lock(m);
      if (!err) err = e;
    }
  };
  std::vector<std::thread> team;
  try {
    for (int t = 1; t < nt; ++t) team.emplace_back(work, true);
  } catch (const std::exception &) { // no thread to be had
  }
  work(false);
  for (std::thread &t : team) t.join();
  return err;
}

} // namespace orstage
