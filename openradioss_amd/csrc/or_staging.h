// Buffers kept between calls, without HIP: the allocator is a template argument (or_capi.hip's, or a
// counting one in the CPU test).
#pragma once
#include <cstddef>
#include <mutex>
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

} // namespace orstage
