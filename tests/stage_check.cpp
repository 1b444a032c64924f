// The kept buffers (openradioss_amd/csrc/or_staging.h) with an allocator that counts, for
// tests/test_staging_pool.py.  Each case returns 0, or the line of the check that failed.
#include "../openradioss_amd/csrc/or_staging.h"

#include <atomic>
#include <cstdint>
#include <cstdlib>
#include <thread>

namespace {
std::atomic<long> g_live{0}, g_allocs{0};
std::atomic<size_t> g_bytes[4]; // host, devices 0..2
std::atomic<size_t> g_room[4];
struct Mem {
  struct Head { size_t bytes; };
  static int alloc(int device, size_t bytes, void **p) {
    if (g_bytes[device + 1] + bytes > g_room[device + 1]) return 2;
    g_bytes[device + 1] += bytes;
    Head *h = (Head *)std::malloc(64); // the bytes themselves are not touched
    h->bytes = bytes;
    *p = h;
    ++g_live;
    ++g_allocs;
    return 0;
  }
  static void free(int device, void *p) {
    g_bytes[device + 1] -= ((Head *)p)->bytes;
    std::free(p);
    --g_live;
  }
};
typedef orstage::BufferPool<Mem> Pool;
constexpr size_t MB = (size_t)1 << 20;
void reset() {
  g_live = 0;
  g_allocs = 0;
  for (int k = 0; k < 4; ++k) { g_bytes[k] = 0; g_room[k] = (size_t)1 << 40; }
}
} // namespace

#define CHECK(x) do { if (!(x)) return __LINE__; } while (0)

extern "C" int pool_keeps_host_buffers_beside_workspaces() {
  reset();
  Pool pool;
  Pool::Buf host[6], ws;
  for (size_t bytes : {Pool::kKeep - MB, Pool::kKeep, Pool::kKeep + MB, 4 * Pool::kKeep})
    for (int call = 0; call < 3; ++call) { // as a nodal call: transfers' buffers back before the workspace
      CHECK(pool.take(0, bytes, ws) == 0);
      for (auto &b : host) CHECK(pool.take(-1, 2 * MB, b) == 0);
      for (auto &b : host) pool.give(b);
      pool.give(ws);
      CHECK(g_bytes[0] == 12 * MB);                     // all six are still there
      CHECK(g_bytes[1] == (bytes <= Pool::kKeep ? bytes : g_bytes[1].load()));
      CHECK(g_bytes[1] <= Pool::kKeep);
    }
  const long before = g_allocs;
  for (auto &b : host) CHECK(pool.take(-1, 2 * MB, b) == 0);
  CHECK(g_allocs == before);
  for (auto &b : host) pool.give(b);
  pool.clear();
  CHECK(g_live == 0);
  return 0;
}

extern "C" int pool_limit_drops_the_oldest() {
  reset();
  Pool pool;
  Pool::Buf b[5];
  for (int k = 0; k < 5; ++k) CHECK(pool.take(-1, (30 + k) * MB, b[k]) == 0);
  for (int k = 0; k < 5; ++k) pool.give(b[k]);
  CHECK(g_bytes[0] == (32 + 33 + 34) * MB); // 30 and 31 are gone: with them 160 MB
  Pool::Buf c;
  CHECK(pool.take(-1, 32 * MB + 1, c) == 0 && c.bytes == 33 * MB); // the smallest that holds it
  pool.give(c);
  Pool::Buf over;
  CHECK(pool.take(-1, Pool::kKeep + 1, over) == 0);
  pool.give(over); // freed at once, nothing pushed out
  CHECK(g_bytes[0] == (32 + 33 + 34) * MB);
  CHECK(pool.take(-1, 0, c) == 0);
  pool.give(c);
  pool.clear();
  CHECK(g_live == 0);
  return 0;
}

extern "C" int pool_frees_idle_buffers_when_memory_runs_out() {
  reset();
  g_room[1] = 100 * MB;
  g_room[0] = 10 * MB;
  Pool pool;
  Pool::Buf a, b, c, h;
  CHECK(pool.take(0, 40 * MB, a) == 0);
  CHECK(pool.take(0, 40 * MB, b) == 0);
  CHECK(pool.take(1, 40 * MB, c) == 0);
  CHECK(pool.take(-1, 8 * MB, h) == 0);
  pool.give(a); pool.give(c); pool.give(h);
  CHECK(pool.take(0, 60 * MB, a) == 0); // 40 idle of this device given up, 40 in use
  CHECK(g_bytes[1] == 100 * MB && g_bytes[2] == 40 * MB && g_bytes[0] == 8 * MB);
  Pool::Buf d;
  CHECK(pool.take(0, 60 * MB, d) != 0 && d.p == nullptr); // nothing idle: the allocator's error
  CHECK(pool.take(-1, 9 * MB, d) == 0 && g_bytes[0] == 9 * MB);
  pool.give(a); pool.give(b); pool.give(d);
  CHECK(g_bytes[1] == 100 * MB && g_bytes[2] == 0); // with the oldest, device 1's, they were 140 MB
  CHECK(pool.take(1, 8 * MB, c) == 0);
  pool.give(c);
  CHECK(pool.drop(0, 0) && g_bytes[1] == 0 && g_bytes[2] == 8 * MB && !pool.drop(0, 0));
  pool.clear();
  CHECK(g_live == 0);
  return 0;
}

extern "C" int pool_threads(int nthreads, int rounds) {
  reset();
  Pool pool;
  std::atomic<int> bad{0};
  std::vector<std::thread> team;
  for (int t = 0; t < nthreads; ++t)
    team.emplace_back([&, t] {
      unsigned s = 12345u + (unsigned)t;
      for (int k = 0; k < rounds; ++k) {
        s = s * 1664525u + 1013904223u;
        const int device = (int)(s >> 16) % 3 - 1;
        const size_t bytes = (size_t)((s >> 8) % 48 + 1) * MB;
        Pool::Buf b;
        if (pool.take(device, bytes, b) || b.device != device || b.bytes < bytes) { ++bad; continue; }
        uintptr_t *mine = (uintptr_t *)b.p + 4; // within the 64 bytes, past the head
        *mine = (uintptr_t)(1000 * t + k);
        std::this_thread::yield();
        if (*mine != (uintptr_t)(1000 * t + k)) ++bad; // another call holds the same buffer
        pool.give(b);
      }
    });
  for (auto &t : team) t.join();
  CHECK(bad == 0);
  CHECK(g_bytes[0] <= Pool::kKeep && g_bytes[1] + g_bytes[2] <= Pool::kKeep);
  pool.clear();
  CHECK(g_live == 0 && g_bytes[0] == 0 && g_bytes[1] == 0 && g_bytes[2] == 0);
  return 0;
}

namespace {
// A worker that counts; helpers are known by their thread.
struct Counter {
  std::atomic<int> *done, *begun, *ended;
  std::thread::id caller;
  int helper_fails, caller_fails, item_fails; // item_fails: from this item on
  int begin() {
    const bool helper = std::this_thread::get_id() != caller;
    if (helper ? helper_fails : caller_fails) return helper ? helper_fails : caller_fails;
    ++*begun;
    return 0;
  }
  int item(size_t k) {
    if ((int)k >= item_fails) return 7;
    std::this_thread::yield();
    ++done[k];
    return 0;
  }
  int end(int e) { ++*ended; return e; }
};
} // namespace

extern "C" int team_takes_every_item_once(int nt, int n) {
  for (int helpers_fail = 0; helpers_fail < 2; ++helpers_fail) {
    std::vector<std::atomic<int>> done((size_t)n);
    std::atomic<int> begun{0}, ended{0};
    const auto me = std::this_thread::get_id();
    const int e = orstage::run_team(nt, (size_t)n, [&] {
      return Counter{done.data(), &begun, &ended, me, helpers_fail ? 5 : 0, 0, n};
    });
    CHECK(e == 0); // also where no helper gets its buffer
    for (auto &d : done) CHECK(d == 1);
    CHECK(begun == ended && begun == (helpers_fail ? 1 : (nt > 0 ? nt : 1)));
  }
  return 0;
}

extern "C" int team_reports_errors() {
  std::vector<std::atomic<int>> done(100);
  std::atomic<int> begun{0}, ended{0};
  const auto me = std::this_thread::get_id();
  CHECK(orstage::run_team(1, 100, [&] { return Counter{done.data(), &begun, &ended, me, 0, 3, 100}; }) == 3);
  for (auto &d : done) CHECK(d == 0);
  CHECK(orstage::run_team(4, 100, [&] { return Counter{done.data(), &begun, &ended, me, 0, 0, 40}; }) == 7);
  for (int k = 0; k < 100; ++k) CHECK(done[(size_t)k] == (k < 40 ? 1 : 0)); // taken in order, none after the failure
  return 0;
}
