// or_capi.hip -- kernels and C ABI of the MI355X explicit hex / Q4 path (gfx950).
//
// Per cycle, on one stream, with every scalar kept on the device:
//   k_hex_forces : SFORC3 chain per 8-node hex -> 4-word skyline rows
//   k_q4_forces  : CFORC3 chain per Q4 shell   -> 8-word skyline rows
//                  (both fold their element time steps into one device word with an
//                  integer atomicMin on the FP64 bit pattern: min is exact, so the
//                  result does not depend on block order)
//   k_elements   : both, in one launch, when a model or batch has more than one family or form
//   k_node_update: ASSPAR4 fixed-order segmented sum per node (hex rows, then Q4 rows,
//                  the FILLCNE order), DT2 pipeline, ACCELE, BCS10, FIXVEL, VELOCITY,
//                  DEPLA; thread 0 advances the cycle scalars (double-buffered by parity)
//
// The file is compiled twice: once with the compiler's default instruction scheduler
// (everything), and once with -DOR_ILP_TU and the ILP-first scheduler
// (-mllvm -amdgpu-sched-strategy=max-ilp), which only provides the element-kernel launches
// of variants 2 and 3 (or_ilp_elements).  Scheduling reorders instructions and never changes
// an operation or its operands, so every variant gives the same bits.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <initializer_list>
#include <mutex>
#include <thread>
#include <numeric>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/or_gpu.h"
#include "or_assembly.h"
#include "or_hex.h"
#include "or_q4.h"
#include "or_staging.h"

using namespace orgpu;

namespace {

thread_local std::string g_err;

int fail(int code, const std::string &msg) {
  g_err = msg;
  return code;
}

#define OR_HIP(call)                                                                         \
  do {                                                                                       \
    hipError_t e_ = (call);                                                                  \
    if (e_ != hipSuccess)                                                                    \
      return fail(OR_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(e_));            \
  } while (0)

constexpr int kBlock = 256;
constexpr double kNoEnd = 1.0e300; // end time of a model advanced by or_model_run

// Launch variants of the element kernels.  Variant v picks the instruction scheduler (default
// for v < 2, ILP-first for v >= 2) and, in the split form, the minimum number of waves per SIMD the
// register allocation is built for (two for even v, three for odd v; a wave's register budget is 512 /
// waves VGPRs and AGPRs together).  Where both budgets give the same kernel, the odd variant is
// the even one: FP64 (three waves spill 316 bytes a lane and take twice the time) and the split
// form's hexes under the default scheduler (156 registers, three waves in either).
// Every element workgroup is one tile of kTile elements, the unit of the LDS assembly.
// Every variant runs the same arithmetic, so the choice (or_model_set_variant,
// or_model_autotune, or_batch_autotune) changes speed only, never a result bit.
constexpr int kVariants = 4;
constexpr int kTile = orasm::kTile;
static_assert(kTile == kBlock, "element tiles and node blocks share the workgroup size");
// The variant that is built for variant v of a family (0: hexes, 1: shells).
constexpr int built_variant(bool fp64, int family, int v) {
  if (fp64) return v & 2;
  return family == 0 && v == 1 ? 0 : v;
}
// Waves per SIMD of built variant v.
constexpr int variant_waves(bool fp64, int v) { return fp64 ? 2 : 2 + (v & 1); }

// MSTOP codes (include/or_gpu.h): an element's non-positive Jacobian, a time step <= 0
constexpr int32_t kMstopJacobian = 1, kMstopTimeStep = 2;

// node code bits (include/or_gpu.h)
constexpr int32_t kTX = 4, kTY = 2, kTZ = 1, kRX = 32, kRY = 16, kRZ = 8, kIX = 256, kIY = 128, kIZ = 64;

// Assembly of the resident model (plan in or_assembly.h).  The rows of a node that
// lead its ASSPAR4 order and whose elements share the tile of its first element are
// summed in that tile's LDS from zero and stored once, in FP64, as the node's prefix
// (pre[n][W]); the node kernel starts from the prefix and adds the node's remaining
// ("rest") rows in order.  Rest rows are stored node after node (CSR, rs[n] ..
// rs[n + 1] - 1), W words each in the storage type: W = 3 (fx, fy, fz) for hexes,
// 6 (plus mx, my, mz) for shells.  Every node with hex rows has a hex prefix; a node
// with shell rows has a shell prefix only when it has no hex rows (its sum does not
// start with a shell row otherwise).  The stiffness words (FSKY 7, 8) have no reader
// on this path (element time step, NODADT=0, no interfaces), so the resident rows
// leave them out; the group drop-ins write them.
constexpr int kHexRowWords = 3; // fx, fy, fz
constexpr int kQ4RowWords = 6;  // fx, fy, fz, mx, my, mz
typedef uint32_t v4u __attribute__((ext_vector_type(4))); // a prefix's 8 LDS sources

// Workgroups of a launch are dispatched to the 8 XCDs in turn (workgroup b runs on
// XCD b mod 8), each XCD with its own L2.  Element kernels renumber their workgroups
// so that each XCD works through one contiguous eighth of the element range:
// neighbouring elements, which share nodes, then gather through the same L2.
// The map is a bijection of [0, nb).
__device__ __forceinline__ int64_t xcd_contiguous_block(int64_t b, int64_t nb) {
  constexpr int64_t kXcd = 8;
  const int64_t q = nb / kXcd, r = nb % kXcd;
  const int64_t x = b % kXcd, j = b / kXcd;
  return x * q + (x < r ? x : r) + j;
}

// Pointers into HBM as the kernels use them: typed in the global address space, so
// that their loads and stores compile to global (not flat) memory instructions even
// though the kernels read them from a descriptor in memory.
template <typename T> using gptr = __attribute__((address_space(1))) T *;
typedef double v2d __attribute__((ext_vector_type(2))); // 16-byte load / store unit
template <typename T> using cptr = const __attribute__((address_space(4))) T *; // read-only: scalar loads
template <typename T> __device__ __forceinline__ gptr<T> to_global(T *p) { return (gptr<T>)p; }
template <typename T> __device__ __forceinline__ gptr<T> to_global(const void *p) { return (gptr<T>)(T *)p; }

// A model's cycle scalars, read field by field with global loads: a flat load among
// an element's global loads makes the compiler wait for all of them at its first use.
static_assert(offsetof(DevTime, ncycle) == 40 && offsetof(DevTime, mstop) == 48 && offsetof(DevTime, done) == 52,
              "DevTime layout");
__device__ __forceinline__ DevTime load_time(const DevTime *t) {
  const gptr<const double> d = to_global<const double>(t);
  DevTime r;
  r.tt = d[0]; r.dt1 = d[1]; r.dt2 = d[2]; r.dt12 = d[3]; r.dt2old = d[4];
  r.ncycle = to_global<const int64_t>(t)[5];
  const gptr<const int32_t> w = to_global<const int32_t>(t);
  r.mstop = w[12]; r.done = w[13];
  return r;
}
__device__ __forceinline__ double time_dt2(const DevTime *t) { return to_global<const double>(t)[2]; }
__device__ __forceinline__ int32_t time_done(const DevTime *t) { return to_global<const int32_t>(t)[13]; }

template <typename S> struct HexPtrs {
  gptr<const int32_t> conn;  // [8][ne]
  gptr<const int32_t> rest;  // [8][ne] rest row of the corner, or -1 (summed in LDS)
  gptr<S> sig;               // [6][ne]
  gptr<S> eint, rho, pla, epsd, offg, qvis;
  gptr<const S> vol0;
  int64_t ne;
};

template <typename S> struct Q4Ptrs {
  gptr<const int32_t> conn;  // [4][ne]
  gptr<const int32_t> rest;  // [4][ne] rest row of the corner, or -1 (summed in LDS)
  gptr<S> offg, thk;
  gptr<const S> thke;
  gptr<S> forc, mom, gstr, hourg, eint, epsd; // [5][ne] [3][ne] [8][ne] [5][ne] [2][ne] [ne]
  gptr<S> sig, pla, epsd_ip;                  // [npt][5][ne] [npt][ne] [npt][ne] (epsd_ip null when israte=0)
  int64_t ne;
};

struct NodePtrs {
  double *xv;            // [nn][6] x,y,z,vx,vy,vz
  double *vr;            // [nn][4] rotational velocity (padded) or null
  double *d;             // [nn][3]
  const double *ms;      // [nn]
  const double *in;      // [nn] or null
  const int32_t *code;   // [nn]
  const double *vimp;    // [nn][3]
  const int32_t *deg_h, *deg_q;    // [nn] rows of each node per family (null when the family is absent)
  const int32_t *rs_h, *rs_q;      // [nn + 1] first rest row of each node per family
  const double *pre_h, *pre_q;     // [nn][3], [nn][6] FP64 prefixes
  double *wext;                    // [2][nn] external work of the node's imposed DOFs, and the part
                                   // each cycle defers to the next (FIXVEL's VEL(4,N)), or null
  int64_t nn;
};

// One model as the cycle kernels see it: pointers into its resident arrays, its
// parameters and its cycle scalars.  Held in device memory, one per model (and one
// per slot of a batch); a launch covers any number of models through a tile list.
struct ModelDev {
  // hexes; element state in the model's storage type (double, or float in the split form)
  const int32_t *hconn, *hrest;
  const int32_t *hfr_start, *hfr_node; // prefixes of each hex tile: [ntiles + 1], [nfr]
  const uint16_t *hfr_src;              // [nfr][8] LDS sources of each prefix
  void *hsig, *heint, *hrho, *hpla, *hepsd, *hoffg, *hqvis;
  const void *hvol0;
  int64_t neh;
  // Q4 shells
  const int32_t *qconn, *qrest;
  const int32_t *qfr_start, *qfr_node;
  const uint16_t *qfr_src;
  void *qoffg, *qthk, *qforc, *qmom, *qgstr, *qhourg, *qeint, *qepsd, *qsig, *qpla, *qepsdip;
  const void *qthke;
  int64_t neq;
  NodePtrs nd;
  void *rowh, *rowq;          // rest rows (storage type)
  double *preh, *preq;        // prefixes (written by the element kernels)
  DevTime *ts;                // [2] cycle scalars, by cycle parity
  unsigned long long *dtmin;  // [2] element time-step minimum (FP64 bits), by parity
  int *flags;                 // bit 0: an element reported MSTOP
  double *ecrit;              // [5][nn] per-node kinetic and momentum terms of ECRIT on output cycles, or null
  const int32_t *th_slot;     // [nn] the node's row in th_node, or -1 (time history), or null
  double *th_node;            // [rows][18] D, V, A, VR, AR, X of the time-history nodes on output cycles
  double *ehou_h, *ehou_q;    // per tile: its elements' hourglass energy summed over the cycles, or null
  double *dtel_h, *dtel_q;    // per-element time-step candidates on output cycles (storage order), or null
  double dtmx;                // DTMX
  double tend;                // the model stops after the cycle whose time reaches tend
  HexConsts hc;
  Q4Consts qc;
};

// One block of a cycle launch: consecutive elements (the launch's workgroup size) or
// kBlock consecutive nodes of one model.
struct Tile {
  int32_t model; // index in the launch's ModelDev array
  int32_t first; // first element (node) of the block
};

template <typename S> __device__ __forceinline__ HexPtrs<S> hex_ptrs(const ModelDev &M) {
  return HexPtrs<S>{to_global(M.hconn), to_global(M.hrest), to_global<S>(M.hsig), to_global<S>(M.heint),
                    to_global<S>(M.hrho), to_global<S>(M.hpla), to_global<S>(M.hepsd), to_global<S>(M.hoffg),
                    to_global<S>(M.hqvis), to_global<const S>(M.hvol0), M.neh};
}
template <typename S> __device__ __forceinline__ Q4Ptrs<S> q4_ptrs(const ModelDev &M) {
  return Q4Ptrs<S>{to_global(M.qconn), to_global(M.qrest), to_global<S>(M.qoffg), to_global<S>(M.qthk),
                   to_global<const S>(M.qthke), to_global<S>(M.qforc), to_global<S>(M.qmom), to_global<S>(M.qgstr),
                   to_global<S>(M.qhourg), to_global<S>(M.qeint), to_global<S>(M.qepsd), to_global<S>(M.qsig),
                   to_global<S>(M.qpla), to_global<S>(M.qepsdip), M.neq};
}

__device__ __forceinline__ unsigned long long dbits(double x) { return (unsigned long long)__double_as_longlong(x); }
__device__ __forceinline__ double bitsd(unsigned long long b) { return __longlong_as_double((long long)b); }

template <int TB> __device__ __forceinline__ double block_min(double v) {
  __shared__ double red[TB / 64];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    double o = __shfl_xor(v, off, 64);
    v = (o < v) ? o : v;
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) red[wid] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < TB / 64; ++w) v = (red[w] < v) ? red[w] : v;
  }
  return v;
}

__device__ __forceinline__ void load_node(gptr<const double> xv, int64_t n, double &x, double &y, double &z,
                                          double &vx, double &vy, double &vz) {
  gptr<const v2d> p = (gptr<const v2d>)(xv + 6 * n);
  const v2d a = p[0], b = p[1], q = p[2];
  x = a.x; y = a.y; z = b.x; vx = b.y; vy = q.x; vz = q.y;
}

// ---------------------------------------------------------------- tile assembly
// The element chains leave every corner's W row words in LDS, in the storage type (the
// value a row holds): corner k, word w of the tile's element t at lds[(k * W + w) * kTile + t].
// After a barrier the tile writes its rest rows from there and sums its prefixes.
template <typename S, int W>
__device__ __forceinline__ void lds_corner(S *lds, int k, const S (&w)[W]) {
#pragma unroll
  for (int c = 0; c < W; ++c) lds[(k * W + c) * kTile + threadIdx.x] = w[c];
}

// The tile's assembly after its element chains: this thread's rest rows (the corners of its
// element whose rest row is >= 0, written from LDS) and the tile's prefixes (each summed in
// row order from zero in FP64, ASSPAR4's running sum A = A + FSKY, stored in pre[n][W]),
// thread t taking prefixes t, t + kTile, ...  The indices are loaded before the tile's
// barrier (prefetch), so that their latency overlaps the wait for the tile's other waves.
template <typename S, int W, int NK> struct TileAssembly {
  int32_t rest[NK];
  int32_t j, j1, node;
  v4u src;

  // The tile's range of the prefix list, read at the kernel's start (uniform: scalar loads),
  // so that prefetch needs no load before its own.
  __device__ __forceinline__ void range(const int32_t *fr_start, int64_t tile) {
    const cptr<int32_t> p = (cptr<int32_t>)(fr_start + tile);
    j = p[0] + (int32_t)threadIdx.x;
    j1 = p[1];
  }

  __device__ __forceinline__ void prefetch(gptr<const int32_t> restp, int64_t ne, int64_t i,
                                           gptr<const int32_t> fr_node, gptr<const v4u> fr_src) {
    __asm__ __volatile__("" ::: "memory"); // where the caller puts it, not hoisted
#pragma unroll
    for (int k = 0; k < NK; ++k) rest[k] = (i < ne) ? restp[(int64_t)k * ne + i] : -1;
    if (j < j1) {
      node = fr_node[j];
      src = fr_src[j];
    }
  }

  __device__ __forceinline__ void finish(const S *lds, gptr<S> rows, gptr<const int32_t> fr_node,
                                         gptr<const v4u> fr_src, gptr<double> pre) {
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      if (rest[k] >= 0) {
        const gptr<S> w = rows + (int64_t)rest[k] * W;
#pragma unroll
        for (int c = 0; c < W; ++c) w[c] = lds[(k * W + c) * kTile + threadIdx.x];
      }
    }
    for (; j < j1; j += kTile) {
      double a[W];
#pragma unroll
      for (int c = 0; c < W; ++c) a[c] = 0.0;
#pragma unroll
      for (int r = 0; r < orasm::kRunCap; ++r) {
        const uint32_t u = (src[r >> 1] >> (16 * (r & 1))) & 0xFFFFu;
        if (u == orasm::kNoSrc) break;
        const int base = (int)(u >> 8) * W * kTile + (int)(u & 0xFFu);
#pragma unroll
        for (int c = 0; c < W; ++c) a[c] = a[c] + double(lds[base + c * kTile]);
      }
      const gptr<double> p = pre + (int64_t)node * W;
#pragma unroll
      for (int c = 0; c < W; ++c) p[c] = a[c];
      if (j + kTile < j1) { // the tile holds more prefixes than threads
        node = fr_node[j + kTile];
        src = fr_src[j + kTile];
      }
    }
  }
};

// The element time-step minimum of a tile: each wave's minimum goes to red[] before the
// tile's barrier, and after it the first thread folds them into the model's word with an
// integer atomicMin on the FP64 bits (min is exact, so the order does not matter).
__device__ __forceinline__ void wave_min_to(double *red, double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const double o = __shfl_xor(v, off, 64);
    v = (o < v) ? o : v;
  }
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
}
template <int TB> __device__ __forceinline__ void tile_min_commit(const double *red, unsigned long long *word) {
  if (threadIdx.x == 0) {
    double v = red[0];
#pragma unroll
    for (int w = 1; w < TB / 64; ++w) v = (red[w] < v) ? red[w] : v;
    atomicMin(word, dbits(v));
  }
}

// The hourglass energy (EHOU) of a tile's elements: each element stores its EHOU in the tile's
// LDS as soon as it is known (no register holds it through the rest of the chain); after the
// tile's barrier the first wave sums them in a fixed order (per lane its elements in order,
// then a shuffle tree) and adds the sum to the tile's accumulator, which only this tile
// writes, so the sum is the same on every run.
template <int TB, typename R> __device__ __forceinline__ void tile_ehou_commit(const R *eh, int64_t first, int64_t ne,
                                                                               double *acc) {
  if (threadIdx.x < 64) {
    double v = 0.0;
#pragma unroll
    for (int k = 0; k < TB / 64; ++k) {
      const int t = threadIdx.x + 64 * k;
      if (first + t < ne) v = v + double(eh[t]);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = v + __shfl_xor(v, off, 64);
    if (threadIdx.x == 0) *to_global(acc) = *to_global(acc) + v;
  }
}

// ---------------------------------------------------------------- element state in LDS
// The element state that the hex chain's material phase reads (SIG(6), EINT, RHO, VOL0, PLA, EPSD,
// QVIS) is copied from HBM to LDS by the wave itself at the start of the chain, with
// global-to-LDS loads that occupy no registers: the copy is in flight during the gather and the
// geometry.  It uses the LDS words in which the same threads leave their force rows at the
// chain's end (24 words per element):
// word a of the tile's element t sits at lds[a * kTile + t], and each wave copies and reads
// its own 64 elements only, so the wave's own wait for its loads orders the copy before its reads
// and its reads precede its writes of the rows.
typedef __attribute__((address_space(3))) void *lds_void;
typedef __attribute__((address_space(3))) char *lds_char;

// One state word (src) of the wave's 64 elements into word a of the tile's LDS.
template <typename S>
__device__ __forceinline__ void stage_word(S *lds, int a, gptr<const S> src, int64_t first, int64_t ne) {
  constexpr int D = sizeof(S) / 4; // dwords per word
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t wfirst = first + 64 * w;
#pragma unroll
  for (int h = 0; h < D; ++h) {
    const int d = h * 64 + l; // dword of the wave's slice
    if (wfirst + d / D < ne)
      __builtin_amdgcn_global_load_lds((gptr<void>)((gptr<const char>)(src + wfirst) + 4 * d),
                                       (lds_void)((char *)(lds + a * kTile + 64 * w) + 256 * h), 4, 0, 0);
  }
}

// The wave's global-to-LDS loads have landed (they count as vector memory loads).
__device__ __forceinline__ void wait_staged() { __asm__ __volatile__("s_waitcnt vmcnt(0)" ::: "memory"); }

// The tables of or_math.h in LDS, one copy for each wave, read from memory when the wave first
// needs them.  A look-up in memory costs a wave 500-600 clocks, and a plastic shell point makes
// ten in one chain: the tube of 72,000 shells, deep in plasticity, takes 38 us instead of 42.
// A wave without a plastic point reads no table (read at the start by every workgroup, they
// cost an elastic plate of 2,304 shells 0.5 us of 16.7).
__device__ __align__(256) constexpr ormath::MathTab kMathTab = ormath::make_math_tab();
struct WaveTab {
  const __attribute__((address_space(3))) double *t;
  bool have; // the same in every lane
  __device__ __forceinline__ explicit WaveTab(double *copies)
      : t((const __attribute__((address_space(3))) double *)(copies +
                                                            ormath::kTabWords * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6))),
        have(false) {}
  // Called by whole waves: the copy is read by all lanes when any of them needs it.
  __device__ __forceinline__ void need(bool cond) {
    if (have || !__any(cond)) return;
    constexpr int kBytes = (int)sizeof(ormath::MathTab);
    static_assert(kBytes % 16 == 0, "16-byte loads");
    const int l = 16 * (threadIdx.x & 63);
    const gptr<const char> src = (gptr<const char>)(gptr<const void>)(const void *)&kMathTab;
#pragma unroll
    for (int o = 0; o < kBytes; o += 1024)
      if (o + l < kBytes) __builtin_amdgcn_global_load_lds((gptr<void>)(src + o + l), (lds_void)((lds_char)t + o), 16, 0, 0);
    wait_staged();
    have = true;
  }
  __device__ __forceinline__ double lg(int i, int k) const { return t[3 * i + k]; }
  __device__ __forceinline__ double ex(int j, int k) const { return t[ormath::kLogWords + 2 * j + k]; }
};

// The tables that a shell chain of type R reads (the split form has none).
template <typename R> __device__ __forceinline__ auto chain_tab(double *copies) {
  if constexpr (sizeof(R) == 8) return WaveTab(copies);
  else return ormath::GlobalTab{};
}

// A tile's LDS: the rows (and the staged state before them), the waves' tables (FP64 shells),
// EHOU per element.
template <typename R, typename S, bool EH, bool TAB> struct TileLds {
  alignas(16) S rows[24 * kTile];
  alignas(16) double tab[TAB ? kTile / 64 * ormath::kTabWords : 1];
  double red[kTile / 64];
  R seh[EH ? kTile : 1];
};
static_assert(8 * kHexRowWords == 24 && 4 * kQ4RowWords == 24, "both families keep 24 row words per element");

// ---------------------------------------------------------------- hex element tile
// The SFORC3 chain of one tile.  Threads past the last element run on the last element's
// nodes and store nothing, so that the whole workgroup reaches its barriers.
template <typename R, typename S, bool EH, bool IDS_FIRST>
__device__ __forceinline__ void hex_tile(const ModelDev &M, int64_t first, int parity_output,
                                         TileLds<R, S, EH, false> &sh) {
  // bit 0: cycle parity; bit 1: an output cycle (each element's time-step candidate is kept)
  const int parity = parity_output & 1;
  const bool output = (parity_output & 2) != 0;
  const DevTime *ts = M.ts;
  // a stopped model computes but stores nothing; the flag is tested only before the
  // stores, so that its load overlaps the element's own loads
  const int stopped = time_done(ts + parity);
  const HexPtrs<S> e = hex_ptrs<S>(M);
  const gptr<const double> xv = to_global<const double>(M.nd.xv);
  const HexConsts &c = M.hc;
  const int64_t i = first + threadIdx.x;
  const bool active = i < e.ne;
  const int64_t ic = active ? i : e.ne - 1;
  // the split form stages its element state through LDS; the FP64 chain, bound by its
  // arithmetic at two waves per SIMD, reads it from HBM after the kinematics (staged, it took
  // 15.2 us against 14.5 at 32,000 elements, and the same at 512,000)
  constexpr bool kStage = sizeof(S) == 4;
  if constexpr (kStage) {
    const gptr<const S> src[12] = {e.sig,          e.sig + e.ne,     e.sig + 2 * e.ne, e.sig + 3 * e.ne,
                                   e.sig + 4 * e.ne, e.sig + 5 * e.ne, e.eint,           e.rho,
                                   e.vol0,         e.pla,            e.epsd,           e.qvis};
#pragma unroll
    for (int a = 0; a < 12; ++a) stage_word<S>(sh.rows, a, src[a], first, e.ne);
  }
  int32_t nc[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) nc[k] = e.conn[(int64_t)k * e.ne + ic];
  // all node ids before the first gather: in k_elements the other order takes 144 us for 140 a cycle
  // (512,000 + 160,000 elements), in the FP64 hexes' own kernel this one 14.2 for 13.7 at
  // 32,000 and 281 for 270 at 2,097,000
  if constexpr (IDS_FIRST || sizeof(R) == 4) __asm__ __volatile__("" ::: "memory");
  TileAssembly<S, kHexRowWords, 8> ta;
  ta.range(M.hfr_start, first / kTile);
  const R DT1 = R(time_dt2(ts + parity));
  HexState<S> st;
  HexOut<R> o;
  // EH: the model keeps EHOUR (its own instantiation, so that the other keeps its registers)
  auto ehou_sink = [&](R v) {
    if constexpr (EH) sh.seh[threadIdx.x] = v;
  };
  double xd[8], yd[8], zd[8];
  R vx[8], vy[8], vz[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    double a, b, cc, u, v, w;
    load_node(xv, nc[k], a, b, cc, u, v, w);
    xd[k] = a; yd[k] = b; zd[k] = cc;
    vx[k] = R(u); vy[k] = R(v); vz[k] = R(w);
  }
  // GBUF%OFF enters the geometry; the rest of the element state is read after the kinematics
  st.offg = e.offg[ic];
  auto load_rest = [&]() {
    if constexpr (kStage) {
      wait_staged();
      const S *s = sh.rows + threadIdx.x;
#pragma unroll
      for (int k = 0; k < 6; ++k) st.sig[k] = s[k * kTile];
      st.eint = s[6 * kTile]; st.rho = s[7 * kTile]; st.vol0 = s[8 * kTile]; st.pla = s[9 * kTile];
      st.epsd = s[10 * kTile]; st.qvis = s[11 * kTile];
    } else {
      __asm__ __volatile__("" ::: "memory");
#pragma unroll
      for (int k = 0; k < 6; ++k) st.sig[k] = e.sig[(int64_t)k * e.ne + ic];
      st.eint = e.eint[ic]; st.rho = e.rho[ic]; st.vol0 = e.vol0[ic]; st.pla = e.pla[ic];
      st.epsd = e.epsd[ic]; st.qvis = e.qvis[ic];
    }
  };
  if constexpr (sizeof(R) == 8) {
    // FP64: each node's force triple leaves for LDS as soon as it is final, which keeps
    // the chain within two waves' register budget
    auto write_row = [&](int k, R fx, R fy, R fz) {
      const S w[3] = {S(fx), S(fy), S(fz)};
      lds_corner<S, 3>(sh.rows, k, w);
    };
    hex_element<R, S>(xd, yd, zd, vx, vy, vz, st, c, DT1, o, write_row, load_rest, ehou_sink);
  } else {
    // FP32: the forces are gathered first and stored together (registers are not the limit)
    R f1[8], f2[8], f3[8];
    auto keep = [&](int k, R fx, R fy, R fz) { f1[k] = fx; f2[k] = fy; f3[k] = fz; };
    hex_element<R, S>(xd, yd, zd, vx, vy, vz, st, c, DT1, o, keep, load_rest, ehou_sink);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const S w[3] = {S(f1[k]), S(f2[k]), S(f3[k])};
      lds_corner<S, 3>(sh.rows, k, w);
    }
  }
  if (stopped) return; // uniform over the workgroup
  if (active) {
#pragma unroll
    for (int k = 0; k < 6; ++k) e.sig[(int64_t)k * e.ne + i] = st.sig[k];
    e.eint[i] = st.eint; e.rho[i] = st.rho; e.pla[i] = st.pla;
    e.epsd[i] = st.epsd; e.offg[i] = st.offg; e.qvis[i] = st.qvis;
    if (output && M.dtel_h) to_global(M.dtel_h)[i] = o.dtx;
  }
  ta.prefetch(e.rest, e.ne, i, to_global(M.hfr_node), to_global<const v4u>(M.hfr_src));
  wave_min_to(sh.red, active ? o.dtx : kEP06);
  if (active && o.mstop) atomicOr(M.flags, kMstopJacobian);
  __syncthreads();
  tile_min_commit<kTile>(sh.red, M.dtmin + parity);
  if constexpr (EH) {
    if (M.ehou_h) tile_ehou_commit<kTile>(sh.seh, first, e.ne, M.ehou_h + first / kTile);
  }
  ta.finish(sh.rows, to_global<S>(M.rowh), to_global(M.hfr_node), to_global<const v4u>(M.hfr_src), to_global(M.preh));
}

// A model's view, in the constant address space: its fields come by scalar loads wherever they are
// used, also behind stores and fences, so that none has to be held (or spilled) from the start:
// 32,000 FP64 hexes 14.1 us for 14.3, 16,428 shells in the split form 14.8 for 15.0.  Not for the
// FP64 shells, whose registers it spills (160,000: 52.2 us for 49.3).
__device__ __forceinline__ const ModelDev &model_of(const ModelDev *md, int32_t model) {
  return *(const ModelDev *)((cptr<ModelDev>)md + model);
}

// The tile of workgroup b of nb: the launch's tile list, or the only model's tiles in order.
__device__ __forceinline__ Tile launch_tile(const Tile *tiles, int64_t b, int64_t nb) {
  const int64_t t = xcd_contiguous_block(b, nb);
  if (!tiles) return Tile{0, (int32_t)(t * kTile)};
  const cptr<Tile> p = (cptr<Tile>)(tiles + t);
  return Tile{p->model, p->first};
}

template <typename R, typename S, int TB, int W, bool EH>
__global__ __launch_bounds__(TB) __attribute__((amdgpu_waves_per_eu(W))) void k_hex_forces(
    const ModelDev *__restrict__ md, const Tile *__restrict__ tiles, int parity_output) {
  static_assert(TB == kTile, "a hex workgroup is one assembly tile");
  __shared__ TileLds<R, S, EH, false> sh;
  const Tile tl = launch_tile(tiles, blockIdx.x, gridDim.x);
  hex_tile<R, S, EH, false>(model_of(md, tl.model), tl.first, parity_output, sh);
}

// ---------------------------------------------------------------- Q4 element kernel
// Per-point state of a resident shell, each point loaded one point ahead, so that its loads
// overlap the previous point's arithmetic.
template <typename R, typename S> struct Q4IpIO {
  const Q4Ptrs<S> &q;
  int64_t i;   // the thread's element, the last one for threads past it
  bool active; // false: past the last element, or the model has stopped: nothing is stored
  int npt;
  R s_next[5], pla_next, epsd_next;
  __device__ __forceinline__ void begin() {
    load(0, s_next, pla_next, epsd_next);
  }
  __device__ __forceinline__ void fetch(int ip, R (&s)[5], R &pla, R &epsd_ip) {
#pragma unroll
    for (int k = 0; k < 5; ++k) s[k] = s_next[k];
    pla = pla_next; epsd_ip = epsd_next;
    if (ip + 1 < npt) load(ip + 1, s_next, pla_next, epsd_next);
  }
  __device__ __forceinline__ void load(int ip, R (&s)[5], R &pla, R &epsd_ip) const {
    const gptr<const S> sg = q.sig + (int64_t)ip * 5 * q.ne + i;
#pragma unroll
    for (int k = 0; k < 5; ++k) s[k] = R(sg[(int64_t)k * q.ne]);
    pla = R(q.pla[(int64_t)ip * q.ne + i]);
    epsd_ip = q.epsd_ip ? R(q.epsd_ip[(int64_t)ip * q.ne + i]) : R(0);
  }
  __device__ __forceinline__ void store(int ip, const R (&s)[5], R pla, R epsd_ip) const {
    if (!active) return;
    const gptr<S> sg = q.sig + (int64_t)ip * 5 * q.ne + i;
#pragma unroll
    for (int k = 0; k < 5; ++k) sg[(int64_t)k * q.ne] = S(s[k]);
    q.pla[(int64_t)ip * q.ne + i] = S(pla);
    if (q.epsd_ip) q.epsd_ip[(int64_t)ip * q.ne + i] = S(epsd_ip);
  }
  __device__ __forceinline__ void late_load(Q4Late<R> &L) const {
#pragma unroll
    for (int k = 0; k < 5; ++k) L.forc[k] = R(q.forc[(int64_t)k * q.ne + i]);
#pragma unroll
    for (int k = 0; k < 3; ++k) L.mom[k] = R(q.mom[(int64_t)k * q.ne + i]);
#pragma unroll
    for (int k = 0; k < 8; ++k) L.gstr[k] = R(q.gstr[(int64_t)k * q.ne + i]);
#pragma unroll
    for (int k = 0; k < 3; ++k) L.hourg[k] = R(q.hourg[(int64_t)k * q.ne + i]);
    L.eint[0] = R(q.eint[i]);
    L.eint[1] = R(q.eint[q.ne + i]);
  }
  __device__ __forceinline__ void late_store(const Q4Late<R> &L) const {
    if (!active) return;
#pragma unroll
    for (int k = 0; k < 5; ++k) q.forc[(int64_t)k * q.ne + i] = S(L.forc[k]);
#pragma unroll
    for (int k = 0; k < 3; ++k) q.mom[(int64_t)k * q.ne + i] = S(L.mom[k]);
#pragma unroll
    for (int k = 0; k < 8; ++k) q.gstr[(int64_t)k * q.ne + i] = S(L.gstr[k]);
    q.eint[i] = S(L.eint[0]);
    q.eint[q.ne + i] = S(L.eint[1]);
  }
  __device__ __forceinline__ void hourg_store(const R (&h)[5]) const {
    if (!active) return;
#pragma unroll
    for (int k = 0; k < 5; ++k) q.hourg[(int64_t)k * q.ne + i] = S(h[k]);
  }
};

// The thread's element, formed again where it stands instead of held in registers from the tile's
// start: two registers of the FP64 shells' 256, which else spill 12 bytes a lane (160,000 elastic shells
// 47.7 us a cycle for 48.8; a kernel with scratch also starts 0.5 us later).  The FP64 hexes spill as
// much but keep theirs: without it the 4,096,000 + 1,000,000 elements in one launch take 1,026 us for 1,004.
__device__ __forceinline__ int64_t element_again(int64_t first) {
  int t = threadIdx.x;
  __asm__ __volatile__("" : "+v"(t));
  return first + t;
}

// ---------------------------------------------------------------- Q4 element tile
// The CFORC3 chain of one tile; threads past the last element as in hex_tile.
template <typename R, typename S, bool EH>
__device__ __forceinline__ void q4_tile(const ModelDev &M, int64_t first, int parity_output,
                                        TileLds<R, S, EH, sizeof(R) == 8> &sh) {
  const int parity = parity_output & 1; // bit 1: an output cycle, as for the hex tile
  const bool output = (parity_output & 2) != 0;
  const DevTime *ts = M.ts;
  const int stopped = time_done(ts + parity); // tested before the stores only
  const Q4Ptrs<S> q = q4_ptrs<S>(M);
  const gptr<const double> xv = to_global<const double>(M.nd.xv);
  const gptr<const double> vr = to_global<const double>(M.nd.vr);
  const Q4Consts &c = M.qc;
  const int64_t ic = std::min<int64_t>(first + threadIdx.x, q.ne - 1);
  int32_t nc[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) nc[k] = q.conn[(int64_t)k * q.ne + ic];
  __asm__ __volatile__("" ::: "memory");
  TileAssembly<S, kQ4RowWords, 4> ta;
  ta.range(M.qfr_start, first / kTile);
  const R DT1 = R(time_dt2(ts + parity));
  double xg[4], yg[4], zg[4];
  R vl[4][3], vrl[4][3];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    double a, b, cc, u, v, w;
    load_node(xv, nc[k], a, b, cc, u, v, w);
    xg[k] = a; yg[k] = b; zg[k] = cc;
    vl[k][0] = R(u); vl[k][1] = R(v); vl[k][2] = R(w);
    const gptr<const v2d> p = (gptr<const v2d>)(vr + 4 * (int64_t)nc[k]);
    const v2d r0 = p[0], r1 = p[1];
    vrl[k][0] = R(r0.x); vrl[k][1] = R(r0.y); vrl[k][2] = R(r1.x);
  }
  Q4Elem<R> st;
  st.offg = R(q.offg[ic]); st.thk = R(q.thk[ic]); st.thke = R(q.thke[ic]); st.epsd = R(q.epsd[ic]);
  Q4IpIO<R, S> io{q, ic, first + threadIdx.x < q.ne && !stopped, c.npt};
  Q4Out<R> o;
  // EH: the model keeps EHOUR (its own instantiation, so that the other keeps its registers)
  auto ehou_sink = [&](R v) {
    if constexpr (EH) sh.seh[threadIdx.x] = v;
  };
  auto nload = [&](int k, double(&x)[3], R(&v)[3]) {
    __asm__ __volatile__("" ::: "memory"); // a fresh load, not the values held since the gather
    double a, b, cc, u, w, z;
    load_node(xv, nc[k], a, b, cc, u, w, z);
    x[0] = a; x[1] = b; x[2] = cc;
    v[0] = R(u); v[1] = R(w); v[2] = R(z);
  };
  q4_element<R>(xg, yg, zg, vl, vrl, nc[2] == nc[3], st, c, DT1, io, nload, o, ehou_sink, chain_tab<R>(sh.tab));
  if (stopped) return; // uniform over the workgroup
  const int64_t i = element_again(first);
  const bool active = i < q.ne;
  if (active) {
    q.offg[i] = S(st.offg); q.thk[i] = S(st.thk); q.epsd[i] = S(st.epsd);
    if (output && M.dtel_q) to_global(M.dtel_q)[i] = o.dt;
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const S w[6] = {S(-o.f[0][k]), S(-o.f[1][k]), S(-o.f[2][k]), S(-o.m[0][k]), S(-o.m[1][k]), S(-o.m[2][k])};
    lds_corner<S, 6>(sh.rows, k, w);
  }
  ta.prefetch(q.rest, q.ne, i, to_global(M.qfr_node), to_global<const v4u>(M.qfr_src));
  wave_min_to(sh.red, active ? o.dt : kEP06);
  __syncthreads();
  tile_min_commit<kTile>(sh.red, M.dtmin + parity);
  if constexpr (EH) {
    if (M.ehou_q) tile_ehou_commit<kTile>(sh.seh, first, q.ne, M.ehou_q + first / kTile);
  }
  ta.finish(sh.rows, to_global<S>(M.rowq), to_global(M.qfr_node), to_global<const v4u>(M.qfr_src), to_global(M.preq));
}

template <typename R, typename S, int TB, int W, bool EH>
__global__ __launch_bounds__(TB) __attribute__((amdgpu_waves_per_eu(W))) void k_q4_forces(
    const ModelDev *__restrict__ md, const Tile *__restrict__ tiles, int parity_output) {
  static_assert(TB == kTile, "a shell workgroup is one assembly tile");
  __shared__ TileLds<R, S, EH, sizeof(R) == 8> sh;
  const Tile tl = launch_tile(tiles, blockIdx.x, gridDim.x);
  if constexpr (sizeof(R) == 8) q4_tile<R, S, EH>(md[tl.model], tl.first, parity_output, sh); // see model_of
  else q4_tile<R, S, EH>(model_of(md, tl.model), tl.first, parity_output, sh);
}

// ---------------------------------------------------------------- all families in one launch
// The element tiles of a cycle whose model (or batch) has more than one family or form, in one
// launch: family f's list is t[f] (null: the only model's tiles in order) of n[f] tiles.
// Shells come first, their chains being the longer ones.  MASK: the families compiled in.
enum { kFamQ4 = 0, kFamHex = 1, kFamQ4Split = 2, kFamHexSplit = 3 };
struct ElemLists {
  const Tile *t[4];
  int32_t n[4];
};
template <int MASK, bool EH>
__global__ __launch_bounds__(kTile) __attribute__((amdgpu_waves_per_eu(2))) void k_elements(
    const ModelDev *__restrict__ md, ElemLists L, int parity_output) {
  typedef TileLds<double, double, EH, true> Lds64;
  typedef TileLds<double, double, EH, false> LdsHex64;
  typedef TileLds<float, float, EH, false> Lds32;
  __shared__ __align__(16) unsigned char buf[(MASK & 3) ? sizeof(Lds64) : sizeof(Lds32)];
  static_assert(sizeof(Lds32) <= sizeof(Lds64), "the FP64 layout is the larger one");
  int32_t b = (int32_t)blockIdx.x;
  if constexpr (MASK & (1 << kFamQ4)) {
    if (b < L.n[kFamQ4]) {
      const Tile tl = launch_tile(L.t[kFamQ4], b, L.n[kFamQ4]);
      q4_tile<double, double, EH>(md[tl.model], tl.first, parity_output, *(Lds64 *)buf);
      return;
    }
    b -= L.n[kFamQ4];
  }
  if constexpr (MASK & (1 << kFamQ4Split)) {
    if (b < L.n[kFamQ4Split]) {
      const Tile tl = launch_tile(L.t[kFamQ4Split], b, L.n[kFamQ4Split]);
      q4_tile<float, float, EH>(model_of(md, tl.model), tl.first, parity_output, *(Lds32 *)buf);
      return;
    }
    b -= L.n[kFamQ4Split];
  }
  if constexpr (MASK & (1 << kFamHex)) {
    if (b < L.n[kFamHex]) {
      const Tile tl = launch_tile(L.t[kFamHex], b, L.n[kFamHex]);
      hex_tile<double, double, EH, true>(model_of(md, tl.model), tl.first, parity_output, *(LdsHex64 *)buf);
      return;
    }
    b -= L.n[kFamHex];
  }
  if constexpr (MASK & (1 << kFamHexSplit)) {
    const Tile tl = launch_tile(L.t[kFamHexSplit], b, L.n[kFamHexSplit]);
    hex_tile<float, float, EH, true>(model_of(md, tl.model), tl.first, parity_output, *(Lds32 *)buf);
  }
}

// ---------------------------------------------------------------- nodal update pieces
// ACCELE (accele.F:65-80, 97-109): A = F / MS, zero where the mass (inertia) is not positive.
__device__ __forceinline__ void accele3(double &a0, double &a1, double &a2, double mass) {
  if (mass > 0.0) {
    const double rtmp = 1.0 / mass;
    a0 = a0 * rtmp; a1 = a1 * rtmp; a2 = a2 * rtmp;
  } else {
    a0 = 0.0; a1 = 0.0; a2 = 0.0;
  }
}

// BCS1V (bcs1.F, global frame) and FIXVEL (fixvel.F:366-379, global frame) on one node:
// fixed DOFs get zero acceleration and velocity, imposed ones A = (VIMP - V) / DT12.
template <typename P>
__device__ __forceinline__ void bcs_fixvel(int32_t code, double &ax, double &ay, double &az, double &vx, double &vy,
                                           double &vz, double &rx, double &ry, double &rz, double &wx, double &wy,
                                           double &wz, P vimp, double DT12, double DT1, double DT2, double msn,
                                           double &work, double &pend) {
  if (code & kTX) { ax = 0.0; vx = 0.0; }
  if (code & kTY) { ay = 0.0; vy = 0.0; }
  if (code & kTZ) { az = 0.0; vz = 0.0; }
  if (code & kRX) { rx = 0.0; wx = 0.0; }
  if (code & kRY) { ry = 0.0; wy = 0.0; }
  if (code & kRZ) { rz = 0.0; wz = 0.0; }
  // the imposed DOF's work (fixvel.F:376-378, 834, 837): DW = FOURTH*MS*AXI*WEIGHT*(A*DT12 +
  // TWO*V)*(A - AOLD) with AXI = WEIGHT = 1; DT1*DW enters WFEXT now, DT2*DW (kept per node in
  // pend) at the next cycle, before the DOF's new work (fixvel.F:342-344)
  const double carried = pend;
  work = work + carried;
  pend = 0.0;
  auto imposed = [&](double &a, double v, double vi) {
    const double aold = a;
    a = (vi - v) / DT12;
    const double dw = ((1.0 / 4.0) * msn) * (a * DT12 + 2.0 * v) * (a - aold);
    work = work + DT1 * dw;
    pend = pend + DT2 * dw;
  };
  if (code & kIX) imposed(ax, vx, vimp[0]);
  if (code & kIY) imposed(ay, vy, vimp[1]);
  if (code & kIZ) imposed(az, vz, vimp[2]);
}

// The DT2 pipeline (resol.F:2826, 6125-6129, 6352, 6494-6497): DT2 from the element
// minimum dt2t, the growth limit on DT2OLD and DTMX.
__host__ __device__ __forceinline__ double dt2_pipeline(double dt2t, double dt2old, double dt_growth, double dtmx) {
  double DT2 = kEP06;
  if (dt2t < DT2) DT2 = dt2t;
  const double g = dt_growth * dt2old;
  DT2 = (g < DT2) ? g : DT2;
  DT2 = (dtmx < DT2) ? dtmx : DT2;
  return DT2;
}

// ---------------------------------------------------------------- node kernel
// Block b of a launch's list, or of the only model's nodes.  FIRST: everything that needs no other
// load is asked for at the start and the rest rows come several at a time; otherwise every load stands
// at its use (node_first chooses).  Both add the same values in the same order.
template <typename S, bool FIRST>
__device__ __forceinline__ void node_tile(const ModelDev *__restrict__ md, const Tile *__restrict__ tiles, int32_t b,
                                          int parity, double dt_growth, int output) {
  const Tile tl = tiles ? tiles[b] : Tile{0, b * kBlock};
  const ModelDev &M = md[tl.model];
  const NodePtrs &nd = M.nd;
  const gptr<const S> rowh = to_global<const S>(M.rowh);
  const gptr<const S> rowq = to_global<const S>(M.rowq);
  DevTime *ts = M.ts;
  unsigned long long *dtmin = M.dtmin;
  const double dtmx = M.dtmx;
  const int64_t n = (int64_t)tl.first + threadIdx.x;
  const bool in_range = n < nd.nn;
  const int64_t m = in_range ? n : nd.nn - 1;
  const DevTime prev = load_time(ts + parity);
  unsigned long long dt2t;
  v2d pa, pb, pc;
  double d0, d1, d2, msn;
  int32_t code, dh = 0, dq = 0, h0 = 0, h1 = 0, q0 = 0, q1 = 0;
  double px = 0.0, py = 0.0, pz = 0.0;
  bool rot = false;
  double wx = 0.0, wy = 0.0, wz = 0.0, inn = 0.0;
  gptr<v2d> pr = nullptr;
  if constexpr (FIRST) {
    dt2t = to_global<const unsigned long long>(dtmin)[parity];
    const gptr<const v2d> p = (gptr<const v2d>)to_global(nd.xv + 6 * m);
    pa = p[0]; pb = p[1]; pc = p[2];
    const gptr<const double> dd = to_global(nd.d) + 3 * m;
    d0 = dd[0]; d1 = dd[1]; d2 = dd[2];
    msn = to_global(nd.ms)[m];
    code = to_global(nd.code)[m];
    if (nd.deg_h) {
      dh = to_global(nd.deg_h)[m];
      h0 = to_global(nd.rs_h)[m]; h1 = to_global(nd.rs_h)[m + 1];
      const gptr<const double> q = to_global(nd.pre_h) + 3 * m; // unused when the node has no hex rows
      px = q[0]; py = q[1]; pz = q[2];
    }
    if (nd.deg_q) {
      dq = to_global(nd.deg_q)[m];
      q0 = to_global(nd.rs_q)[m]; q1 = to_global(nd.rs_q)[m + 1];
    }
    // A node without shell rows and without rotational BCs has AR = 0, so VELOCITY leaves
    // its VR as it is: its VR and IN are not touched.
    rot = nd.vr && (dq > 0 || (code & (kRX | kRY | kRZ)));
    if (rot) {
      inn = to_global(nd.in)[m];
      pr = (gptr<v2d>)to_global(nd.vr + 4 * m);
      const v2d r0 = pr[0], r1 = pr[1];
      wx = r0.x; wy = r0.y; wz = r1.x;
    }
  } else if (nd.deg_h && in_range) {
    dh = to_global(nd.deg_h)[n];
    if (dh > 0) {
      const gptr<const double> q = to_global(nd.pre_h) + 3 * n;
      px = q[0]; py = q[1]; pz = q[2];
      h0 = to_global(nd.rs_h)[n]; h1 = to_global(nd.rs_h)[n + 1];
    }
  }
  // ASSPAR4: rows of this node in skyline order (solids, then shells), from zero: the
  // prefix the element tiles summed, then the rest rows in order
  double ax = 0.0, ay = 0.0, az = 0.0, rx = 0.0, ry = 0.0, rz = 0.0;
  if (dh > 0) { ax = px; ay = py; az = pz; }
  if (FIRST && dq > 0 && dh == 0) { // the node's sum starts with its shell rows: their prefix
    const gptr<const v2d> q = (gptr<const v2d>)(to_global(nd.pre_q) + 6 * m);
    const v2d p0 = q[0], p1 = q[1], p2 = q[2];
    ax = p0.x; ay = p0.y; az = p1.x; rx = p1.y; ry = p2.x; rz = p2.y;
  }
  constexpr int kHexAhead = FIRST ? 4 : 1, kQ4Ahead = FIRST ? 3 : 1; // rest rows in flight at once
  for (int32_t r = h0; r < h1; r += kHexAhead) {
    S w[kHexAhead][kHexRowWords];
#pragma unroll
    for (int k = 0; k < kHexAhead; ++k) {
      const gptr<const S> q = rowh + (int64_t)(r + k < h1 ? r + k : r) * kHexRowWords;
#pragma unroll
      for (int c = 0; c < kHexRowWords; ++c) w[k][c] = q[c];
    }
#pragma unroll
    for (int k = 0; k < kHexAhead; ++k)
      if (r + k < h1) { ax = ax + double(w[k][0]); ay = ay + double(w[k][1]); az = az + double(w[k][2]); }
  }
  if constexpr (!FIRST) {
    if (nd.deg_q && in_range) {
      dq = to_global(nd.deg_q)[n];
      if (dq > 0) {
        if (dh == 0) {
          const gptr<const v2d> q = (gptr<const v2d>)(to_global(nd.pre_q) + 6 * n);
          const v2d p0 = q[0], p1 = q[1], p2 = q[2];
          ax = p0.x; ay = p0.y; az = p1.x; rx = p1.y; ry = p2.x; rz = p2.y;
        }
        q0 = to_global(nd.rs_q)[n]; q1 = to_global(nd.rs_q)[n + 1];
      }
    }
  }
  for (int32_t r = q0; r < q1; r += kQ4Ahead) {
    S w[kQ4Ahead][kQ4RowWords];
#pragma unroll
    for (int k = 0; k < kQ4Ahead; ++k) {
      const gptr<const S> q = rowq + (int64_t)(r + k < q1 ? r + k : r) * kQ4RowWords;
#pragma unroll
      for (int c = 0; c < kQ4RowWords; ++c) w[k][c] = q[c];
    }
#pragma unroll
    for (int k = 0; k < kQ4Ahead; ++k)
      if (r + k < q1) {
        ax = ax + double(w[k][0]); ay = ay + double(w[k][1]); az = az + double(w[k][2]);
        rx = rx + double(w[k][3]); ry = ry + double(w[k][4]); rz = rz + double(w[k][5]);
      }
  }
  if (prev.done) {
    // a stopped model keeps its state; its scalars are carried to the other parity
    if (n == 0) {
      ts[parity ^ 1] = prev;
      dtmin[parity ^ 1] = dbits(kEP06);
    }
    return;
  }
  // DT2 pipeline (resol.F:2721-2722, 2826, 6125-6129, 6352, 6494-6497)
  if constexpr (!FIRST) dt2t = to_global<const unsigned long long>(dtmin)[parity];
  const double DT1 = prev.dt2;
  const double DT2 = dt2_pipeline(bitsd(dt2t), prev.dt2old, dt_growth, dtmx);
  const double DT12 = (1.0 / 2.0) * (DT1 + DT2);
  if (n == 0) {
    DevTime nx;
    nx.tt = prev.tt + DT2;
    nx.dt1 = DT1;
    nx.dt2 = DT2;
    nx.dt12 = DT12;
    nx.dt2old = DT2;
    nx.ncycle = prev.ncycle + 1;
    // a time step <= 0 stops the run (resol.F:8575, 9599)
    nx.mstop = prev.mstop | *M.flags | (DT2 <= 0.0 ? kMstopTimeStep : 0);
    nx.done = (nx.mstop != 0 || nx.tt >= M.tend) ? 1 : 0;
    ts[parity ^ 1] = nx;
    dtmin[parity ^ 1] = dbits(kEP06);
  }
  if (!in_range) return;
  // ACCELE (accele.F:65-80, 97-109)
  if constexpr (!FIRST) msn = to_global(nd.ms)[n];
  accele3(ax, ay, az, msn);
  if constexpr (!FIRST) {
    code = to_global(nd.code)[n];
    rot = nd.vr && (dq > 0 || (code & (kRX | kRY | kRZ)));
    if (rot) {
      inn = to_global(nd.in)[n];
      pr = (gptr<v2d>)to_global(nd.vr + 4 * n);
      const v2d r0 = pr[0], r1 = pr[1];
      wx = r0.x; wy = r0.y; wz = r1.x;
    }
  }
  if (rot) accele3(rx, ry, rz, inn);
  const gptr<v2d> p = (gptr<v2d>)to_global(nd.xv + 6 * n);
  if constexpr (!FIRST) { pa = p[0]; pb = p[1]; pc = p[2]; }
  double x = pa.x, y = pa.y, z = pb.x, vx = pb.y, vy = pc.x, vz = pc.y;
  if (code) {
    // the node's external work (WFEXT) accumulates in wext[n] when its DOFs are imposed
    const bool imp = (code & (kIX | kIY | kIZ)) && nd.wext;
    double work = imp ? to_global(nd.wext)[n] : 0.0, pend = imp ? to_global(nd.wext)[nd.nn + n] : 0.0;
    bcs_fixvel(code, ax, ay, az, vx, vy, vz, rx, ry, rz, wx, wy, wz, to_global(nd.vimp) + 3 * n, DT12, DT1, DT2,
               msn, work, pend);
    if (imp) {
      to_global(nd.wext)[n] = work;
      to_global(nd.wext)[nd.nn + n] = pend;
    }
  }
  if (output && M.ecrit) {
    // ECRIT's kinetic energies at its output point, between FIXVEL and VELOCITY
    // (sortie_main.F:368 from resol.F:8523): V + DT05*A with DT05 = HALF*DT1 (ecrit.F:193,
    // 221-225, 319-324; MAS = MS*WEIGHT_MD, WEIGHT_MD = 1 on one domain)
    const double DT05 = (1.0 / 2.0) * DT1;
    const double ux = vx + DT05 * ax, uy = vy + DT05 * ay, uz = vz + DT05 * az;
    const gptr<double> ke = to_global(M.ecrit);
    ke[n] = (ux * ux + uy * uy + uz * uz) * (1.0 / 2.0) * msn;
    double kr = 0.0;
    if (nd.vr) {
      double qx = wx, qy = wy, qz = wz;
      if (!pr) { // rotational work skipped: AR = 0, VR as stored
        const gptr<const v2d> q = (gptr<const v2d>)to_global(nd.vr + 4 * n);
        const v2d q0 = q[0], q1 = q[1];
        qx = q0.x; qy = q0.y; qz = q1.x;
      }
      inn = to_global(nd.in)[n];
      const double sx = qx + DT05 * rx, sy = qy + DT05 * ry, sz = qz + DT05 * rz;
      kr = (sx * sx + sy * sy + sz * sz) * (1.0 / 2.0) * inn;
    }
    ke[nd.nn + n] = kr;
    // XMOMT, YMOMT, ZMOMT (ecrit.F:226-228)
    ke[2 * nd.nn + n] = ux * msn;
    ke[3 * nd.nn + n] = uy * msn;
    ke[4 * nd.nn + n] = uz * msn;
    // the time history's nodal values at the same point (thnod.F:59-97): D and X before
    // DEPLA, V after BCS10, A after FIXVEL, VR and AR (zero without rotational DOFs)
    const int32_t slot = M.th_slot ? to_global(M.th_slot)[n] : -1;
    if (slot >= 0) {
      const gptr<double> t = to_global(M.th_node) + 18 * (int64_t)slot;
      const gptr<const double> dn = to_global(nd.d) + 3 * n;
      double qx = 0.0, qy = 0.0, qz = 0.0;
      if (nd.vr) {
        qx = wx; qy = wy; qz = wz;
        if (!pr) {
          const gptr<const v2d> q = (gptr<const v2d>)to_global(nd.vr + 4 * n);
          const v2d q0 = q[0], q1 = q[1];
          qx = q0.x; qy = q0.y; qz = q1.x;
        }
      }
      t[0] = dn[0]; t[1] = dn[1]; t[2] = dn[2];
      t[3] = vx; t[4] = vy; t[5] = vz;
      t[6] = ax; t[7] = ay; t[8] = az;
      t[9] = qx; t[10] = qy; t[11] = qz;
      t[12] = rx; t[13] = ry; t[14] = rz;
      t[15] = x; t[16] = y; t[17] = z;
    }
  }
  // VELOCITY (velocity.F:58-86)
  vx = vx + DT12 * ax; vy = vy + DT12 * ay; vz = vz + DT12 * az;
  if (pr) {
    wx = wx + DT12 * rx; wy = wy + DT12 * ry; wz = wz + DT12 * rz;
    pr[0] = v2d{wx, wy};
    pr[1] = v2d{wz, 0.0};
  }
  // DEPLA (displacement.F:108-118, IRESP=0 form in FP64)
  const gptr<double> dd = to_global(nd.d) + 3 * n;
  if constexpr (!FIRST) { d0 = dd[0]; d1 = dd[1]; d2 = dd[2]; }
  double vdt;
  vdt = DT2 * vx; dd[0] = d0 + vdt; x = x + vdt;
  vdt = DT2 * vy; dd[1] = d1 + vdt; y = y + vdt;
  vdt = DT2 * vz; dd[2] = d2 + vdt; z = z + vdt;
  p[0] = v2d{x, y};
  p[1] = v2d{z, vx};
  p[2] = v2d{vy, vz};
}

template <typename S, bool FIRST>
__global__ __launch_bounds__(kBlock) void k_node_update(const ModelDev *__restrict__ md,
                                                        const Tile *__restrict__ tiles, int parity,
                                                        double dt_growth, int output) {
  node_tile<S, FIRST>(md, tiles, (int32_t)blockIdx.x, parity, dt_growth, output);
}

// The node update of a batch with members of both forms, in one launch: n64 blocks of FP64
// members, then those of the split form.  98 registers, four waves a SIMD; still the fastest at every
// size (12 bars and tubes: 41.6 us a cycle against 45.6 in a launch for each form at 98,000 nodes, 110
// and 115 at 515,000, 498 and 506 at 2,586,000, 1,508 and 1,515 at 8,072,000; held to five waves 1,513).
__global__ __launch_bounds__(kBlock) void k_node_update_both(const ModelDev *__restrict__ md,
                                                             const Tile *__restrict__ t64, int32_t n64,
                                                             const Tile *__restrict__ t32, int parity,
                                                             double dt_growth) {
  const int32_t b = (int32_t)blockIdx.x;
  if (b < n64) node_tile<double, true>(md, t64, b, parity, dt_growth, 0);
  else node_tile<float, true>(md, t32, b - n64, parity, dt_growth, 0);
}

// ---------------------------------------------------------------- energies (fixed-order)
// ENINT, ENCIN, ENROT, WFEXT, XMOMT, YMOMT, ZMOMT
constexpr int kEnergySums = 7;
__device__ __forceinline__ double block_sum(double v) {
  __shared__ double red[kBlock];
  red[threadIdx.x] = v;
  __syncthreads();
  for (int s = kBlock / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] = red[threadIdx.x] + red[threadIdx.x + s];
    __syncthreads();
  }
  double r = red[0];
  __syncthreads();
  return r;
}

template <typename S>
__global__ __launch_bounds__(kBlock) void k_energy_partial(const S *heint, const S *hvol0, int64_t neh,
                                                           const S *qeint, int64_t neq, const double *xv,
                                                           const double *vr, const double *ms, const double *in,
                                                           const double *ecrit, const double *wext, int64_t nn,
                                                           int64_t per_block, double *partial) {
  double ie = 0.0, ke = 0.0, kr = 0.0, we = 0.0, mx = 0.0, my = 0.0, mz = 0.0;
  const int64_t b0 = (int64_t)blockIdx.x * per_block;
  for (int64_t j = b0 + threadIdx.x; j < b0 + per_block; j += kBlock) {
    if (j < nn && wext) we = we + wext[j];
    if (j < neh) ie = ie + double(heint[j]) * double(hvol0[j]);
    if (j < neq) ie = ie + (double(qeint[j]) + double(qeint[neq + j]));
    if (j < nn && ecrit) {
      // per-node terms written by the node kernel on an output cycle
      ke = ke + ecrit[j];
      kr = kr + ecrit[nn + j];
      mx = mx + ecrit[2 * nn + j];
      my = my + ecrit[3 * nn + j];
      mz = mz + ecrit[4 * nn + j];
    } else if (j < nn) {
      const double *p = xv + 6 * j;
      ke = ke + ms[j] * (p[3] * p[3] + p[4] * p[4] + p[5] * p[5]);
      if (vr) {
        const double *w = vr + 4 * j;
        kr = kr + in[j] * (w[0] * w[0] + w[1] * w[1] + w[2] * w[2]);
      }
    }
  }
  const double v[kEnergySums] = {block_sum(ie), block_sum(ke), block_sum(kr), block_sum(we),
                                 block_sum(mx), block_sum(my), block_sum(mz)};
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < kEnergySums; ++k) partial[kEnergySums * blockIdx.x + k] = v[k];
  }
}

__global__ __launch_bounds__(kBlock) void k_energy_final(const double *partial, int nb, double kin_factor,
                                                         double *out) {
  double a[kEnergySums];
#pragma unroll
  for (int k = 0; k < kEnergySums; ++k) a[k] = 0.0;
  for (int j = threadIdx.x; j < nb; j += kBlock) {
#pragma unroll
    for (int k = 0; k < kEnergySums; ++k) a[k] = a[k] + partial[kEnergySums * j + k];
  }
#pragma unroll
  for (int k = 0; k < kEnergySums; ++k) a[k] = block_sum(a[k]);
  if (threadIdx.x == 0) {
    out[0] = a[0];
    out[1] = kin_factor * a[1];
    out[2] = kin_factor * a[2];
    for (int k = 3; k < kEnergySums; ++k) out[k] = a[k];
  }
}

template <typename T> __global__ __launch_bounds__(kBlock) void k_fill(T *p, int64_t n, T v) {
  for (int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x; j < n; j += (int64_t)gridDim.x * kBlock) p[j] = v;
}
// A launch holds fewer than 2^32 threads, a state array of ten points more values than that from 86
// million shells on: 16,384 blocks at most, which fill the chip eight times over.
template <typename T> hipError_t fill(hipStream_t st, T *p, int64_t n, T v) {
  if (n <= 0) return hipSuccess;
  const unsigned g = (unsigned)std::min<int64_t>((n + kBlock - 1) / kBlock, 16384);
  hipLaunchKernelGGL(k_fill<T>, dim3(g), dim3(kBlock), 0, st, p, n, v);
  return hipGetLastError();
}

// The element that controls the time step of an output cycle, as MQVISCB and CDT3 name it
// (NELTS, ITYPTS): with DT2T = EP06 on entry (resol.F:2826), the solids in element order
// replace it when DTX <= DT2T (mqviscb.F:622-630), so the last solid with the smallest DTX;
// then the shells when DT < DT2T (cdt3.F:205-215), so the first shell whose DT is below
// every solid's.  Elements that cannot control the step carry EP06.  w[0], w[1]: the
// minimum of each family (FP64 bits, integer atomicMin); w[2]: the largest solid index at
// the solid minimum (atomicMax); w[3]: the smallest shell index at the shell minimum.
__global__ __launch_bounds__(64) void k_ctrl_init(unsigned long long *w) {
  if (threadIdx.x < 4) w[threadIdx.x] = threadIdx.x < 2 ? dbits(kEP06) : threadIdx.x == 2 ? 0ull : ~0ull;
}
__global__ __launch_bounds__(kBlock) void k_ctrl_min(const double *dt, int64_t ne, unsigned long long *w) {
  double v = kEP06;
  for (int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x; j < ne; j += (int64_t)gridDim.x * kBlock)
    v = (dt[j] < v) ? dt[j] : v;
  const double b = block_min<kBlock>(v);
  if (threadIdx.x == 0 && b < kEP06) atomicMin(w, dbits(b));
}
__global__ __launch_bounds__(kBlock) void k_ctrl_pick(const double *dt, const int32_t *logical, int64_t ne,
                                                      const unsigned long long *wmin, int last,
                                                      unsigned long long *pick) {
  const double m = bitsd(*wmin);
  for (int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x; j < ne; j += (int64_t)gridDim.x * kBlock) {
    if (dt[j] == m && m < kEP06) {
      const unsigned long long e = (unsigned long long)logical[j];
      if (last) atomicMax(pick, e);
      else atomicMin(pick, e);
    }
  }
}

// ---------------------------------------------------------------- time history
// The element values of THSOL (thsol.F:189-200, 511-548) and THCOQ (thcoq.F:296-340, 452-520)
// that the time-history file reads from the element buffers, for the listed elements (storage
// slots): hexes OFF, SIG(6), EINT, RHO, QVIS, VOL0, PLA, EPSD; shells FOR(5), MOM(3), EINT(2),
// OFF, THK and the PLA of each through-thickness point.
template <typename S>
__global__ __launch_bounds__(kBlock) void k_th_elements(const ModelDev *__restrict__ md, const int32_t *hex,
                                                        int64_t nh, const int32_t *q4, int64_t nq, int npt,
                                                        double *hout, double *qout) {
  const ModelDev &M = md[0];
  const int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (j < nh) {
    const HexPtrs<S> e = hex_ptrs<S>(M);
    const int64_t i = hex[j];
    const gptr<double> o = to_global(hout) + 13 * j;
    o[0] = double(e.offg[i]);
#pragma unroll
    for (int k = 0; k < 6; ++k) o[1 + k] = double(e.sig[(int64_t)k * e.ne + i]);
    o[7] = double(e.eint[i]); o[8] = double(e.rho[i]); o[9] = double(e.qvis[i]); o[10] = double(e.vol0[i]);
    o[11] = double(e.pla[i]); o[12] = double(e.epsd[i]);
  } else if (j < nh + nq) {
    const Q4Ptrs<S> q = q4_ptrs<S>(M);
    const int64_t i = q4[j - nh];
    const gptr<double> o = to_global(qout) + (12 + npt) * (j - nh);
#pragma unroll
    for (int k = 0; k < 5; ++k) o[k] = double(q.forc[(int64_t)k * q.ne + i]);
#pragma unroll
    for (int k = 0; k < 3; ++k) o[5 + k] = double(q.mom[(int64_t)k * q.ne + i]);
    o[8] = double(q.eint[i]); o[9] = double(q.eint[q.ne + i]);
    o[10] = double(q.offg[i]); o[11] = double(q.thk[i]);
    for (int k = 0; k < npt; ++k) o[12 + k] = double(q.pla[(int64_t)k * q.ne + i]);
  }
}

// EHOUR: the tiles' accumulators, solid tiles then shell tiles, summed in a fixed order.
__global__ __launch_bounds__(kBlock) void k_th_ehour(const double *h, int64_t nh, const double *q, int64_t nq,
                                                     double *out) {
  double v = 0.0;
  for (int64_t j = threadIdx.x; j < nh + nq; j += kBlock) v = v + (j < nh ? h[j] : q[j - nh]);
  v = block_sum(v);
  if (threadIdx.x == 0) *out = v;
}

// ---------------------------------------------------------------- group drop-in kernels
// SFORC3 on one group with the reference host layouts (X(3,*), V(3,*), IXS(11,*),
// SIG(NEL,6), FSKY(8,*), IADS(8,*) 1-based).
__global__ __launch_bounds__(kBlock) void k_sforc3_group(int nel, int64_t nft, const double *x, const double *v,
                                                         const int32_t *ixs, double *sig, double *eint, double *rho,
                                                         const double *vol, double *pla, double *epsd,
                                                         double *off, double *qvis, double *fsky,
                                                         const int32_t *iads, HexConsts c, double dt1,
                                                         double *dtx_out, int *mstop_out) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= nel) return;
  const int64_t col = nft + i; // 0-based column of IXS / IADS
  double xd[8], yd[8], zd[8], vx[8], vy[8], vz[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int64_t n = (int64_t)ixs[11 * col + 1 + k] - 1;
    xd[k] = x[3 * n]; yd[k] = x[3 * n + 1]; zd[k] = x[3 * n + 2];
    vx[k] = v[3 * n]; vy[k] = v[3 * n + 1]; vz[k] = v[3 * n + 2];
  }
  HexState<double> st;
#pragma unroll
  for (int k = 0; k < 6; ++k) st.sig[k] = sig[(int64_t)k * nel + i];
  st.eint = eint[i]; st.rho = rho[i]; st.vol0 = vol[i]; st.pla = pla[i];
  st.epsd = epsd[i]; st.offg = off[i]; st.qvis = qvis[i];
  HexOut<double> o;
  auto write_row = [&](int k, double fx, double fy, double fz) {
    const int64_t K = (int64_t)iads[8 * col + k] - 1;
    fsky[8 * K + 0] = fx;
    fsky[8 * K + 1] = fy;
    fsky[8 * K + 2] = fz;
    fsky[8 * K + 6] = o.sti4;
  };
  hex_element<double, double>(xd, yd, zd, vx, vy, vz, st, c, dt1, o, write_row, [] {});
#pragma unroll
  for (int k = 0; k < 6; ++k) sig[(int64_t)k * nel + i] = st.sig[k];
  eint[i] = st.eint; rho[i] = st.rho; pla[i] = st.pla;
  epsd[i] = st.epsd; off[i] = st.offg; qvis[i] = st.qvis;
  dtx_out[i] = o.dtx;
  mstop_out[i] = o.mstop;
}

// SFORC3 on one group staged in page-locked host memory, which the kernel reads and writes
// over the bus: w holds, nel values each, X and V of the elements' nodes (8 corners x 3), the
// GBUF arrays (SIG 6, EINT, RHO, VOL, PLA, EPSD, OFF, QVIS; updated in place), then the rows'
// written words (8 corners x FX, FY, FZ, STI), DTX and MSTOP.  About 0.9 KB an element cross the
// bus in two round trips; two copies and a kernel on device memory need two launches more.
constexpr int kHexStageState = 48, kHexStageRows = 61, kHexStageDt = 93, kHexStageWords = 95;
__global__ __launch_bounds__(kBlock) void k_sforc3_staged(int nel, double *w, HexConsts c, double dt1) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= nel) return;
  const gptr<double> p = to_global(w) + i;
  double xd[8], yd[8], zd[8], vx[8], vy[8], vz[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    xd[k] = p[(3 * k) * nel]; yd[k] = p[(3 * k + 1) * nel]; zd[k] = p[(3 * k + 2) * nel];
    vx[k] = p[(24 + 3 * k) * nel]; vy[k] = p[(25 + 3 * k) * nel]; vz[k] = p[(26 + 3 * k) * nel];
  }
  const gptr<double> g = p + kHexStageState * nel;
  HexState<double> st;
#pragma unroll
  for (int k = 0; k < 6; ++k) st.sig[k] = g[k * nel];
  st.eint = g[6 * nel]; st.rho = g[7 * nel]; st.vol0 = g[8 * nel]; st.pla = g[9 * nel];
  st.epsd = g[10 * nel]; st.offg = g[11 * nel]; st.qvis = g[12 * nel];
  HexOut<double> o;
  const gptr<double> r = p + kHexStageRows * nel;
  auto write_row = [&](int k, double fx, double fy, double fz) {
    r[(4 * k) * nel] = fx; r[(4 * k + 1) * nel] = fy; r[(4 * k + 2) * nel] = fz; r[(4 * k + 3) * nel] = o.sti4;
  };
  hex_element<double, double>(xd, yd, zd, vx, vy, vz, st, c, dt1, o, write_row, [] {});
#pragma unroll
  for (int k = 0; k < 6; ++k) g[k * nel] = st.sig[k];
  g[6 * nel] = st.eint; g[7 * nel] = st.rho; g[9 * nel] = st.pla;
  g[10 * nel] = st.epsd; g[11 * nel] = st.offg; g[12 * nel] = st.qvis;
  p[kHexStageDt * nel] = o.dtx;
  p[(kHexStageDt + 1) * nel] = o.mstop;
}

// Per-point state of the CFORC3 drop-in: LBUF arrays of one group, SIG(NEL,5) per point.
struct GroupIpIO {
  double *sig, *pla, *epsd_ip, *gstr, *hourg, *eint, *forc, *mom;
  int nel, i;
  double s_next[5], pla_next, epsd_next; // each point's state, loaded one point ahead
  int npt;
  __device__ __forceinline__ void begin() { load(0, s_next, pla_next, epsd_next); }
  __device__ __forceinline__ void fetch(int ip, double (&s)[5], double &p, double &e) {
#pragma unroll
    for (int k = 0; k < 5; ++k) s[k] = s_next[k];
    p = pla_next; e = epsd_next;
    if (ip + 1 < npt) load(ip + 1, s_next, pla_next, epsd_next);
  }
  __device__ __forceinline__ void late_load(Q4Late<double> &L) const {
#pragma unroll
    for (int k = 0; k < 5; ++k) L.forc[k] = forc[(int64_t)k * nel + i];
#pragma unroll
    for (int k = 0; k < 3; ++k) L.mom[k] = mom[(int64_t)k * nel + i];
#pragma unroll
    for (int k = 0; k < 8; ++k) L.gstr[k] = gstr[(int64_t)k * nel + i];
#pragma unroll
    for (int k = 0; k < 3; ++k) L.hourg[k] = hourg[(int64_t)k * nel + i];
    L.eint[0] = eint[i];
    L.eint[1] = eint[nel + i];
  }
  __device__ __forceinline__ void late_store(const Q4Late<double> &L) const {
#pragma unroll
    for (int k = 0; k < 5; ++k) forc[(int64_t)k * nel + i] = L.forc[k];
#pragma unroll
    for (int k = 0; k < 3; ++k) mom[(int64_t)k * nel + i] = L.mom[k];
#pragma unroll
    for (int k = 0; k < 8; ++k) gstr[(int64_t)k * nel + i] = L.gstr[k];
    eint[i] = L.eint[0];
    eint[nel + i] = L.eint[1];
  }
  __device__ __forceinline__ void hourg_store(const double (&h)[5]) const {
#pragma unroll
    for (int k = 0; k < 5; ++k) hourg[(int64_t)k * nel + i] = h[k];
  }
  __device__ __forceinline__ void load(int ip, double (&s)[5], double &p, double &e) const {
#pragma unroll
    for (int k = 0; k < 5; ++k) s[k] = sig[((int64_t)ip * 5 + k) * nel + i];
    p = pla[(int64_t)ip * nel + i];
    e = epsd_ip[(int64_t)ip * nel + i];
  }
  __device__ __forceinline__ void store(int ip, const double (&s)[5], double p, double e) const {
#pragma unroll
    for (int k = 0; k < 5; ++k) sig[((int64_t)ip * 5 + k) * nel + i] = s[k];
    pla[(int64_t)ip * nel + i] = p;
    epsd_ip[(int64_t)ip * nel + i] = e;
  }
};

// CFORC3 on one group staged in page-locked host memory as k_sforc3_staged's: X, V and VR of the
// nodes (4 corners x 3 each), whether the element is a triangle, OFF, THK, THKE, EPSD, FOR 5,
// MOM 3, STRA 8, HOURG 5, EINT 2, the rows' words 1..7 (4 corners) and DT; then for each point
// SIG 5, and after them all PLA and all EPSD, as LBUF lays them out.
constexpr int kQ4StageState = 36, kQ4StageRows = 64, kQ4StageDt = 92, kQ4StagePoints = 93;
__host__ __device__ constexpr int q4_stage_words(int npt) { return kQ4StagePoints + 7 * npt; }
__global__ __launch_bounds__(kBlock) void k_cforc3_staged(int nel, double *w, Q4Consts c, double dt1) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= nel) return;
  const gptr<double> p = to_global(w) + i;
  double xg[4], yg[4], zg[4], vl[4][3], vrl[4][3];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    xg[k] = p[(3 * k) * nel]; yg[k] = p[(3 * k + 1) * nel]; zg[k] = p[(3 * k + 2) * nel];
#pragma unroll
    for (int d = 0; d < 3; ++d) { vl[k][d] = p[(12 + 3 * k + d) * nel]; vrl[k][d] = p[(24 + 3 * k + d) * nel]; }
  }
  const gptr<double> g = p + kQ4StageState * nel;
  const bool tri = g[0] != 0.0;
  Q4Elem<double> st;
  st.offg = g[nel]; st.thk = g[2 * nel]; st.thke = g[3 * nel]; st.epsd = g[4 * nel];
  double *s = w + kQ4StageState * (int64_t)nel;
  double *q = w + kQ4StagePoints * (int64_t)nel;
  GroupIpIO io{q, q + 5 * c.npt * nel, q + 6 * c.npt * nel, s + 13 * nel, s + 21 * nel, s + 26 * nel, s + 5 * nel,
               s + 10 * nel, nel, i};
  io.npt = c.npt;
  Q4Out<double> o;
  auto nload = [&](int k, double(&x)[3], double(&v)[3]) {
#pragma unroll
    for (int d = 0; d < 3; ++d) { x[d] = p[(3 * k + d) * nel]; v[d] = p[(12 + 3 * k + d) * nel]; }
  };
  q4_element<double>(xg, yg, zg, vl, vrl, tri, st, c, dt1, io, nload, o);
  g[nel] = st.offg; g[2 * nel] = st.thk; g[4 * nel] = st.epsd;
  const gptr<double> r = p + kQ4StageRows * nel;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
#pragma unroll
    for (int d = 0; d < 3; ++d) { r[(7 * k + d) * nel] = -o.f[d][k]; r[(7 * k + 3 + d) * nel] = -o.m[d][k]; }
    r[(7 * k + 6) * nel] = o.sti;
  }
  p[kQ4StageDt * nel] = o.dt;
}

// Nodal half of a cycle on the reference host layouts: ASSPAR4 over FSKY(8,LSKY) rows
// listed by ADSKY (1-based CSR, FILLCNE order), ACCELE, BCS10, FIXVEL, VELOCITY, DEPLA on
// X/V/VR/D(3,NUMNOD).  DT12 and DT2 are the cycle's, from the DT2 pipeline on the host.
__global__ __launch_bounds__(kBlock) void k_nodal_dropin(int64_t nn, const int64_t *adsky, const double *fsky,
                                                         const double *ms, const double *in, const int32_t *code,
                                                         const double *vimp, double *x, double *v, double *vr,
                                                         double *d, double *stifn, double *stifr, double DT12,
                                                         double DT2) {
  const int64_t n = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (n >= nn) return;
  // ASSPAR4 (asspar4.F:164-180)
  double ax = 0.0, ay = 0.0, az = 0.0, rx = 0.0, ry = 0.0, rz = 0.0, sn = 0.0, sr = 0.0;
  for (int64_t k = adsky[n] - 1; k < adsky[n + 1] - 1; ++k) {
    const double *f = fsky + 8 * k;
    ax = ax + f[0]; ay = ay + f[1]; az = az + f[2];
    rx = rx + f[3]; ry = ry + f[4]; rz = rz + f[5];
    sn = sn + f[6]; sr = sr + f[7];
  }
  if (stifn) stifn[n] = sn;
  if (stifr) stifr[n] = sr;
  accele3(ax, ay, az, ms[n]);
  const bool rot = vr != nullptr;
  double wx = 0.0, wy = 0.0, wz = 0.0;
  if (rot) {
    accele3(rx, ry, rz, in[n]);
    wx = vr[3 * n]; wy = vr[3 * n + 1]; wz = vr[3 * n + 2];
  }
  double vx = v[3 * n], vy = v[3 * n + 1], vz = v[3 * n + 2];
  const int32_t cd = code ? code[n] : 0;
  if (cd) {
    double work = 0.0, pend = 0.0; // the drop-in reports no external work (the caller's FIXVEL keeps WFEXT)
    bcs_fixvel(cd, ax, ay, az, vx, vy, vz, rx, ry, rz, wx, wy, wz, vimp + 3 * n, DT12, 0.0, 0.0, ms[n], work, pend);
  }
  // VELOCITY (velocity.F:58-86)
  vx = vx + DT12 * ax; vy = vy + DT12 * ay; vz = vz + DT12 * az;
  v[3 * n] = vx; v[3 * n + 1] = vy; v[3 * n + 2] = vz;
  if (rot) {
    wx = wx + DT12 * rx; wy = wy + DT12 * ry; wz = wz + DT12 * rz;
    vr[3 * n] = wx; vr[3 * n + 1] = wy; vr[3 * n + 2] = wz;
  }
  // DEPLA (displacement.F:108-118)
  double vdt;
  vdt = DT2 * vx; d[3 * n] = d[3 * n] + vdt; x[3 * n] = x[3 * n] + vdt;
  vdt = DT2 * vy; d[3 * n + 1] = d[3 * n + 1] + vdt; x[3 * n + 1] = x[3 * n + 1] + vdt;
  vdt = DT2 * vz; d[3 * n + 2] = d[3 * n + 2] + vdt; x[3 * n + 2] = x[3 * n + 2] + vdt;
}

// ---------------------------------------------------------------- read-back
// Values [i0, i1) of an array as the caller lays it out, written to page-locked host memory over
// the bus.  Element arrays [ncomp][ne] leave in element order (slot: element -> storage slot),
// widened to FP64; node arrays [n][3] leave from records of `stride` words.
template <typename S>
__global__ __launch_bounds__(kBlock) void k_export_elements(double *dst, const S *src, const int32_t *slot, int64_t ne,
                                                            int64_t i0, int64_t i1) {
  for (int64_t i = i0 + (int64_t)blockIdx.x * kBlock + threadIdx.x; i < i1; i += (int64_t)gridDim.x * kBlock) {
    const int64_t k = i / ne;
    to_global(dst)[i - i0] = double(to_global(src)[k * ne + to_global(slot)[i - k * ne]]);
  }
}
__global__ __launch_bounds__(kBlock) void k_export_nodes(double *dst, const double *src, int stride, int64_t i0,
                                                         int64_t i1) {
  for (int64_t i = i0 + (int64_t)blockIdx.x * kBlock + threadIdx.x; i < i1; i += (int64_t)gridDim.x * kBlock) {
    const int64_t n = i / 3;
    to_global(dst)[i - i0] = to_global(src)[n * stride + (i - 3 * n)];
  }
}

// ---------------------------------------------------------------- host helpers
double host_onep333() {
  volatile double zep3 = 3.0 / 10.0, zep03 = 3.0 / 100.0, threeem3 = 3.0 / 1000.0;
  volatile double onep3 = 1.0 + zep3;
  volatile double onep33 = onep3 + zep03;
  return onep33 + threeem3;
}

HexConsts make_hex_consts(const or_hex_params &p) {
  HexConsts c;
  c.rho0 = p.rho0; c.bulk = p.bulk; c.shear = p.shear; c.ca = p.ca; c.cb = p.cb; c.cn = p.cn;
  c.epmx = p.epmx; c.sigmx = p.sigmx; c.cc = p.cc; c.epdr = p.epdr; c.fisokin = p.fisokin;
  c.asrate = p.asrate; c.m_exp = p.m_exp; c.icc = p.icc; c.vp = p.vp; c.israte = p.israte;
  c.iform = p.iform; c.qa = p.qa; c.qb = p.qb; c.qh = p.qh; c.vns1 = p.vns1; c.vns2 = p.vns2;
  c.dtfac = p.dtfac; c.dtmx = p.dtmx;
  c.onep333 = host_onep333();
  c.dt_growth = (double)1.1f;
  return c;
}

int check_hex_params(const or_hex_params &p) {
  if (p.fisokin != 0.0) return fail(OR_ERR_ARG, "law 2 kinematic hardening (FISOKIN>0) is not on this path");
  if (p.iform != 0) return fail(OR_ERR_ARG, "law 2 Zerilli form (IFORM=1) is not on this path");
  // VP=1 (plastic strain rate) filters EPSD after the return (m2law.F:536-544) with the Starter's
  // default cut-off frequency; that update is not on this path
  if (p.vp != 2 && p.vp != 3) return fail(OR_ERR_ARG, "law 2 hexes: VP must be 2 (total) or 3 (deviatoric strain rate)");
  if (!(p.rho0 > 0.0) || !(p.dtfac > 0.0)) return fail(OR_ERR_ARG, "rho0 and dtfac must be positive");
  return OR_OK;
}

// Tables of COQINI (coqini.F:46-152), single-precision DATA literals.
const float kZ0[11][11] = {
    {0.f}, {-.5f, 0.5f}, {-.5f, 0.f, 0.5f}, {-.5f, -.1666667f, 0.1666667f, 0.5f}, {-.5f, -.25f, 0.f, 0.25f, 0.5f},
    {-.5f, -.3f, -.1f, 0.1f, 0.3f, 0.5f}, {-.5f, -.3333333f, -.1666667f, 0.0f, 0.1666667f, 0.3333333f, 0.5f},
    {-.5f, -.3571429f, -.2142857f, -.0714286f, 0.0714286f, 0.2142857f, 0.3571429f, 0.5f},
    {-.5f, -.375f, -.25f, -.125f, 0.0f, 0.125f, 0.25f, 0.375f, 0.5f},
    {-.5f, -.3888889f, -.2777778f, -.1666667f, -.0555555f, 0.0555555f, 0.1666667f, 0.2777778f, 0.3888889f, 0.5f},
    {-.5f, -.4f, -.3f, -.2f, -.1f, 0.f, 0.1f, 0.2f, 0.3f, 0.4f, 0.5f}};
const float kWF[11][11] = {
    {1.f}, {0.5f, 0.5f}, {0.25f, 0.5f, 0.25f}, {0.1666667f, 0.3333333f, 0.3333333f, 0.1666667f},
    {0.125f, 0.25f, 0.25f, 0.25f, 0.125f}, {0.1f, 0.2f, 0.2f, 0.2f, 0.2f, 0.1f},
    {0.0833333f, 0.1666667f, 0.1666667f, 0.1666667f, 0.1666667f, 0.1666667f, 0.0833333f},
    {0.0714286f, 0.1428571f, 0.1428571f, 0.1428571f, 0.1428571f, 0.1428571f, 0.1428571f, 0.0714286f},
    {0.0625f, 0.125f, 0.125f, 0.125f, 0.125f, 0.125f, 0.125f, 0.125f, 0.0625f},
    {0.0555556f, 0.1111111f, 0.1111111f, 0.1111111f, 0.1111111f, 0.1111111f, 0.1111111f, 0.1111111f, 0.1111111f,
     0.0555556f},
    {0.05f, 0.1f, 0.1f, 0.1f, 0.1f, 0.1f, 0.1f, 0.1f, 0.1f, 0.1f, 0.05f}};
const float kWM[11][11] = {
    {0.f}, {-.0833333f, 0.0833333f}, {-.0833333f, 0.f, 0.0833333f}, {-.0648148f, -.0555556f, 0.0555556f, 0.0648148f},
    {-.0520833f, -.0625f, 0.f, 0.0625f, 0.0520833f},
    {-.0433333f, -.0600000f, -.0200000f, 0.0200000f, 0.0600000f, 0.0433333f},
    {-.0370370f, -.0555556f, -.0277778f, 0.0000000f, 0.0277778f, 0.0555556f, 0.0370370f},
    {-.0323129f, -.0510204f, -.0306122f, -.0102041f, 0.0102041f, 0.0306122f, 0.0510204f, 0.0323129f},
    {-.0286458f, -.0468750f, -.0312500f, -.0156250f, 0.0000000f, 0.0156250f, 0.0312500f, 0.0468750f, 0.0286458f},
    {-.0257202f, -.0432099f, -.0308642f, -.0185185f, -.0061728f, 0.0061728f, 0.0185185f, 0.0308642f, 0.0432099f,
     0.0257202f},
    {-.0233333f, -.0400000f, -.0300000f, -.0200000f, -.0100000f, 0.0000000f, 0.0100000f, 0.0200000f, 0.0300000f,
     0.0400000f, 0.0233333f}};

int make_q4_consts(const or_q4_params &p, Q4Consts &c) {
  if (p.npt < 2 || p.npt > 10) return fail(OR_ERR_ARG, "shell NPT must be in 2..10 (NPT=1 uses MHVIS3, not on this path)");
  if (p.ipla < 0 || p.ipla > 2) return fail(OR_ERR_ARG, "Iplas must be 0, 1 or 2");
  if (p.iform != 0) return fail(OR_ERR_ARG, "law 2 Zerilli form (IFORM=1) is not on this path");
  if (p.vp != 2) return fail(OR_ERR_ARG, "law 2 shells: only VP=2 (total strain rate) is on this path");
  if (!(p.rho > 0.0) || !(p.young > 0.0) || !(p.dtfac > 0.0) || !(p.ssp > 0.0))
    return fail(OR_ERR_ARG, "rho, young, ssp and dtfac must be positive");
  std::memset(&c, 0, sizeof(c));
  c.rho = p.rho; c.young = p.young; c.nu = p.nu; c.shear = p.shear; c.ssp = p.ssp; c.ca = p.ca; c.cb = p.cb;
  c.cn = p.cn; c.epmx = p.epmx; c.ymax = p.ymax; c.cc = p.cc; c.epdr = p.epdr; c.m_exp = p.m_exp;
  c.asrate = p.asrate; c.icc = p.icc; c.vp = p.vp; c.israte = p.israte; c.npt = p.npt; c.ipla = p.ipla;
  c.ithk = p.ithk; c.ishear = p.ishear; c.hm = p.hm; c.hf = p.hf; c.hr = p.hr; c.fsh = p.fsh; c.dtfac = p.dtfac;
  c.dtmin = p.dtmin;
  {
    volatile double a1 = p.young / (1.0 - p.nu * p.nu);
    c.a1 = a1;
    c.a2 = a1 * p.nu;
  }
  {
    volatile double zep1 = 1.0 / 10.0, zep01 = 1.0 / 100.0, zep03 = 3.0 / 100.0;
    volatile double zep09 = zep1 - zep01;
    volatile double zep19 = zep1 + zep09;
    c.zep81 = 1.0 - zep19;
    volatile double zep07 = zep1 - zep03, twoem3 = 2.0 / 1000.0;
    volatile double ep04 = (100.0 * 10.0) * 10.0, ep05 = ep04 * 10.0, ep06 = ep05 * 10.0;
    volatile double em04 = 1.0 / ep04, em05 = 1.0 / ep05, em06 = 1.0 / ep06;
    volatile double sixem5 = em04 - 4.0 / ep05, nineem6 = em05 - em06;
    volatile double s = zep07 + twoem3;
    s = s + em04;
    s = s + sixem5;
    c.zep072169 = s + nineem6;
    volatile double two = 2.0;
    c.sr2d2 = std::sqrt(two) * 0.5;
  }
  c.srh1 = std::sqrt(p.hm); c.srh2 = std::sqrt(p.hf); c.srh3 = std::sqrt(p.hr);
  for (int k = 0; k < p.npt; ++k) {
    c.z0[k] = (double)kZ0[p.npt - 1][k];
    c.wf[k] = (double)kWF[p.npt - 1][k];
    c.wm[k] = (double)kWM[p.npt - 1][k];
  }
  return OR_OK;
}

#ifndef OR_ILP_TU
// The buffers kept between calls (or_staging.h): allocating and freeing one costs more than a group's
// whole call (2.0 ms with 15 of them, 0.05 ms now, of which the kernel is 0.02).
struct HipMem {
  static int alloc(int device, size_t bytes, void **p) {
    const hipError_t e = device < 0 ? hipHostMalloc(p, bytes, hipHostMallocPortable | hipHostMallocMapped)
                                    : hipMalloc(p, bytes);
    if (e != hipSuccess) (void)hipGetLastError(); // reported here, not by the thread's next launch
    return (int)e;
  }
  static void free(int device, void *p) { (void)(device < 0 ? hipHostFree(p) : hipFree(p)); }
};
typedef orstage::BufferPool<HipMem> StagePool;
StagePool &stage_pool() {
  static StagePool *pool = new StagePool; // outlives every static object
  return *pool;
}

// hipMalloc on the current device; when memory runs out, once more without the idle workspaces.
hipError_t device_alloc(void **p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  int device = 0;
  if (e == hipErrorOutOfMemory && hipGetDevice(&device) == hipSuccess && stage_pool().drop(device, 0)) {
    (void)hipGetLastError();
    e = hipMalloc(p, bytes);
  }
  return e;
}

template <typename T> int dalloc(T **p, int64_t n, int64_t &acc) {
  if (n <= 0) { *p = nullptr; return OR_OK; }
  OR_HIP(device_alloc((void **)p, sizeof(T) * (size_t)n));
  acc += (int64_t)(sizeof(T) * (size_t)n);
  return OR_OK;
}

#endif // OR_ILP_TU

} // namespace

#ifndef OR_ILP_TU
// ============================================================== staging
namespace {

struct Lease {
  StagePool::Buf b; // given back at the end of the scope
  Lease() = default;
  Lease(const Lease &) = delete;
  Lease &operator=(const Lease &) = delete;
  ~Lease() {
    static std::once_flag exit_handler; // runs before the HIP runtime's own, which is there by now
    if (b.p) std::call_once(exit_handler, [] { (void)std::atexit([] { stage_pool().clear(); }); });
    stage_pool().give(b);
  }
  hipError_t take(int device, size_t bytes) { return (hipError_t)stage_pool().take(device, bytes, b); }
  double *d() const { return (double *)b.p; }
};

// Transfers between the caller's pageable arrays and device memory, cut into chunks of at most
// kChunk doubles that go through page-locked buffers.  A transfer of some MB is bound by the
// CPU's copies (and the first touch of the caller's fresh pages), 10 GB/s a thread against 50 of
// the bus, so a few threads take the chunks in turn, each with its own buffer and event.
struct Chunk {
  enum Kind { kUp, kUpElem64, kUpElem32, kDown, kNodes, kElem64, kElem32 } kind;
  void *host;        // the caller's memory
  void *dev;         // device array (kUp, kDown: the chunk's bytes; else the whole array)
  size_t bytes;      // of the chunk, at most 8 * kChunk
  int64_t i0;        // element and node arrays: first value
  int64_t ne;        // kNodes: record stride; element arrays: elements
  const int32_t *slot; // kElem*: element -> slot (device); kUpElem*: slot -> element (host)
};
class Chunks {
 public:
  static constexpr int64_t kChunk = 1 << 18; // 2 MB
  static constexpr int kThreads = 6;
  void bytes(Chunk::Kind kind, const void *host, void *dev, size_t n) {
    for (size_t o = 0; o < n; o += 8 * kChunk)
      c_.push_back(Chunk{kind, (char *)const_cast<void *>(host) + o, (char *)dev + o, std::min<size_t>(n - o, 8 * kChunk), 0, 0, nullptr});
  }
  void values(Chunk::Kind kind, double *host, const void *dev, int64_t n, int64_t ne, const int32_t *slot) {
    if (!host) return;
    const bool up = kind == Chunk::kUpElem64 || kind == Chunk::kUpElem32; // these index the whole array
    for (int64_t o = 0; o < n; o += kChunk)
      c_.push_back(Chunk{kind, host + (up ? 0 : o), const_cast<void *>(dev), 8 * (size_t)std::min<int64_t>(n - o, kChunk), o, ne, slot});
  }
  hipError_t run(int device, hipStream_t st) {
    if (c_.empty()) return hipSuccess;
    size_t total = 0;
    for (const Chunk &c : c_) total += c.bytes;
    // a thread costs some 30 us to start, the time of 0.3 MB
    const int nt = (int)std::min<size_t>({(size_t)kThreads, c_.size(), 1 + (total >> 20)});
    const int e = orstage::run_team(nt, c_.size(), [&] { return Worker{c_, device, st}; });
    c_.clear();
    return (hipError_t)e;
  }

 private:
  // One thread's buffer and event.  Chunks follow each other in the buffer; when it has no room for the next,
  // and at the end, the thread waits for those in it and hands the downloads among them to the caller, so
  // that a small model's arrays cost one wait together (the four node arrays of 64 hexes and 64 shells 27 us, 85
  // with a wait for each, 53 by blocking copies; 15,000 nodes 98, 144 and 135).
  struct Worker {
    const std::vector<Chunk> &chunks;
    int device;
    hipStream_t st;
    Lease buf{};
    hipEvent_t ev = nullptr;
    size_t used = 0;          // of the buffer
    bool recorded = false;    // ev stands behind the chunks in the buffer
    static constexpr int kHeld = 32;
    struct { size_t chunk, at; } held[kHeld] = {}; // downloads in the buffer
    int nheld = 0;

    int begin() {
      hipError_t e = hipSetDevice(device);
      if (e == hipSuccess) e = buf.take(-1, 8 * kChunk);
      if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
      return (int)e;
    }
    int flush() {
      hipError_t e = hipSuccess;
      if (used == 0) return (int)e;
      if (!recorded) e = hipEventRecord(ev, st);
      if (e == hipSuccess) e = hipEventSynchronize(ev);
      for (int k = 0; k < nheld && e == hipSuccess; ++k)
        std::memcpy(chunks[held[k].chunk].host, (char *)buf.b.p + held[k].at, chunks[held[k].chunk].bytes);
      if (e != hipSuccess) (void)hipStreamSynchronize(st); // nothing may still use the buffer
      used = 0;
      nheld = 0;
      recorded = false;
      return (int)e;
    }
    int item(size_t index) {
      const Chunk &c = chunks[index];
      hipError_t e = hipSuccess;
      if (used + c.bytes > 8 * (size_t)kChunk || nheld == kHeld) e = (hipError_t)flush();
      if (e != hipSuccess) return (int)e;
      char *const at = (char *)buf.b.p + used;
      double *const d = (double *)at;
      const int64_t n = (int64_t)(c.bytes / 8);
      if (c.kind == Chunk::kUp || c.kind == Chunk::kUpElem64 || c.kind == Chunk::kUpElem32) {
        size_t b = c.bytes, to = 0;
        if (c.kind == Chunk::kUp) std::memcpy(at, c.host, c.bytes);
        else if (c.kind == Chunk::kUpElem64) permuted(c, (size_t)n, d), to = 8 * (size_t)c.i0;
        else permuted(c, (size_t)n, (float *)at), b = 4 * (size_t)n, to = 4 * (size_t)c.i0;
        e = hipMemcpyAsync((char *)c.dev + to, at, b, hipMemcpyHostToDevice, st);
      } else {
        const dim3 g((unsigned)std::min<int64_t>((n + kBlock - 1) / kBlock, 512));
        if (c.kind == Chunk::kDown) e = hipMemcpyAsync(at, c.dev, c.bytes, hipMemcpyDeviceToHost, st);
        else if (c.kind == Chunk::kNodes)
          hipLaunchKernelGGL(k_export_nodes, g, dim3(kBlock), 0, st, d, (const double *)c.dev, (int)c.ne, c.i0, c.i0 + n);
        else if (c.kind == Chunk::kElem64)
          hipLaunchKernelGGL(k_export_elements<double>, g, dim3(kBlock), 0, st, d, (const double *)c.dev, c.slot, c.ne, c.i0, c.i0 + n);
        else
          hipLaunchKernelGGL(k_export_elements<float>, g, dim3(kBlock), 0, st, d, (const float *)c.dev, c.slot, c.ne, c.i0, c.i0 + n);
        held[nheld].chunk = index;
        held[nheld++].at = used;
      }
      used += (c.bytes + 63) / 64 * 64;
      if (e == hipSuccess) e = hipGetLastError();
      // a full buffer: other threads' chunks on the stream are not waited for
      if (e == hipSuccess && used > 4 * (size_t)kChunk) {
        e = hipEventRecord(ev, st);
        recorded = true;
      } else {
        recorded = false;
      }
      return (int)e;
    }
    int end(int e) {
      const int f = e ? 0 : flush();
      if (e && used) (void)hipStreamSynchronize(st); // nothing of this call may still use the buffer
      return e ? e : f;
    }
    ~Worker() {
      if (ev) (void)hipEventDestroy(ev);
    }
  };
  template <typename S> static void permuted(const Chunk &c, size_t n, S *out) {
    const double *src = (const double *)c.host;
    int64_t k = c.i0 / c.ne, s = c.i0 - k * c.ne;
    for (size_t j = 0; j < n; ++j) {
      out[j] = (S)src[k * c.ne + c.slot[s]];
      if (++s == c.ne) { s = 0; ++k; }
    }
  }
  std::vector<Chunk> c_;
};

} // namespace

// ============================================================== model object
struct or_model {
  int device = 0;
  int prec = OR_PREC_FP64;
  int64_t nn = 0, neh = 0, neq = 0;
  int npt = 0;
  int64_t lsky_h = 0, lsky_q = 0;
  int64_t bytes = 0;
  hipStream_t stream = nullptr;
  bool have_hparams = false, have_qparams = false, have_nodes = false, have_hex = false, have_q4 = false,
       have_sky = false;
  HexConsts hc{};
  Q4Consts qc{};
  // nodes
  double *xv = nullptr, *vr = nullptr, *d = nullptr, *ms = nullptr, *in = nullptr, *vimp = nullptr;
  int32_t *code = nullptr, *deg_h = nullptr, *deg_q = nullptr, *rs_h = nullptr, *rs_q = nullptr;
  double *preh = nullptr, *preq = nullptr;
  int64_t sky_bytes = 0;               // rest rows and prefix lists, sized at upload_skyline
  // element storage order of each family: slot -> element (or_assembly.h tile_order); empty
  // until the first element upload, fixed after it
  std::vector<int32_t> hperm, qperm;
  int32_t *hslot = nullptr, *qslot = nullptr; // on the device: element -> slot
  int64_t asm_stats[4] = {0, 0, 0, 0}; // prefixes and rest rows of the hex and shell plans
  // hex (storage type depends on precision)
  int32_t *hconn = nullptr, *hrest = nullptr, *hfr_start = nullptr, *hfr_node = nullptr;
  uint16_t *hfr_src = nullptr;
  void *hsig = nullptr, *heint = nullptr, *hrho = nullptr, *hvol0 = nullptr, *hpla = nullptr, *hepsd = nullptr,
       *hoffg = nullptr, *hqvis = nullptr, *rowh = nullptr;
  // Q4
  int32_t *qconn = nullptr, *qrest = nullptr, *qfr_start = nullptr, *qfr_node = nullptr;
  uint16_t *qfr_src = nullptr;
  void *qoffg = nullptr, *qthk = nullptr, *qthke = nullptr, *qforc = nullptr, *qmom = nullptr, *qgstr = nullptr,
       *qhourg = nullptr, *qeint = nullptr, *qepsd = nullptr, *qsig = nullptr, *qpla = nullptr, *qepsdip = nullptr,
       *rowq = nullptr;
  // scalars
  DevTime *ts = nullptr;               // [2]
  unsigned long long *dtmin = nullptr; // [2]
  int *flags = nullptr;
  double *energy = nullptr;            // [kEnergySums * (1 + nb)]
  double *ecrit = nullptr;             // [5][nn] per-node ECRIT terms, allocated at the first output cycle
  double momentum[3] = {0.0, 0.0, 0.0}; // XMOMT, YMOMT, ZMOMT of the last output cycle
  // time history: the rows of its nodes (th_slot), their output-cycle values and the sampled
  // elements (th_buf: nodes [n][18], hexes [n][13], shells [n][12 + npt]), EHOUR per tile
  int32_t *th_slot = nullptr, *th_hex = nullptr, *th_q4 = nullptr;
  double *th_buf = nullptr, *ehou_h = nullptr, *ehou_q = nullptr;
  int64_t th_nn = 0, th_nh = 0, th_nq = 0;
  double *wext = nullptr;              // [2][nn] external work per node (and its deferred part), when
                                       // the model has imposed DOFs
  // the controlling element of output cycles: per-element candidates (storage order), the
  // element index of each storage slot, and the scan's words; allocated at the first output cycle
  double *dtel_h = nullptr, *dtel_q = nullptr;
  int32_t *lidx_h = nullptr, *lidx_q = nullptr;
  unsigned long long *ctrl = nullptr;  // [4]
  int64_t parity = 0;
  // what the kernels see (host copy, device copy) and the numbers of its tiles
  ModelDev hdev{};
  ModelDev *dev = nullptr;
  bool dev_dirty = true;
  int32_t nt_h = 0, nt_q = 0, nt_n = 0;
  int var_h = 0, var_q = 0;            // element kernel variants, as built
  or_batch *batch = nullptr;           // set while the model belongs to a batch
  // timing
  bool timing = false;
  std::vector<hipEvent_t> ev;          // ring of 4 events per cycle (hex | q4 | node)
  int ring_used = 0;
  double t_hex = 0.0, t_q4 = 0.0, t_node = 0.0;
  int64_t t_cycles = 0;
};

// A set of resident models advanced together: every cycle launches each kernel once
// per precision class over the tile lists of all live members (or_batch_*).
struct or_batch {
  int device = 0;
  hipStream_t stream = nullptr;
  std::vector<or_model *> members; // slot order
  std::vector<double> tend;        // per slot
  std::vector<char> live;          // per slot: still cycling (cleared by or_batch_active)
  ModelDev *md = nullptr;          // device array of the slots' kernel views
  int64_t md_cap = 0;
  Tile *tiles[2][3] = {};          // [precision][hex, q4, node]
  int var[2][2] = {};              // element kernel variants, as built [precision][hex, q4]
  int32_t nt[2][3] = {};
  int64_t tcap[2][3] = {};
  bool dirty = true;
  int64_t parity = 0;
  int64_t cycles = 0;              // cycles launched
};

// Wait for every stream that may hold work of the model (its own, and its batch's).
static hipError_t quiesce(or_model *m) {
  if (m->batch) {
    hipError_t e = hipStreamSynchronize(m->batch->stream);
    if (e != hipSuccess) return e;
  }
  return hipStreamSynchronize(m->stream);
}

// Small results of the model's work so far, read back behind it with one synchronisation: each
// blocking copy to pageable memory costs 13-25 us, as much as a cycle of a small model (400 cycles
// of 13,824 hexes + 2,304 shells with 19 time-history records: 22.2 ms, 17.7 with this).
struct ReadBack {
  void *dst;
  const void *src;
  size_t bytes;
};
static int read_back(or_model *m, std::initializer_list<ReadBack> items) {
  size_t total = 0;
  for (const ReadBack &r : items) total += (r.bytes + 15) / 16 * 16;
  Lease buf;
  OR_HIP(buf.take(-1, total));
  if (m->batch) OR_HIP(hipStreamSynchronize(m->batch->stream));
  char *at = (char *)buf.b.p;
  hipError_t e = hipSuccess;
  for (const ReadBack &r : items) {
    if (r.bytes && e == hipSuccess) e = hipMemcpyAsync(at, r.src, r.bytes, hipMemcpyDeviceToHost, m->stream);
    at += (r.bytes + 15) / 16 * 16;
  }
  const hipError_t f = hipStreamSynchronize(m->stream); // also after an error: the buffer goes back
  OR_HIP(e);
  OR_HIP(f);
  at = (char *)buf.b.p;
  for (const ReadBack &r : items) {
    if (r.bytes) std::memcpy(r.dst, at, r.bytes);
    at += (r.bytes + 15) / 16 * 16;
  }
  return OR_OK;
}

// Pointers or parameters of the model changed: its kernel views must be rebuilt.
static void mark_changed(or_model *m) {
  m->dev_dirty = true;
  if (m->batch) m->batch->dirty = true;
}

static size_t ssize(const or_model *m) { return m->prec == OR_PREC_FP64 ? sizeof(double) : sizeof(float); }

// Entry points: C linkage comes from their declarations in or_gpu.h.

int or_version(void) { return 200; }

const char *or_last_error(void) { return g_err.c_str(); }

int or_device_count(int *count) {
  if (!count) return fail(OR_ERR_ARG, "null count");
  int n = 0;
  hipError_t e = hipGetDeviceCount(&n);
  if (e != hipSuccess) { *count = 0; return fail(OR_ERR_NODEV, hipGetErrorString(e)); }
  *count = n;
  return OR_OK;
}

int or_device_memory(int device, int64_t *free_bytes, int64_t *total_bytes) {
  if (!free_bytes || !total_bytes) return fail(OR_ERR_ARG, "null argument");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return fail(OR_ERR_NODEV, "no HIP device");
  if (device < 0 || device >= ndev) return fail(OR_ERR_ARG, "device index out of range");
  OR_HIP(hipSetDevice(device));
  size_t f = 0, t = 0;
  OR_HIP(hipMemGetInfo(&f, &t));
  *free_bytes = (int64_t)f;
  *total_bytes = (int64_t)t;
  return OR_OK;
}

int or_model_create(or_model **out, int device, int64_t nn, int64_t ne_hex, int64_t ne_q4, int32_t npt,
                    int precision) {
  if (!out) return fail(OR_ERR_ARG, "null out");
  *out = nullptr;
  if (nn <= 0 || ne_hex < 0 || ne_q4 < 0) return fail(OR_ERR_ARG, "nn must be > 0, ne_hex and ne_q4 >= 0");
  if (ne_q4 > 0 && (npt < 2 || npt > 10)) return fail(OR_ERR_ARG, "shell NPT must be in 2..10");
  if (precision != OR_PREC_FP64 && precision != OR_PREC_SPLIT) return fail(OR_ERR_ARG, "bad precision");
  if (8 * ne_hex >= (int64_t)1 << 31 || 4 * ne_q4 >= (int64_t)1 << 31 || nn >= (int64_t)1 << 31)
    return fail(OR_ERR_ARG, "skyline rows and node ids must fit in int32");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return fail(OR_ERR_NODEV, "no HIP device");
  if (device < 0 || device >= ndev) return fail(OR_ERR_ARG, "device index out of range");
  OR_HIP(hipSetDevice(device));
  or_model *m = new or_model();
  m->device = device;
  m->prec = precision;
  m->nn = nn;
  m->neh = ne_hex;
  m->neq = ne_q4;
  m->npt = ne_q4 > 0 ? npt : 0;
  m->lsky_h = 8 * ne_hex;
  m->lsky_q = 4 * ne_q4;
  int rc = OR_OK;
  auto A = [&](auto **p, int64_t n) { if (rc == OR_OK) rc = dalloc(p, n, m->bytes); };
  const size_t ss = ssize(m);
  auto AS = [&](void **p, int64_t n) {
    if (rc != OR_OK || n <= 0) return;
    if (device_alloc(p, ss * (size_t)n) != hipSuccess) { rc = fail(OR_ERR_HIP, "hipMalloc state"); return; }
    m->bytes += (int64_t)(ss * (size_t)n);
  };
  A(&m->xv, 6 * nn);
  A(&m->d, 3 * nn);
  A(&m->ms, nn);
  A(&m->vimp, 3 * nn);
  A(&m->code, nn);
  if (ne_q4 > 0) {
    A(&m->vr, 4 * nn);
    A(&m->in, nn);
  }
  if (ne_hex > 0) {
    A(&m->deg_h, nn);
    A(&m->rs_h, nn + 1);
    A(&m->preh, 3 * nn);
    A(&m->hfr_start, (ne_hex + kTile - 1) / kTile + 1);
    A(&m->hconn, 8 * ne_hex);
    A(&m->hrest, 8 * ne_hex);
    A(&m->hslot, ne_hex);
    AS(&m->hsig, 6 * ne_hex);
    AS(&m->heint, ne_hex); AS(&m->hrho, ne_hex); AS(&m->hvol0, ne_hex); AS(&m->hpla, ne_hex);
    AS(&m->hepsd, ne_hex); AS(&m->hoffg, ne_hex); AS(&m->hqvis, ne_hex);
  }
  if (ne_q4 > 0) {
    A(&m->deg_q, nn);
    A(&m->rs_q, nn + 1);
    A(&m->preq, 6 * nn);
    A(&m->qfr_start, (ne_q4 + kTile - 1) / kTile + 1);
    A(&m->qconn, 4 * ne_q4);
    A(&m->qrest, 4 * ne_q4);
    A(&m->qslot, ne_q4);
    AS(&m->qoffg, ne_q4); AS(&m->qthk, ne_q4); AS(&m->qthke, ne_q4); AS(&m->qepsd, ne_q4);
    AS(&m->qforc, 5 * ne_q4); AS(&m->qmom, 3 * ne_q4); AS(&m->qgstr, 8 * ne_q4); AS(&m->qhourg, 5 * ne_q4);
    AS(&m->qeint, 2 * ne_q4);
    AS(&m->qsig, (int64_t)npt * 5 * ne_q4);
    AS(&m->qpla, (int64_t)npt * ne_q4);
  }
  A(&m->ts, 2);
  A(&m->dtmin, 2);
  A(&m->flags, 1);
  A(&m->dev, 1);
  m->nt_n = (int32_t)((nn + kBlock - 1) / kBlock);
  m->nt_h = (int32_t)((ne_hex + kTile - 1) / kTile);
  m->nt_q = (int32_t)((ne_q4 + kTile - 1) / kTile);
  const int64_t nb = 1024;
  A(&m->energy, kEnergySums * (1 + nb));
  if (rc == OR_OK && hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess)
    rc = fail(OR_ERR_HIP, "hipStreamCreate");
  if (rc == OR_OK) {
    if (hipMemsetAsync(m->d, 0, sizeof(double) * 3 * nn, m->stream) != hipSuccess ||
        hipMemsetAsync(m->code, 0, sizeof(int32_t) * nn, m->stream) != hipSuccess ||
        (m->hslot && hipMemsetAsync(m->hslot, 0, sizeof(int32_t) * ne_hex, m->stream) != hipSuccess) ||
        (m->qslot && hipMemsetAsync(m->qslot, 0, sizeof(int32_t) * ne_q4, m->stream) != hipSuccess) ||
        hipMemsetAsync(m->vimp, 0, sizeof(double) * 3 * nn, m->stream) != hipSuccess ||
        (m->vr && hipMemsetAsync(m->vr, 0, sizeof(double) * 4 * nn, m->stream) != hipSuccess) ||
        hipMemsetAsync(m->flags, 0, sizeof(int), m->stream) != hipSuccess)
      rc = fail(OR_ERR_HIP, "hipMemsetAsync init");
    DevTime t0{};
    t0.dt2old = 1.0e6 / (1.0 + 1.0 / 10.0); // DTINI/ONEP1 (starter contrl.F:1125-1127)
    DevTime tsh[2] = {t0, t0};
    unsigned long long dm[2];
    double big = kEP06;
    std::memcpy(&dm[0], &big, 8);
    dm[1] = dm[0];
    if (rc == OR_OK && (hipMemcpyAsync(m->ts, tsh, sizeof(tsh), hipMemcpyHostToDevice, m->stream) != hipSuccess ||
                        hipMemcpyAsync(m->dtmin, dm, sizeof(dm), hipMemcpyHostToDevice, m->stream) != hipSuccess ||
                        hipStreamSynchronize(m->stream) != hipSuccess))
      rc = fail(OR_ERR_HIP, "init scalars");
  }
  if (rc != OR_OK) {
    std::string keep = g_err;
    or_model_destroy(m);
    g_err = keep;
    return rc;
  }
  *out = m;
  return OR_OK;
}

int or_model_destroy(or_model *m) {
  if (!m) return OR_OK;
  if (m->batch) (void)or_batch_remove(m->batch, m);
  (void)hipSetDevice(m->device);
  if (m->stream) (void)hipStreamSynchronize(m->stream);
  void *ptrs[] = {m->xv, m->vr, m->d, m->ms, m->in, m->vimp, m->code, m->deg_h, m->deg_q, m->rs_h, m->rs_q,
                  m->preh, m->preq, m->hconn, m->hrest, m->hslot, m->qslot, m->hfr_start, m->hfr_node, m->hfr_src,
                  m->hsig, m->heint, m->hrho, m->hvol0, m->hpla, m->hepsd, m->hoffg, m->hqvis, m->rowh, m->qconn,
                  m->qrest, m->qfr_start, m->qfr_node, m->qfr_src, m->qoffg, m->qthk, m->qthke, m->qforc, m->qmom,
                  m->qgstr, m->qhourg, m->qeint, m->qepsd,
                  m->qsig, m->qpla, m->qepsdip, m->rowq, m->ts, m->dtmin, m->flags, m->energy, m->dev,
                  m->ecrit, m->wext, m->dtel_h, m->dtel_q, m->lidx_h,
                  m->lidx_q, m->ctrl, m->th_slot, m->th_hex, m->th_q4, m->th_buf, m->ehou_h, m->ehou_q};
  for (void *p : ptrs)
    if (p) (void)hipFree(p);
  for (hipEvent_t e : m->ev) (void)hipEventDestroy(e);
  if (m->stream) (void)hipStreamDestroy(m->stream);
  delete m;
  return OR_OK;
}

int or_model_set_hex_params(or_model *m, const or_hex_params *p) {
  if (!m || !p) return fail(OR_ERR_ARG, "null argument");
  int rc = check_hex_params(*p);
  if (rc) return rc;
  m->hc = make_hex_consts(*p);
  m->have_hparams = true;
  mark_changed(m);
  return OR_OK;
}

int or_model_set_q4_params(or_model *m, const or_q4_params *p) {
  if (!m || !p) return fail(OR_ERR_ARG, "null argument");
  if (m->neq > 0 && p->npt != m->npt) return fail(OR_ERR_ARG, "q4 params NPT differs from the model's NPT");
  Q4Consts c;
  int rc = make_q4_consts(*p, c);
  if (rc) return rc;
  // LBUF%EPSD is only distinct from GBUF%EPSD when the strain-rate filter is on (ASRATE < 1)
  if (c.israte > 0 && m->neq > 0 && !m->qepsdip) {
    const size_t ss = ssize(m);
    OR_HIP(hipSetDevice(m->device));
    OR_HIP(device_alloc(&m->qepsdip, ss * (size_t)(m->npt * m->neq)));
    OR_HIP(hipMemsetAsync(m->qepsdip, 0, ss * (size_t)(m->npt * m->neq), m->stream));
    OR_HIP(quiesce(m));
    m->bytes += (int64_t)(ss * (size_t)(m->npt * m->neq));
  }
  m->qc = c;
  m->have_qparams = true;
  mark_changed(m);
  return OR_OK;
}

int or_model_upload_nodes(or_model *m, const double *x, const double *v, const double *vr, const double *ms,
                          const double *in, const int32_t *code, const double *vimp) {
  if (!m || !x || !v || !ms) return fail(OR_ERR_ARG, "null argument");
  if (m->neq > 0 && !in) return fail(OR_ERR_ARG, "a model with shells needs nodal inertias IN");
  OR_HIP(hipSetDevice(m->device));
  const int64_t nn = m->nn;
  std::vector<double> xv((size_t)(6 * nn));
  for (int64_t n = 0; n < nn; ++n) {
    xv[6 * n + 0] = x[3 * n]; xv[6 * n + 1] = x[3 * n + 1]; xv[6 * n + 2] = x[3 * n + 2];
    xv[6 * n + 3] = v[3 * n]; xv[6 * n + 4] = v[3 * n + 1]; xv[6 * n + 5] = v[3 * n + 2];
    if (code && (code[n] & ~511)) return fail(OR_ERR_ARG, "node code has bits outside 0..511");
    if (code && (code[n] & (kIX | kIY | kIZ)) && !vimp)
      return fail(OR_ERR_ARG, "imposed-velocity bits given without vimp");
  }
  OR_HIP(hipMemcpyAsync(m->xv, xv.data(), sizeof(double) * 6 * nn, hipMemcpyHostToDevice, m->stream));
  OR_HIP(hipMemcpyAsync(m->ms, ms, sizeof(double) * nn, hipMemcpyHostToDevice, m->stream));
  if (code) OR_HIP(hipMemcpyAsync(m->code, code, sizeof(int32_t) * nn, hipMemcpyHostToDevice, m->stream));
  if (vimp) OR_HIP(hipMemcpyAsync(m->vimp, vimp, sizeof(double) * 3 * nn, hipMemcpyHostToDevice, m->stream));
  std::vector<double> vr4;
  if (m->vr) {
    vr4.assign((size_t)(4 * nn), 0.0);
    if (vr)
      for (int64_t n = 0; n < nn; ++n) {
        vr4[4 * n] = vr[3 * n]; vr4[4 * n + 1] = vr[3 * n + 1]; vr4[4 * n + 2] = vr[3 * n + 2];
      }
    OR_HIP(hipMemcpyAsync(m->vr, vr4.data(), sizeof(double) * 4 * nn, hipMemcpyHostToDevice, m->stream));
    OR_HIP(hipMemcpyAsync(m->in, in, sizeof(double) * nn, hipMemcpyHostToDevice, m->stream));
  }
  OR_HIP(hipMemsetAsync(m->d, 0, sizeof(double) * 3 * nn, m->stream));
  // external work of the imposed DOFs (FIXVEL's WFEXT), from zero at this upload
  bool imposed = false;
  for (int64_t n = 0; code && n < nn && !imposed; ++n) imposed = (code[n] & (kIX | kIY | kIZ)) != 0;
  if (imposed && !m->wext) {
    OR_HIP(quiesce(m));
    OR_HIP(device_alloc((void **)&m->wext, sizeof(double) * 2 * (size_t)nn));
    m->bytes += (int64_t)(sizeof(double) * 2 * nn);
    mark_changed(m);
  }
  if (m->wext) OR_HIP(hipMemsetAsync(m->wext, 0, sizeof(double) * 2 * (size_t)nn, m->stream));
  OR_HIP(quiesce(m));
  m->have_nodes = true;
  return OR_OK;
}

int or_model_upload_displacement(or_model *m, const double *d) {
  if (!m || !d) return fail(OR_ERR_ARG, "null argument");
  if (!m->have_nodes) return fail(OR_ERR_STATE, "upload the nodes before their displacements");
  OR_HIP(hipSetDevice(m->device));
  OR_HIP(quiesce(m));
  OR_HIP(hipMemcpyAsync(m->d, d, sizeof(double) * 3 * m->nn, hipMemcpyHostToDevice, m->stream));
  OR_HIP(quiesce(m));
  return OR_OK;
}

// Element arrays [ncomp][ne] move between the caller's element order and the storage
// order of slots (perm: slot -> element).  An absent one is filled with its default.
static int put_state(or_model *m, Chunks &io, void *dst, const double *src, int64_t n, double dflt,
                     const std::vector<int32_t> &perm) {
  if (!dst || n <= 0) return OR_OK;
  if (src) {
    io.values(m->prec == OR_PREC_FP64 ? Chunk::kUpElem64 : Chunk::kUpElem32, const_cast<double *>(src), dst, n,
              (int64_t)perm.size(), perm.data());
    return OR_OK;
  }
  if (m->prec == OR_PREC_FP64) OR_HIP(fill(m->stream, (double *)dst, n, dflt));
  else OR_HIP(fill(m->stream, (float *)dst, n, (float)dflt));
  return OR_OK;
}
// An element array of the caller's order, read back by the export kernels.
static int get_state(or_model *m, Chunks &io, double *dst, const void *src, int64_t n, int64_t ne, const int32_t *slot) {
  if (!dst || n <= 0) return OR_OK;
  if (!src) return fail(OR_ERR_STATE, "state array not held by this model");
  io.values(m->prec == OR_PREC_FP64 ? Chunk::kElem64 : Chunk::kElem32, dst, src, n, ne, slot);
  return OR_OK;
}

// The storage slot of every element, for the export kernels.
static std::vector<int32_t> slots_of(const std::vector<int32_t> &perm) {
  std::vector<int32_t> slot(perm.size());
  for (size_t s = 0; s < perm.size(); ++s) slot[(size_t)perm[s]] = (int32_t)s;
  return slot;
}

// Node coordinates on the host ([nn][3]), or empty before the nodes are uploaded.
static int host_coords(or_model *m, std::vector<double> &x) {
  x.clear();
  if (!m->have_nodes) return OR_OK;
  const int64_t nn = m->nn;
  std::vector<double> xv((size_t)(6 * nn));
  OR_HIP(quiesce(m));
  OR_HIP(hipMemcpy(xv.data(), m->xv, sizeof(double) * 6 * nn, hipMemcpyDeviceToHost));
  x.resize((size_t)(3 * nn));
  for (int64_t n = 0; n < nn; ++n)
    for (int d = 0; d < 3; ++d) x[(size_t)(3 * n + d)] = xv[(size_t)(6 * n + d)];
  return OR_OK;
}

// The storage order of a family is chosen at its first element upload: tiles from the
// node coordinates when the nodes are already uploaded, the caller's order otherwise.
static int choose_order(or_model *m, int nk, int64_t ne, const int32_t *conn, std::vector<int32_t> &perm) {
  if (!perm.empty() || ne == 0) return OR_OK;
  std::vector<double> x;
  int rc = host_coords(m, x);
  if (rc) return rc;
  perm = orasm::tile_order(nk, ne, conn, x.empty() ? nullptr : x.data());
  return OR_OK;
}

int or_model_upload_hex(or_model *m, const int32_t *conn, const double *sig, const double *eint, const double *rho,
                        const double *vol0, const double *pla, const double *epsd, const double *offg,
                        const double *qvis) {
  if (!m) return fail(OR_ERR_ARG, "null model");
  const int64_t ne = m->neh;
  if (ne == 0) { m->have_hex = true; return OR_OK; }
  if (!conn || !vol0 || !rho) return fail(OR_ERR_ARG, "conn, rho and vol0 are required");
  OR_HIP(hipSetDevice(m->device));
  for (int64_t j = 0; j < 8 * ne; ++j)
    if (conn[j] < 0 || conn[j] >= m->nn) return fail(OR_ERR_ARG, "connectivity node id out of range");
  if (m->have_hex && m->have_sky) {
    // the assembly plan holds this connectivity: a later upload may change the state only
    std::vector<int32_t> cur((size_t)(8 * ne));
    OR_HIP(hipMemcpy(cur.data(), m->hconn, sizeof(int32_t) * 8 * ne, hipMemcpyDeviceToHost));
    for (int64_t s = 0; s < ne; ++s)
      for (int k = 0; k < 8; ++k)
        if (cur[(size_t)(k * ne + s)] != conn[8 * (int64_t)m->hperm[(size_t)s] + k])
          return fail(OR_ERR_ARG, "hex connectivity differs from the one the skyline was uploaded for");
  }
  int rc = choose_order(m, 8, ne, conn, m->hperm);
  if (rc) return rc;
  const std::vector<int32_t> &perm = m->hperm;
  std::vector<int32_t> soa((size_t)(8 * ne));
  for (int64_t s = 0; s < ne; ++s)
    for (int k = 0; k < 8; ++k) soa[(size_t)(k * ne + s)] = conn[8 * (int64_t)perm[(size_t)s] + k];
  const std::vector<int32_t> slot = slots_of(perm);
  OR_HIP(quiesce(m)); // cycles of the model that still run use what is replaced here
  Chunks io;
  io.bytes(Chunk::kUp, soa.data(), m->hconn, sizeof(int32_t) * soa.size());
  io.bytes(Chunk::kUp, slot.data(), m->hslot, sizeof(int32_t) * slot.size());
  if ((rc = put_state(m, io, m->hsig, sig, 6 * ne, 0.0, perm))) return rc;
  if ((rc = put_state(m, io, m->heint, eint, ne, 0.0, perm))) return rc;
  if ((rc = put_state(m, io, m->hrho, rho, ne, 0.0, perm))) return rc;
  if ((rc = put_state(m, io, m->hvol0, vol0, ne, 0.0, perm))) return rc;
  if ((rc = put_state(m, io, m->hpla, pla, ne, 0.0, perm))) return rc;
  if ((rc = put_state(m, io, m->hepsd, epsd, ne, 0.0, perm))) return rc;
  if ((rc = put_state(m, io, m->hoffg, offg, ne, 1.0, perm))) return rc;
  if ((rc = put_state(m, io, m->hqvis, qvis, ne, 0.0, perm))) return rc;
  OR_HIP(io.run(m->device, m->stream));
  OR_HIP(quiesce(m));
  m->have_hex = true;
  return OR_OK;
}

int or_model_upload_q4(or_model *m, const int32_t *conn, const double *thke, const double *offg, const double *thk,
                       const double *forc, const double *mom, const double *gstr, const double *hourg,
                       const double *eint, const double *epsd, const double *sig, const double *pla,
                       const double *epsd_ip) {
  if (!m) return fail(OR_ERR_ARG, "null model");
  const int64_t ne = m->neq;
  if (ne == 0) { m->have_q4 = true; return OR_OK; }
  if (!conn || !thke) return fail(OR_ERR_ARG, "conn and thke are required");
  OR_HIP(hipSetDevice(m->device));
  for (int64_t e = 0; e < ne; ++e) {
    if (!(thke[e] > 0.0)) return fail(OR_ERR_ARG, "shell thickness must be positive");
    for (int k = 0; k < 4; ++k)
      if (conn[4 * e + k] < 0 || conn[4 * e + k] >= m->nn) return fail(OR_ERR_ARG, "connectivity node id out of range");
  }
  if (m->have_q4 && m->have_sky) {
    std::vector<int32_t> cur((size_t)(4 * ne));
    OR_HIP(hipMemcpy(cur.data(), m->qconn, sizeof(int32_t) * 4 * ne, hipMemcpyDeviceToHost));
    for (int64_t s = 0; s < ne; ++s)
      for (int k = 0; k < 4; ++k)
        if (cur[(size_t)(k * ne + s)] != conn[4 * (int64_t)m->qperm[(size_t)s] + k])
          return fail(OR_ERR_ARG, "shell connectivity differs from the one the skyline was uploaded for");
  }
  int rc = choose_order(m, 4, ne, conn, m->qperm);
  if (rc) return rc;
  const std::vector<int32_t> &perm = m->qperm;
  std::vector<int32_t> soa((size_t)(4 * ne));
  for (int64_t s = 0; s < ne; ++s)
    for (int k = 0; k < 4; ++k) soa[(size_t)(k * ne + s)] = conn[4 * (int64_t)perm[(size_t)s] + k];
  const std::vector<int32_t> slot = slots_of(perm);
  OR_HIP(quiesce(m)); // cycles of the model that still run use what is replaced here
  const int64_t np = m->npt;
  Chunks io;
  io.bytes(Chunk::kUp, soa.data(), m->qconn, sizeof(int32_t) * soa.size());
  io.bytes(Chunk::kUp, slot.data(), m->qslot, sizeof(int32_t) * slot.size());
  if ((rc = put_state(m, io, m->qthke, thke, ne, 0.0, perm))) return rc;
  if ((rc = put_state(m, io, m->qoffg, offg, ne, 1.0, perm))) return rc;
  if ((rc = put_state(m, io, m->qthk, thk ? thk : thke, ne, 0.0, perm))) return rc;
  if ((rc = put_state(m, io, m->qforc, forc, 5 * ne, 0.0, perm))) return rc;
  if ((rc = put_state(m, io, m->qmom, mom, 3 * ne, 0.0, perm))) return rc;
  if ((rc = put_state(m, io, m->qgstr, gstr, 8 * ne, 0.0, perm))) return rc;
  if ((rc = put_state(m, io, m->qhourg, hourg, 5 * ne, 0.0, perm))) return rc;
  if ((rc = put_state(m, io, m->qeint, eint, 2 * ne, 0.0, perm))) return rc;
  if ((rc = put_state(m, io, m->qepsd, epsd, ne, 0.0, perm))) return rc;
  if ((rc = put_state(m, io, m->qsig, sig, np * 5 * ne, 0.0, perm))) return rc;
  if ((rc = put_state(m, io, m->qpla, pla, np * ne, 0.0, perm))) return rc;
  if (m->qepsdip && (rc = put_state(m, io, m->qepsdip, epsd_ip, np * ne, 0.0, perm))) return rc;
  OR_HIP(io.run(m->device, m->stream));
  OR_HIP(quiesce(m));
  m->have_q4 = true;
  return OR_OK;
}

int or_model_upload_skyline(or_model *m, const int64_t *adsky, const int64_t *iads, const int64_t *iadc) {
  if (!m || !adsky) return fail(OR_ERR_ARG, "null argument");
  if ((m->neh > 0 && !iads) || (m->neq > 0 && !iadc)) return fail(OR_ERR_ARG, "missing iads / iadc");
  OR_HIP(hipSetDevice(m->device));
  const int64_t nn = m->nn, neh = m->neh, neq = m->neq;
  const int64_t lsky = m->lsky_h + m->lsky_q;
  if (adsky[0] != 0 || adsky[nn] != lsky) return fail(OR_ERR_ARG, "adsky must start at 0 and end at 8*ne_hex+4*ne_q4");
  for (int64_t n = 0; n < nn; ++n)
    if (adsky[n + 1] < adsky[n]) return fail(OR_ERR_ARG, "adsky must be non-decreasing");
  // owner node of every global row, and the family of every row
  std::vector<int32_t> owner((size_t)lsky);
  for (int64_t n = 0; n < nn; ++n)
    for (int64_t k = adsky[n]; k < adsky[n + 1]; ++k) owner[(size_t)k] = (int32_t)n;
  std::vector<int8_t> fam((size_t)lsky, -1);
  std::vector<int32_t> nh((size_t)nn, 0), nq((size_t)nn, 0);
  auto claim = [&](int64_t K, int f) -> int {
    if (K < 0 || K >= lsky) return fail(OR_ERR_ARG, "skyline row out of range");
    if (fam[(size_t)K] != -1) return fail(OR_ERR_ARG, "skyline rows must be distinct");
    fam[(size_t)K] = (int8_t)f;
    return OR_OK;
  };
  int rc;
  for (int64_t e = 0; e < neh; ++e)
    for (int k = 0; k < 8; ++k) {
      const int64_t K = iads[8 * e + k];
      if ((rc = claim(K, 0))) return rc;
      nh[(size_t)owner[(size_t)K]] += 1;
    }
  for (int64_t e = 0; e < neq; ++e)
    for (int k = 0; k < 4; ++k) {
      const int64_t K = iadc[4 * e + k];
      if ((rc = claim(K, 1))) return rc;
      nq[(size_t)owner[(size_t)K]] += 1;
    }
  // FILLCNE order: the solid rows of a node come before its shell rows
  for (int64_t n = 0; n < nn; ++n)
    for (int64_t k = adsky[n]; k < adsky[n + 1]; ++k)
      if ((k - adsky[n] < nh[(size_t)n]) != (fam[(size_t)k] == 0))
        return fail(OR_ERR_ARG, "skyline rows of a node must list solid rows before shell rows (FILLCNE order)");
  // element and corner of every row
  std::vector<int32_t> relem((size_t)lsky);
  std::vector<int8_t> rcorner((size_t)lsky);
  for (int64_t e = 0; e < neh; ++e)
    for (int k = 0; k < 8; ++k) { relem[(size_t)iads[8 * e + k]] = (int32_t)e; rcorner[(size_t)iads[8 * e + k]] = (int8_t)k; }
  for (int64_t e = 0; e < neq; ++e)
    for (int k = 0; k < 4; ++k) { relem[(size_t)iadc[4 * e + k]] = (int32_t)e; rcorner[(size_t)iadc[4 * e + k]] = (int8_t)k; }
  // the storage orders (chosen here if no element upload has chosen them yet)
  Chunks orders;
  std::vector<int32_t> slots[2];
  for (int f = 0; f < 2; ++f) {
    std::vector<int32_t> &perm = f == 0 ? m->hperm : m->qperm;
    const int64_t ne = f == 0 ? neh : neq;
    if (ne == 0 || (f == 0 ? m->have_hex : m->have_q4)) continue;
    if (perm.empty()) {
      perm.resize((size_t)ne);
      std::iota(perm.begin(), perm.end(), 0);
    }
    slots[f] = slots_of(perm);
    orders.bytes(Chunk::kUp, slots[f].data(), f == 0 ? m->hslot : m->qslot, sizeof(int32_t) * slots[f].size());
  }
  OR_HIP(orders.run(m->device, m->stream));
  // release the previous plan's arrays
  for (void **q : {&m->rowh, &m->rowq, (void **)&m->hfr_node, (void **)&m->hfr_src, (void **)&m->qfr_node,
                   (void **)&m->qfr_src})
    if (*q) { (void)hipFree(*q); *q = nullptr; }
  m->bytes -= m->sky_bytes;
  m->sky_bytes = 0;
  const size_t ss = ssize(m);
  for (int f = 0; f < 2; ++f) {
    const int64_t ne = f == 0 ? neh : neq;
    if (ne == 0) continue;
    const int nk = f == 0 ? 8 : 4, W = f == 0 ? kHexRowWords : kQ4RowWords;
    // the family's rows of every node, in the node's row order
    std::vector<int64_t> rptr((size_t)nn + 1, 0);
    std::vector<int32_t> fe;
    std::vector<int8_t> fk;
    std::vector<char> ok((size_t)nn);
    fe.reserve((size_t)(nk * ne));
    fk.reserve((size_t)(nk * ne));
    for (int64_t n = 0; n < nn; ++n) {
      const int64_t k0 = f == 0 ? adsky[n] : adsky[n] + nh[(size_t)n];
      const int64_t k1 = f == 0 ? adsky[n] + nh[(size_t)n] : adsky[n + 1];
      for (int64_t K = k0; K < k1; ++K) { fe.push_back(relem[(size_t)K]); fk.push_back(rcorner[(size_t)K]); }
      rptr[(size_t)n + 1] = (int64_t)fe.size();
      ok[(size_t)n] = (f == 0 || nh[(size_t)n] == 0) ? 1 : 0;
    }
    orasm::FamilyPlan plan;
    orasm::plan_family(plan, nk, ne, nn, f == 0 ? m->hperm : m->qperm, rptr, fe, fk, ok);
    const int64_t nfr = (int64_t)plan.fr_node.size();
    m->asm_stats[2 * f] = nfr;
    m->asm_stats[2 * f + 1] = plan.nrest;
    void **rows = f == 0 ? &m->rowh : &m->rowq;
    int32_t **frn = f == 0 ? &m->hfr_node : &m->qfr_node;
    uint16_t **frs = f == 0 ? &m->hfr_src : &m->qfr_src;
    const size_t nrow = ss * (size_t)(plan.nrest * W);
    OR_HIP(device_alloc(rows, nrow ? nrow : ss));
    OR_HIP(device_alloc((void **)frn, sizeof(int32_t) * (size_t)std::max<int64_t>(nfr, 1)));
    OR_HIP(device_alloc((void **)frs, sizeof(uint16_t) * orasm::kRunCap * (size_t)std::max<int64_t>(nfr, 1)));
    m->sky_bytes += (int64_t)(nrow + (4 + 2 * orasm::kRunCap) * (size_t)nfr);
    const std::vector<int32_t> &deg = f == 0 ? nh : nq;
    hipStream_t st = m->stream;
    OR_HIP(hipMemcpyAsync(f == 0 ? m->deg_h : m->deg_q, deg.data(), sizeof(int32_t) * nn, hipMemcpyHostToDevice, st));
    OR_HIP(hipMemcpyAsync(f == 0 ? m->rs_h : m->rs_q, plan.rs.data(), sizeof(int32_t) * (nn + 1), hipMemcpyHostToDevice, st));
    OR_HIP(hipMemcpyAsync(f == 0 ? m->hfr_start : m->qfr_start, plan.fr_start.data(),
                          sizeof(int32_t) * plan.fr_start.size(), hipMemcpyHostToDevice, st));
    if (nfr > 0) {
      OR_HIP(hipMemcpyAsync(*frn, plan.fr_node.data(), sizeof(int32_t) * nfr, hipMemcpyHostToDevice, st));
      OR_HIP(hipMemcpyAsync(*frs, plan.fr_src.data(), sizeof(uint16_t) * orasm::kRunCap * nfr, hipMemcpyHostToDevice, st));
    }
    OR_HIP(hipMemcpyAsync(f == 0 ? m->hrest : m->qrest, plan.rest.data(), sizeof(int32_t) * nk * ne,
                          hipMemcpyHostToDevice, st));
    OR_HIP(quiesce(m));
  }
  m->bytes += m->sky_bytes;
  m->have_sky = true;
  mark_changed(m);
  return OR_OK;
}

int or_model_set_time(or_model *m, const or_time_state *t) {
  if (!m || !t) return fail(OR_ERR_ARG, "null argument");
  OR_HIP(hipSetDevice(m->device));
  OR_HIP(quiesce(m));
  DevTime dt{};
  dt.tt = t->tt; dt.dt1 = t->dt1; dt.dt2 = t->dt2; dt.dt12 = t->dt12; dt.dt2old = t->dt2old;
  dt.ncycle = t->ncycle; dt.mstop = t->mstop; dt.done = t->mstop ? 1 : 0;
  DevTime two[2] = {dt, dt};
  OR_HIP(hipMemcpy(m->ts, two, sizeof(two), hipMemcpyHostToDevice));
  unsigned long long dm[2];
  const double big = kEP06;
  std::memcpy(&dm[0], &big, 8);
  dm[1] = dm[0];
  OR_HIP(hipMemcpy(m->dtmin, dm, sizeof(dm), hipMemcpyHostToDevice));
  int zero = 0;
  OR_HIP(hipMemcpy(m->flags, &zero, sizeof(int), hipMemcpyHostToDevice));
  m->parity = 0;
  return OR_OK;
}

int or_model_get_time(or_model *m, or_time_state *t) {
  if (!m || !t) return fail(OR_ERR_ARG, "null argument");
  OR_HIP(hipSetDevice(m->device));
  DevTime dt;
  int flags = 0;
  const int rc = read_back(m, {{&dt, m->ts + (m->parity & 1), sizeof(DevTime)}, {&flags, m->flags, sizeof(int)}});
  if (rc) return rc;
  t->tt = dt.tt; t->dt1 = dt.dt1; t->dt2 = dt.dt2; t->dt12 = dt.dt12; t->dt2old = dt.dt2old;
  t->ncycle = dt.ncycle; t->mstop = dt.mstop | flags;
  return OR_OK;
}

static int flush_timing(or_model *m) {
  if (m->ring_used == 0) return OR_OK;
  OR_HIP(hipEventSynchronize(m->ev[4 * (m->ring_used - 1) + 3]));
  for (int j = 0; j < m->ring_used; ++j) {
    float a = 0.f, b = 0.f, c = 0.f;
    OR_HIP(hipEventElapsedTime(&a, m->ev[4 * j], m->ev[4 * j + 1]));
    OR_HIP(hipEventElapsedTime(&b, m->ev[4 * j + 1], m->ev[4 * j + 2]));
    OR_HIP(hipEventElapsedTime(&c, m->ev[4 * j + 2], m->ev[4 * j + 3]));
    m->t_hex += a;
    m->t_q4 += b;
    m->t_node += c;
    m->t_cycles += 1;
  }
  m->ring_used = 0;
  return OR_OK;
}

// Refresh the device copy of a model's kernel view after uploads or parameter changes.
static void fill_dev(or_model *m, ModelDev &d, double tend) {
  d = ModelDev{};
  d.hconn = m->hconn; d.hrest = m->hrest; d.hfr_start = m->hfr_start; d.hfr_node = m->hfr_node;
  d.hfr_src = m->hfr_src; d.hsig = m->hsig; d.heint = m->heint; d.hrho = m->hrho;
  d.hpla = m->hpla; d.hepsd = m->hepsd; d.hoffg = m->hoffg; d.hqvis = m->hqvis; d.hvol0 = m->hvol0;
  d.neh = m->neh;
  d.qconn = m->qconn; d.qrest = m->qrest; d.qfr_start = m->qfr_start; d.qfr_node = m->qfr_node;
  d.qfr_src = m->qfr_src; d.qoffg = m->qoffg; d.qthk = m->qthk; d.qforc = m->qforc;
  d.qmom = m->qmom; d.qgstr = m->qgstr; d.qhourg = m->qhourg; d.qeint = m->qeint; d.qepsd = m->qepsd;
  d.qsig = m->qsig; d.qpla = m->qpla; d.qepsdip = m->qepsdip; d.qthke = m->qthke; d.neq = m->neq;
  d.nd = NodePtrs{m->xv, m->vr, m->d, m->ms, m->in, m->code, m->vimp, m->deg_h, m->deg_q, m->rs_h, m->rs_q,
                  m->preh, m->preq, m->wext, m->nn};
  d.rowh = m->rowh; d.rowq = m->rowq;
  d.preh = m->preh; d.preq = m->preq;
  d.ts = m->ts; d.dtmin = m->dtmin; d.flags = m->flags; d.ecrit = m->ecrit;
  d.dtel_h = m->dtel_h; d.dtel_q = m->dtel_q;
  d.th_slot = m->th_slot; d.th_node = m->th_buf; d.ehou_h = m->ehou_h; d.ehou_q = m->ehou_q;
  d.dtmx = m->neh > 0 ? m->hc.dtmx : 1.0e20;
  d.tend = tend;
  d.hc = m->hc;
  d.qc = m->qc;
}

static int refresh_dev(or_model *m) {
  if (!m->dev_dirty) return OR_OK;
  fill_dev(m, m->hdev, kNoEnd);
  OR_HIP(quiesce(m));
  OR_HIP(hipMemcpy(m->dev, &m->hdev, sizeof(ModelDev), hipMemcpyHostToDevice));
  m->dev_dirty = false;
  return OR_OK;
}

#endif // OR_ILP_TU

// The launches of one cycle for a set of models of one precision: element forces (hexes and
// shells) and the node update, each over the set's tile list (null: one model's own tiles).
struct LaunchSet {
  const ModelDev *md = nullptr;
  const Tile *th = nullptr, *tq = nullptr, *tn = nullptr;
  int32_t nth = 0, ntq = 0, ntn = 0;
  int vh = 0, vq = 0; // element kernel variants, as built
  bool eh = false, eq = false; // the set keeps EHOUR (hexes, shells): one model with a time history
};

// v & 1 selects the register budget; the caller routes v >= 2 to the unit built with the
// ILP-first scheduler.
#ifdef OR_ILP_TU
constexpr int kUnitFirst = 2; // this unit's first variant
#else
constexpr int kUnitFirst = 0;
#endif
template <typename R, typename S, bool EH>
static void launch_hex_eh(int v, hipStream_t st, const LaunchSet &L, int parity) {
  constexpr bool fp64 = sizeof(R) == 8;
  constexpr int W0 = variant_waves(fp64, built_variant(fp64, 0, kUnitFirst)),
                W1 = variant_waves(fp64, built_variant(fp64, 0, kUnitFirst + 1));
  const dim3 g((unsigned)L.nth);
  if ((v & 1) == 0) hipLaunchKernelGGL((k_hex_forces<R, S, kTile, W0, EH>), g, dim3(kTile), 0, st, L.md, L.th, parity);
  else hipLaunchKernelGGL((k_hex_forces<R, S, kTile, W1, EH>), g, dim3(kTile), 0, st, L.md, L.th, parity);
}
template <typename R, typename S>
static void launch_hex(int v, hipStream_t st, const LaunchSet &L, int parity) {
  if (L.eh) launch_hex_eh<R, S, true>(v, st, L, parity);
  else launch_hex_eh<R, S, false>(v, st, L, parity);
}

template <typename R, typename S, bool EH>
static void launch_q4_eh(int v, hipStream_t st, const LaunchSet &L, int parity) {
  constexpr bool fp64 = sizeof(R) == 8;
  constexpr int W0 = variant_waves(fp64, built_variant(fp64, 1, kUnitFirst)),
                W1 = variant_waves(fp64, built_variant(fp64, 1, kUnitFirst + 1));
  const dim3 g((unsigned)L.ntq);
  if ((v & 1) == 0) hipLaunchKernelGGL((k_q4_forces<R, S, kTile, W0, EH>), g, dim3(kTile), 0, st, L.md, L.tq, parity);
  else hipLaunchKernelGGL((k_q4_forces<R, S, kTile, W1, EH>), g, dim3(kTile), 0, st, L.md, L.tq, parity);
}
template <typename R, typename S>
static void launch_q4(int v, hipStream_t st, const LaunchSet &L, int parity) {
  if (L.eq) launch_q4_eh<R, S, true>(v, st, L, parity);
  else launch_q4_eh<R, S, false>(v, st, L, parity);
}

// Element launches of variants 2..3 (variant - 2 in the unit built with the ILP-first
// scheduler): family 0 hexes, 1 shells; fp64 selects <double,double> or <float,float>.
void or_ilp_elements(int family, int fp64, int variant, hipStream_t st, const void *md, const void *tiles,
                     int32_t ntiles, int parity, bool ehour)
#ifdef OR_ILP_TU
{
  LaunchSet L;
  L.md = (const ModelDev *)md;
  L.eh = L.eq = ehour;
  if (family == 0) {
    L.th = (const Tile *)tiles; L.nth = ntiles;
    if (fp64) launch_hex<double, double>(variant, st, L, parity);
    else launch_hex<float, float>(variant, st, L, parity);
  } else {
    L.tq = (const Tile *)tiles; L.ntq = ntiles;
    if (fp64) launch_q4<double, double>(variant, st, L, parity);
    else launch_q4<float, float>(variant, st, L, parity);
  }
}
#else
;

static LaunchSet model_set(const or_model *m) {
  LaunchSet L;
  L.md = m->dev;
  L.nth = m->nt_h; L.vh = m->var_h;
  L.eh = m->ehou_h != nullptr; L.eq = m->ehou_q != nullptr;
  L.ntq = m->nt_q; L.vq = m->var_q;
  L.ntn = m->nt_n;
  return L;
}

// A set's element kernels run in one launch (k_elements) when both families are there, their
// variants are the default one and nobody asked for the families' own times: the tiles of one
// family fill the compute units that the other leaves idle.  Against one launch each, us a cycle: 13,824
// hexes + 2,304 shells 19.8 (29.8), 512,000 + 160,000 137 (151; split form 95 and 102), 4,096,000 +
// 1,000,000 1,000 (1,027; 740 and 731, where the tuner finds the separate launches), a batch of 12 bars and
// tubes in both forms 47.0 (103.2).
static bool one_launch(const LaunchSet &L) { return L.nth > 0 && L.ntq > 0 && L.vh == 0 && L.vq == 0; }

// Which form of the node update a launch of nb blocks takes.  A small model's update is a chain of
// memory round trips (it fits in L2, one wave a SIMD), so its loads come first (76 registers, six waves
// a SIMD; 70 and seven in the split form); a large one is bound by HBM and takes the loads at their uses
// (64 registers, eight waves).  us at FP64 / split form, loads first against at their uses: 45,000
// nodes 7.8 / 7.9 and 8.9 / 8.2; 373,000 21.3 / 20.0 and 22.6 / 20.4; 1,264,000 82 / 62 and 83 / 64;
// 1,921,000 123 / 97 and 123 / 96; 2,771,000 172 / 140 and 172 / 134; 5,149,000 310 / 255 and 302 / 242
// (4.4 TB/s).
static bool node_first(int64_t nb) { return nb < 8192; }

template <typename S> static void launch_nodes(hipStream_t st, const LaunchSet &L, int parity, int output) {
  const dim3 g((unsigned)L.ntn);
  const double growth = (double)1.1f;
  if (node_first(L.ntn)) hipLaunchKernelGGL((k_node_update<S, true>), g, dim3(kBlock), 0, st, L.md, L.tn, parity, growth, output);
  else hipLaunchKernelGGL((k_node_update<S, false>), g, dim3(kBlock), 0, st, L.md, L.tn, parity, growth, output);
}

template <typename R, typename S>
static int launch_cycle(hipStream_t st, const LaunchSet &L, int parity, hipEvent_t after_hex, hipEvent_t after_q4,
                        int output = 0) {
  constexpr int fp64 = sizeof(R) == 8 ? 1 : 0;
  const int po = parity | (output ? 2 : 0); // element kernels: parity and the output-cycle bit
  if (one_launch(L) && !after_hex && !after_q4) {
    constexpr int q = fp64 ? kFamQ4 : kFamQ4Split, h = fp64 ? kFamHex : kFamHexSplit;
    constexpr int mask = (1 << q) | (1 << h);
    ElemLists E{};
    E.t[q] = L.tq; E.n[q] = L.ntq;
    E.t[h] = L.th; E.n[h] = L.nth;
    const dim3 g((unsigned)(L.ntq + L.nth));
    if (L.eh || L.eq) hipLaunchKernelGGL((k_elements<mask, true>), g, dim3(kTile), 0, st, L.md, E, po);
    else hipLaunchKernelGGL((k_elements<mask, false>), g, dim3(kTile), 0, st, L.md, E, po);
    OR_HIP(hipGetLastError());
    launch_nodes<S>(st, L, parity, output);
    OR_HIP(hipGetLastError());
    return OR_OK;
  }
  if (L.nth > 0) {
    if (L.vh >= 2) or_ilp_elements(0, fp64, L.vh - 2, st, L.md, L.th, L.nth, po, L.eh);
    else launch_hex<R, S>(L.vh, st, L, po);
    OR_HIP(hipGetLastError());
  }
  if (after_hex) OR_HIP(hipEventRecord(after_hex, st));
  if (L.ntq > 0) {
    if (L.vq >= 2) or_ilp_elements(1, fp64, L.vq - 2, st, L.md, L.tq, L.ntq, po, L.eq);
    else launch_q4<R, S>(L.vq, st, L, po);
    OR_HIP(hipGetLastError());
  }
  if (after_q4) OR_HIP(hipEventRecord(after_q4, st));
  if (L.ntn > 0) {
    launch_nodes<S>(st, L, parity, output);
    OR_HIP(hipGetLastError());
  }
  return OR_OK;
}

int or_model_run(or_model *m, int64_t ncycles) {
  if (!m) return fail(OR_ERR_ARG, "null model");
  if (ncycles < 0) return fail(OR_ERR_ARG, "ncycles < 0");
  if (!m->have_nodes || !m->have_sky || (m->neh > 0 && (!m->have_hparams || !m->have_hex)) ||
      (m->neq > 0 && (!m->have_qparams || !m->have_q4)))
    return fail(OR_ERR_STATE, "params, nodes, element state and skyline must be uploaded before run");
  if (m->batch) return fail(OR_ERR_STATE, "the model belongs to a batch: advance it with or_batch_run");
  OR_HIP(hipSetDevice(m->device));
  int rc0 = refresh_dev(m);
  if (rc0) return rc0;
  const LaunchSet L = model_set(m);
  for (int64_t c = 0; c < ncycles; ++c) {
    if (m->timing) {
      if (m->ring_used * 4 + 4 > (int)m->ev.size()) {
        int rc = flush_timing(m);
        if (rc) return rc;
      }
      OR_HIP(hipEventRecord(m->ev[4 * m->ring_used], m->stream));
    }
    hipEvent_t e1 = m->timing ? m->ev[4 * m->ring_used + 1] : nullptr;
    hipEvent_t e2 = m->timing ? m->ev[4 * m->ring_used + 2] : nullptr;
    const int p = (int)(m->parity & 1);
    int rc = (m->prec == OR_PREC_FP64) ? launch_cycle<double, double>(m->stream, L, p, e1, e2)
                                       : launch_cycle<float, float>(m->stream, L, p, e1, e2);
    if (rc) return rc;
    m->parity ^= 1;
    if (m->timing) {
      OR_HIP(hipEventRecord(m->ev[4 * m->ring_used + 3], m->stream));
      m->ring_used += 1;
    }
  }
  return OR_OK;
}

static int energy_launch(or_model *m, const double *ecrit);

// Per-element candidates of the controlling element and each storage slot's element index,
// allocated (and the slot indices uploaded) at the first output cycle.
static int ensure_ctrl(or_model *m) {
  if (m->ctrl) return OR_OK;
  OR_HIP(quiesce(m));
  auto put = [&](double **dt, int32_t **lidx, const std::vector<int32_t> &perm, int64_t ne) -> int {
    if (ne <= 0) return OR_OK;
    std::vector<int32_t> li((size_t)ne);
    for (int64_t s = 0; s < ne; ++s) li[(size_t)s] = perm.empty() ? (int32_t)s : perm[(size_t)s];
    OR_HIP(device_alloc((void **)dt, sizeof(double) * (size_t)ne));
    OR_HIP(device_alloc((void **)lidx, sizeof(int32_t) * (size_t)ne));
    OR_HIP(hipMemcpy(*lidx, li.data(), sizeof(int32_t) * (size_t)ne, hipMemcpyHostToDevice));
    m->bytes += (int64_t)(12 * ne);
    return OR_OK;
  };
  int rc = put(&m->dtel_h, &m->lidx_h, m->hperm, m->neh);
  if (rc == OR_OK) rc = put(&m->dtel_q, &m->lidx_q, m->qperm, m->neq);
  if (rc) return rc;
  OR_HIP(device_alloc((void **)&m->ctrl, 4 * sizeof(unsigned long long)));
  m->bytes += 32;
  mark_changed(m);
  return OR_OK;
}

int or_model_run_ecrit(or_model *m, or_ecrit *out) {
  if (!m || !out) return fail(OR_ERR_ARG, "null argument");
  if (!m->have_nodes || !m->have_sky || (m->neh > 0 && (!m->have_hparams || !m->have_hex)) ||
      (m->neq > 0 && (!m->have_qparams || !m->have_q4)))
    return fail(OR_ERR_STATE, "params, nodes, element state and skyline must be uploaded before run");
  if (m->batch) return fail(OR_ERR_STATE, "the model belongs to a batch: advance it with or_batch_run");
  OR_HIP(hipSetDevice(m->device));
  if (!m->ecrit) {
    OR_HIP(quiesce(m));
    OR_HIP(device_alloc((void **)&m->ecrit, sizeof(double) * 5 * (size_t)m->nn));
    m->bytes += (int64_t)(sizeof(double) * 5 * m->nn);
    mark_changed(m);
  }
  int rc = ensure_ctrl(m);
  if (rc) return rc;
  // candidates of elements that cannot control the step (and of a stopped model) stay EP06
  OR_HIP(fill(m->stream, m->dtel_h, m->neh, kEP06));
  OR_HIP(fill(m->stream, m->dtel_q, m->neq, kEP06));
  rc = refresh_dev(m);
  if (rc) return rc;
  const LaunchSet L = model_set(m);
  const int p = (int)(m->parity & 1);
  rc = (m->prec == OR_PREC_FP64) ? launch_cycle<double, double>(m->stream, L, p, nullptr, nullptr, 1)
                                 : launch_cycle<float, float>(m->stream, L, p, nullptr, nullptr, 1);
  if (rc) return rc;
  m->parity ^= 1;
  if ((rc = energy_launch(m, m->ecrit))) return rc;
  // the controlling element (k_ctrl_min / k_ctrl_pick); a grid of 1,024 blocks, or what the
  // larger family fills
  hipLaunchKernelGGL(k_ctrl_init, dim3(1), dim3(64), 0, m->stream, m->ctrl);
  const unsigned nb = (unsigned)std::min<int64_t>(1024, std::max(m->nt_h, m->nt_q));
  if (m->neh > 0) {
    hipLaunchKernelGGL(k_ctrl_min, dim3(nb), dim3(kBlock), 0, m->stream, m->dtel_h, m->neh, m->ctrl);
    hipLaunchKernelGGL(k_ctrl_pick, dim3(nb), dim3(kBlock), 0, m->stream, m->dtel_h, m->lidx_h, m->neh, m->ctrl, 1,
                       m->ctrl + 2);
  }
  if (m->neq > 0) {
    hipLaunchKernelGGL(k_ctrl_min, dim3(nb), dim3(kBlock), 0, m->stream, m->dtel_q, m->neq, m->ctrl + 1);
    hipLaunchKernelGGL(k_ctrl_pick, dim3(nb), dim3(kBlock), 0, m->stream, m->dtel_q, m->lidx_q, m->neq, m->ctrl + 1,
                       0, m->ctrl + 3);
  }
  OR_HIP(hipGetLastError());
  unsigned long long w[4];
  double e[kEnergySums];
  if ((rc = read_back(m, {{w, m->ctrl, sizeof(w)}, {e, m->energy, sizeof(e)}}))) return rc;
  out->enint = e[0]; out->encin = e[1]; out->enrot = e[2]; out->wfext = e[3];
  m->momentum[0] = e[4]; m->momentum[1] = e[5]; m->momentum[2] = e[6];
  double mh, mq;
  std::memcpy(&mh, &w[0], 8);
  std::memcpy(&mq, &w[1], 8);
  out->itypts = 0;
  out->pad = 0;
  out->nelts = -1;
  if (mh < kEP06) { out->itypts = 1; out->nelts = (int64_t)w[2]; }
  if (mq < mh) { out->itypts = 3; out->nelts = (int64_t)w[3]; }
  return OR_OK;
}

int or_model_run_output(or_model *m, double out[3]) {
  or_ecrit e;
  const int rc = or_model_run_ecrit(m, &e);
  if (rc) return rc;
  out[0] = e.enint; out[1] = e.encin; out[2] = e.enrot;
  return OR_OK;
}

// ---------------------------------------------------------------- time history (HIST2)
int or_model_th_setup(or_model *m, int64_t n_node, const int32_t *node, int64_t n_hex, const int32_t *hex,
                      int64_t n_q4, const int32_t *q4) {
  if (!m) return fail(OR_ERR_ARG, "null model");
  if (n_node < 0 || n_hex < 0 || n_q4 < 0 || (n_node && !node) || (n_hex && !hex) || (n_q4 && !q4))
    return fail(OR_ERR_ARG, "entity counts must be >= 0 with their lists given");
  if (m->batch) return fail(OR_ERR_STATE, "the model belongs to a batch");
  if (!m->have_nodes || !m->have_sky || (m->neh > 0 && !m->have_hex) || (m->neq > 0 && !m->have_q4))
    return fail(OR_ERR_STATE, "nodes, element state and skyline must be uploaded before the time history");
  std::vector<int32_t> slot((size_t)m->nn, -1);
  for (int64_t j = 0; j < n_node; ++j) {
    if (node[j] < 0 || node[j] >= m->nn) return fail(OR_ERR_ARG, "time-history node out of range");
    if (slot[(size_t)node[j]] >= 0) return fail(OR_ERR_ARG, "time-history node listed twice");
    slot[(size_t)node[j]] = (int32_t)j;
  }
  auto slots = [&](const int32_t *ids, int64_t n, int64_t ne, const std::vector<int32_t> &perm,
                   std::vector<int32_t> &out) -> int {
    std::vector<int32_t> inv((size_t)ne);
    for (int64_t s = 0; s < ne; ++s) inv[(size_t)(perm.empty() ? s : perm[(size_t)s])] = (int32_t)s;
    out.resize((size_t)n);
    for (int64_t j = 0; j < n; ++j) {
      if (ids[j] < 0 || ids[j] >= ne) return fail(OR_ERR_ARG, "time-history element out of range");
      out[(size_t)j] = inv[(size_t)ids[j]];
    }
    return OR_OK;
  };
  std::vector<int32_t> hs, qs;
  int rc = slots(hex, n_hex, m->neh, m->hperm, hs);
  if (rc == OR_OK) rc = slots(q4, n_q4, m->neq, m->qperm, qs);
  if (rc) return rc;
  OR_HIP(hipSetDevice(m->device));
  OR_HIP(quiesce(m));
  for (void **p : {(void **)&m->th_slot, (void **)&m->th_hex, (void **)&m->th_q4, (void **)&m->th_buf})
    if (*p) { (void)hipFree(*p); *p = nullptr; }
  const int64_t words = 18 * n_node + 13 * n_hex + (12 + m->npt) * n_q4 + 1;
  OR_HIP(device_alloc((void **)&m->th_slot, sizeof(int32_t) * (size_t)m->nn));
  OR_HIP(hipMemcpy(m->th_slot, slot.data(), sizeof(int32_t) * (size_t)m->nn, hipMemcpyHostToDevice));
  OR_HIP(device_alloc((void **)&m->th_buf, sizeof(double) * (size_t)words));
  OR_HIP(hipMemset(m->th_buf, 0, sizeof(double) * (size_t)words));
  if (n_hex) {
    OR_HIP(device_alloc((void **)&m->th_hex, sizeof(int32_t) * (size_t)n_hex));
    OR_HIP(hipMemcpy(m->th_hex, hs.data(), sizeof(int32_t) * (size_t)n_hex, hipMemcpyHostToDevice));
  }
  if (n_q4) {
    OR_HIP(device_alloc((void **)&m->th_q4, sizeof(int32_t) * (size_t)n_q4));
    OR_HIP(hipMemcpy(m->th_q4, qs.data(), sizeof(int32_t) * (size_t)n_q4, hipMemcpyHostToDevice));
  }
  // EHOUR accumulates from the first setup on (a later setup keeps it)
  if (m->nt_h > 0 && !m->ehou_h) {
    OR_HIP(device_alloc((void **)&m->ehou_h, sizeof(double) * (size_t)m->nt_h));
    OR_HIP(hipMemset(m->ehou_h, 0, sizeof(double) * (size_t)m->nt_h));
    m->bytes += 8 * (int64_t)m->nt_h;
  }
  if (m->nt_q > 0 && !m->ehou_q) {
    OR_HIP(device_alloc((void **)&m->ehou_q, sizeof(double) * (size_t)m->nt_q));
    OR_HIP(hipMemset(m->ehou_q, 0, sizeof(double) * (size_t)m->nt_q));
    m->bytes += 8 * (int64_t)m->nt_q;
  }
  m->bytes += 4 * m->nn + 8 * words + 4 * (n_hex + n_q4);
  m->th_nn = n_node; m->th_nh = n_hex; m->th_nq = n_q4;
  mark_changed(m);
  return OR_OK;
}

static double *th_ehour_word(or_model *m) { return m->th_buf + 18 * m->th_nn + 13 * m->th_nh + (12 + m->npt) * m->th_nq; }

static int th_ehour_launch(or_model *m) {
  double *w = th_ehour_word(m);
  hipLaunchKernelGGL(k_th_ehour, dim3(1), dim3(kBlock), 0, m->stream, m->ehou_h, (int64_t)(m->ehou_h ? m->nt_h : 0),
                     m->ehou_q, (int64_t)(m->ehou_q ? m->nt_q : 0), w);
  OR_HIP(hipGetLastError());
  return OR_OK;
}

static int th_ehour(or_model *m, double *ehour) {
  const int rc = th_ehour_launch(m);
  return rc ? rc : read_back(m, {{ehour, th_ehour_word(m), sizeof(double)}});
}

int or_model_run_th(or_model *m, or_ecrit *ec, double glob[4], double *node_out, double *hex_out, double *q4_out) {
  if (!m || !ec || !glob) return fail(OR_ERR_ARG, "null argument");
  if (!m->th_buf) return fail(OR_ERR_STATE, "or_model_th_setup first");
  if ((m->th_nn && !node_out) || (m->th_nh && !hex_out) || (m->th_nq && !q4_out))
    return fail(OR_ERR_ARG, "an output array of the listed entities is null");
  int rc = or_model_run_ecrit(m, ec);
  if (rc) return rc;
  OR_HIP(hipSetDevice(m->device));
  double *hb = m->th_buf + 18 * m->th_nn, *qb = hb + 13 * m->th_nh;
  const int64_t ne = m->th_nh + m->th_nq;
  if (ne > 0) {
    const dim3 g((unsigned)((ne + kBlock - 1) / kBlock));
    if (m->prec == OR_PREC_FP64)
      hipLaunchKernelGGL(k_th_elements<double>, g, dim3(kBlock), 0, m->stream, m->dev, m->th_hex, m->th_nh, m->th_q4,
                         m->th_nq, m->npt, hb, qb);
    else
      hipLaunchKernelGGL(k_th_elements<float>, g, dim3(kBlock), 0, m->stream, m->dev, m->th_hex, m->th_nh, m->th_q4,
                         m->th_nq, m->npt, hb, qb);
    OR_HIP(hipGetLastError());
  }
  glob[0] = m->momentum[0]; glob[1] = m->momentum[1]; glob[2] = m->momentum[2];
  if ((rc = th_ehour_launch(m))) return rc;
  return read_back(m, {{node_out, m->th_buf, sizeof(double) * 18 * (size_t)m->th_nn},
                       {hex_out, hb, sizeof(double) * 13 * (size_t)m->th_nh},
                       {q4_out, qb, sizeof(double) * (size_t)((12 + m->npt) * m->th_nq)},
                       {&glob[3], th_ehour_word(m), sizeof(double)}});
}

int or_model_ehour(or_model *m, double *ehour) {
  if (!m || !ehour) return fail(OR_ERR_ARG, "null argument");
  if (!m->th_buf) return fail(OR_ERR_STATE, "or_model_th_setup first");
  OR_HIP(hipSetDevice(m->device));
  return th_ehour(m, ehour);
}

int or_model_set_ehour(or_model *m, double ehour) {
  if (!m) return fail(OR_ERR_ARG, "null model");
  if (!m->th_buf) return fail(OR_ERR_STATE, "or_model_th_setup first");
  OR_HIP(hipSetDevice(m->device));
  OR_HIP(quiesce(m));
  if (m->ehou_h) OR_HIP(hipMemset(m->ehou_h, 0, sizeof(double) * (size_t)m->nt_h));
  if (m->ehou_q) OR_HIP(hipMemset(m->ehou_q, 0, sizeof(double) * (size_t)m->nt_q));
  double *first = m->ehou_h ? m->ehou_h : m->ehou_q;
  if (first) OR_HIP(hipMemcpy(first, &ehour, sizeof(double), hipMemcpyHostToDevice));
  return OR_OK;
}

int or_model_sync(or_model *m) {
  if (!m) return fail(OR_ERR_ARG, "null model");
  OR_HIP(hipSetDevice(m->device));
  int flags = 0;
  const int rc = read_back(m, {{&flags, m->flags, sizeof(int)}});
  if (rc) return rc;
  if (flags & 1) return fail(OR_ERR_MSTOP, "non-positive Jacobian: element deleted and MSTOP raised");
  return OR_OK;
}

int or_model_set_timing(or_model *m, int enable) {
  if (!m) return fail(OR_ERR_ARG, "null model");
  OR_HIP(hipSetDevice(m->device));
  if (enable && m->ev.empty()) {
    m->ev.resize(4 * 256);
    for (auto &e : m->ev) OR_HIP(hipEventCreate(&e));
  }
  m->timing = enable != 0;
  return OR_OK;
}

int or_model_kernel_times(or_model *m, int reset, double *hex_ms, double *q4_ms, double *node_ms, int64_t *cycles) {
  if (!m) return fail(OR_ERR_ARG, "null model");
  OR_HIP(hipSetDevice(m->device));
  int rc = flush_timing(m);
  if (rc) return rc;
  const double nc = m->t_cycles > 0 ? (double)m->t_cycles : 1.0;
  if (hex_ms) *hex_ms = m->t_hex / nc;
  if (q4_ms) *q4_ms = m->t_q4 / nc;
  if (node_ms) *node_ms = m->t_node / nc;
  if (cycles) *cycles = m->t_cycles;
  if (reset) { m->t_hex = 0.0; m->t_q4 = 0.0; m->t_node = 0.0; m->t_cycles = 0; }
  return OR_OK;
}

int or_model_download_nodes(or_model *m, double *x, double *v, double *vr, double *d) {
  if (!m) return fail(OR_ERR_ARG, "null model");
  OR_HIP(hipSetDevice(m->device));
  OR_HIP(quiesce(m));
  const int64_t n = 3 * m->nn;
  Chunks io;
  io.values(Chunk::kNodes, x, m->xv, n, 6, nullptr);
  io.values(Chunk::kNodes, v, m->xv + 3, n, 6, nullptr);
  if (vr && m->vr) io.values(Chunk::kNodes, vr, m->vr, n, 4, nullptr);
  if (vr && !m->vr) std::memset(vr, 0, sizeof(double) * (size_t)n);
  io.values(Chunk::kNodes, d, m->d, n, 3, nullptr);
  OR_HIP(io.run(m->device, m->stream));
  return OR_OK;
}

int or_model_download_hex(or_model *m, double *sig, double *eint, double *rho, double *pla, double *epsd,
                          double *offg, double *qvis) {
  if (!m) return fail(OR_ERR_ARG, "null model");
  OR_HIP(hipSetDevice(m->device));
  OR_HIP(quiesce(m));
  const int64_t ne = m->neh;
  Chunks io;
  int rc;
  if ((rc = get_state(m, io, sig, m->hsig, 6 * ne, ne, m->hslot))) return rc;
  if ((rc = get_state(m, io, eint, m->heint, ne, ne, m->hslot))) return rc;
  if ((rc = get_state(m, io, rho, m->hrho, ne, ne, m->hslot))) return rc;
  if ((rc = get_state(m, io, pla, m->hpla, ne, ne, m->hslot))) return rc;
  if ((rc = get_state(m, io, epsd, m->hepsd, ne, ne, m->hslot))) return rc;
  if ((rc = get_state(m, io, offg, m->hoffg, ne, ne, m->hslot))) return rc;
  if ((rc = get_state(m, io, qvis, m->hqvis, ne, ne, m->hslot))) return rc;
  OR_HIP(io.run(m->device, m->stream));
  return OR_OK;
}

int or_model_download_q4(or_model *m, double *offg, double *thk, double *forc, double *mom, double *gstr,
                         double *hourg, double *eint, double *epsd, double *sig, double *pla, double *epsd_ip) {
  if (!m) return fail(OR_ERR_ARG, "null model");
  OR_HIP(hipSetDevice(m->device));
  OR_HIP(quiesce(m));
  const int64_t ne = m->neq, np = m->npt;
  Chunks io;
  int rc;
  if ((rc = get_state(m, io, offg, m->qoffg, ne, ne, m->qslot))) return rc;
  if ((rc = get_state(m, io, thk, m->qthk, ne, ne, m->qslot))) return rc;
  if ((rc = get_state(m, io, forc, m->qforc, 5 * ne, ne, m->qslot))) return rc;
  if ((rc = get_state(m, io, mom, m->qmom, 3 * ne, ne, m->qslot))) return rc;
  if ((rc = get_state(m, io, gstr, m->qgstr, 8 * ne, ne, m->qslot))) return rc;
  if ((rc = get_state(m, io, hourg, m->qhourg, 5 * ne, ne, m->qslot))) return rc;
  if ((rc = get_state(m, io, eint, m->qeint, 2 * ne, ne, m->qslot))) return rc;
  if ((rc = get_state(m, io, epsd, m->qepsd, ne, ne, m->qslot))) return rc;
  if ((rc = get_state(m, io, sig, m->qsig, np * 5 * ne, ne, m->qslot))) return rc;
  if ((rc = get_state(m, io, pla, m->qpla, np * ne, ne, m->qslot))) return rc;
  if (epsd_ip) {
    if (m->qepsdip) {
      if ((rc = get_state(m, io, epsd_ip, m->qepsdip, np * ne, ne, m->qslot))) return rc;
    } else {
      // ASRATE = 1: LBUF%EPSD = 1*EPSD_PG + 0*LBUF%EPSD equals GBUF%EPSD at every point
      for (int64_t ip = 0; ip < np; ++ip)
        if ((rc = get_state(m, io, epsd_ip + ip * ne, m->qepsd, ne, ne, m->qslot))) return rc;
    }
  }
  OR_HIP(io.run(m->device, m->stream));
  return OR_OK;
}

// Fixed-order reduction of the internal energy and of the kinetic terms: 0.5*MS*|V|^2 from the
// resident state, or the per-node ECRIT terms of the last output cycle (ecrit != null, which
// also gives the momentum sums out[4..6]).
static int energy_launch(or_model *m, const double *ecrit) {
  int64_t n = m->nn;
  if (m->neh > n) n = m->neh;
  if (m->neq > n) n = m->neq;
  const int nb = 1024;
  const int64_t per = (n + nb - 1) / nb;
  const int64_t per_block = ((per + kBlock - 1) / kBlock) * kBlock;
  double *partial = m->energy + kEnergySums;
  if (m->batch) OR_HIP(hipStreamSynchronize(m->batch->stream));
  if (m->prec == OR_PREC_FP64)
    hipLaunchKernelGGL((k_energy_partial<double>), dim3(nb), dim3(kBlock), 0, m->stream, (const double *)m->heint,
                       (const double *)m->hvol0, m->neh, (const double *)m->qeint, m->neq, m->xv, m->vr, m->ms, m->in,
                       ecrit, m->wext, m->nn, per_block, partial);
  else
    hipLaunchKernelGGL((k_energy_partial<float>), dim3(nb), dim3(kBlock), 0, m->stream, (const float *)m->heint,
                       (const float *)m->hvol0, m->neh, (const float *)m->qeint, m->neq, m->xv, m->vr, m->ms, m->in,
                       ecrit, m->wext, m->nn, per_block, partial);
  OR_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_energy_final, dim3(1), dim3(kBlock), 0, m->stream, (const double *)partial, nb,
                     ecrit ? 1.0 : 0.5, m->energy);
  OR_HIP(hipGetLastError());
  return OR_OK;
}
static int energy_sums(or_model *m, const double *ecrit, double out[kEnergySums]) {
  const int rc = energy_launch(m, ecrit);
  return rc ? rc : read_back(m, {{out, m->energy, kEnergySums * sizeof(double)}});
}


int or_model_energy(or_model *m, double out[3]) {
  if (!m || !out) return fail(OR_ERR_ARG, "null argument");
  OR_HIP(hipSetDevice(m->device));
  double e[kEnergySums];
  const int rc = energy_sums(m, nullptr, e);
  if (rc) return rc;
  out[0] = e[0]; out[1] = e[1]; out[2] = e[2];
  return OR_OK;
}

int or_model_wfext(or_model *m, double *wfext) {
  if (!m || !wfext) return fail(OR_ERR_ARG, "null argument");
  OR_HIP(hipSetDevice(m->device));
  double e[kEnergySums];
  const int rc = energy_sums(m, nullptr, e);
  if (rc) return rc;
  *wfext = e[3];
  return OR_OK;
}

int or_model_footprint_estimate(int64_t nn, int64_t ne_hex, int64_t ne_q4, int32_t npt, int precision,
                                int strain_rate_filter, const int32_t *rows_hex, const int32_t *rows_q4,
                                int64_t *bytes) {
  if (!bytes) return fail(OR_ERR_ARG, "null argument");
  if (nn <= 0 || ne_hex < 0 || ne_q4 < 0) return fail(OR_ERR_ARG, "nn must be > 0, ne_hex and ne_q4 >= 0");
  if (ne_q4 > 0 && (npt < 2 || npt > 10)) return fail(OR_ERR_ARG, "shell NPT must be in 2..10");
  if (precision != OR_PREC_FP64 && precision != OR_PREC_SPLIT) return fail(OR_ERR_ARG, "bad precision");
  if ((ne_hex > 0 && !rows_hex) || (ne_q4 > 0 && !rows_q4)) return fail(OR_ERR_ARG, "missing row counts");
  const int64_t ss = precision == OR_PREC_FP64 ? 8 : 4;
  const int64_t th = (ne_hex + kTile - 1) / kTile, tq = (ne_q4 + kTile - 1) / kTile;
  // the allocations of or_model_create, in the same order
  int64_t b = 8 * (6 * nn + 3 * nn + nn + 3 * nn) + 4 * nn;             // xv, d, ms, vimp, code
  b += 16 * nn;                                                          // wext (models with imposed DOFs)
  if (ne_q4 > 0) b += 8 * (4 * nn + nn);                                 // vr, in
  if (ne_hex > 0)                                                        // deg, rs, prefix, tiles, conn, rest, state
    b += 4 * (nn + nn + 1) + 8 * 3 * nn + 4 * (th + 1) + 4 * 17 * ne_hex + ss * 13 * ne_hex;
  if (ne_q4 > 0) {
    b += 4 * (nn + nn + 1) + 8 * 6 * nn + 4 * (tq + 1) + 4 * 9 * ne_q4 + ss * (4 + 5 + 3 + 8 + 5 + 2) * ne_q4 +
         ss * 6 * (int64_t)npt * ne_q4;
    if (strain_rate_filter) b += ss * (int64_t)npt * ne_q4;              // LBUF EPSD (or_model_set_q4_params)
  }
  b += (int64_t)sizeof(DevTime) * 2 + 8 * 2 + 4 + 8 * (kEnergySums * (1 + 1024)) + (int64_t)sizeof(ModelDev);
  // or_model_upload_skyline: rest rows (at most every row of the family) and the prefix lists
  // (at most one prefix per node and family)
  for (int f = 0; f < 2; ++f) {
    const int32_t *rows = f == 0 ? rows_hex : rows_q4;
    if ((f == 0 ? ne_hex : ne_q4) == 0) continue;
    int64_t nrow = 0, nodes = 0;
    for (int64_t n = 0; n < nn; ++n) { nrow += rows[n]; nodes += rows[n] > 0; }
    b += ss * nrow * (f == 0 ? kHexRowWords : kQ4RowWords) + (4 + 2 * orasm::kRunCap) * nodes;
  }
  *bytes = b;
  return OR_OK;
}

int or_model_assembly_stats(const or_model *m, int64_t out[4]) {
  if (!m || !out) return fail(OR_ERR_ARG, "null argument");
  if (!m->have_sky) return fail(OR_ERR_STATE, "upload the skyline first");
  for (int k = 0; k < 4; ++k) out[k] = m->asm_stats[k];
  return OR_OK;
}

int or_model_footprint(const or_model *m, int64_t *bytes) {
  if (!m || !bytes) return fail(OR_ERR_ARG, "null argument");
  *bytes = m->bytes;
  return OR_OK;
}

// ============================================================== group drop-ins
namespace {
// Device buffers of one diagnostic call: allocated, copied and freed here.
struct Stage {
  std::vector<void *> ptrs;
  hipError_t e = hipSuccess;
  ~Stage() {
    for (void *p : ptrs)
      if (p) (void)hipFree(p);
  }
  template <typename T> T *up(const T *h, size_t n) {
    T *d = nullptr;
    if (e == hipSuccess) e = device_alloc((void **)&d, sizeof(T) * (n ? n : 1));
    ptrs.push_back(d);
    if (e == hipSuccess && h && n) e = hipMemcpy(d, h, sizeof(T) * n, hipMemcpyHostToDevice);
    return d;
  }
  template <typename T> void down(T *h, const T *d, size_t n) {
    if (e == hipSuccess && h && n) e = hipMemcpy(h, d, sizeof(T) * n, hipMemcpyDeviceToHost);
  }
};
} // namespace

int or_sforc3_group(int device, const or_hex_params *p, int64_t numnod, int32_t nel, int64_t nft, const double *x,
                    const double *v, const int32_t *ixs, double *sig, double *eint, double *rho, const double *vol,
                    double *pla, double *epsd, double *off, double *qvis, int64_t lsky, double *fsky,
                    const int32_t *iads, double dt1, double *dt2t, int32_t *mstop) {
  if (!p || !x || !v || !ixs || !sig || !eint || !rho || !vol || !pla || !epsd || !off || !qvis || !fsky || !iads ||
      !dt2t || !mstop)
    return fail(OR_ERR_ARG, "null argument");
  if (nel <= 0 || nel > 128) return fail(OR_ERR_ARG, "nel must be in 1..128 (MVSIZ-1)");
  if (numnod <= 0 || lsky <= 0 || nft < 0) return fail(OR_ERR_ARG, "bad sizes");
  int rc = check_hex_params(*p);
  if (rc) return rc;
  for (int i = 0; i < nel; ++i)
    for (int k = 0; k < 8; ++k) {
      const int32_t nid = ixs[11 * (nft + i) + 1 + k];
      if (nid < 1 || nid > numnod) return fail(OR_ERR_ARG, "IXS node id out of range");
      const int32_t K = iads[8 * (nft + i) + k];
      if (K < 1 || K > lsky) return fail(OR_ERR_ARG, "IADS row out of range");
    }
  OR_HIP(hipSetDevice(device));
  const HexConsts c = make_hex_consts(*p);
  Lease buf;
  OR_HIP(buf.take(-1, sizeof(double) * kHexStageWords * (size_t)nel));
  double *w = buf.d(), *g = w + kHexStageState * nel, *r = w + kHexStageRows * nel, *dt = w + kHexStageDt * nel;
  for (int i = 0; i < nel; ++i)
    for (int k = 0; k < 8; ++k) {
      const int64_t n = 3 * ((int64_t)ixs[11 * (nft + i) + 1 + k] - 1);
      for (int d = 0; d < 3; ++d) {
        w[(3 * k + d) * nel + i] = x[n + d];
        w[(24 + 3 * k + d) * nel + i] = v[n + d];
      }
    }
  const double *in[] = {eint, rho, vol, pla, epsd, off, qvis};
  double *out[] = {eint, rho, nullptr, pla, epsd, off, qvis};
  std::memcpy(g, sig, sizeof(double) * 6 * (size_t)nel);
  for (int k = 0; k < 7; ++k) std::memcpy(g + (6 + k) * nel, in[k], sizeof(double) * (size_t)nel);
  hipLaunchKernelGGL(k_sforc3_staged, dim3((nel + kBlock - 1) / kBlock), dim3(kBlock), 0, 0, (int)nel, w, c, dt1);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
  if (e != hipSuccess) return fail(OR_ERR_HIP, std::string("or_sforc3_group: ") + hipGetErrorString(e));
  std::memcpy(sig, g, sizeof(double) * 6 * (size_t)nel);
  for (int k = 0; k < 7; ++k)
    if (out[k]) std::memcpy(out[k], g + (6 + k) * nel, sizeof(double) * (size_t)nel);
  for (int i = 0; i < nel; ++i) {
    for (int k = 0; k < 8; ++k) {
      double *f = fsky + 8 * ((int64_t)iads[8 * (nft + i) + k] - 1);
      for (int d = 0; d < 3; ++d) f[d] = r[(4 * k + d) * nel + i];
      f[6] = r[(4 * k + 3) * nel + i];
    }
    if (dt[i] < *dt2t) *dt2t = dt[i];
    if (dt[nel + i] != 0.0) *mstop = 1;
  }
  return OR_OK;
}

// ---------------------------------------------------------------------------
// SFORC3 group drop-in without allocation.  The group is staged through one file-scope
// device array instead of per-call device buffers: its own nodes (at most 8 per element,
// renumbered in order of first appearance), its GBUF arrays and its FSKY rows (8 per
// element, gathered from the caller's FSKY and scattered back, so that words the kernel
// does not write keep their values).  k_sforc3_group runs on the staged copy with
// nft = 0.  The array holds kStaticGroupBytes per device, for the whole process.
namespace {
constexpr int kStaticNel = 128;                                   // MVSIZ - 1
constexpr size_t kStaticGroupDoubles = 6 * 8 * kStaticNel         // x, v of the group's nodes
                                       + 13 * kStaticNel           // GBUF (SIG 6, 7 scalars)
                                       + 64 * kStaticNel           // FSKY rows (8 words x 8)
                                       + kStaticNel;               // element time steps
constexpr size_t kStaticGroupInts = 11 * kStaticNel + 8 * kStaticNel + kStaticNel; // IXS, IADS, MSTOP
constexpr size_t kStaticGroupBytes = 8 * kStaticGroupDoubles + 4 * kStaticGroupInts;

static __device__ __align__(256) unsigned char scratch[kStaticGroupBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
unsigned char *g_scratch[kMaxDevices] = {};

// The device address of this device's copy of `scratch` (host code never uses the array's
// name as an address): looked up once per device, with that device current.
int scratch_of(int device, unsigned char **out) {
  if (device < 0 || device >= kMaxDevices) return fail(OR_ERR_ARG, "device index out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch[device]) {
    void *ptr = nullptr;
    hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
      return fail(OR_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    g_scratch[device] = (unsigned char *)ptr;
  }
  *out = g_scratch[device];
  return OR_OK;
}
} // namespace

int or_sforc3_group_static(int device, const or_hex_params *p, int64_t numnod, int32_t nel, int64_t nft,
                           const double *x, const double *v, const int32_t *ixs, double *sig, double *eint,
                           double *rho, const double *vol, double *pla, double *epsd, double *off, double *qvis,
                           int64_t lsky, double *fsky, const int32_t *iads, double dt1, double *dt2t,
                           int32_t *mstop) {
  if (!p || !x || !v || !ixs || !sig || !eint || !rho || !vol || !pla || !epsd || !off || !qvis || !fsky || !iads ||
      !dt2t || !mstop)
    return fail(OR_ERR_ARG, "null argument");
  if (nel <= 0 || nel > kStaticNel)
    return fail(OR_ERR_ARG, "nel must be in 1..128: the staging array holds one group of at most 128 hexes");
  if (numnod <= 0 || lsky <= 0 || nft < 0) return fail(OR_ERR_ARG, "bad sizes");
  int rc = check_hex_params(*p);
  if (rc) return rc;
  for (int i = 0; i < nel; ++i)
    for (int k = 0; k < 8; ++k) {
      const int32_t nid = ixs[11 * (nft + i) + 1 + k];
      if (nid < 1 || nid > numnod) return fail(OR_ERR_ARG, "IXS node id out of range");
      const int32_t K = iads[8 * (nft + i) + k];
      if (K < 1 || K > lsky) return fail(OR_ERR_ARG, "IADS row out of range");
    }
  OR_HIP(hipSetDevice(device));
  unsigned char *base = nullptr;
  if ((rc = scratch_of(device, &base))) return rc;
  const HexConsts c = make_hex_consts(*p);
  // the staged group on the host, laid out as in the device array
  double hd[kStaticGroupDoubles];
  int32_t hi[kStaticGroupInts];
  double *lx = hd, *lv = hd + 24 * kStaticNel, *lsig = hd + 48 * kStaticNel;
  double *leint = lsig + 6 * nel, *lrho = leint + nel, *lvol = lrho + nel, *lpla = lvol + nel, *lepsd = lpla + nel,
         *loff = lepsd + nel, *lqvis = loff + nel;
  double *lfsky = hd + 61 * kStaticNel, *ldtx = hd + 125 * kStaticNel;
  int32_t *lixs = hi, *liads = hi + 11 * kStaticNel, *lms = hi + 19 * kStaticNel;
  int32_t nloc = 0;
  int32_t gid[8 * kStaticNel]; // global (1-based) id of each local node
  for (int i = 0; i < nel; ++i) {
    for (int k = 0; k < 8; ++k) {
      const int32_t g = ixs[11 * (nft + i) + 1 + k];
      int32_t l = 0;
      while (l < nloc && gid[l] != g) ++l;
      if (l == nloc) {
        gid[nloc++] = g;
        for (int d = 0; d < 3; ++d) {
          lx[3 * l + d] = x[3 * (int64_t)(g - 1) + d];
          lv[3 * l + d] = v[3 * (int64_t)(g - 1) + d];
        }
      }
      lixs[11 * i + 1 + k] = l + 1;
      liads[8 * i + k] = 8 * i + k + 1;
      const int64_t K = iads[8 * (nft + i) + k] - 1;
      for (int w = 0; w < 8; ++w) lfsky[8 * (8 * i + k) + w] = fsky[8 * K + w];
    }
    lixs[11 * i] = ixs[11 * (nft + i)];
    for (int w = 9; w < 11; ++w) lixs[11 * i + w] = ixs[11 * (nft + i) + w];
  }
  for (int k = 0; k < 6; ++k)
    for (int i = 0; i < nel; ++i) lsig[k * nel + i] = sig[(int64_t)k * nel + i];
  for (int i = 0; i < nel; ++i) {
    leint[i] = eint[i]; lrho[i] = rho[i]; lvol[i] = vol[i]; lpla[i] = pla[i];
    lepsd[i] = epsd[i]; loff[i] = off[i]; lqvis[i] = qvis[i];
  }
  double *dd = (double *)base;
  int32_t *di = (int32_t *)(base + 8 * kStaticGroupDoubles);
  OR_HIP(hipMemcpy(dd, hd, sizeof(hd), hipMemcpyHostToDevice));
  OR_HIP(hipMemcpy(di, hi, sizeof(hi), hipMemcpyHostToDevice));
  double *dsig = dd + 48 * kStaticNel;
  double *deint = dsig + 6 * nel, *drho = deint + nel, *dvol = drho + nel, *dpla = dvol + nel, *depsd = dpla + nel,
         *doff = depsd + nel, *dq = doff + nel;
  hipLaunchKernelGGL(k_sforc3_group, dim3(1), dim3(kBlock), 0, 0, nel, (int64_t)0, (const double *)dd,
                     (const double *)(dd + 24 * kStaticNel), (const int32_t *)di, dsig, deint, drho,
                     (const double *)dvol, dpla, depsd, doff, dq, dd + 61 * kStaticNel,
                     (const int32_t *)(di + 11 * kStaticNel), c, dt1, dd + 125 * kStaticNel, (int *)(di + 19 * kStaticNel));
  OR_HIP(hipGetLastError());
  OR_HIP(hipMemcpy(hd, dd, sizeof(hd), hipMemcpyDeviceToHost)); // synchronous after the launch
  OR_HIP(hipMemcpy(hi, di, sizeof(hi), hipMemcpyDeviceToHost));
  for (int k = 0; k < 6; ++k)
    for (int i = 0; i < nel; ++i) sig[(int64_t)k * nel + i] = lsig[k * nel + i];
  for (int i = 0; i < nel; ++i) {
    eint[i] = leint[i]; rho[i] = lrho[i]; pla[i] = lpla[i]; epsd[i] = lepsd[i]; off[i] = loff[i];
    qvis[i] = lqvis[i];
    for (int k = 0; k < 8; ++k) {
      const int64_t K = iads[8 * (nft + i) + k] - 1;
      for (int w = 0; w < 8; ++w) fsky[8 * K + w] = lfsky[8 * (8 * i + k) + w];
    }
    if (ldtx[i] < *dt2t) *dt2t = ldtx[i];
    if (lms[i]) *mstop = 1;
  }
  return OR_OK;
}

int or_cforc3_group(int device, const or_q4_params *p, int64_t numnod, int32_t nel, int64_t nft, const double *x,
                    const double *v, const double *vr, const int32_t *ixc, double *offg, double *thk,
                    const double *thke, double *forc, double *mom, double *gstr, double *hourg, double *eint,
                    double *epsd, double *sig, double *pla, double *epsd_ip, int64_t lsky, double *fsky,
                    const int32_t *iadc, double dt1, double *dt2t) {
  if (!p || !x || !v || !vr || !ixc || !offg || !thk || !thke || !forc || !mom || !gstr || !hourg || !eint ||
      !epsd || !sig || !pla || !epsd_ip || !fsky || !iadc || !dt2t)
    return fail(OR_ERR_ARG, "null argument");
  if (nel <= 0 || nel > 128) return fail(OR_ERR_ARG, "nel must be in 1..128 (MVSIZ-1)");
  if (numnod <= 0 || lsky <= 0 || nft < 0) return fail(OR_ERR_ARG, "bad sizes");
  Q4Consts c;
  int rc = make_q4_consts(*p, c);
  if (rc) return rc;
  for (int i = 0; i < nel; ++i)
    for (int k = 0; k < 4; ++k) {
      const int32_t nid = ixc[7 * (nft + i) + 1 + k];
      if (nid < 1 || nid > numnod) return fail(OR_ERR_ARG, "IXC node id out of range");
      const int32_t K = iadc[4 * (nft + i) + k];
      if (K < 1 || K > lsky) return fail(OR_ERR_ARG, "IADC row out of range");
    }
  OR_HIP(hipSetDevice(device));
  const int np = p->npt;
  Lease buf;
  OR_HIP(buf.take(-1, sizeof(double) * (size_t)(q4_stage_words(np) * nel)));
  double *w = buf.d(), *r = w + kQ4StageRows * nel, *dt = w + kQ4StageDt * nel;
  for (int i = 0; i < nel; ++i) {
    const int32_t *node = ixc + 7 * (nft + i) + 1;
    for (int k = 0; k < 4; ++k) {
      const int64_t n = 3 * ((int64_t)node[k] - 1);
      for (int d = 0; d < 3; ++d) {
        w[(3 * k + d) * nel + i] = x[n + d];
        w[(12 + 3 * k + d) * nel + i] = v[n + d];
        w[(24 + 3 * k + d) * nel + i] = vr[n + d];
      }
    }
    w[kQ4StageState * nel + i] = node[2] == node[3] ? 1.0 : 0.0;
  }
  // the arrays in their staged order; thke is read only
  struct {
    const double *in;
    double *out;
    int words, at;
  } const arr[] = {{offg, offg, 1, kQ4StageState + 1},    {thk, thk, 1, kQ4StageState + 2},
                   {thke, nullptr, 1, kQ4StageState + 3}, {epsd, epsd, 1, kQ4StageState + 4},
                   {forc, forc, 5, kQ4StageState + 5},    {mom, mom, 3, kQ4StageState + 10},
                   {gstr, gstr, 8, kQ4StageState + 13},   {hourg, hourg, 5, kQ4StageState + 21},
                   {eint, eint, 2, kQ4StageState + 26},   {sig, sig, 5 * np, kQ4StagePoints},
                   {pla, pla, np, kQ4StagePoints + 5 * np}, {epsd_ip, epsd_ip, np, kQ4StagePoints + 6 * np}};
  for (const auto &a : arr) std::memcpy(w + a.at * nel, a.in, sizeof(double) * (size_t)(a.words * nel));
  hipLaunchKernelGGL(k_cforc3_staged, dim3((nel + kBlock - 1) / kBlock), dim3(kBlock), 0, 0, (int)nel, w, c, dt1);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
  if (e != hipSuccess) return fail(OR_ERR_HIP, std::string("or_cforc3_group: ") + hipGetErrorString(e));
  for (const auto &a : arr)
    if (a.out) std::memcpy(a.out, w + a.at * nel, sizeof(double) * (size_t)(a.words * nel));
  for (int i = 0; i < nel; ++i) {
    for (int k = 0; k < 4; ++k) {
      double *f = fsky + 8 * ((int64_t)iadc[4 * (nft + i) + k] - 1);
      for (int d = 0; d < 7; ++d) f[d] = r[(7 * k + d) * nel + i];
      f[7] = 0.0;
    }
    if (dt[i] < *dt2t) *dt2t = dt[i];
  }
  return OR_OK;
}

// ---------------------------------------------------------------------------
// Device evaluation of the FP64 elementary functions (diagnostic).
namespace {
__global__ void k_math_eval(int fn, int64_t n, const double *__restrict__ x, const double *__restrict__ y,
                            double *__restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double a = x[i];
  out[i] = fn == 0 ? ormath::or_log(a) : fn == 1 ? ormath::or_exp(a) : ormath::or_pow(a, y[i]);
}
} // namespace

int or_math_eval(int device, int fn, int64_t n, const double *x, const double *y, double *out) {
  if (fn < 0 || fn > 2) return fail(OR_ERR_ARG, "fn must be 0 (log), 1 (exp) or 2 (pow)");
  if (n < 0 || n > (int64_t(1) << 30)) return fail(OR_ERR_ARG, "n must be in 0..2^30");
  if (n == 0) return OR_OK;
  if (!x || !out || (fn == 2 && !y)) return fail(OR_ERR_ARG, "null argument");
  OR_HIP(hipSetDevice(device));
  Stage s;
  double *dx = s.up(x, n), *dy = fn == 2 ? s.up(y, n) : nullptr, *dout = s.up<double>(nullptr, n);
  if (s.e == hipSuccess) {
    hipLaunchKernelGGL(k_math_eval, dim3((unsigned)((n + kBlock - 1) / kBlock)), dim3(kBlock), 0, 0, fn, n, dx, dy,
                       dout);
    s.e = hipGetLastError();
  }
  if (s.e == hipSuccess) s.e = hipDeviceSynchronize();
  s.down(out, dout, n);
  if (s.e != hipSuccess) return fail(OR_ERR_HIP, std::string("or_math_eval: ") + hipGetErrorString(s.e));
  return OR_OK;
}

// ---------------------------------------------------------------------------
// Batches: many resident models in one launch per kernel and precision class.
namespace {

int read_time(or_model *m, int slot, DevTime &t) {
  OR_HIP(hipMemcpy(&t, m->ts + slot, sizeof(DevTime), hipMemcpyDeviceToHost));
  return OR_OK;
}

// Move a model's cycle scalars to the slot of the given parity, and set its stop flag
// for the end time tend.
int align_model(or_model *m, int64_t parity, double tend) {
  const int from = (int)(m->parity & 1), to = (int)(parity & 1);
  DevTime t;
  int rc = read_time(m, from, t);
  if (rc) return rc;
  t.done = (t.mstop != 0 || t.tt >= tend) ? 1 : 0;
  OR_HIP(hipMemcpy(m->ts + to, &t, sizeof(DevTime), hipMemcpyHostToDevice));
  unsigned long long dm;
  const double big = kEP06;
  std::memcpy(&dm, &big, 8);
  OR_HIP(hipMemcpy(m->dtmin + to, &dm, sizeof(dm), hipMemcpyHostToDevice));
  m->parity = parity & 1;
  return OR_OK;
}

int batch_rebuild(or_batch *b) {
  if (!b->dirty) return OR_OK;
  OR_HIP(hipStreamSynchronize(b->stream));
  const int64_t ns = (int64_t)b->members.size();
  if (ns > b->md_cap) {
    if (b->md) OR_HIP(hipFree(b->md));
    b->md = nullptr;
    b->md_cap = 0;
    OR_HIP(device_alloc((void **)&b->md, sizeof(ModelDev) * (size_t)ns));
    b->md_cap = ns;
  }
  std::vector<ModelDev> hd((size_t)ns);
  std::vector<Tile> tl[2][3];
  for (int64_t i = 0; i < ns; ++i) {
    or_model *m = b->members[(size_t)i];
    fill_dev(m, hd[(size_t)i], b->tend[(size_t)i]);
    if (!b->live[(size_t)i]) continue;
    const int c = m->prec == OR_PREC_FP64 ? 0 : 1;
    const int64_t cnt[3] = {m->neh, m->neq, m->nn};
    const int step[3] = {kTile, kTile, kBlock};
    for (int f = 0; f < 3; ++f)
      for (int64_t first = 0; first < cnt[f]; first += step[f]) tl[c][f].push_back(Tile{(int32_t)i, (int32_t)first});
  }
  if (ns > 0) OR_HIP(hipMemcpy(b->md, hd.data(), sizeof(ModelDev) * (size_t)ns, hipMemcpyHostToDevice));
  for (int c = 0; c < 2; ++c)
    for (int f = 0; f < 3; ++f) {
      const int64_t n = (int64_t)tl[c][f].size();
      if (n > b->tcap[c][f]) {
        if (b->tiles[c][f]) OR_HIP(hipFree(b->tiles[c][f]));
        b->tiles[c][f] = nullptr;
        b->tcap[c][f] = 0;
        OR_HIP(device_alloc((void **)&b->tiles[c][f], sizeof(Tile) * (size_t)n));
        b->tcap[c][f] = n;
      }
      if (n > 0) OR_HIP(hipMemcpy(b->tiles[c][f], tl[c][f].data(), sizeof(Tile) * (size_t)n, hipMemcpyHostToDevice));
      b->nt[c][f] = (int32_t)n;
    }
  b->dirty = false;
  return OR_OK;
}

} // namespace

int or_batch_create(or_batch **out, int device) {
  if (!out) return fail(OR_ERR_ARG, "null out");
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return fail(OR_ERR_NODEV, "no HIP device");
  if (device < 0 || device >= ndev) return fail(OR_ERR_ARG, "device index out of range");
  OR_HIP(hipSetDevice(device));
  or_batch *b = new or_batch();
  b->device = device;
  if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess) {
    delete b;
    return fail(OR_ERR_HIP, "hipStreamCreate");
  }
  *out = b;
  return OR_OK;
}

int or_batch_destroy(or_batch *b) {
  if (!b) return OR_OK;
  (void)hipSetDevice(b->device);
  (void)hipStreamSynchronize(b->stream);
  while (!b->members.empty()) (void)or_batch_remove(b, b->members.back());
  if (b->md) (void)hipFree(b->md);
  for (auto &row : b->tiles)
    for (Tile *t : row)
      if (t) (void)hipFree(t);
  (void)hipStreamDestroy(b->stream);
  delete b;
  return OR_OK;
}

int or_batch_add(or_batch *b, or_model *m, double t_end) {
  if (!b || !m) return fail(OR_ERR_ARG, "null argument");
  if (m->batch) return fail(OR_ERR_STATE, "the model already belongs to a batch");
  if (m->device != b->device) return fail(OR_ERR_ARG, "the model lives on another device");
  if (!(t_end > 0.0)) return fail(OR_ERR_ARG, "t_end must be > 0");
  if (!m->have_nodes || !m->have_sky || (m->neh > 0 && (!m->have_hparams || !m->have_hex)) ||
      (m->neq > 0 && (!m->have_qparams || !m->have_q4)))
    return fail(OR_ERR_STATE, "params, nodes, element state and skyline must be uploaded before add");
  OR_HIP(hipSetDevice(b->device));
  OR_HIP(hipStreamSynchronize(m->stream));
  OR_HIP(hipStreamSynchronize(b->stream));
  int rc = align_model(m, b->parity, t_end);
  if (rc) return rc;
  m->batch = b;
  b->members.push_back(m);
  b->tend.push_back(t_end);
  b->live.push_back(1);
  b->dirty = true;
  return OR_OK;
}

int or_batch_remove(or_batch *b, or_model *m) {
  if (!b || !m) return fail(OR_ERR_ARG, "null argument");
  size_t i = 0;
  while (i < b->members.size() && b->members[i] != m) ++i;
  if (i == b->members.size()) return fail(OR_ERR_ARG, "the model is not in this batch");
  OR_HIP(hipSetDevice(b->device));
  OR_HIP(hipStreamSynchronize(b->stream));
  b->members.erase(b->members.begin() + (ptrdiff_t)i);
  b->tend.erase(b->tend.begin() + (ptrdiff_t)i);
  b->live.erase(b->live.begin() + (ptrdiff_t)i);
  m->batch = nullptr;
  m->dev_dirty = true;
  b->dirty = true;
  // alone again: the model runs without an end time unless MSTOP was raised
  return align_model(m, m->parity, kNoEnd);
}

int or_batch_run(or_batch *b, int64_t ncycles) {
  if (!b) return fail(OR_ERR_ARG, "null batch");
  if (ncycles < 0) return fail(OR_ERR_ARG, "ncycles < 0");
  OR_HIP(hipSetDevice(b->device));
  int rc = batch_rebuild(b);
  if (rc) return rc;
  LaunchSet L[2];
  for (int c = 0; c < 2; ++c) {
    L[c].md = b->md;
    L[c].th = b->tiles[c][0]; L[c].nth = b->nt[c][0]; L[c].vh = b->var[c][0];
    L[c].tq = b->tiles[c][1]; L[c].ntq = b->nt[c][1]; L[c].vq = b->var[c][1];
    L[c].tn = b->tiles[c][2]; L[c].ntn = b->nt[c][2];
  }
  // members of both forms and default variants: one element and one node launch for all of them
  const bool both = L[0].ntn > 0 && L[1].ntn > 0 && !b->var[0][0] && !b->var[0][1] && !b->var[1][0] && !b->var[1][1];
  ElemLists E{};
  for (int c = 0; c < 2; ++c) {
    E.t[2 * c + kFamQ4] = L[c].tq; E.n[2 * c + kFamQ4] = L[c].ntq;
    E.t[2 * c + kFamHex] = L[c].th; E.n[2 * c + kFamHex] = L[c].nth;
  }
  const dim3 ge((unsigned)(E.n[0] + E.n[1] + E.n[2] + E.n[3])), gn((unsigned)(L[0].ntn + L[1].ntn));
  for (int64_t k = 0; k < ncycles; ++k) {
    const int p = (int)(b->parity & 1);
    if (both) {
      if (ge.x > 0) hipLaunchKernelGGL((k_elements<15, false>), ge, dim3(kTile), 0, b->stream, (const ModelDev *)b->md, E, p);
      hipLaunchKernelGGL(k_node_update_both, gn, dim3(kBlock), 0, b->stream, (const ModelDev *)b->md, L[0].tn,
                         L[0].ntn, L[1].tn, p, (double)1.1f);
      OR_HIP(hipGetLastError());
    } else {
      if ((rc = launch_cycle<double, double>(b->stream, L[0], p, nullptr, nullptr))) return rc;
      if ((rc = launch_cycle<float, float>(b->stream, L[1], p, nullptr, nullptr))) return rc;
    }
    b->parity ^= 1;
    b->cycles += 1;
  }
  // members still in the tile lists follow the batch parity; stopped ones keep their slot
  for (size_t i = 0; i < b->members.size(); ++i)
    if (b->live[i]) b->members[i]->parity = b->parity & 1;
  return OR_OK;
}

int or_batch_sync(or_batch *b) {
  if (!b) return fail(OR_ERR_ARG, "null batch");
  OR_HIP(hipSetDevice(b->device));
  OR_HIP(hipStreamSynchronize(b->stream));
  return OR_OK;
}

int or_batch_active(or_batch *b, int32_t *nactive) {
  if (!b || !nactive) return fail(OR_ERR_ARG, "null argument");
  OR_HIP(hipSetDevice(b->device));
  OR_HIP(hipStreamSynchronize(b->stream));
  int32_t n = 0;
  for (size_t i = 0; i < b->members.size(); ++i) {
    DevTime t;
    int rc = read_time(b->members[i], (int)(b->members[i]->parity & 1), t);
    if (rc) return rc;
    const char alive = t.done ? 0 : 1;
    if (alive != b->live[i]) {
      b->live[i] = alive;
      b->dirty = true; // stopped models leave the tile lists
    }
    n += alive;
  }
  *nactive = n;
  return OR_OK;
}

// ---------------------------------------------------------------------------
// Kernel variants and their autotuning
namespace {

// Device time of `ncycles` cycles launched by `launch` on `st` (events around the loop).  Of several
// cycles the first, which may have to load its kernels' code, is not in the time.
template <typename F> int time_cycles(hipStream_t st, int ncycles, F launch, float &ms) {
  hipEvent_t e0, e1;
  OR_HIP(hipEventCreate(&e0));
  OR_HIP(hipEventCreate(&e1));
  int rc = OR_OK;
  const int untimed = ncycles > 1 ? 1 : 0;
  for (int k = 0; k < ncycles && rc == OR_OK; ++k) {
    if (k == untimed && hipEventRecord(e0, st) != hipSuccess) rc = fail(OR_ERR_HIP, "hipEventRecord");
    if (rc == OR_OK) rc = launch();
  }
  if (rc == OR_OK && (hipEventRecord(e1, st) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
                      hipEventElapsedTime(&ms, e0, e1) != hipSuccess))
    rc = fail(OR_ERR_HIP, "event timing");
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return rc;
}

// The variants of a model's (or a batch form's) families: trial(h, q, ms) runs cycles_per_variant
// cycles with variants h and q.  The default pair, whose families share a launch, is measured
// against pairs with a launch each: hexes' other variants, shells' with the best of those, the default
// hexes with the best shells.  kVariants trials a family in all; those left over repeat the default and
// the best other pair, whose shortest times count.  Where a joint launch is at stake another pair is
// taken only when it is 1 % faster, which is what two measurements of one pair differ by.
template <typename F> int tune_variants(bool fp64, bool has_hex, bool has_q4, bool joint, F trial, int best[2]) {
  constexpr float kNone = 1.0e30f;
  float t[kVariants][kVariants];
  for (auto &row : t) std::fill(std::begin(row), std::end(row), kNone);
  int left = kVariants * ((has_hex ? 1 : 0) + (has_q4 ? 1 : 0));
  int rc = OR_OK;
  auto run = [&](int h, int q) {
    if (rc != OR_OK || left == 0) return;
    --left;
    float ms = kNone;
    rc = trial(h, q, ms);
    t[h][q] = std::min(t[h][q], ms);
  };
  auto fastest_other = [&](int &h, int &q) { // of the pairs measured, the default one apart
    h = q = 0;
    float ms = kNone;
    for (int a = 0; a < kVariants; ++a)
      for (int b = 0; b < kVariants; ++b)
        if ((a || b) && t[a][b] < ms) { h = a; q = b; ms = t[a][b]; }
    return ms;
  };
  run(0, 0);
  int h = 0, q = 0;
  for (int v = 1; has_hex && v < kVariants; ++v)
    if (built_variant(fp64, 0, v) == v) run(v, 0);
  fastest_other(h, q);
  const int hs = h;
  for (int v = 1; has_q4 && v < kVariants; ++v)
    if (built_variant(fp64, 1, v) == v) run(hs, v);
  fastest_other(h, q);
  if (has_hex && has_q4) run(0, q ? q : 2);
  while (left > 0 && rc == OR_OK) {
    run(0, 0);
    fastest_other(h, q);
    run(h, q);
  }
  const float ms = fastest_other(h, q);
  const bool take = rc == OR_OK && ms < (joint ? 0.99f : 1.0f) * t[0][0];
  best[0] = take ? h : 0;
  best[1] = take ? q : 0;
  return rc;
}

} // namespace

int or_model_set_variant(or_model *m, int family, int variant) {
  if (!m) return fail(OR_ERR_ARG, "null model");
  if (family < 0 || family > 1 || variant < 0 || variant >= kVariants) return fail(OR_ERR_ARG, "bad family / variant");
  OR_HIP(hipSetDevice(m->device));
  OR_HIP(quiesce(m));
  (family == 0 ? m->var_h : m->var_q) = built_variant(m->prec == OR_PREC_FP64, family, variant);
  return OR_OK;
}

int or_model_autotune(or_model *m, int32_t cycles_per_variant, int32_t chosen[2]) {
  if (!m || !chosen) return fail(OR_ERR_ARG, "null argument");
  if (cycles_per_variant < 1) return fail(OR_ERR_ARG, "cycles_per_variant must be >= 1");
  if (m->batch) return fail(OR_ERR_STATE, "the model belongs to a batch: use or_batch_autotune");
  if (!m->have_nodes || !m->have_sky || (m->neh > 0 && (!m->have_hparams || !m->have_hex)) ||
      (m->neq > 0 && (!m->have_qparams || !m->have_q4)))
    return fail(OR_ERR_STATE, "params, nodes, element state and skyline must be uploaded before autotune");
  OR_HIP(hipSetDevice(m->device));
  int rc = refresh_dev(m);
  if (rc) return rc;
  auto trial = [&](int h, int q, float &ms) -> int {
    m->var_h = h;
    m->var_q = q;
    const LaunchSet L = model_set(m);
    auto one = [&]() -> int {
      const int p = (int)(m->parity & 1);
      int r = (m->prec == OR_PREC_FP64) ? launch_cycle<double, double>(m->stream, L, p, nullptr, nullptr)
                                        : launch_cycle<float, float>(m->stream, L, p, nullptr, nullptr);
      m->parity ^= 1;
      return r;
    };
    return time_cycles(m->stream, cycles_per_variant, one, ms);
  };
  int best[2];
  rc = tune_variants(m->prec == OR_PREC_FP64, m->neh > 0, m->neq > 0, m->neh > 0 && m->neq > 0, trial, best);
  m->var_h = best[0];
  m->var_q = best[1];
  if (rc) return rc;
  chosen[0] = m->var_h;
  chosen[1] = m->var_q;
  return OR_OK;
}

int or_batch_autotune(or_batch *b, int32_t cycles_per_variant, int32_t chosen[4]) {
  if (!b || !chosen) return fail(OR_ERR_ARG, "null argument");
  if (cycles_per_variant < 1) return fail(OR_ERR_ARG, "cycles_per_variant must be >= 1");
  OR_HIP(hipSetDevice(b->device));
  int rc = batch_rebuild(b);
  if (rc) return rc;
  for (auto &v : b->var) v[0] = v[1] = 0;
  for (int c = 0; c < 2; ++c) {
    auto trial = [&](int h, int q, float &ms) -> int {
      b->var[c][0] = h;
      b->var[c][1] = q;
      return time_cycles(b->stream, cycles_per_variant, [&]() { return or_batch_run(b, 1); }, ms);
    };
    const bool hexes = b->nt[c][0] > 0, shells = b->nt[c][1] > 0;
    const bool joint = (hexes && shells) || (b->nt[0][2] > 0 && b->nt[1][2] > 0);
    rc = tune_variants(c == 0, hexes, shells, joint, trial, b->var[c]);
    if (rc) return rc;
  }
  for (int c = 0; c < 2; ++c)
    for (int f = 0; f < 2; ++f) chosen[2 * c + f] = b->var[c][f];
  return OR_OK;
}

// ---------------------------------------------------------------------------
// Nodal half of a cycle with host arrays (ASSPAR4 -> DEPLA drop-in)
int or_nodal_update(int device, int64_t numnod, int64_t lsky, const int64_t *adsky, const double *fsky,
                    const double *ms, const double *in, const int32_t *code, const double *vimp, double *x,
                    double *v, double *vr, double *d, double *stifn, double *stifr, double dt2t, double dtmx,
                    or_time_state *ts) {
  if (!adsky || !fsky || !ms || !x || !v || !d || !ts) return fail(OR_ERR_ARG, "null argument");
  if (vr && !in) return fail(OR_ERR_ARG, "rotational velocities need the nodal inertias IN");
  if (numnod <= 0 || lsky < 0) return fail(OR_ERR_ARG, "bad sizes");
  if (adsky[0] != 1 || adsky[numnod] != lsky + 1) return fail(OR_ERR_ARG, "ADSKY must run from 1 to LSKY+1");
  for (int64_t n = 0; n < numnod; ++n) {
    if (adsky[n + 1] < adsky[n]) return fail(OR_ERR_ARG, "ADSKY must be non-decreasing");
    if (code && (code[n] & ~511)) return fail(OR_ERR_ARG, "node code has bits outside 0..511");
    if (code && (code[n] & (kIX | kIY | kIZ)) && !vimp) return fail(OR_ERR_ARG, "imposed-velocity bits without vimp");
  }
  OR_HIP(hipSetDevice(device));
  // DT2 pipeline on the host (resol.F:2721-2722, 6125-6129, 6352, 6494-6497)
  const double DT1 = ts->dt2;
  const double DT2 = dt2_pipeline(dt2t, ts->dt2old, (double)1.1f, dtmx);
  const double DT12 = (1.0 / 2.0) * (DT1 + DT2);
  // one device workspace, filled and read back through page-locked chunks
  const size_t nn = (size_t)numnod;
  struct Array {
    const void *in;
    void *out;
    size_t bytes;
    char *dev;
  } arr[] = {{adsky, nullptr, 8 * (nn + 1), nullptr}, {fsky, nullptr, 64 * (size_t)lsky, nullptr}, {ms, nullptr, 8 * nn, nullptr},
             {in, nullptr, 8 * nn, nullptr},          {code, nullptr, 4 * nn, nullptr},            {vimp, nullptr, 24 * nn, nullptr},
             {x, x, 24 * nn, nullptr},                {v, v, 24 * nn, nullptr},                    {d, d, 24 * nn, nullptr},
             {vr, vr, 24 * nn, nullptr},              {nullptr, stifn, 8 * nn, nullptr},           {nullptr, stifr, 8 * nn, nullptr}};
  size_t total = 0;
  for (Array &a : arr)
    if (a.in || a.out) total += (a.bytes + 255) / 256 * 256;
  Lease work;
  OR_HIP(work.take(device, total));
  char *at = (char *)work.b.p;
  Chunks io;
  for (Array &a : arr) {
    if (!a.in && !a.out) continue;
    a.dev = at;
    at += (a.bytes + 255) / 256 * 256;
    if (a.in) io.bytes(Chunk::kUp, a.in, a.dev, a.bytes);
  }
  // up to one chunk the whole workspace is one copy each way: below that a copy's fixed cost
  // (10 us) counts, above it the threads of Chunks pay (72,240 nodes: 1.85 ms by pageable copies,
  // 1.25 now; 1 MB in one image each way 0.12 ms, by arrays 0.34)
  const bool image = total <= 8 * (size_t)Chunks::kChunk;
  Lease host;
  hipError_t e = hipSuccess;
  char *const base = (char *)work.b.p;
  if (image) {
    OR_HIP(host.take(-1, total));
    for (const Array &a : arr)
      if (a.in) std::memcpy((char *)host.b.p + (a.dev - base), a.in, a.bytes);
    e = hipMemcpyAsync(base, host.b.p, total, hipMemcpyHostToDevice, nullptr);
  } else {
    e = io.run(device, nullptr);
  }
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_nodal_dropin, dim3((unsigned)((numnod + kBlock - 1) / kBlock)), dim3(kBlock), 0, 0, numnod,
                       (const int64_t *)arr[0].dev, (const double *)arr[1].dev, (const double *)arr[2].dev,
                       (const double *)arr[3].dev, (const int32_t *)arr[4].dev, (const double *)arr[5].dev,
                       (double *)arr[6].dev, (double *)arr[7].dev, (double *)arr[9].dev, (double *)arr[8].dev,
                       (double *)arr[10].dev, (double *)arr[11].dev, DT12, DT2);
    e = hipGetLastError();
  }
  if (image) {
    const size_t o = (size_t)(arr[6].dev - base); // X and the arrays after it come back
    if (e == hipSuccess) e = hipMemcpyAsync((char *)host.b.p + o, base + o, total - o, hipMemcpyDeviceToHost, nullptr);
    if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
    for (const Array &a : arr)
      if (a.out && e == hipSuccess) std::memcpy(a.out, (char *)host.b.p + (a.dev - base), a.bytes);
  } else {
    Chunks back;
    for (const Array &a : arr)
      if (a.out) back.bytes(Chunk::kDown, a.out, a.dev, a.bytes);
    if (e == hipSuccess) e = back.run(device, nullptr);
  }
  if (e != hipSuccess) {
    (void)hipStreamSynchronize(nullptr); // the workspace goes back only when nothing uses it
    return fail(OR_ERR_HIP, std::string("or_nodal_update: ") + hipGetErrorString(e));
  }
  ts->dt1 = DT1;
  ts->dt2 = DT2;
  ts->dt12 = DT12;
  ts->dt2old = DT2;
  ts->tt = ts->tt + DT2;
  ts->ncycle += 1;
  if (DT2 <= 0.0) ts->mstop |= kMstopTimeStep; // resol.F:8575, 9599
  return OR_OK;
}
#endif // OR_ILP_TU
