// Rows longer than 32 elements, first stage: one workgroup per group of up to 16384 consecutive
// elements of a row, whose lower hull it builds (the first merge level's nodes; the rows' final
// hulls where a row is one group, which the workgroup then expands).
//
// Replaces the reference's chunk stage and its first merge rounds (reference src/torchisotonic/
// csrc/tiles.cuh:665-913, 1326-1743). Instead of hulls of small pieces merged pairwise, nearly
// every point is dropped by one test against a chord that is known to lie under it:
//
//   1. each thread holds E consecutive elements in registers; their sums, scanned over the
//      workgroup with their rounding errors, place the threads' first points (the coarse points);
//   2. a lower hull of the coarse points, roughly: per wave, a few rounds in which every point
//      above a chord of two other points drops out, all at once, on a 64-bit mask of the lanes;
//      then the same over the points that are left of all waves, at most 64 of them (more, on
//      rising data, keep their waves' chords);
//   3. each thread's elements lie under one chord of that hull: a point is a candidate only where
//      it lies below the chord (or within rounding of it) and y rises into it. Noise leaves
//      tens of candidates in a group of 16384, a noisy trend hundreds;
//   4. the candidates, compacted into LDS with their exact sums, lose every point on or above the
//      chord of its neighbours (or clearly above one of three longer chords), all at once, round
//      after round until none goes: five rounds or so. What is left is the group's hull.
//
// A chord between two points of the diagram never drops a vertex of its hull, whichever points
// they are, so steps 2 and 3 need no exactness beyond a margin for rounding, and only step 4's
// neighbour test decides ties (the filtered exact predicate). Groups of more candidates than LDS
// holds (rising data, where most points are vertices) are built a chunk at a time and merged in
// global memory by reference to the chunks' hulls (merge_global), by a second launch.
//
// What bounds it: VALU issue, about 1500 instructions a wave of 2048 weighted float32 elements, and
// the latency of the load, three barriers and the candidates' rounds at two workgroups a CU. One
// lane a span of 80 to 256 elements with a stack in LDS, the form before, was bound by the chain of
// each stack operation. Forward calls, before and now: 20000 rows of 200 float32 107 -> 36 us; 10000
// of 1000 131 -> 56 us; 1000 of 5000 60 -> 27 us, weighted float64 81 -> 51 us; 500 of 20000 120 ->
// 60 us; one weighted row of 1e8 (the kernel) 346 -> 233 us; rising rows, all overflowing (1000 of
// 10000, a vertex at every element) 468 -> 187 us.
#include <algorithm>

#include "ti_common.h"
#include "ti_expand.h"
#include "ti_gmerge.h"
#include "ti_kernels.h"
#include "ti_points.h"
#include "ti_tile.h"

namespace ti {

namespace {

struct GroupArgs {
  const void* y;
  const void* w;
  uint32_t* bad_weight;
  int64_t n, batch;
  int64_t gpr;      // groups per row
  int g_elems;      // elements per group
  int span0;        // elements per span of level 0 (a chunk's hull lies in its spans' slots)
  int nt;           // group_kernel's threads
  int cap;          // point slots in LDS
  int chunk, cpg;   // (overflow_kernel) spans per chunk, chunks per group
  int parts;        // and workgroups that share a group's
  NodeLevel chunks;  // level 0, a chunk a node: its hull, and in tot the sums before it; a group's
                     // first node's bad counts its parts done
  int expand_at;    // the expansion's LDS, from the region's start
  unsigned flags;
  NodeLevel spans;  // level 0
  NodeLevel out;    // the groups' level
  bool expand;      // rows of one group: the workgroup expands its row
  int repair_passes;  // (overflow_kernel, such rows of float32 data) see repair_row
  RowExpand xp;
  RowMap map;
  uint32_t* mark;   // (where given) mark_value stored to *mark by the kernel's first thread
  uint32_t mark_value;
};

// A group's candidates: sums in the group's frame, indices within the group.
template <bool W, bool PR>
using GPoints = Points<W, PR, uint16_t>;

// Per group: the waves' totals and flags, candidate counts, the coarse list.
template <int NW>
struct GroupShared {
  double tot[4][NW];  // per wave: W hi, lo, S hi, lo
  double maxabs[NW];
  int bad[NW];
  int live[NW];
  int count[NW];
  int wc[NW];
  int result;
  double ls[kWave + 1], lw[kWave + 1];
  double end[2];  // the group's end, its pad included: W and S
};

__host__ __device__ constexpr int group_head_bytes(int nw) {
  return (nw * (5 * 8 + 4 * 4) + 8 + 2 * (kWave + 2) * 8 + 63) & ~63;
}

// E consecutive elements a thread from the wave's 64 * E: loaded in 16-byte pieces, each load
// instruction of the wave on one contiguous 1 KiB (load_pieces), and handed to their threads
// through the wave's slab of LDS (own_pieces; 16 * 64 * P bytes); with at most two pieces a
// thread each thread loads its own. Piece q of thread t lies at t * P + (q ^ sw(t)), which
// spreads the reads of 16 lanes over all banks.
template <typename T, int E>
struct Pieces {
  static constexpr int V = 16 / sizeof(T);
  static constexpr int P = E / V;
  static constexpr bool kDirect = P <= 2;
  static_assert(E % V == 0 && (P & (P - 1)) == 0 && P <= 16, "whole 16-byte pieces");
  using VT = T __attribute__((ext_vector_type(V)));
  VT buf[P];

  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r) {
    const int lane = threadIdx.x & (kWave - 1);
    const int w0 = wave_index() * kWave * E;
#pragma unroll
    for (int j = 0; j < P; ++j) {
      const int e = w0 + (kDirect ? lane * P + j : j * kWave + lane) * V;
      buf[j] = __builtin_bit_cast(
          VT, __builtin_amdgcn_raw_buffer_load_b128(r, static_cast<uint32_t>(e * sizeof(T)), 0, 0));
    }
  }
  __device__ __forceinline__ void own(char* slab, T (&v)[E]) {
    if constexpr (!kDirect) {
      const int lane = threadIdx.x & (kWave - 1);
      auto sw = [](int t) { return (t / (16 / P)) & (P - 1); };
      VT* const s = reinterpret_cast<VT*>(slab);
#pragma unroll
      for (int j = 0; j < P; ++j) {
        const int c = j * kWave + lane, t = c / P;
        s[t * P + ((c % P) ^ sw(t))] = buf[j];
      }
      wave_fence();
#pragma unroll
      for (int q = 0; q < P; ++q) buf[q] = s[lane * P + (q ^ sw(lane))];
      wave_fence();
    }
#pragma unroll
    for (int q = 0; q < P; ++q) {
#pragma unroll
      for (int t = 0; t < V; ++t) v[q * V + t] = buf[q][t];
    }
  }
};

// After every fourth (float64: every) of many unrolled elements: the scheduler would otherwise
// start dozens of their conversions at once, and spill.
template <typename T, int E>
__device__ __forceinline__ void element_end(int k) {
  if constexpr (E >= 16 || sizeof(T) == 8) {
    if (sizeof(T) == 8 || (k & 3) == 3) __builtin_amdgcn_sched_barrier(0);
  }
}

__device__ __forceinline__ float abs_t(float v) { return __builtin_fabsf(v); }
__device__ __forceinline__ double abs_t(double v) { return __builtin_fabs(v); }
__device__ __forceinline__ float signed_t(float v, uint32_t sign) {
  return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v) ^ sign);
}
__device__ __forceinline__ double signed_t(double v, uint32_t sign) {
  return __builtin_bit_cast(double, __builtin_bit_cast(uint64_t, v) ^ (static_cast<uint64_t>(sign) << 32));
}
__device__ __forceinline__ float max_t(float a, float b) { return __builtin_fmaxf(a, b); }
__device__ __forceinline__ double max_t(double a, double b) { return __builtin_fmax(a, b); }

// The values as they are in registers, opaque to the compiler: it would otherwise keep their
// float64 conversions from one use to the next, in twice the registers.
template <typename T, int N>
__device__ __forceinline__ void opaque(T (&v)[N]) {
#pragma unroll
  for (int k = 0; k < N; ++k) asm volatile("" : "+v"(v[k]));
}

// The final hull in LDS, for expand_hull.
template <bool W, bool PR>
struct LdsHull {
  GPoints<W, PR> v;
  __device__ __forceinline__ int idx(int k) const { return v.i[k]; }
  __device__ __forceinline__ void edge(int k, double& dW, double& dS) const {
    const HPt a = pget(v, k), b = pget(v, k + 1);
    dS = dd_diff(DD{b.s, b.sl}, DD{a.s, a.sl});
    if constexpr (W) dW = dd_diff(DD{b.w, b.wl}, DD{a.w, a.wl});
    else dW = static_cast<double>(b.i - a.i);
  }
};

// One thread's part of a group: its place and its elements.
template <typename T, bool W, int NT, int E, bool MAP>
struct GroupThread {
  int64_t row;
  int grp;
  int len;    // the group's elements
  int glen;   // those that are the row's own (ragged rows: the pad is the rest, and never read)
  int t0;     // the thread's first element
  int64_t base;

  // (g: the group, of all rows; 32-bit: the grid fits)
  __device__ __forceinline__ GroupThread(const GroupArgs& a, unsigned g) {
    const unsigned row32 = a.gpr == 1 ? g : g / static_cast<unsigned>(a.gpr);
    row = row32;
    grp = static_cast<int>(g - row32 * static_cast<unsigned>(a.gpr));
    const int64_t goff = static_cast<int64_t>(grp) * a.g_elems;
    len = static_cast<int>(min<int64_t>(a.g_elems, a.n - goff));
    int64_t mfirst = row * a.n, mlen = a.n;
    if constexpr (MAP) map_row(a.map, row, a.n, mfirst, mlen);
    glen = static_cast<int>(wave_uniform(max<int64_t>(0, min<int64_t>(len, mlen - goff))));
    base = wave_uniform(glen > 0 ? mfirst + goff : 0);
    t0 = threadIdx.x * E;
  }

  // The thread's elements of the group's [p0, p0 + n), signed (a decreasing fit is the increasing
  // fit of -y), through the wave's slab. Past their end, where the buffer resources end, y = 0 and
  // w = 0.
  __device__ __forceinline__ void load_at(const GroupArgs& a, int p0, int n, char* slab, T (&y)[E],
                                          T (&w)[W ? E : 1]) const {
    const int64_t bytes = n * static_cast<int64_t>(sizeof(T));
    Pieces<T, E> py;
    py.load(make_rsrc(static_cast<const T*>(a.y) + base + p0, bytes));
    if constexpr (W) {
      Pieces<T, E> pw;
      pw.load(make_rsrc(static_cast<const T*>(a.w) + base + p0, bytes));
      py.own(slab, y);
      pw.own(slab, w);
    } else {
      py.own(slab, y);
    }
    // (without a branch, whose two sides' copies of the elements would spill)
    const uint32_t sign = (a.flags & TI_INCREASING) ? 0u : 0x80000000u;
#pragma unroll
    for (int k = 0; k < E; ++k) y[k] = signed_t(y[k], sign);
  }
};

// A thread's running sums of w y (s) and w; float64 data carries their rounding errors.
template <typename T, bool W>
struct RunSums {
  static constexpr bool PR = sizeof(T) == 8;
  double s = 0.0, sl = 0.0, w = 0.0, wl = 0.0;
  __device__ __forceinline__ void add(T yk, T wk) {
    if constexpr (PR) {
      const DD t = two_sum(s, W ? static_cast<double>(wk) * static_cast<double>(yk) : static_cast<double>(yk));
      s = t.hi;
      sl += t.lo;
      if constexpr (W) {
        const DD u = two_sum(w, static_cast<double>(wk));
        w = u.hi;
        wl += u.lo;
      }
    } else if constexpr (W) {
      s = __builtin_fma(static_cast<double>(wk), static_cast<double>(yk), s);
      w += static_cast<double>(wk);
    } else {
      s += static_cast<double>(yk);
    }
  }
};

// The sums before the thread's first element (x), and before its wave (b). A thread's own sums (32
// elements at most) of float32 data are float64, of float64 data double-double; from there on,
// across lanes and waves, both are pairs whose second part holds the first's rounding errors, and a
// point's sums are rounded once at the end (float32) or not at all. Where values cancel (2^60 and
// -2^60 beside ordinary ones) a plain float64 scan lost the rest: errors of up to six times the
// largest other value.
struct BaseSums {
  DD xs, xw, bs, bw;
};
// v, the same in every lane, in scalar registers.
__device__ __forceinline__ double uniform_f64(double v) {
  return __builtin_bit_cast(double, wave_uniform(__builtin_bit_cast(int64_t, v)));
}
__device__ __forceinline__ DD uniform_dd(DD v) { return DD{uniform_f64(v.hi), uniform_f64(v.lo)}; }

// (float32: the errors summed and the pair not renormalised, eight operations in place of eleven:
// an error under 2^-104 of the terms' magnitudes either way)
template <bool PR>
__device__ __forceinline__ DD sums_plus(DD a, DD b) {
  if constexpr (PR) {
    return dd_add(a, b);
  } else {
    const DD t = two_sum(a.hi, b.hi);
    return DD{t.hi, t.lo + (a.lo + b.lo)};
  }
}
// x and a thread's sum after it.
template <bool PR>
__device__ __forceinline__ DD sums_point(DD x, double t, double tl) {
  if constexpr (PR) {
    return dd_add(x, DD{t, tl});
  } else {
    const DD s = two_sum(x.hi, t);
    return DD{s.hi + (s.lo + x.lo), 0.0};
  }
}

// The lanes' sums (hi, lo) before each lane, and of the whole wave (see wave_incl_dd).
template <bool PR>
__device__ __forceinline__ void wave_scan(double hi, double lo, DD& before, DD& all) {
  DD v{hi, lo};
  if constexpr (PR) v = dd_add(dpp_dd<0x111, 0xF>(v), v);
  else v = two_sum(dpp_f64<0x111, 0xF>(hi), hi);  // (lo is zero)
  v = sums_plus<PR>(dpp_dd<0x112, 0xF>(v), v);
  v = sums_plus<PR>(dpp_dd<0x114, 0xF>(v), v);
  v = sums_plus<PR>(dpp_dd<0x118, 0xF>(v), v);
  v = sums_plus<PR>(dpp_dd<0x142, 0xA>(v), v);
  v = sums_plus<PR>(dpp_dd<0x143, 0xC>(v), v);
  before = wave_shr1_dd(v);
  all = wave_last_dd(v);
}

// The points of `mine` (bit k: the point after element k) to slots pos, pos + 1, ...: the thread's
// own sums at each, what comes before them added. With 32 elements a thread the adding waits until
// the thread's points are all in their slots: at the elements, where any lane's point takes the
// whole wave through it, a wave did it up to 32 times for a lane's one or two (1000 weighted rows
// of 65536 with gradients 505 us, 498 so; with 8 or 16 elements no faster).
template <typename T, bool W, int E>
__device__ __forceinline__ void emit(const GPoints<W, sizeof(T) == 8>& pts, int pos, uint32_t mine, int t0, bool bad,
                                     const BaseSums& b, T (&y)[E], T (&w)[W ? E : 1]) {
  constexpr bool PR = sizeof(T) == 8;
  constexpr bool kLate = E >= 32;
  if (mine == 0) return;
  const auto point = [&](const HPt& own) {
    const DD S = bad ? DD{0.0, 0.0} : sums_point<PR>(b.xs, own.s, own.sl);
    const DD Wd = W ? sums_point<PR>(b.xw, own.w, own.wl) : DD{0.0, 0.0};
    return HPt{own.i, S.hi, S.lo, Wd.hi, Wd.lo};
  };
  const int first = pos;
  RunSums<T, W> t;
#pragma unroll
  for (int k = 0; k < E; ++k) {
    t.add(y[k], w[W ? k : 0]);
    if ((mine >> k) & 1) {
      const HPt own{t0 + k + 1, t.s, t.sl, t.w, t.wl};
      pput(pts, pos, kLate ? own : point(own));
      ++pos;
    }
    element_end<T, E>(k);
  }
  if constexpr (kLate) {
    for (int q = first; q < pos; ++q) pput(pts, q, point(pget(pts, q)));
  }
}

// (ragged rows) the pad's value, signed as the elements are
__device__ __forceinline__ double signed_pad(const GroupArgs& a) {
  return (a.flags & TI_INCREASING) ? a.map.pad : -a.map.pad;
}

// Where the thread's points go: its first slot, and the points of all threads (have: its own).
template <int NT, class SH>
__device__ __forceinline__ int place(int have, int& all, SH& sh, int nt = NT) {
  const int wave = wave_index();
  const int incl = wave_incl_i32(have);
  if ((threadIdx.x & (kWave - 1)) == kWave - 1) sh.count[wave] = incl;
  __syncthreads();
  int pos = incl - have;
  all = 0;
  for (int q = 0; q < nt / kWave; ++q) {
    pos += q < wave ? sh.count[q] : 0;
    all += sh.count[q];
  }
  return pos;
}

// What a thread knows of its group once its sums are scanned.
struct GroupSums {
  BaseSums b;
  DD wave_s, wave_w;    // the wave's totals
  double maxabs, wsum;  // the group's largest |y|, and its weight
  bool bad;             // it holds a NaN
};

// The thread's sums, scanned over the workgroup; the group's totals and NaN flag go to its node.
template <typename T, bool W, int NT, int E, bool MAP, class SH>
__device__ __forceinline__ GroupSums group_sums(const GroupArgs& a, const GroupThread<T, W, NT, E, MAP>& g, SH& sh,
                                                const NodeOut& out, T (&y)[E], T (&w)[W ? E : 1], int nt = NT) {
  constexpr bool PR = sizeof(T) == 8;
  const int lane = threadIdx.x & (kWave - 1), wave = wave_index();
  GroupSums r{};
  if constexpr (W) {
    if (a.bad_weight != nullptr) {
      bool wbad = false;
      if (__any(g.t0 + E > g.glen)) {
#pragma unroll
        for (int k = 0; k < E; ++k) wbad |= k < g.glen - g.t0 && !(w[W ? k : 0] > T(0));
      } else if constexpr (PR) {
#pragma unroll
        for (int k = 0; k < E; ++k) wbad |= !(w[W ? k : 0] > T(0));
      } else {
        // (positive floats are positive integers; a NaN's sum is seen below)
        int least = 1;
#pragma unroll
        for (int k = 0; k < E; ++k) least = min(least, __builtin_bit_cast(int, w[W ? k : 0]));
        wbad = least <= 0;
      }
      if (wbad) *a.bad_weight = 1u;
    }
    opaque(w);
  }
  opaque(y);
  T big = T(0);
#pragma unroll
  for (int k = 0; k < E; ++k) big = max_t(big, abs_t(y[k]));
  RunSums<T, W> t;
#pragma unroll
  for (int k = 0; k < E; ++k) {
    t.add(y[k], w[W ? k : 0]);
    element_end<T, E>(k);
  }
  // (the sums formed whole here: a test of one of them would otherwise come before the others are,
  // with every partial sum kept for those)
  asm volatile("" : "+v"(t.s), "+v"(t.sl), "+v"(t.w), "+v"(t.wl));
  if (W && a.bad_weight != nullptr && t.w != t.w) *a.bad_weight = 1u;
  bool nan = false;
  if (t.s != t.s) {
#pragma unroll
    for (int k = 0; k < E; ++k) nan |= y[k] != y[k];
  }
  wave_scan<PR>(t.s, t.sl, r.b.xs, r.wave_s);
  if constexpr (W) wave_scan<PR>(t.w, t.wl, r.b.xw, r.wave_w);
  const double mx = wave_max_f64(static_cast<double>(big));
  const bool anynan = __any(nan);
  if (lane == 0) {
    sh.tot[0][wave] = r.wave_w.hi;
    sh.tot[1][wave] = r.wave_w.lo;
    sh.tot[2][wave] = r.wave_s.hi;
    sh.tot[3][wave] = r.wave_s.lo;
    sh.maxabs[wave] = mx;
    sh.bad[wave] = anynan ? 1 : 0;
  }
  __syncthreads();
  r.wsum = W ? 0.0 : static_cast<double>(g.glen);
  for (int q = 0; q < nt / kWave; ++q) {
    if (q < wave) {
      r.b.bs = sums_plus<PR>(r.b.bs, DD{sh.tot[2][q], sh.tot[3][q]});
      if constexpr (W) r.b.bw = sums_plus<PR>(r.b.bw, DD{sh.tot[0][q], sh.tot[1][q]});
    }
    if constexpr (W) r.wsum += sh.tot[0][q];
    r.maxabs = __builtin_fmax(r.maxabs, sh.maxabs[q]);
    r.bad |= sh.bad[q] != 0;
  }
  r.b.bs = uniform_dd(r.b.bs);
  if constexpr (W) {
    r.b.bw = uniform_dd(r.b.bw);
    r.wsum = uniform_f64(r.wsum);
  }
  r.maxabs = uniform_f64(r.maxabs);
  r.bad = __builtin_amdgcn_readfirstlane(r.bad ? 1 : 0) != 0;
  r.b.xs = sums_plus<PR>(r.b.bs, r.b.xs);
  if constexpr (W) r.b.xw = sums_plus<PR>(r.b.bw, r.b.xw);
  if (threadIdx.x == nt - 1) {  // (the last wave's: every element is in its sums)
    const int pad = g.len - g.glen;  // (ragged rows: the pad, of weight 1)
    const DD S = r.bad ? DD{0.0, 0.0} : dd_add(r.b.bs, r.wave_s);
    const DD Wd = W ? dd_add(r.b.bw, r.wave_w) : DD{static_cast<double>(g.glen), 0.0};
    const DD Sp = MAP && !r.bad ? dd_add(S, pad * signed_pad(a)) : S;
    const DD Wp = MAP ? dd_add(Wd, static_cast<double>(pad)) : Wd;
    *out.bad = r.bad ? 1 : 0;
    out.tot[0] = Wp.hi;
    out.tot[1] = Wp.lo;
    out.tot[2] = Sp.hi;
    out.tot[3] = Sp.lo;
    sh.end[0] = Wp.hi + Wp.lo;
    sh.end[1] = Sp.hi + Sp.lo;
  }
  return r;
}

// A group's points wait for overflow_kernel: they are more than its slots.
constexpr int kOverflow = -1;

template <typename T, bool W, int NT, int E, bool MAP>
__global__ __launch_bounds__(NT, 4) void group_kernel(GroupArgs a) {
  constexpr bool PR = sizeof(T) == 8;
  constexpr int NW = NT / kWave;
  extern __shared__ __align__(64) char group_lds[];
  GroupShared<NW>& sh = *reinterpret_cast<GroupShared<NW>*>(group_lds);
  static_assert(sizeof(GroupShared<NW>) <= group_head_bytes(NW), "the shared head's size");
  char* const region = group_lds + group_head_bytes(NW);
  // (at most two waves: always all)
  const int nt = NT <= 2 * kWave ? NT : a.nt;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = wave_index();
  if (a.mark != nullptr && blockIdx.x == 0 && tid == 0)
    __hip_atomic_store(a.mark, a.mark_value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  const GroupThread<T, W, NT, E, MAP> g(a, blockIdx.x);
  const int len = g.glen, t0 = g.t0;
  const NodeOut out = node_at(a.out, W, g.row, g.grp);

  // 1. the thread's elements and their sums
  T y[E], w[W ? E : 1];
  g.load_at(a, 0, len, region + wave * (kWave * E * static_cast<int>(sizeof(T))), y, w);
  const GroupSums q = group_sums(a, g, sh, out, y, w, nt);
  const BaseSums& b = q.b;
  const CPt me{b.xs.hi, W ? b.xw.hi : static_cast<double>(min(t0, len))};
  opaque(y);
  if constexpr (W) opaque(w);

  // 2. the coarse points: 65 a wave (its threads' first points and its end)
  double* const cs = reinterpret_cast<double*>(region);
  double* const cw = cs + NW * (kWave + 1);
  T* const fy = reinterpret_cast<T*>(cw + NW * (kWave + 1));
  const int c0 = wave * (kWave + 1);
  cs[c0 + lane] = me.s;
  cw[c0 + lane] = me.w;
  if (lane == kWave - 1) {
    cs[c0 + kWave] = sums_plus<PR>(b.bs, q.wave_s).hi;
    cw[c0 + kWave] = W ? sums_plus<PR>(b.bw, q.wave_w).hi : static_cast<double>(min((wave + 1) * kWave * E, len));
  }
  fy[tid] = y[0];
  wave_fence();
  const int nact = max(0, min(kWave, (len - wave * kWave * E + E - 1) / E));
  uint64_t alive = nact == kWave ? ~uint64_t{0} : (uint64_t{1} << nact) - 1;
  auto wave_point = [&](int j) { return CPt{cs[c0 + j], cw[c0 + j]}; };
  if (nact > 0) alive = coarse_rounds(alive, me, wave_point);
  CPt ca{0.0, 0.0}, cb{0.0, 1.0};  // the chord over the thread's elements
  bool own = true;                 // (the wave's own)
  if constexpr (NW > 1) {
    if (lane == 0) sh.live[wave] = __popcll(alive);
    __syncthreads();
    int before = 0, live = 0;
    for (int q = 0; q < nt / kWave; ++q) {
      before += q < wave ? sh.live[q] : 0;
      live += sh.live[q];
    }
    own = live > kWave;
    if (!own) {
      const int at = before + __popcll(alive & ((uint64_t{1} << lane) - 1));
      if ((alive >> lane) & 1) {
        sh.ls[at] = me.s;
        sh.lw[at] = me.w;
      }
      if (tid == 0) {
        const int last = (len - 1) / (kWave * E) * (kWave + 1) + kWave;
        sh.ls[kWave] = cs[last];
        sh.lw[kWave] = cw[last];
      }
      __syncthreads();
      if (nact > 0) {
        auto list_point = [&](int j) { return CPt{sh.ls[j], sh.lw[j]}; };
        uint64_t all = live == kWave ? ~uint64_t{0} : (uint64_t{1} << live) - 1;
        all = coarse_rounds(all, list_point(min(lane, live - 1)), list_point);
        const int r = before + __popcll(alive & ((uint64_t{2} << lane) - 1)) - 1;
        ca = list_point(at_or_below(all, r));
        cb = list_point(beyond(all, r));
      }
    }
  }
  if (own && nact > 0) {
    ca = wave_point(at_or_below(alive, lane));
    cb = wave_point(beyond(alive, lane));
  }

  // 3. the candidates: bit k, the point after element k. The margin bounds what rounding can move a
  // point's height over the chord by: the sums' (32 terms a thread, the scan's steps) and this
  // loop's, under 2^-48 of the largest |y| and |slope| times the weight, 16-fold.
  uint32_t bits = 0;
  {
    const double m = slope_div(cb.s - ca.s, cb.w - ca.w);
    const double margin = (q.maxabs + __builtin_fabs(m)) * q.wsum * 0x1p-44;
    double d = __builtin_fma(-m, me.w - ca.w, me.s - ca.s);
    const T ynext = fy[min(tid + 1, nt - 1)];
#pragma unroll
    for (int k = 0; k < E; ++k) {
      if constexpr (W) d = __builtin_fma(static_cast<double>(w[W ? k : 0]), static_cast<double>(y[k]) - m, d);
      else d += static_cast<double>(y[k]) - m;
      const bool rises = y[k] < (k + 1 < E ? y[k + 1 < E ? k + 1 : 0] : ynext);
      bits |= (rises && !(d > margin)) ? 1u << k : 0u;
      element_end<T, E>(k);
    }
    if (q.bad) bits = 0;  // (a NaN group: its ends only)
    const int inner = max(0, min(E, len - 1 - t0));  // (the group's end comes below)
    bits &= inner == 32 ? ~0u : (1u << inner) - 1u;
    // the group's end, in the thread that holds its last element (a NaN row's pad is in its one
    // block)
    const int jend = len - 1 - t0;
    if (jend >= 0 && jend < E && !(MAP && q.bad && g.len > len)) bits |= 1u << jend;
  }

  // 4. the hull of the candidates and both ends, in LDS
  const GPoints<W, PR> pts = points_carve<W, PR, uint16_t>(region, a.cap);
  const int extra = tid == 0 ? 1 : 0;  // point 0, before every element
  int all;
  int pos = place<NT>(__popc(bits) + extra, all, sh, nt);
  if (all + 1 > a.cap) {
    // (a chunk begins where a thread's elements do: see overflow_shape)
    const int ce = a.chunk * a.span0;
    const int64_t c0 = static_cast<int64_t>(g.grp) * a.cpg;
    if (t0 < len && t0 % ce == 0) {
      double* const tot = node_at(a.chunks, W, g.row, c0 + t0 / ce).tot;
      tot[0] = W ? b.xw.hi : 0.0;
      tot[1] = W ? b.xw.lo : 0.0;
      tot[2] = b.xs.hi;
      tot[3] = b.xs.lo;
    }
    if (tid == 0) {
      *node_at(a.chunks, W, g.row, c0).bad = 0;
      *out.count = kOverflow;
    }
    return;
  }
  if (extra != 0) pput(pts, pos++, HPt{0, 0.0, 0.0, 0.0, 0.0});
  opaque(y);
  if constexpr (W) opaque(w);
  emit<T, W, E>(pts, pos, bits, t0, q.bad, b, y, w);
  __syncthreads();
  int cnt = prune_all<NT>(pts, all, sh.wc, &sh.result, nt);
  if constexpr (MAP) {
    // the pad, beyond the row's extreme, is a block of its own (ti_fwd_rows: float32 only)
    if (g.len > len) {
      if (tid == 0) pput(pts, cnt, HPt{g.len, sh.end[1], 0.0, sh.end[0], 0.0});
      ++cnt;
      __syncthreads();
    }
  }
  for (int k = tid; k < cnt; k += nt) {
    const HPt p = pget(pts, k);
    out.idx[k] = p.i;
    put_dd(out.shi, out.slo, k, p.s, p.sl);
    if constexpr (W) put_dd(out.whi, out.wlo, k, p.w, p.wl);
  }
  if (tid == 0) *out.count = cnt;
  if (a.expand) {
    RowExpand x = a.xp;
    x.lds_bytes -= a.expand_at;
    expand_hull<T, W, MAP, NT, (E < 16 ? E : 16)>(x, LdsHull<W, PR>{pts}, cnt, q.bad, g.row, region + a.expand_at, nt);
  }
}

// The groups of more candidates than slots (kOverflow): the points at every rise, a chunk of spans
// at a time, each chunk's hull to its spans' slots in the group's frame, then those merged by
// reference (merge_global). A workgroup a group, or several, which share its chunks, where groups
// are few. Where none overflowed (noisy data) the launch is one read of the counts. (A kernel of
// its own: in group_kernel its registers would halve every group's occupancy. Few threads a
// workgroup, as most of the merge keeps a few busy, and up to four workgroups a CU.)
//
// What bounds it: a chunk's rounds and the merge's chains of reads. With a workgroup a group
// whatever their number, and float64 in 128 threads of 8 elements: one weighted rising row of 16384
// 166 us (float64 377), now 128 (154); 200 of them 203 (484), now 207 (289); 1000 float64 ones of
// 5000 317, now 253 (float64: with the conversion of float32 inputs).
template <typename T, bool W, int NT, int E, bool MAP>
__global__ __launch_bounds__(NT, 4) void overflow_kernel(GroupArgs a) {
  constexpr bool PR = sizeof(T) == 8;
  constexpr int NW = NT / kWave;
  extern __shared__ __align__(64) char group_lds[];
  GroupShared<NW>& sh = *reinterpret_cast<GroupShared<NW>*>(group_lds);
  char* const region = group_lds + group_head_bytes(NW);
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = wave_index();
  // (part p of a group's `parts`: chunks p, p + parts, ...)
  const unsigned parts = static_cast<unsigned>(a.parts);
  const unsigned items = static_cast<unsigned>(a.batch * a.gpr) * parts;
  const int* const counts = node_at(a.out, W, 0, 0).count;
  bool any = false;
  for (unsigned k = blockIdx.x + gridDim.x * tid; k < items; k += gridDim.x * NT) any |= counts[k / parts] == kOverflow;
  if (!__syncthreads_or(any)) return;
  const int ce = a.chunk * a.span0;
  const GPoints<W, PR> pts = points_carve<W, PR, uint16_t>(region, a.cap);
  char* const slab = region + wave * (kWave * E * static_cast<int>(sizeof(T)));
  for (unsigned item = blockIdx.x; item < items; item += gridDim.x) {
    const unsigned gi = item / parts;
    const int part = static_cast<int>(item - gi * parts);
    // (the same in every thread: overwritten once all of the group's parts, this one too, are done)
    if (counts[gi] != kOverflow) continue;
    const GroupThread<T, W, NT, E, MAP> g(a, gi);
    const int len = g.glen;
    const int nch = (len + ce - 1) / ce;
    if (part >= nch) continue;  // (a group at its row's end)
    const int64_t c0 = static_cast<int64_t>(g.grp) * a.cpg;
    for (int chunk = part; chunk < nch; chunk += a.parts) {
      __syncthreads();  // (the points, counts and totals before read by every thread)
      const int p0 = chunk * ce, clen = min(ce, len - p0);
      const double* const tot = node_at(a.chunks, W, g.row, c0 + chunk).tot;
      const DD cs{tot[2], tot[3]}, cw{tot[0], tot[1]};  // the sums before the chunk
      T y[E], w[W ? E : 1];
      g.load_at(a, p0, clen, slab, y, w);
      RunSums<T, W> t;
#pragma unroll
      for (int k = 0; k < E; ++k) t.add(y[k], w[W ? k : 0]);
      BaseSums b{};
      DD wave_s, wave_w{0.0, 0.0};
      wave_scan<PR>(t.s, t.sl, b.xs, wave_s);
      if constexpr (W) wave_scan<PR>(t.w, t.wl, b.xw, wave_w);
      if (lane == 0) {
        sh.tot[0][wave] = wave_w.hi;
        sh.tot[1][wave] = wave_w.lo;
        sh.tot[2][wave] = wave_s.hi;
        sh.tot[3][wave] = wave_s.lo;
      }
      T* const fy = reinterpret_cast<T*>(region + NW * (kWave * E * static_cast<int>(sizeof(T))));
      fy[tid] = y[0];
      __syncthreads();
      b.bs = cs;
      b.bw = cw;
      for (int q = 0; q < wave; ++q) {
        b.bs = sums_plus<PR>(b.bs, DD{sh.tot[2][q], sh.tot[3][q]});
        if constexpr (W) b.bw = sums_plus<PR>(b.bw, DD{sh.tot[0][q], sh.tot[1][q]});
      }
      b.xs = sums_plus<PR>(b.bs, b.xs);
      if constexpr (W) b.xw = sums_plus<PR>(b.bw, b.xw);
      const T ynext = fy[min(tid + 1, NT - 1)];
      uint32_t bits = 0;
#pragma unroll
      for (int k = 0; k < E; ++k) bits |= y[k] < (k + 1 < E ? y[k + 1 < E ? k + 1 : 0] : ynext) ? 1u << k : 0u;
      const int t0 = tid * E, inner = max(0, min(E, clen - 1 - t0));
      bits &= (1u << inner) - 1u;
      int all;
      int pos = place<NT>(__popc(bits) + (tid == 0 ? 1 : 0), all, sh);
      // The chunk's ends: where the next chunk begins, from that chunk's own sums, so that the point
      // where two chunks meet is one point, to its last bit (summed otherwise in each, 34 of 600
      // weighted rows of 3840 stepped down). (float32: the pair's sum, rounded once)
      const auto end = [](int i, DD s, DD w) {
        return PR ? HPt{i, s.hi, s.lo, w.hi, w.lo} : HPt{i, s.hi + s.lo, 0.0, w.hi + w.lo, 0.0};
      };
      if (tid == 0) pput(pts, pos++, end(p0, cs, cw));
      if (tid == NT - 1) {
        DD es = sums_plus<PR>(b.bs, wave_s), ew = W ? sums_plus<PR>(b.bw, wave_w) : DD{0.0, 0.0};
        if (chunk + 1 < nch) {
          const double* const next = tot + 4;  // (the next chunk's)
          es = DD{next[2], next[3]};
          ew = DD{next[0], next[1]};
        }
        pput(pts, all, end(p0 + clen, es, ew));
      }
      ++all;
      emit<T, W, E>(pts, pos, bits, p0 + t0, false, b, y, w);
      __syncthreads();
      const int cnt = prune_all<NT>(pts, all, sh.wc, &sh.result);
      const NodeOut o = node_at(a.chunks, W, g.row, c0 + chunk);
      for (int k = tid; k < cnt; k += NT) {
        const HPt p = pget(pts, k);
        o.idx[k] = p.i;
        put_dd(o.shi, o.slo, k, p.s, p.sl);
        if constexpr (W) put_dd(o.whi, o.wlo, k, p.w, p.wl);
      }
      if (tid == 0) *o.count = cnt;
    }
    // The last of the group's parts to be done merges the chunks' hulls: every part's stores are
    // made visible to the device before it is counted, and read after the last one was.
    __syncthreads();
    if (parts > 1) {
      if (tid == 0)
        sh.result = __hip_atomic_fetch_add(node_at(a.chunks, W, g.row, c0).bad, 1, __ATOMIC_ACQ_REL,
                                           __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      if (sh.result != min(a.parts, nch) - 1) continue;
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    const NodeOut out = node_at(a.out, W, g.row, g.grp);
    MergeSmall& sm = *reinterpret_cast<MergeSmall*>(region);
    MergeRanges& mr = *reinterpret_cast<MergeRanges*>(region + ((sizeof(MergeSmall) + 63) & ~size_t(63)));
    for (int c = tid; c < nch; c += NT) {
      sm.cnt[c] = *node_at(a.chunks, W, g.row, c0 + c).count;
#pragma unroll
      for (int i = 0; i < 4; ++i) sm.tot[i][c] = 0.0;  // (the chunks are in the group's frame)
    }
    __syncthreads();
    MergeArgs ma;
    ma.in = a.chunks;
    ma.out = a.out;
    ma.child_elems = 0;
    merge_global<W, true, NT>(ma, sm, mr.rlo, mr.rhi, mr.pre, g.row, c0, nch, out);
    __syncthreads();
    // A row's final hull of float32 data convex in its stored values: the chunks' hulls are, and
    // share their points, but a bridge found by a search over nearly collinear points can miss by
    // their rounding. A triple that holds vertices of two chunks is tested; where one fails, the
    // whole hull is. (Longer rows: their hulls, after the last merge.)
    if constexpr (!PR) {
      if (a.expand) {
        const VArr v = dvarr_of(out);
        bool dented = false;
        for (int c = 1 + tid; c < nch; c += NT) {
          for (int k = max(mr.pre[c] - 1, 1); k <= min(mr.pre[c], sm.total - 2); ++k)
            dented |= vpools<W>(vload<W>(v, k - 1), vload<W>(v, k), vload<W>(v, k + 1));
        }
        if (__syncthreads_or(dented)) {
          VPt* tile = reinterpret_cast<VPt*>(region);
          int* wcount = reinterpret_cast<int*>(tile + NT + 2);
          repair_row<W, NT, 1>(out, tile, wcount, wcount[NT / kWave], a.repair_passes);
          __syncthreads();
        }
      }
    }
    if constexpr (MAP) {
      // (the pad's block: see group_kernel)
      if (g.len > len) {
        if (tid == 0) {
          const int cnt = *out.count;
          out.idx[cnt] = g.len;
          out.shi[cnt] = out.tot[2] + out.tot[3];
          if constexpr (W) out.whi[cnt] = out.tot[0] + out.tot[1];
          *out.count = cnt + 1;
        }
      }
    }
    if (a.expand) expand_row<T, W, MAP, NT>(a.xp, out, false, g.row, region);
    __syncthreads();
  }
}

// LDS of a launch: the head; then the slabs, the coarse points, or the point slots with the
// expansion's (bitmap, counts, a table of every edge the slots can hold) behind them, whichever
// is largest.
template <class K>
hipError_t launch_lds(K k, const GroupArgs& a, int64_t blocks, int threads, int lds, hipStream_t stream) {
  if (lds > 65536) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
  }
  k<<<dim3(static_cast<unsigned>(blocks)), dim3(threads), static_cast<size_t>(lds), stream>>>(a);
  return hipGetLastError();
}

// Chunks of at most 2048 elements (float64: 1024, in as many threads: its merge keeps more of them
// busy), a multiple of 8 spans (float64: 4) of a multiple of 4 elements each (float64 groups of up
// to 2048 elements: of 8; float32 ones never overflow), so a chunk begins where one of
// group_kernel's threads does, whose sums it starts from.
template <typename T>
constexpr int kOverflowThreads = 256;
template <typename T>
constexpr int kOverflowElems = sizeof(T) == 8 ? 4 : 8;
template <typename T>
void overflow_shape(GroupArgs& a) {
  a.chunk = std::min(kGroup, kOverflowThreads<T> * kOverflowElems<T> / a.span0 & (sizeof(T) == 8 ? ~3 : ~7));
  a.cpg = (a.g_elems + a.chunk * a.span0 - 1) / (a.chunk * a.span0);
  a.chunks = a.spans;
  a.chunks.npr = a.gpr * a.cpg;
  a.chunks.spn = a.chunk;
}

// The groups that overflowed. Several workgroups share a group where that gives up to a workgroup a
// CU; each is counted by an atomic that first writes its XCD's L2 back, which many groups cannot
// afford (1000 rising rows of 10000, a workgroup a chunk: 1795 us, a workgroup a group 180).
constexpr int64_t kOverflowShare = 256;
template <typename T, bool W, bool MAP>
hipError_t overflow_launch(GroupArgs a, hipStream_t stream) {
  constexpr bool PR = sizeof(T) == 8;
  constexpr int tb = static_cast<int>(sizeof(T));
  constexpr int NT = kOverflowThreads<T>, E = kOverflowElems<T>;
  const int64_t groups = a.batch * a.gpr;
  a.parts = static_cast<int>(std::min<int64_t>(a.cpg, std::max<int64_t>(1, kOverflowShare / groups)));
  a.mark = nullptr;
  a.cap = (a.chunk * a.span0 + 1 + 3) & ~3;
  int region = std::max(a.cap * point_bytes<W, PR, uint16_t>(), (NT * E + NT) * tb);
  region = std::max(region, static_cast<int>(((sizeof(MergeSmall) + 63) & ~size_t(63)) + sizeof(MergeRanges)));
  if (a.expand) region = std::max({region, expand_lds_min(a.g_elems, NT, tb), static_cast<int>(repair_lds_bytes(NT))});
  region = (region + 63) & ~63;
  a.xp.lds_bytes = region;
  return launch_lds(overflow_kernel<T, W, NT, E, MAP>, a, std::min<int64_t>(groups * a.parts, 2048), NT,
                    group_head_bytes(NT / kWave) + region, stream);
}

template <typename T, bool W, int NT, int E, bool MAP>
hipError_t group_launch(GroupArgs a, hipStream_t stream) {
  constexpr bool PR = sizeof(T) == 8;
  constexpr int NW = NT / kWave;
  constexpr int tb = static_cast<int>(sizeof(T));
  constexpr int P = E * tb / 16;
  constexpr int G = NT * E;
  const int64_t grid = a.batch * a.gpr;
  if (grid > 0x7FFFFFFF) return hipErrorInvalidConfiguration;
  // (as many waves as the groups' elements fill: an idle wave takes its registers all the same)
  a.nt = NT <= 2 * kWave ? NT : (a.g_elems + E * kWave - 1) / (E * kWave) * kWave;
  // Slots: every point of a group of up to 2048 elements (float64: half); beyond, one for every
  // four elements (noisy trends leave a candidate in eight or fewer), float64 one for every eight
  // and at least 1028: what lets two workgroups or more share a CU's LDS. Weighted groups of over
  // 8192: three for every sixteen (18 bytes a slot and 4 in the expansion's table: with 4100 one
  // workgroup would take 94 KB of the CU's 160).
  constexpr int kMost = PR ? std::max(1028, G / 8 + 4) : G <= 2048 ? 2052 : G >= 16384 ? (W ? 3076 : 4100) : G / 4 + 4;
  a.cap = (std::min(a.g_elems + 3, kMost) + 3) & ~3;
  overflow_shape<T>(a);
  a.expand_at = (a.cap * point_bytes<W, PR, uint16_t>() + 63) & ~63;
  const int words4 = (((a.g_elems + 31) / 32) + 3) & ~3;
  int region = std::max(P > 2 ? a.nt * E * tb : 0, NW * (kWave + 1) * 16 + NT * tb);
  region = std::max(region, a.expand_at + (a.expand ? 64 + 2 * words4 * 4 + a.cap * tb : 0));
  region = (region + 63) & ~63;
  a.xp.lds_bytes = region;
  const bool may_overflow = a.cap < a.g_elems + 3;
  if (may_overflow && a.chunk * a.span0 % E != 0) return hipErrorInvalidConfiguration;  // (see overflow_shape)
  const hipError_t e = launch_lds(group_kernel<T, W, NT, E, MAP>, a, grid, a.nt, group_head_bytes(NW) + region, stream);
  if (e != hipSuccess || !may_overflow) return e;
  return overflow_launch<T, W, MAP>(a, stream);
}

// Threads and elements a thread by the group's size: a thread's eight to 32 elements share its scan
// steps and its chord (fewer leave the fixed work of a wave, about 500 instructions, to fewer
// elements; 32 float64 elements, or 32 weighted ones in more than 128 registers, would spill).
template <typename T, bool W, bool MAP>
hipError_t group_shape(const GroupArgs& a, hipStream_t stream) {
  const int g = a.g_elems;
  if (g <= 256) return group_launch<T, W, 64, 4, MAP>(a, stream);
  if (g <= 512) return group_launch<T, W, 64, 8, MAP>(a, stream);
  if (g <= 1024) return group_launch<T, W, 128, 8, MAP>(a, stream);
  if (g <= 2048) return group_launch<T, W, 256, 8, MAP>(a, stream);
  if (g <= 4096) return group_launch<T, W, 256, 16, MAP>(a, stream);
  if (g <= 8192) return group_launch<T, W, 512, 16, MAP>(a, stream);
  if constexpr (sizeof(T) == 4) return group_launch<T, W, 512, 32, MAP>(a, stream);
  else return group_launch<T, W, 1024, 16, MAP>(a, stream);
}

}  // namespace

hipError_t group_run(const TileArgs& t, const NodeLevel& spans, int64_t span0, const NodeLevel& out, int64_t g_elems,
                     TileRec* tiles, int repair_passes) {
  GroupArgs a{};
  a.y = t.y;
  a.w = t.w;
  a.bad_weight = t.bad_weight;
  a.n = t.n;
  a.batch = t.batch;
  a.gpr = (t.n + g_elems - 1) / g_elems;
  a.g_elems = static_cast<int>(g_elems);
  a.span0 = static_cast<int>(span0);
  a.flags = t.flags;
  a.spans = spans;
  a.out = out;
  a.expand = tiles != nullptr;
  a.repair_passes = repair_passes;
  a.xp.n = t.n;
  a.xp.out = t.out;
  a.xp.starts = t.starts;
  a.xp.tiles = tiles;
  a.xp.tile_n = static_cast<int>(tile_elems(t.w != nullptr));
  a.xp.tpr = (t.n + a.xp.tile_n - 1) / a.xp.tile_n;
  a.xp.flags = t.flags;
  a.xp.lo = t.lo;
  a.xp.hi = t.hi;
  a.xp.map = t.map;
  a.map = t.map;
  a.mark = t.start_mark;
  a.mark_value = t.mark_value;
  if (t.dtype == TI_F32) {
    if (t.map.rows != nullptr)  // (ragged rows of a block: float32 only)
      return t.w != nullptr ? group_shape<float, true, true>(a, t.stream) : group_shape<float, false, true>(a, t.stream);
    return t.w != nullptr ? group_shape<float, true, false>(a, t.stream) : group_shape<float, false, false>(a, t.stream);
  }
  return t.w != nullptr ? group_shape<double, true, false>(a, t.stream) : group_shape<double, false, false>(a, t.stream);
}

}  // namespace ti
