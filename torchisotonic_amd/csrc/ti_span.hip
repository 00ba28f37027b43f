// Rows of 33 to 256 elements in batches of thousands (LongPlan::levels == 0): one lane per row.
//
// Takes the place of the reference's packed kernel for such rows (reference src/torchisotonic/
// csrc/tiles.cuh:920-1112). A lane runs the monotone chain over its whole row by itself: no
// scans, no merges, no barriers. The row streams through registers C elements at a time (the next
// block of LC loading meanwhile), in two phases:
//
//   1. uniform work per chunk: the cumulative sums (float64, relative to the row's start;
//      float64 data also carries their rounding errors, two-sum) at every point, and the
//      candidate points appended to the lane's queue of Q slots in LDS;
//   2. before each chunk, an event loop in which every lane with queued candidates does one
//      stack operation per iteration - pop the top vertex, or push its next candidate - until
//      every queue has room for the chunk. Lanes advance independently, so one lane's run of
//      pops does not hold the others at a data-dependent loop, and a lane's queue lets it fall
//      behind by up to Q candidates before the wave waits for it.
//
// (Longer rows, and smaller batches, which would leave most lanes idle, take ti_group.hip: a
// workgroup or wave per row; 100000 rows of 128: 103 us here, 149 there; 20000 rows of 200, two
// lanes a row then: 107 us, 36 there.)
//
// The stack lives in a ring of R LDS slots per lane; positions that fall out of it go to the
// row's hull array in global memory, where the finished hull ends anyway (noisy data seldom
// gets that deep).
//
// A point is a candidate only where the data rises into it (y_{k-1} < y_k): elsewhere the slope
// into it is at least the slope out of it, and equal slopes pool, so it is never a vertex. Grids
// of at most two waves a SIMD (FILT) also drop a point that lies clearly above the chord of its
// neighbours two elements away on either side: about 0.68 loop iterations per element of noisy
// data instead of 0.98, for some twenty more float64 operations per element.
//
// Output: the rows' final hulls, which xpack_kernel (ti_merge.hip) expands.
#include <atomic>

#include "ti_common.h"
#include "ti_kernels.h"
#include "ti_tile.h"

namespace ti {

namespace {

constexpr int kSpanLanes = 64;

struct SpanArgs {
  const void* y;
  const void* w;
  uint32_t* bad_weight;
  int64_t n, batch;
  NodeLevel hulls;  // level 0: one node a row
  RowMap map;       // ragged rows of one block: y and w read from the packed arrays
  // (where given) mark_value stored to *mark by the kernel's first thread as it starts: the
  // caller's mark that a kernel before this one has read every weight
  uint32_t* mark;
  uint32_t mark_value;
};

// Per lane (columns [slot][lane], so lanes never share a bank row): the candidate queue (index
// and sums of each queued point) and the stack ring. Arrays a configuration does not use have
// no rows (a zero-length array, which only code under a false `if constexpr` or condition names).
template <typename T, bool W, int Q, int R>
struct SpanLds {
  static constexpr bool PR = sizeof(T) == 8;
  int qi[Q][kSpanLanes];
  double qs[Q][kSpanLanes];
  double qsl[PR ? Q : 0][kSpanLanes];
  double qw[W ? Q : 0][kSpanLanes];
  double qwl[W && PR ? Q : 0][kSpanLanes];
  int ri[R][kSpanLanes];
  double rs[R][kSpanLanes];
  double rsl[PR ? R : 0][kSpanLanes];
  double rw[W ? R : 0][kSpanLanes];
  double rwl[W && PR ? R : 0][kSpanLanes];
};

// N consecutive values at byte offset `off` of a buffer resource, 16 bytes per load. Reads past
// the resource's end return zero and never fault, so a block is always loaded whole (its values
// past the span's end are never used) and the loads stay straight-line code.
template <typename T, int N>
__device__ __forceinline__ void load_block(__amdgpu_buffer_rsrc_t r, uint32_t off, T (&v)[N]) {
  constexpr int V = 16 / sizeof(T);
  using VT = T __attribute__((ext_vector_type(V)));
#pragma unroll
  for (int j = 0; j < N / V; ++j) {
    // (taken as a vector of T at once: element access on the builtin's integer-vector result
    // is what this compiler narrows to a single-dword load)
    const VT x = __builtin_bit_cast(VT, __builtin_amdgcn_raw_buffer_load_b128(r, off + j * 16, 0, 0));
#pragma unroll
    for (int t = 0; t < V; ++t) v[j * V + t] = x[t];
  }
}

template <typename T, bool W, int C, int Q, int R, int LC, bool INC, bool MAP = false, bool FILT = false>
__global__ __launch_bounds__(kSpanLanes) void span_kernel(SpanArgs a) {
  static_assert((R & (R - 1)) == 0 && (Q & (Q - 1)) == 0 && R >= 4, "ring and queue slots: powers of two");
  static_assert(C < Q, "a chunk's candidates fit the queue");
  static_assert(LC % C == 0, "a load block is a whole number of chunks");
  // PR: the row's sums carry their rounding errors (float64 data).
  constexpr bool PR = sizeof(T) == 8;
  __shared__ SpanLds<T, W, Q, R> L;
  const int lane = threadIdx.x;
  if (a.mark != nullptr && blockIdx.x == 0 && lane == 0)
    __hip_atomic_store(a.mark, a.mark_value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kSpanLanes + lane;
  const bool active = row < a.batch;
  const int64_t node = active ? row : 0;
  const int len = active ? static_cast<int>(a.n) : 0;
  constexpr double sgn = INC ? 1.0 : -1.0;
  // Ragged rows (MAP, a.map): the lane's row in the packed arrays, and rlim, the elements that
  // are the row's own; from rlim on the row holds the pad (weight 1), made in registers: a
  // block wholly past rlim is never read (its loads take an offset past the buffer's end, which
  // returns zeros without a memory access).
  int64_t mfirst = 0, mlen = a.n;
  if constexpr (MAP) map_row(a.map, node, a.n, mfirst, mlen);
  const int rlim = MAP ? static_cast<int>(max<int64_t>(mlen, 0)) : 0x7FFFFFFF;
  const T tpad = static_cast<T>(a.map.pad);
  // The wave's rows are consecutive elements, so one buffer resource based at the first of them
  // serves every lane (ragged rows: one resource over the whole packed arrays, under 2 GB).
  // (read from the first lane: the compiler then keeps the buffer resources in scalar registers,
  // where a per-lane value would put every load in a loop over the lanes' distinct resources)
  const int64_t base = wave_uniform(MAP ? int64_t{0} : static_cast<int64_t>(blockIdx.x) * kSpanLanes * a.n);
  const int64_t total = MAP ? a.map.total : a.batch * a.n;  // elements of the arrays
  const __amdgpu_buffer_rsrc_t ry = make_rsrc(static_cast<const T*>(a.y) + base, (total - base) * sizeof(T));
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(W ? static_cast<const T*>(a.w) + base : a.y, (total - base) * sizeof(T));
  // this lane's row in memory, an element offset from base
  const int64_t lmem = MAP ? mfirst : lane * a.n;
  // block b's byte offset (a block wholly past rlim: past the resource, never read)
  auto boff = [&](int b) -> uint32_t {
    if constexpr (!MAP) return static_cast<uint32_t>((lmem + b) * static_cast<int64_t>(sizeof(T)));
    return b < rlim ? static_cast<uint32_t>((lmem + b) * static_cast<int64_t>(sizeof(T))) : 0x80000000u;
  };
  const NodeOut o = node_out(a.hulls, W, node);

  auto ring_put = [&](int q, const HPt& p) {
    const int r = q & (R - 1);
    L.ri[r][lane] = p.i;
    L.rs[r][lane] = p.s;
    if constexpr (PR) L.rsl[r][lane] = p.sl;
    if constexpr (W) L.rw[r][lane] = p.w;
    if constexpr (W && PR) L.rwl[r][lane] = p.wl;
  };
  auto ring_get = [&](int q) -> HPt {
    const int r = q & (R - 1);
    HPt p;
    p.i = L.ri[r][lane];
    p.s = L.rs[r][lane];
    p.sl = PR ? L.rsl[PR ? r : 0][lane] : 0.0;
    p.w = W ? L.rw[W ? r : 0][lane] : 0.0;
    p.wl = (W && PR) ? L.rwl[(W && PR) ? r : 0][lane] : 0.0;
    return p;
  };
  // node arrays hold double-double sums; float32 data has no rounding errors to carry (lo = 0)
  auto node_put = [&](int q, const HPt& p) {
    o.idx[q] = p.i;
    put_dd(o.shi, o.slo, q, p.s, p.sl);
    if constexpr (W) put_dd(o.whi, o.wlo, q, p.w, p.wl);
  };
  auto node_get = [&](int q) -> HPt {
    HPt p;
    p.i = o.idx[q];
    p.s = o.shi[q];
    p.sl = PR ? lo_at(o.slo, q) : 0.0;
    p.w = W ? o.whi[q] : 0.0;
    p.wl = (W && PR) ? lo_at(o.wlo, q) : 0.0;
    return p;
  };

  auto q_put = [&](int q, const HPt& p) {
    const int r = q & (Q - 1);
    L.qi[r][lane] = p.i;
    L.qs[r][lane] = p.s;
    if constexpr (PR) L.qsl[r][lane] = p.sl;
    if constexpr (W) L.qw[r][lane] = p.w;
    if constexpr (W && PR) L.qwl[r][lane] = p.wl;
  };
  auto q_get = [&](int q) -> HPt {
    const int r = q & (Q - 1);
    HPt p;
    p.i = L.qi[r][lane];
    p.s = L.qs[r][lane];
    p.sl = PR ? L.qsl[PR ? r : 0][lane] : 0.0;
    p.w = W ? L.qw[W ? r : 0][lane] : 0.0;
    p.wl = (W && PR) ? L.qwl[(W && PR) ? r : 0][lane] : 0.0;
    return p;
  };

  // The stack holds positions [0, depth): [r0, depth) in the ring (1 <= depth - r0 <= R), [0, r0)
  // in the node array. The queue holds the candidates [qh, qt).
  int depth = 1, r0 = 0;
  ring_put(0, HPt{0, 0.0, 0.0, 0.0, 0.0});
  int qh = 0, qt = 0;

  double S = 0.0, SL = 0.0, P = 0.0, PL = 0.0;
  bool bad = false, wbad = false;
  // 2. one stack operation per lane and iteration - pop the top vertex B, or push the first
  // queued candidate c - until every lane holds at most `limit` queued candidates. An iteration's
  // reads depend on the previous iteration's depth and queue position only, and its one ring
  // write needs no branch: a push writes c above B, any other lane writes B back into its own
  // slot (a pop frees it next). The loop touches LDS only (and stores spills), so the next loads
  // stay in flight; a lane whose second vertex went to the node array makes the wave leave it,
  // refill that lane's ring from the node array, and come back (rare).
  // (at a raised issue priority: a wave in its chain wins the SIMD over the other wave's uniform
  // chunk work, so the chains, the kernel's bound, wait less)
  auto run = [&](int limit) {
    __builtin_amdgcn_s_setprio(1);
    for (;;) {
      while (__any(qt - qh > limit)) {
        const bool act = qt != qh;
        const bool two = act && depth >= 2;
        if (__any(two && depth - 2 < r0)) break;
        const HPt c = q_get(qh);
        const HPt A = ring_get(depth - 2), B = ring_get(depth - 1);
        // pools(A, B, c): a filtered fma test, exact where it cannot decide (see pools<true>)
        double dS1 = B.s - A.s, dS2 = c.s - B.s, dW1, dW2;
        if constexpr (PR) {
          dS1 += B.sl - A.sl;
          dS2 += c.sl - B.sl;
        }
        if constexpr (W) {
          dW1 = B.w - A.w;
          dW2 = c.w - B.w;
          if constexpr (PR) {
            dW1 += B.wl - A.wl;
            dW2 += c.wl - B.wl;
          }
        } else {
          dW1 = static_cast<double>(B.i - A.i);
          dW2 = static_cast<double>(c.i - B.i);
        }
        const double qq = dS2 * dW1;
        const double dd = __builtin_fma(dS1, dW2, -qq);
        const bool close = !(__builtin_fabs(dd) > 0x1p-52 * __builtin_fabs(qq));
        bool pop = two && dd > 0.0;
        if (__any(two && close)) {
          // (an empty statement with side effects: it keeps this rare path a branch, where the
          // compiler would otherwise compute the exact test in every iteration and select)
          asm volatile("");
          if (two && close) pop = cross_sign(dS1, dW2, dS2, dW1) >= 0;
        }
        const bool push = act && !pop;
        if (__any(push && depth - r0 == R)) {
          // a full ring: its oldest position leaves for the node array
          asm volatile("");
          if (push && depth - r0 == R) {
            node_put(r0, ring_get(r0));
            ++r0;
          }
        }
        ring_put(push ? depth : depth - 1, hsel(push, c, B));
        depth += push ? 1 : (pop ? -1 : 0);
        qh += push ? 1 : 0;
      }
      if (!__any(qt - qh > limit)) break;
      if (qt != qh && depth >= 2 && depth - 2 < r0) {
        // only the top is in the ring (depth - 1 == r0): bring back up to R / 2 positions below
        const int lo = r0 > R / 2 ? r0 - R / 2 : 0;
        for (int q = lo; q < r0; ++q) ring_put(q, node_get(q));
        r0 = lo;
      }
    }
    __builtin_amdgcn_s_setprio(0);
  };

  // loads come in blocks of LC elements (the next block in flight while this one is processed),
  // processed in chunks of C: before a chunk, the loop makes room in every queue for its
  // candidates
  T yc[LC], yn[LC];
  T wc[W ? LC : 1], wn[W ? LC : 1];
  load_block<T, LC>(ry, boff(0), yc);
  if constexpr (W) load_block<T, LC>(rw, boff(0), wc);
  // FILT: a point is queued one element late, for the stronger test below, which needs the
  // element after it. Carried from element to element: the last three elements' terms (t1 the
  // newest), their weights and signed values, the running sum of |term| (the rounding margin's
  // scale), and the sums of the point waiting to be queued.
  double t1 = 0.0, t2 = 0.0, t3 = 0.0, w1 = 1.0, w2 = 1.0, w3 = 1.0, v1 = 0.0, v2 = 0.0, A = 0.0;
  HPt pend{0, 0.0, 0.0, 0.0, 0.0};
  // (FILT) Point e - 1 (between elements e - 2 and e - 1; e the element just summed, its term t0
  // and weight w0) is a candidate where the data rises into it (v2 < v1) and it does not lie
  // above the chord from point e - 3 to point e (b, from e >= 3) or from point e - 2 to point
  // e + 1 (c, where e is in the span). Such a point is no vertex of the exact hull; it is dropped
  // only where its height above the chord exceeds 2^-39 x A x the chord's width, which bounds
  // what the rounding of the span's sums (and of this test) can move, so that near-ties stay
  // candidates and the event loop decides them as without the test.
  auto keep = [&](bool use_b, bool use_c, double t0, double w0) {
    const double thr = A * 0x1p-39;
    bool k = v2 < v1;
    if constexpr (W) {
      const double d3 = w3 + w2;
      const double db = __builtin_fma(t3 + t2, w1, -(t1 * d3));
      const double wc1 = w1 + w0;
      const double dc = __builtin_fma(t2, wc1, -((t1 + t0) * w2));
      k &= !(use_b && db > thr * (d3 + w1));
      k &= !(use_c && dc > thr * (w2 + wc1));
    } else {
      const double db = (t3 + t2) - 2.0 * t1;
      const double dc = 2.0 * t2 - (t1 + t0);
      k &= !(use_b && db > 3.0 * thr);
      k &= !(use_c && dc > 3.0 * thr);
    }
    return k;
  };
  for (int b0 = 0; b0 < len; b0 += LC) {
    // the next block, whole, whether or not the span reaches it
    load_block<T, LC>(ry, boff(b0 + LC), yn);
    if constexpr (W) load_block<T, LC>(rw, boff(b0 + LC), wn);
    // (ragged rows: the pad past the row's end, in the one block a lane's row ends in or after)
    if (MAP && __any(b0 + LC > rlim)) {
#pragma unroll
      for (int k = 0; k < LC; ++k) {
        if (b0 + k >= rlim) {
          yc[k] = tpad;
          if constexpr (W) wc[W ? k : 0] = T(1);
        }
      }
    }
    // the element after the block: the next block's first, or the pad
    auto after_block = [&]() { return MAP && b0 + LC >= rlim ? tpad : yn[0]; };
#pragma unroll
    for (int sub = 0; sub < LC; sub += C) {
      const int c0 = b0 + sub;
      run(Q - C);
      // 1. sums at every point of the chunk; each point goes to the queue's next free slot,
      // which it keeps if it is a candidate (so the stores need no branch). Without FILT, point
      // e + 1 as element e is summed, a candidate where y rises into element e + 1 (or at the
      // span's end); with FILT, point e - 1.
      auto element = [&](int k, bool cand) {
        const int e = c0 + k;
        const double ye = sgn * static_cast<double>(yc[sub + k]);
        bad |= ye != ye;
        double term = ye, we = 1.0;
        if constexpr (W) {
          we = static_cast<double>(wc[W ? sub + k : 0]);
          wbad |= !(we > 0.0);
          term = we * ye;
        }
        if constexpr (FILT) {
          A += __builtin_fabs(term);
          const bool kept = e >= 2 && keep(e >= 3, true, term, we);
          q_put(qt, pend);
          qt += kept ? 1 : 0;
          pend = HPt{e, S, PR ? SL : 0.0, W ? P : 0.0, (W && PR) ? PL : 0.0};
        }
        if constexpr (W) {
          if constexpr (PR) {
            const DD t = two_sum(P, we);
            P = t.hi;
            PL += t.lo;
          } else {
            P += we;
          }
        }
        if constexpr (PR) {
          const DD t = two_sum(S, term);
          S = t.hi;
          SL += t.lo;
        } else {
          S += term;
        }
        if constexpr (FILT) {
          t3 = t2;
          t2 = t1;
          t1 = term;
          w3 = w2;
          w2 = w1;
          w1 = we;
          v2 = v1;
          v1 = ye;
        } else {
          q_put(qt, HPt{e + 1, S, PR ? SL : 0.0, W ? P : 0.0, (W && PR) ? PL : 0.0});
          qt += cand ? 1 : 0;
        }
      };
      // the point after element e is a candidate where y rises into e + 1, or at the span's end
      auto rises = [&](T u, T v) { return INC ? u < v : v < u; };
      if (__all(c0 + C <= len)) {
        // whole chunks (all but a row's last span): no per-element bounds
#pragma unroll
        for (int k = 0; k < C; ++k) {
          if constexpr (FILT) {
            element(k, false);
          } else {
            const int kk = sub + k;
            const T ynext = kk + 1 < LC ? yc[kk + 1 < LC ? kk + 1 : 0] : after_block();
            // (the span can end only after a chunk's last element here)
            element(k, k + 1 < C ? rises(yc[kk], ynext) : ((c0 + C == len) | rises(yc[kk], ynext)));
          }
        }
      } else {
#pragma unroll
        for (int k = 0; k < C; ++k) {
          const int e = c0 + k;
          if (e < len) {
            if constexpr (FILT) {
              element(k, false);
            } else {
              const int kk = sub + k;
              const T ynext = kk + 1 < LC ? yc[kk + 1 < LC ? kk + 1 : 0] : after_block();
              element(k, (e + 1 == len) | (e + 1 < len && rises(yc[kk], ynext)));
            }
          }
        }
      }
    }
#pragma unroll
    for (int k = 0; k < LC; ++k) {
      yc[k] = yn[k];
      if constexpr (W) wc[W ? k : 0] = wn[W ? k : 0];
    }
  }
  if constexpr (FILT) {
    // the span's last two points: point len - 1 (tests a and b: there is no point len + 1), and
    // the span's end, always a vertex
    run(Q - 2);
    if (len >= 1) {
      const bool kept = len >= 2 && keep(len >= 3, false, 0.0, 1.0);
      q_put(qt, pend);
      qt += kept ? 1 : 0;
      q_put(qt, HPt{len, S, PR ? SL : 0.0, W ? P : 0.0, (W && PR) ? PL : 0.0});
      ++qt;
    }
  }
  // the last candidates
  run(0);
  if (W && wbad && a.bad_weight != nullptr) *a.bad_weight = 1u;

  // the row's hull
  if (active) {
    for (int q = r0; q < depth; ++q) node_put(q, ring_get(q));
    *o.count = depth;
    *o.bad = bad ? 1 : 0;
    o.tot[0] = W ? P : static_cast<double>(len);
    o.tot[1] = W ? PL : 0.0;
    o.tot[2] = S;
    o.tot[3] = SL;
  }
}

// SIMDs of the current device (four a CU), read once per device
int simd_count() {
  static std::atomic<int> cache[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 1024;
  int v = cache[dev].load(std::memory_order_relaxed);
  if (v == 0) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
    v = 4 * cus;
    cache[dev].store(v, std::memory_order_relaxed);
  }
  return v;
}

}  // namespace

hipError_t span_run(const TileArgs& t, const NodeLevel& hulls) {
  SpanArgs a;
  a.y = t.y;
  a.w = t.w;
  a.bad_weight = t.bad_weight;
  a.n = t.n;
  a.batch = t.batch;
  a.hulls = hulls;
  a.map = t.map;
  a.mark = t.start_mark;
  a.mark_value = t.mark_value;
  const unsigned grid = static_cast<unsigned>((t.batch + kSpanLanes - 1) / kSpanLanes);
  const bool W = t.w != nullptr;
  const bool inc = (t.flags & TI_INCREASING) != 0;
  // A grid the GPU holds in one round at two waves a SIMD or fewer is latency-bound: each wave's
  // event loop sets the time, and the stronger candidate test (FILT: fewer loop iterations for
  // more arithmetic per element) pays; over several rounds it costs more than it saves (5-7 %).
  const bool filt = t.map.rows == nullptr && grid <= 2u * static_cast<unsigned>(simd_count());
  auto go = [&](auto k_inc, auto k_dec) {
    if (inc) k_inc<<<dim3(grid), dim3(kSpanLanes), 0, t.stream>>>(a);
    else k_dec<<<dim3(grid), dim3(kSpanLanes), 0, t.stream>>>(a);
  };
  if (t.dtype == TI_F32) {
    if (t.map.rows != nullptr) {  // (ragged rows of a block: float32 only)
      if (W) go(span_kernel<float, true, 4, 8, 8, 32, true, true>, span_kernel<float, true, 4, 8, 8, 32, false, true>);
      else go(span_kernel<float, false, 4, 8, 16, 32, true, true>, span_kernel<float, false, 4, 8, 16, 32, false, true>);
    } else if (W) {
      if (filt) go(span_kernel<float, true, 4, 8, 8, 32, true, false, true>, span_kernel<float, true, 4, 8, 8, 32, false, false, true>);
      else go(span_kernel<float, true, 4, 8, 8, 32, true>, span_kernel<float, true, 4, 8, 8, 32, false>);
    } else {
      if (filt) go(span_kernel<float, false, 4, 8, 16, 32, true, false, true>, span_kernel<float, false, 4, 8, 16, 32, false, false, true>);
      else go(span_kernel<float, false, 4, 8, 16, 32, true>, span_kernel<float, false, 4, 8, 16, 32, false>);
    }
  } else {
    if (W) {
      if (filt) go(span_kernel<double, true, 4, 8, 8, 8, true, false, true>, span_kernel<double, true, 4, 8, 8, 8, false, false, true>);
      else go(span_kernel<double, true, 4, 8, 8, 8, true>, span_kernel<double, true, 4, 8, 8, 8, false>);
    } else {
      if (filt) go(span_kernel<double, false, 4, 8, 16, 8, true, false, true>, span_kernel<double, false, 4, 8, 16, 8, false, false, true>);
      else go(span_kernel<double, false, 4, 8, 16, 8, true>, span_kernel<double, false, 4, 8, 16, 8, false>);
    }
  }
  return hipGetLastError();
}

}  // namespace ti
