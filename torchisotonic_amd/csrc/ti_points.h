// Hulls of points in LDS by rounds that drop points all at once, shared by the group kernel (a
// group's candidates) and the merge kernel (the vertices of a parent's children).
//
// A chord between two points of a diagram never drops a vertex of its lower hull, whichever points
// they are. So coarse_rounds (a rough hull of at most 64 points, one a lane, as a bit mask) needs
// no exactness, and prune drops every point on or above the chord of its neighbours by the exact
// predicate, and clearly above longer chords, until a round drops none: five rounds or so on
// noise, trends and rising data alike.
#pragma once

#include "ti_common.h"
#include "ti_tile.h"

namespace ti {
namespace {

template <bool W, bool PR>
__device__ __forceinline__ void hdiff(const HPt& a, const HPt& b, double& dS, double& dW) {
  dS = b.s - a.s;
  if constexpr (PR) dS += b.sl - a.sl;
  if constexpr (W) {
    dW = b.w - a.w;
    if constexpr (PR) dW += b.wl - a.wl;
  } else {
    dW = static_cast<double>(b.i - a.i);
  }
}

// Points in LDS, structure of arrays: sums (PR: double-double) and the index (of type I).
template <bool W, bool PR, typename I>
struct Points {
  double *s, *sl, *w, *wl;
  I* i;
};

template <bool W, bool PR, typename I>
constexpr int point_bytes() {
  return static_cast<int>(sizeof(I)) + 8 * (W ? 2 : 1) * (PR ? 2 : 1);
}

// (cap a multiple of 4)
template <bool W, bool PR, typename I>
__device__ __forceinline__ Points<W, PR, I> points_carve(char* p, int cap) {
  Points<W, PR, I> v;
  v.s = reinterpret_cast<double*>(p);
  p += cap * 8;
  v.sl = v.w = v.wl = nullptr;
  if constexpr (PR) {
    v.sl = reinterpret_cast<double*>(p);
    p += cap * 8;
  }
  if constexpr (W) {
    v.w = reinterpret_cast<double*>(p);
    p += cap * 8;
  }
  if constexpr (W && PR) {
    v.wl = reinterpret_cast<double*>(p);
    p += cap * 8;
  }
  v.i = reinterpret_cast<I*>(p);
  return v;
}

template <bool W, bool PR, typename I>
__device__ __forceinline__ HPt pget(const Points<W, PR, I>& v, int k) {
  HPt p;
  p.i = v.i[k];
  p.s = v.s[k];
  p.sl = PR ? v.sl[k] : 0.0;
  p.w = W ? v.w[k] : 0.0;
  p.wl = (W && PR) ? v.wl[k] : 0.0;
  return p;
}

template <bool W, bool PR, typename I>
__device__ __forceinline__ void pput(const Points<W, PR, I>& v, int k, const HPt& p) {
  v.i[k] = static_cast<I>(p.i);
  v.s[k] = p.s;
  if constexpr (PR) v.sl[k] = p.sl;
  if constexpr (W) v.w[k] = p.w;
  if constexpr (W && PR) v.wl[k] = p.wl;
}

// The wave's index in its workgroup, known uniform.
__device__ __forceinline__ int wave_index() { return __builtin_amdgcn_readfirstlane(threadIdx.x / kWave); }

// LDS written by this wave is read by its other lanes next (one wave's LDS operations run in
// order: only the compiler must keep them so).
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <int NT>
__device__ __forceinline__ void group_sync() {
  if constexpr (NT == kWave) wave_fence();
  else __syncthreads();
}

// b lies above the chord a-c by more than rounding can move it.
template <bool W, bool PR>
__device__ __forceinline__ bool clearly_above(const HPt& a, const HPt& b, const HPt& c) {
  double dS1, dW1, dS2, dW2;
  hdiff<W, PR>(a, b, dS1, dW1);
  hdiff<W, PR>(b, c, dS2, dW2);
  const double q = dS2 * dW1;
  return __builtin_fma(dS1, dW2, -q) > 0x1p-48 * __builtin_fabs(q);
}

constexpr int kPrunePasses = 64;

// The lower hull of points [0, cnt), by nt threads (all of a workgroup, or its first wave): each
// pass drops every point on or above the chord of its neighbours, or clearly above the chord of
// its left neighbour and the point d to its right, or of the point d to its left and its right
// neighbour (d = 2, 4, 8, 16 in turn; from the ninth pass up to 2048, as a far low point would
// otherwise take its neighbours a few a pass), until a pass drops none. A point is tested against
// the array as it stands, where earlier blocks of the pass may have been compacted already: any
// points left and right of it give a valid chord. Stops early with at most `stop` points left
// (done false). wc: NT / 64 ints of LDS. Returns the count; all threads have passed a barrier.
template <int NT, bool W, bool PR, typename I>
__device__ int prune(const Points<W, PR, I>& v, int cnt, int stop, int* wc, bool& done, int nt = NT) {
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = wave_index();
  done = true;
  for (int pass = 0; pass < kPrunePasses; ++pass) {
    if (cnt <= 2) return cnt;
    if (cnt <= stop) {
      done = false;
      return cnt;
    }
    const int d = 2 << (pass < 8 ? pass & 3 : pass % 11);
    int out = 0;
    for (int b0 = 0; b0 < cnt; b0 += nt) {
      const int k = b0 + tid;
      const bool in = k < cnt;
      bool keep = in;
      HPt x = pget(v, in ? k : 0);
      if (in && k > 0 && k < cnt - 1) {
        const HPt l = pget(v, k - 1), r = pget(v, k + 1);
        const HPt L = pget(v, max(k - d, 0)), R = pget(v, min(k + d, cnt - 1));
        keep = !clearly_above<W, PR>(l, x, R) && !clearly_above<W, PR>(L, x, r) && !hpools<W, PR>(l, x, r);
      }
      const uint64_t m = __ballot(keep);
      int before = out, all = __popcll(m);
      if constexpr (NT > kWave) {
        if (lane == 0) wc[wave] = all;
        __syncthreads();
        all = 0;
        for (int q = 0; q < nt / kWave; ++q) {
          before += q < wave ? wc[q] : 0;
          all += wc[q];
        }
      } else {
        wave_fence();
      }
      const int at = before + __popcll(m & ((uint64_t{1} << lane) - 1));
      if (keep && at != k) pput(v, at, x);
      out += all;
      group_sync<NT>();
    }
    if (out == cnt) return cnt;
    cnt = out;
  }
  // (not convex after that many passes: one thread's monotone chain, in place. Sorted runs in
  // random order come here, one permutation in 15 at 2048 points, 934 of them left at most of the
  // 160 tried: the worst weighted row of 2048 took 169 us in all, where pairwise merges took 543)
  if (tid == 0) {
    int top = 0;
    for (int k = 0; k < cnt; ++k) {
      const HPt x = pget(v, k);
      while (top >= 2 && hpools<W, PR>(pget(v, top - 2), pget(v, top - 1), x)) --top;
      pput(v, top, x);
      ++top;
    }
    wc[0] = top;
  }
  group_sync<NT>();
  cnt = wc[0];
  group_sync<NT>();
  return cnt;
}

struct CPt {
  double s, w;
};

// q lies above the chord a-b (as rounded: a coarse point dropped or kept wrongly costs only
// candidates)
__device__ __forceinline__ bool coarse_above(CPt a, CPt q, CPt b) {
  return (q.s - a.s) * (b.w - q.w) > (b.s - q.s) * (q.w - a.w);
}

// The points 0 .. 63 of a wave (one a lane, those in `alive`; point 0 alive) and an end point 64:
// a few rounds of dropping, all at once, every point above the chord of its neighbours, of its
// left neighbour and the end, or of point 0 and its right neighbour. Returns the points left.
constexpr int kCoarseRounds = 3;
template <class G>
__device__ __forceinline__ uint64_t coarse_rounds(uint64_t alive, CPt me, G get) {
  const int lane = threadIdx.x & (kWave - 1);
  const CPt first = get(0), end = get(kWave);
  for (int it = 0; it < kCoarseRounds; ++it) {
    const bool act = lane > 0 && ((alive >> lane) & 1) != 0;
    const uint64_t below = alive & ((uint64_t{1} << lane) - 1);
    const uint64_t above = (alive >> lane) >> 1;
    const int prev = below ? 63 - __builtin_clzll(below) : 0;
    const int next = above ? lane + 1 + __builtin_ctzll(above) : kWave;
    const CPt a = get(prev), b = get(next);
    const bool dead = act && (coarse_above(a, me, b) || coarse_above(a, me, end) || coarse_above(first, me, b));
    const uint64_t kill = __ballot(dead);
    if (kill == 0) break;
    alive &= ~kill;
  }
  return alive;
}

// The last point of the mask at or below j; the first beyond j (the end point, 64, where none is).
__device__ __forceinline__ int at_or_below(uint64_t m, int j) {
  return 63 - __builtin_clzll(m & ((uint64_t{2} << j) - 1));
}
__device__ __forceinline__ int beyond(uint64_t m, int j) {
  const uint64_t h = (m >> j) >> 1;
  return h ? j + 1 + __builtin_ctzll(h) : kWave;
}

// The hull of points [0, cnt): its count, in every thread.
template <int NT, bool W, bool PR, typename I>
__device__ __forceinline__ int prune_all(const Points<W, PR, I>& pts, int cnt, int* wc, int* result, int nt = NT) {
  bool done = false;
  if constexpr (NT > kWave) cnt = prune<NT>(pts, cnt, 2 * kWave, wc, done, nt);
  if (done) return cnt;  // (the same in every thread)
  if (threadIdx.x < kWave) {
    const int c = prune<kWave>(pts, cnt, 0, wc, done);
    if (threadIdx.x == 0) *result = c;
  }
  __syncthreads();
  return *result;
}

}  // namespace
}  // namespace ti
