// The calibration steps around an isotonic fit: equal keys pooled into one point before it, and
// after it the piecewise-linear interpolation of the fitted curve (xp, fp) at new points, constant
// beyond its ends (np.interp's semantics).
//
// Replaces the reference's interp (reference examples/ctr_calibration/calibrate.py:163-168),
// five tensor operations and their launches (searchsorted, four gathers, then the arithmetic),
// with one kernel: per point, a binary search over xp (the first knot at or above x, clamped to
// [1, m - 1]) and the same arithmetic in the same order, each operation rounded once
// (contraction off), so the result is the reference's bit for bit:
//
//   t = clamp((x - x0) / max(x1 - x0, 1e-300), 0, 1),   out = f0 + t * (f1 - f0).
//
// A NaN x gives NaN (the clamp keeps it); one knot gives fp[0] everywhere.
//
// A search over millions of knots is a chain of ~23 dependent reads a query, most of them
// misses. The knot index (interp_index) cuts it to about three: buckets of equal width over
// [xp[0], xp[m - 1]], about kKnotsPerBucket knots each,
//
//   bucket(v) = clamp(floor((v - xp[0]) * scale), 0, B - 1),   scale = B / (xp[m - 1] - xp[0]),
//   first[b]  = the first knot i with bucket(xp[i]) >= b        (first[B] = m).
//
// bucket() is monotone in v (a subtraction, a product with scale >= 0, a clamp and a floor, each
// rounding a monotone function), so xp[i] < v gives bucket(xp[i]) <= bucket(v) and xp[i] >= v
// gives bucket(xp[i]) >= bucket(v): the first knot at or above v lies in [first[b], first[b + 1]]
// for b = bucket(v), and only those knots are searched - the same index as the full search, so
// the output is ti_interp's bit for bit. Knot ranges that are not finite and positive (an
// infinite or NaN end, all knots equal) give scale 0, and every query then searches all knots.
#include <hip/hip_runtime.h>

#include <cmath>

#include "ti_kernels.h"

namespace ti {

namespace {

// The reference formula at the first knot i at or above v (m after the last), i clamped to
// [1, m - 1]; each operation rounded once.
template <typename T>
__device__ __forceinline__ T interp_at(const T* __restrict__ xp, const T* __restrict__ fp, int64_t i, int64_t m,
                                       T v) {
#pragma clang fp contract(off)
  i = i < 1 ? 1 : (i > m - 1 ? m - 1 : i);
  const T x0 = xp[i - 1], x1 = xp[i], f0 = fp[i - 1], f1 = fp[i];
  T dx = x1 - x0;
  dx = dx < T(1e-300) ? T(1e-300) : dx;
  T t = (v - x0) / dx;
  t = t < T(0) ? T(0) : (t > T(1) ? T(1) : t);
  return f0 + t * (f1 - f0);
}

// The first i in [lo, hi) with !(xp[i] < v) (hi if none), as searchsorted(side="left").
template <typename T>
__device__ __forceinline__ int64_t lower_bound(const T* __restrict__ xp, int64_t lo, int64_t hi, T v) {
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (xp[mid] < v) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

template <typename T>
__global__ __launch_bounds__(256) void interp_kernel(const T* __restrict__ x, const T* __restrict__ xp,
                                                     const T* __restrict__ fp, T* __restrict__ out,
                                                     int64_t n, int64_t m) {
#pragma clang fp contract(off)
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t e = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; e < n; e += stride) {
    const T v = x[e];
    if (m == 1) {
      out[e] = v == v ? fp[0] : v;
      continue;
    }
    out[e] = interp_at(xp, fp, lower_bound(xp, int64_t{0}, m, v), m, v);
  }
}

// The index's header, then first[0..B] (uint32). m and dtype name the knots it was built from:
// a search through an index of another knot count or dtype would narrow to the wrong buckets.
struct InterpIndex {
  double lo, scale;
  int64_t buckets, m, dtype;
};

template <typename T>
constexpr int64_t dtype_code() {
  return sizeof(T) == 4 ? TI_F32 : TI_F64;
}
constexpr size_t kIndexHead = 256;
constexpr int64_t kKnotsPerBucket = 4;
constexpr int kCountMax = 8;  // buckets of at most this many knots are counted, not searched

__device__ __forceinline__ int64_t bucket_of(double v, double lo, double scale, int64_t buckets) {
#pragma clang fp contract(off)
  double d = (v - lo) * scale;
  d = d >= 0.0 ? d : 0.0;  // NaN and below the first knot: bucket 0
  const double top = static_cast<double>(buckets - 1);
  d = d < top ? d : top;
  return static_cast<int64_t>(d);
}

// One thread a bucket b in [0, B]: first[b] by a search over the knots' buckets.
template <typename T>
__global__ __launch_bounds__(256) void interp_index_kernel(const T* __restrict__ xp, int64_t m, int64_t buckets,
                                                           InterpIndex* __restrict__ head,
                                                           uint32_t* __restrict__ first) {
  const double lo = static_cast<double>(xp[0]);
  const double range = static_cast<double>(xp[m - 1]) - lo;
  double scale = range > 0.0 && range < INFINITY ? static_cast<double>(buckets) / range : 0.0;
  scale = scale < INFINITY ? scale : 0.0;
  const int64_t b = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (b == 0) {
    head->lo = lo;
    head->scale = scale;
    head->buckets = buckets;
    head->m = m;
    head->dtype = dtype_code<T>();
  }
  if (b > buckets) return;
  int64_t l = 0, h = b == 0 ? 0 : m;
  while (l < h) {
    const int64_t mid = (l + h) >> 1;
    if (bucket_of(static_cast<double>(xp[mid]), lo, scale, buckets) < b) l = mid + 1;
    else h = mid;
  }
  first[b] = static_cast<uint32_t>(l);
}

// interp_kernel through the index: the bucket's knots [a, c) are counted (at most kCountMax) or
// searched. The header is read as stored, with the bucket count capped at what the buffer holds
// (cap) and the bounds clamped to [0, m], so every read stays in the buffers whatever they hold;
// an index built from another knot count or dtype is not used (every query searches all knots).
template <typename T>
__global__ __launch_bounds__(256) void interp_indexed_kernel(const T* __restrict__ x, const T* __restrict__ xp,
                                                             const T* __restrict__ fp,
                                                             const InterpIndex* __restrict__ head,
                                                             const uint32_t* __restrict__ first, int64_t cap,
                                                             T* __restrict__ out, int64_t n, int64_t m) {
  const double lo = head->lo, scale = head->scale;
  int64_t buckets = head->buckets;
  buckets = buckets < cap ? buckets : cap;
  const bool indexed = scale > 0.0 && buckets >= 1 && head->m == m && head->dtype == dtype_code<T>();
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t e = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; e < n; e += stride) {
    const T v = x[e];
    if (m == 1) {
      out[e] = v == v ? fp[0] : v;
      continue;
    }
    int64_t i;
    if (indexed) {
      const int64_t b = bucket_of(static_cast<double>(v), lo, scale, buckets);
      int64_t c = first[b + 1];
      c = c < m ? c : m;
      int64_t a = first[b];
      a = a < c ? a : c;
      if (c - a <= kCountMax) {
        int cnt = 0;
#pragma unroll
        for (int j = 0; j < kCountMax; ++j)
          if (j < c - a) cnt += xp[a + j] < v ? 1 : 0;
        i = a + cnt;
      } else {
        i = lower_bound(xp, a, c, v);
      }
    } else {
      i = lower_bound(xp, int64_t{0}, m, v);
    }
    out[e] = interp_at(xp, fp, i, m, v);
  }
}

// --- pooling equal keys -----------------------------------------------------------------------
//
// Sorted keys, each run of equal keys pooled into one point: its key, the (weighted) mean of its
// values and its total weight, in four launches over tiles of kPoolE * 64 elements, one wave each:
//
//   pool_heads_kernel   the runs that start in each tile, and whether all weights are positive;
//   pool_scan_kernel    (one workgroup) the runs before each tile, and their total;
//   pool_kernel         each run that starts and ends in one tile; of the others, each tile's part
//                       of the run it begins in the middle of (lead) and of its last run (tail);
//   pool_tail_kernel    (a wave a tile) each tile's last run: its tail and the leads that follow.
//
// A step of a wave is 64 elements: the runs' sums by a segmented scan over the lanes, as many
// doublings as the step's longest run needs, the sum of a run that began in an earlier step carried
// on. Sums are formed in a fixed order (no atomics), in float64, each from its own run's values
// only.
//
// What bounds it: the gather of the values in key order, a cache line an element. 6.5M keys, 6.0M
// distinct: a library's segmented reduction, which gives each run a workgroup of 256 threads, took
// 3739 us, and finding the runs, their lengths and their starts 200 us.
constexpr int kPoolThreads = 256;
constexpr int kPoolE = 16;
constexpr int kPoolTile = 64 * kPoolE;
constexpr int kPoolScan = 1024;
constexpr int64_t kBadWeight = int64_t{1} << 62;

// (the header: the runs' total, and whether a weight is not positive)
struct PoolHead {
  int64_t runs, bad;
};
struct PoolWork {
  PoolHead* head;
  int64_t* before;  // per tile: the runs it starts, then the runs before it
  int* runs;        // per tile: the runs it starts
  double *lead_s, *lead_w, *tail_s, *tail_w;
};

constexpr int64_t pool_tiles(int64_t n) { return (n + kPoolTile - 1) / kPoolTile; }

PoolWork pool_work(void* work, int64_t n) {
  const int64_t tiles = pool_tiles(n);
  PoolWork p;
  p.head = static_cast<PoolHead*>(work);
  p.before = reinterpret_cast<int64_t*>(p.head + 1);
  p.lead_s = reinterpret_cast<double*>(p.before + tiles);
  p.lead_w = p.lead_s + tiles;
  p.tail_s = p.lead_w + tiles;
  p.tail_w = p.tail_s + tiles;
  p.runs = reinterpret_cast<int*>(p.tail_w + tiles);
  return p;
}

// Whether element i of n begins a run (a NaN key equals none); false past the end.
template <typename K>
__device__ __forceinline__ bool run_head(const K* __restrict__ keys, int64_t i, int64_t n) {
  const int64_t j = i < n ? i : n - 1;
  const K k = keys[j], q = keys[j > 0 ? j - 1 : 0];
  return i < n && (i == 0 || k != q);
}

template <typename K, typename Y>
__global__ __launch_bounds__(kPoolThreads) void pool_heads_kernel(const K* __restrict__ keys,
                                                                  const Y* __restrict__ w, int64_t n,
                                                                  int64_t tiles, PoolWork p) {
  const int lane = threadIdx.x & 63;
  const int64_t t = (static_cast<int64_t>(blockIdx.x) * kPoolThreads + threadIdx.x) >> 6;
  if (t >= tiles) return;
  int runs = 0;
  bool bad = false;
#pragma unroll
  for (int u = 0; u < kPoolE; ++u) {
    const int64_t i = t * kPoolTile + u * 64 + lane;
    runs += __popcll(__ballot(run_head(keys, i, n)));
    if (w != nullptr && i < n) bad |= !(w[i] > Y(0));
  }
  const bool anybad = __any(bad);
  if (lane == 0) {
    p.before[t] = runs + (anybad ? kBadWeight : 0);
    p.runs[t] = runs;
  }
}

__global__ __launch_bounds__(kPoolScan) void pool_scan_kernel(int64_t tiles, PoolWork p) {
  __shared__ int64_t wsum[kPoolScan / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int64_t base = 0;
  bool bad = false;
  for (int64_t t0 = 0; t0 < tiles; t0 += kPoolScan) {
    const int64_t t = t0 + tid;
    int64_t v = t < tiles ? p.before[t] : 0;
    bad |= v >= kBadWeight;
    v &= kBadWeight - 1;
    int64_t incl = v;
    for (int d = 1; d < 64; d <<= 1) {
      const int64_t q = __shfl_up(incl, d);
      if (lane >= d) incl += q;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int64_t before = base;
    for (int q = 0; q < kPoolScan / 64; ++q) {
      before += q < wave ? wsum[q] : 0;
      base += wsum[q];
    }
    if (t < tiles) p.before[t] = before + incl - v;
    __syncthreads();
  }
  const bool anybad = __syncthreads_or(bad);
  if (tid == 0) {
    p.head->runs = base;
    p.head->bad = anybad ? 1 : 0;
  }
}

struct PoolOut {
  int64_t knots;
  double *xp, *mean, *weight;
  int64_t* inverse;  // per sorted element, its run (or null)
};

// (a run's sum starts from +0, as a sum over a list does)
__device__ __forceinline__ void put_run(const PoolOut& o, int64_t r, double s, double w) {
  if (r >= o.knots) return;
  o.mean[r] = (s + 0.0) / w;
  o.weight[r] = w;
}

template <typename K, typename Y, bool W>
__global__ __launch_bounds__(kPoolThreads) void pool_kernel(const K* __restrict__ keys,
                                                            const int64_t* __restrict__ order,
                                                            const Y* __restrict__ y, const Y* __restrict__ w,
                                                            int64_t n, int64_t tiles, PoolWork p, PoolOut o) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  const int64_t t = (static_cast<int64_t>(blockIdx.x) * kPoolThreads + threadIdx.x) >> 6;
  if (t >= tiles) return;
  const int64_t i0 = t * kPoolTile;
  uint64_t head[kPoolE];
  double s[kPoolE], wt[kPoolE];
#pragma unroll
  for (int u = 0; u < kPoolE; ++u) {
    const int64_t i = i0 + u * 64 + lane;
    const int64_t at = order[i < n ? i : n - 1];
    s[u] = static_cast<double>(y[at]);
    wt[u] = 1.0;
    if constexpr (W) wt[u] = static_cast<double>(w[at]);
    head[u] = __ballot(run_head(keys, i, n));
  }
  const int64_t before = p.before[t];
  const uint64_t upto = (uint64_t{2} << lane) - 1;
  double cs = 0.0, cw = 0.0;  // the run open at the step's start
  int seen = 0;               // the tile's runs begun before the step
#pragma unroll
  for (int u = 0; u < kPoolE; ++u) {
    const int64_t i = i0 + u * 64 + lane;
    const uint64_t m = head[u];
    double vs = i < n ? (W ? wt[u] * s[u] : s[u]) : 0.0;
    double vw = i < n ? wt[u] : 0.0;
    const uint64_t own = m & upto;
    const int off = lane - (own != 0 ? 63 - __builtin_clzll(own) : 0);
    uint64_t longer = ~m & ~uint64_t{1};  // the elements at offset d or more of their runs
    for (int d = 1; longer != 0; d <<= 1) {
      const double qs = __shfl_up(vs, d), qw = __shfl_up(vw, d);
      if (off >= d) {
        vs += qs;
        vw += qw;
      }
      longer &= longer << d;
    }
    if (own == 0) {
      vs += cs;
      vw += cw;
    }
    const int64_t r = before + seen + __popcll(own) - 1;
    if (i < n) {
      if ((m >> lane) & 1u) {
        if (r < o.knots) o.xp[r] = static_cast<double>(keys[i]);
      }
      if (o.inverse != nullptr) o.inverse[i] = r;
    }
    // the element ends its run where the next begins one (the tile's last run: pool_tail_kernel)
    const uint64_t next = (m >> 1) | (u + 1 < kPoolE ? head[u + 1 < kPoolE ? u + 1 : u] << 63 : 0);
    if ((next >> lane) & 1u) {
      if (seen + __popcll(own) > 0) {
        put_run(o, r, vs, vw);
      } else {
        p.lead_s[t] = vs;
        p.lead_w[t] = vw;
      }
    }
    cs = __shfl(vs, 63);
    cw = __shfl(vw, 63);
    seen += __popcll(m);
  }
  if (lane == 0) {
    p.tail_s[t] = cs;
    p.tail_w[t] = cw;
    if (seen == 0 || (head[0] & 1u)) {
      p.lead_s[t] = seen == 0 ? cs : 0.0;
      p.lead_w[t] = seen == 0 ? cw : 0.0;
    }
  }
}

__global__ __launch_bounds__(kPoolThreads) void pool_tail_kernel(int64_t tiles, PoolWork p, PoolOut o) {
  const int lane = threadIdx.x & 63;
  const int64_t t = (static_cast<int64_t>(blockIdx.x) * kPoolThreads + threadIdx.x) >> 6;
  if (t >= tiles) return;
  const int runs = p.runs[t];
  if (runs == 0) return;
  double s = p.tail_s[t], w = p.tail_w[t];
  for (int64_t t0 = t + 1; t0 < tiles; t0 += 64) {
    const int64_t q = t0 + lane;
    const bool in = q < tiles;
    const uint64_t starts = __ballot(in && p.runs[in ? q : t] != 0);
    const int last = starts != 0 ? __builtin_ctzll(starts) : 63;  // (its lead is the run's too)
    double vs = in && lane <= last ? p.lead_s[q] : 0.0;
    double vw = in && lane <= last ? p.lead_w[q] : 0.0;
    for (int d = 32; d > 0; d >>= 1) {
      vs += __shfl_xor(vs, d);
      vw += __shfl_xor(vw, d);
    }
    s += vs;
    w += vw;
    if (starts != 0) break;
  }
  if (lane == 0) put_run(o, p.before[t] + runs - 1, s, w);
}

unsigned pool_grid(int64_t tiles) {
  constexpr int waves = kPoolThreads / 64;
  return static_cast<unsigned>((tiles + waves - 1) / waves);
}

unsigned grid_for(int64_t n) {
  const int64_t blocks64 = (n + 255) / 256;
  return static_cast<unsigned>(blocks64 < 65536 ? blocks64 : 65536);
}

}  // namespace

int64_t interp_buckets(int64_t m) {
  const int64_t b = (m + kKnotsPerBucket - 1) / kKnotsPerBucket;
  return b < 1 ? 1 : b;
}

size_t interp_index_bytes(int64_t m) {
  return (kIndexHead + 4 * static_cast<size_t>(interp_buckets(m) + 1) + 255) & ~size_t{255};
}

hipError_t interp_index(const void* xp, int64_t m, int dtype, void* index, hipStream_t stream) {
  const int64_t buckets = interp_buckets(m);
  auto* head = static_cast<InterpIndex*>(index);
  auto* first = reinterpret_cast<uint32_t*>(static_cast<char*>(index) + kIndexHead);
  const unsigned blocks = static_cast<unsigned>((buckets + 1 + 255) / 256);
  if (dtype == TI_F32)
    interp_index_kernel<float><<<dim3(blocks), dim3(256), 0, stream>>>(static_cast<const float*>(xp), m, buckets,
                                                                        head, first);
  else
    interp_index_kernel<double><<<dim3(blocks), dim3(256), 0, stream>>>(static_cast<const double*>(xp), m, buckets,
                                                                         head, first);
  return hipGetLastError();
}

hipError_t interp_indexed(const void* x, const void* xp, const void* fp, const void* index, size_t index_bytes,
                          void* out, int64_t n, int64_t m, int dtype, hipStream_t stream) {
  const auto* head = static_cast<const InterpIndex*>(index);
  const auto* first = reinterpret_cast<const uint32_t*>(static_cast<const char*>(index) + kIndexHead);
  const int64_t cap = static_cast<int64_t>((index_bytes - kIndexHead) / 4) - 1;
  const unsigned blocks = grid_for(n);
  if (dtype == TI_F32)
    interp_indexed_kernel<float><<<dim3(blocks), dim3(256), 0, stream>>>(
        static_cast<const float*>(x), static_cast<const float*>(xp), static_cast<const float*>(fp), head, first, cap,
        static_cast<float*>(out), n, m);
  else
    interp_indexed_kernel<double><<<dim3(blocks), dim3(256), 0, stream>>>(
        static_cast<const double*>(x), static_cast<const double*>(xp), static_cast<const double*>(fp), head, first,
        cap, static_cast<double*>(out), n, m);
  return hipGetLastError();
}

hipError_t interp(const void* x, const void* xp, const void* fp, void* out, int64_t n, int64_t m, int dtype,
                  hipStream_t stream) {
  const unsigned blocks = grid_for(n);
  if (dtype == TI_F32)
    interp_kernel<float><<<dim3(blocks), dim3(256), 0, stream>>>(
        static_cast<const float*>(x), static_cast<const float*>(xp), static_cast<const float*>(fp),
        static_cast<float*>(out), n, m);
  else
    interp_kernel<double><<<dim3(blocks), dim3(256), 0, stream>>>(
        static_cast<const double*>(x), static_cast<const double*>(xp), static_cast<const double*>(fp),
        static_cast<double*>(out), n, m);
  return hipGetLastError();
}

size_t pool_bytes(int64_t n) {
  const size_t tiles = static_cast<size_t>(pool_tiles(n));
  return sizeof(PoolHead) + tiles * (sizeof(int64_t) + 4 * sizeof(double) + sizeof(int));
}

hipError_t pool_count(const void* keys, const void* w, int64_t n, int key_dtype, int dtype, void* work,
                      hipStream_t stream) {
  const int64_t tiles = pool_tiles(n);
  const PoolWork p = pool_work(work, n);
  auto go = [&](auto k, auto v) {
    using K = decltype(k);
    using Y = decltype(v);
    pool_heads_kernel<K, Y><<<dim3(pool_grid(tiles)), dim3(kPoolThreads), 0, stream>>>(
        static_cast<const K*>(keys), static_cast<const Y*>(w), n, tiles, p);
  };
  if (key_dtype == TI_F32) dtype == TI_F32 ? go(float{}, float{}) : go(float{}, double{});
  else dtype == TI_F32 ? go(double{}, float{}) : go(double{}, double{});
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  pool_scan_kernel<<<dim3(1), dim3(kPoolScan), 0, stream>>>(tiles, p);
  return hipGetLastError();
}

hipError_t pool(const void* keys, const int64_t* order, const void* y, const void* w, int64_t n, int key_dtype,
                int dtype, void* work, int64_t knots, double* xp, double* mean, double* weight, int64_t* inverse,
                hipStream_t stream) {
  const int64_t tiles = pool_tiles(n);
  const PoolWork p = pool_work(work, n);
  const PoolOut o{knots, xp, mean, weight, inverse};
  auto go = [&](auto k, auto v) {
    using K = decltype(k);
    using Y = decltype(v);
    auto kernel = w != nullptr ? pool_kernel<K, Y, true> : pool_kernel<K, Y, false>;
    kernel<<<dim3(pool_grid(tiles)), dim3(kPoolThreads), 0, stream>>>(
        static_cast<const K*>(keys), order, static_cast<const Y*>(y), static_cast<const Y*>(w), n, tiles, p, o);
  };
  if (key_dtype == TI_F32) dtype == TI_F32 ? go(float{}, float{}) : go(float{}, double{});
  else dtype == TI_F32 ? go(double{}, float{}) : go(double{}, double{});
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  pool_tail_kernel<<<dim3(pool_grid(tiles)), dim3(kPoolThreads), 0, stream>>>(tiles, p, o);
  return hipGetLastError();
}

}  // namespace ti
