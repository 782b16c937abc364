// select.hip -- exact median and MAD (reference src/utils.cpp:166-203) of
// the values a SelSrc names, bit-exact: a median is an order statistic, and
// the final 0.5 (a + b) and 1.4826 m are the reference's operations.
//
// Both middle order statistics are found from a sorted sample.  Positions of
// equal strata (one hashed position each) give kSelSample keys; the sorted
// keys around the sample's middle are the edges of buckets: below, equal to
// edge 0, between edges 0 and 1, ... , above.  One pass counts every value
// into them (only the values near the middle need the search), and the
// buckets that hold the middle ranks follow from the counts: an equality
// bucket is the answer itself (heavily tied values are edges with near
// certainty), and an open bucket holds about count / kSelSample values
// whatever the distribution, since the edges are quantiles.  A second pass
// gathers those, and one workgroup ranks them.  The counts decide, not the
// sample: a rank outside the bracket (4.6 standard deviations of the
// sample's middle) or a bucket beyond the buffer is resolved by 11-bit
// digits over the values.  The deviations' sample is the same sample with
// the median taken off.
//
// What bounds it: launches and latency up to 2^20 values, then two reads of
// the values per median.  MAD of 2^18 FP64 details, kernel times: 56 us in
// seven launches (sample 8, counts 6, gather 5, ranking 12, and the last
// three again) against 87 in sixteen for selection digit by digit, whose
// first digit of an FP64 key is the sign and ten exponent bits, a handful of
// crowded buckets; 2.6 M values: 91 us against 149.  The sample is small
// because one workgroup sorts it (2048 keys took 20 us, 512 take 5 of the 8),
// and the counters have kReplicas copies on lines of their own because
// device-scope atomics on one line serialise at about 14 ns each (gather of
// 2.6 M values by 1024 workgroups: 20 us with one line, 11 with eight).  Up
// to kOneMax values one workgroup does all of it in one launch, the values
// held in registers.
#include <algorithm>

#include "wh_common.h"
#include "wh_internal.h"
#include "wh_stats.h"

namespace wh {

namespace {

constexpr int kNT = 256;    // threads of the passes over the values
constexpr int kNTB = 1024;  // threads of the one-workgroup steps
constexpr int kFly = 4;     // loads in flight per thread of the passes
constexpr int kHold = 8;    // values a thread of the one-workgroup kernel holds
constexpr int kOneMax = kHold * kNTB;
// a third pass beyond: where the open bucket is too full, and always (sel_refines)
constexpr int64_t kRefineMin = int64_t(1) << 23, kRefineAll = int64_t(1) << 24;
constexpr int kRefineFull = 1, kRefineAlways = 2;
constexpr int kBits = 11;
constexpr int kBins = 1 << kBits;
constexpr int kDirect = 256;  // keys ranked by counting
constexpr int kReplicas = kSelReplicas;
constexpr unsigned kRegion = kSelCandCap / kReplicas;  // of the candidate buffer
constexpr int kEdge0 = (kSelSample - kSelEdges) / 2;  // first edge in the sorted sample
using u64 = unsigned long long;

template <typename T>
__device__ __forceinline__ T value_from_key(uint64_t k);
template <>
__device__ __forceinline__ double value_from_key<double>(uint64_t k) {
  return __longlong_as_double(int64_t((k >> 63) ? (k & 0x7fffffffffffffffull) : ~k));
}
template <>
__device__ __forceinline__ float value_from_key<float>(uint64_t k) {
  const uint32_t kk = uint32_t(k);
  return __uint_as_float((kk >> 31) ? (kk & 0x7fffffffu) : ~kk);
}

// Element e of the positions a pass walks (count of them, or n for mode 2,
// which filters by level); false when the position is not selected.
template <typename T, int MODE>
__device__ __forceinline__ bool sel_value(const SelSrc& s, int64_t e, T& v) {
  const T* __restrict__ b = static_cast<const T*>(s.base);
  if constexpr (MODE == 0) {
    v = b[s.off + e];
    return true;
  } else if constexpr (MODE == 1) {  // MODWT detail blocks: block e / n starts at 2 n blk + n
    v = b[e + s.n * ((e >> s.lgn) + 1)];
    return true;
  } else {  // DWT details of 0-based levels [lmin, lmax]
    v = b[e];
    if (e == 0) return false;
    const int l = __builtin_ctzll(uint64_t(e));
    return l < s.J && l >= s.lmin && l <= s.lmax;
  }
}

// selected value t of 0..count-1 (mode 2: level by level)
template <typename T>
__device__ __forceinline__ T sel_at(const SelSrc& s, int64_t t) {
  T v;
  if (s.mode == 2) {
    int l = s.lmin;
    while (l < s.lmax && t >= (s.n >> (l + 1))) {
      t -= s.n >> (l + 1);
      ++l;
    }
    return static_cast<const T*>(s.base)[(2 * t + 1) << l];
  }
  if (s.mode == 1) (void)sel_value<T, 1>(s, t, v);
  else (void)sel_value<T, 0>(s, t, v);
  return v;
}

// position of sample i of m: stratum i of m equal ones, a hashed place in it
__device__ __forceinline__ int64_t sample_pos(int i, int m, int64_t count) {
  const int lg = 31 - __clz(m);
  const int64_t lo = (int64_t(i) * count) >> lg, hi = (int64_t(i + 1) * count) >> lg;
  uint64_t h = uint64_t(i + 1) * 0x9e3779b97f4a7c15ull;
  h ^= h >> 29;
  h *= 0xbf58476d1ce4e5b9ull;
  return lo + int64_t(((h >> 32) * uint64_t(hi - lo)) >> 32);
}

// every selected value's key (of the value, or of its deviation from med)
// of positions first, first + stride, ...: kFly loads in flight
template <typename T, int MODE, typename F>
__device__ __forceinline__ void for_keys_of(const SelSrc& s, int64_t first, int64_t stride,
                                            int deviation, T med, F fn) {
  const int64_t E = MODE == 2 ? s.n : s.count;
  for (int64_t e0 = first; e0 < E; e0 += kFly * stride) {
    T v[kFly];
    bool ok[kFly];
#pragma unroll
    for (int u = 0; u < kFly; ++u) {
      const int64_t e = e0 + u * stride;
      ok[u] = sel_value<T, MODE>(s, e < E ? e : E - 1, v[u]) && e < E;
    }
#pragma unroll
    for (int u = 0; u < kFly; ++u)
      if (ok[u]) fn(sel_key(deviation ? T(fabs(v[u] - med)) : v[u]));
  }
}
template <typename T, typename F>
__device__ __forceinline__ void for_keys(const SelSrc& s, int64_t first, int64_t stride,
                                         int deviation, T med, F fn) {
  // the mode is the launch's: a loop for each keeps the loads of one together
  if (s.mode == 0) for_keys_of<T, 0>(s, first, stride, deviation, med, fn);
  else if (s.mode == 1) for_keys_of<T, 1>(s, first, stride, deviation, med, fn);
  else for_keys_of<T, 2>(s, first, stride, deviation, med, fn);
}

// bitonic sort of the sample s[0..kSelSample) in LDS (one key per thread
// of the first kSelSample): partners within a wave by shuffles, across waves
// through s
__device__ void sample_sort(uint64_t* s) {
  const int tid = threadIdx.x;
  const bool on = tid < kSelSample;
  __syncthreads();
  uint64_t v = on ? s[tid] : 0;
  for (int k = 2; k <= kSelSample; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      uint64_t p;
      if (j >= 64) {
        __syncthreads();
        if (on) s[tid] = v;
        __syncthreads();
        p = on ? s[tid ^ j] : 0;
      } else {
        p = __shfl_xor((u64)v, j, 64);
      }
      const bool small = ((tid & j) == 0) == ((tid & k) == 0);
      v = (small == (p < v)) ? p : v;
    }
  }
  __syncthreads();
  if (on) s[tid] = v;
  __syncthreads();
}

// s holds the sorted keys of the sample's values; left in s: the sorted keys
// of their deviations from med.  The deviations fall towards the median
// and rise after it, so each one's rank is its place on its own side plus a
// search of the other; where rounding to NaN breaks that order, sort.
template <typename T>
__device__ void sample_deviations(uint64_t* s, T med) {
  __shared__ uint64_t d[kSelSample];
  const int tid = threadIdx.x;
  const bool on = tid < kSelSample;
  const T v = on ? value_from_key<T>(s[tid]) : T(0);
  const uint64_t key = sel_key(T(fabs(v - med)));
  if (on) d[tid] = key;
  const int c = __syncthreads_count(on && v < med);
  if (on) {
    // of the other side, the keys below (left side: or equal)
    int lo = tid < c ? c : 0, hi = tid < c ? kSelSample : c;
    const int from = lo, own = tid < c ? c - 1 - tid : tid - c;
    int other;
    if (tid < c) {  // right side rises
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (d[mid] <= key) lo = mid + 1;
        else hi = mid;
      }
      other = lo - from;
    } else {  // left side falls
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (d[mid] < key) hi = mid;
        else lo = mid + 1;
      }
      other = c - lo;
    }
    s[own + other] = key;
  }
  __syncthreads();
  // every rank taken once and in order?
  const bool bad = on && (d[tid] != key || (tid > 0 && s[tid - 1] > s[tid]) ||
                          (tid < c ? (tid > 0 && d[tid - 1] < key)
                                   : (tid > c && d[tid - 1] > key)));
  if (__syncthreads_or(bad)) {
    if (on) s[tid] = key;
    sample_sort(s);
  }
}

// bucket of a key among the sorted edges: 2 i + 1 equal to edge i, 2 i between
// edges i - 1 and i
__device__ __forceinline__ int bucket_of(const uint64_t* edges, uint64_t key) {
  int lo = 0, len = kSelEdges;
  while (len > 0) {
    const int half = len >> 1;
    if (edges[lo + half] < key) {
      lo += half + 1;
      len -= half + 1;
    } else {
      len = half;
    }
  }
  return 2 * lo + ((lo < kSelEdges && edges[lo] == key) ? 1 : 0);
}

// inclusive scan over the workgroup's NT threads
template <int NT>
__device__ __forceinline__ u64 block_scan(u64 v, u64* wsum) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const u64 t = __shfl_up(v, o, 64);
    if (lane >= o) v += t;
  }
  __syncthreads();
  if (lane == 63) wsum[wave] = v;
  __syncthreads();
  u64 add = 0;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) add += (w < wave) ? wsum[w] : 0;
  return v + add;
}

// What is known of the two middle ranks: found (key), or rank k among the
// keys with key - base < width (unsigned), `inside` of them.  Two ranks not
// found share that range: an open bucket is followed by an equality bucket
// that holds at least its edge.
struct Pick {
  long long k[2];
  uint64_t key[2];
  int found[2];
  uint64_t base, width;
  u64 inside;
};

template <int NT, int REP, typename B>
__device__ void block_pick(const B* bins, const uint64_t* edges, int64_t count, Pick* p,
                           u64* wsum) {
  constexpr int nb = 2 * kSelEdges;  // the last bucket (above) is what the others leave
  constexpr int per = (nb + NT - 1) / NT;
  const int b0 = int(threadIdx.x) * per;
  u64 cnt[per], loc = 0;
#pragma unroll
  for (int i = 0; i < per; ++i) {
    cnt[i] = 0;
#pragma unroll
    for (int r = 0; r < REP; ++r) cnt[i] += b0 + i < nb ? u64(bins[r * kSelBuckets + b0 + i]) : 0;
    loc += cnt[i];
  }
  const u64 incl = block_scan<NT>(loc, wsum);
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const u64 K = u64(r == 0 ? (count - 1) / 2 : count / 2);
    u64 below = incl - loc, in = 0;
    int hit = -1;
    if (below <= K && K < incl) {
#pragma unroll
      for (int i = 0; i < per; ++i) {
        if (hit >= 0) continue;
        if (K < below + cnt[i]) {
          hit = b0 + i;
          in = cnt[i];
        } else {
          below += cnt[i];
        }
      }
    } else if (int(threadIdx.x) == NT - 1 && K >= incl) {
      hit = nb;
      below = incl;
    }
    if (hit < 0) continue;
    const int i = hit >> 1;
    p->found[r] = hit & 1;
    p->k[r] = (long long)(K - below);
    if (hit & 1) {
      p->key[r] = edges[i];
    } else {
      const uint64_t lo = hit == 0 ? ~0ull : edges[i - 1];  // exclusive; ~0: none
      const uint64_t hi = hit == nb ? 0ull : edges[i];      // exclusive; 0: none
      p->base = lo + 1;
      p->width = hi - lo - 1;
      // of the open bucket alone: the other rank may sit in an equality one
      p->inside = hit == nb ? u64(count) - below : in;
    }
  }
  __syncthreads();
}

__device__ __forceinline__ int width_bits(uint64_t width) {
  return width <= 1 ? 0 : 64 - __clzll(width - 1);
}

// p narrowed by the counts of the leading digit (kBins of them) of key -
// base, from the first digit that holds a rank to the last; true when that
// is one digit
template <int NT>
__device__ bool block_narrow(const u64* hist, Pick* p, u64* wsum) {
  constexpr int per = kBins / NT;
  const int bits = width_bits(p->width), sh = bits > kBits ? bits - kBits : 0;
  const long long kmin = p->found[0] ? p->k[1] : p->k[0], kmax = p->found[1] ? p->k[0] : p->k[1];
  __shared__ int dig[2];
  __shared__ u64 cut[2];  // keys below the first digit, keys up to the last
  u64 cnt[per], loc = 0;
#pragma unroll
  for (int i = 0; i < per; ++i) {
    cnt[i] = hist[threadIdx.x * per + i];
    loc += cnt[i];
  }
  const u64 incl = block_scan<NT>(loc, wsum);
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const u64 k = u64(r == 0 ? kmin : kmax);
    u64 below = incl - loc;
    if (below <= k && k < incl) {
      bool hit = false;
#pragma unroll
      for (int i = 0; i < per; ++i) {
        if (hit) continue;
        if (k < below + cnt[i]) {
          hit = true;
          dig[r] = int(threadIdx.x) * per + i;
          cut[r] = r == 0 ? below : below + cnt[i];
        } else {
          below += cnt[i];
        }
      }
    }
  }
  __syncthreads();
  const bool one = dig[0] == dig[1];
  if (threadIdx.x == 0) {
    const uint64_t off = uint64_t(dig[0]) << sh;
    const uint64_t end = uint64_t(dig[1] + 1) << sh;  // 0 when it wraps: the range's end
    p->width = ((end == 0 || end > p->width) ? p->width : end) - off;
    p->base += off;
    p->inside = cut[1] - cut[0];
    p->k[0] -= (long long)cut[0];
    p->k[1] -= (long long)cut[0];
  }
  __syncthreads();
  return one;
}

// The ranks of p not found yet -> p->key.  each(fn) calls fn with every key
// of a set that holds all keys of p's range; the threads share the calls.
// Leading digits narrow the range until a few keys are left, which are
// ranked by counting.
template <typename EACH>
__device__ void block_resolve(Pick* p, uint64_t* buf /* kDirect */, u64* hist /* kBins */,
                              u64* wsum, EACH each) {
  __shared__ unsigned n;
  __shared__ uint64_t ends[2];
  const int tid = threadIdx.x;
  while (!(p->found[0] && p->found[1])) {
    const uint64_t base = p->base, width = p->width;
    if (width == 1) {
      if (tid < 2 && !p->found[tid]) p->key[tid] = base;
      break;
    }
    if (p->inside <= u64(kDirect)) {
      if (tid == 0) n = 0;
      __syncthreads();
      each([&](uint64_t key) {
        if (key - base < width) buf[atomicAdd(&n, 1u)] = key;
      });
      __syncthreads();
      // four threads per key, each counting against a quarter of them
      const int i = tid >> 2, m = int(n);
      const uint64_t ki = i < m ? buf[i] : 0;
      int less = 0, upto = 0;
      if (i < m) {
        for (int j = tid & 3; j < m; j += 4) {
          const uint64_t kj = buf[j];
          less += kj < ki;
          upto += kj <= ki;
        }
      }
      less += __shfl_xor(less, 1, 64);
      upto += __shfl_xor(upto, 1, 64);
      less += __shfl_xor(less, 2, 64);
      upto += __shfl_xor(upto, 2, 64);
      if (i < m && (tid & 3) == 0) {
#pragma unroll
        for (int r = 0; r < 2; ++r)  // equal keys write the same value
          if (!p->found[r] && less <= p->k[r] && p->k[r] < upto) p->key[r] = ki;
      }
      break;
    }
    const int bits = width_bits(width), sh = bits > kBits ? bits - kBits : 0;
    for (int i = tid; i < kBins; i += kNTB) hist[i] = 0;
    __syncthreads();
    each([&](uint64_t key) {
      if (key - base < width) atomicAdd(&hist[(key - base) >> sh], u64(1));
    });
    __syncthreads();
    const bool one = block_narrow<kNTB>(hist, p, wsum);
    if (one) continue;
    // the ranks follow one another across digits: the last key of the
    // first digit and the first key of the last
    if (tid == 0) {
      ends[0] = p->base;
      ends[1] = p->base + (p->width - 1);
    }
    __syncthreads();
    const uint64_t b2 = p->base, w2 = p->width;
    const uint64_t d0 = (b2 - base) >> sh;
    each([&](uint64_t key) {
      if (key - b2 >= w2) return;
      if (((key - base) >> sh) == d0) atomicMax((u64*)&ends[0], (u64)key);
      else atomicMin((u64*)&ends[1], (u64)key);
    });
    __syncthreads();
    if (tid < 2) p->key[tid] = ends[tid];
    break;
  }
  __syncthreads();
}

// 0.5 (a + b) of the two keys
template <typename T>
__device__ __forceinline__ double middle(const uint64_t* key) {
  return 0.5 * (double(value_from_key<T>(key[0])) + double(value_from_key<T>(key[1])));
}

// the result to every place that wants it
__device__ void deliver(double m, const SelOut& o) {
  double v = m;
  if (o.mad) {
    v = 1.4826 * m;
    if (o.factor > 0.0) v = v * o.factor;
  }
  if (threadIdx.x == 0) {
    if (o.out) *o.out = v;
    if (o.cv) cv_start(o.cv, v, o.levels, o.J);
  }
  if (o.levels && !o.cv && int(threadIdx.x) < o.J) o.levels[threadIdx.x] = v;
}

// ------------------------------------------------------- one workgroup
// count <= kOneMax: sample, counts, gather and ranking in one launch
template <typename T>
__global__ __launch_bounds__(kNTB) void sel_one_k(SelSrc s, SelOut o) {
  __shared__ uint64_t smp[kSelSample];
  __shared__ uint64_t buf[kDirect];
  __shared__ u64 hist[kBins];
  __shared__ unsigned bins[kSelBuckets];
  __shared__ u64 wsum[kNTB / 64];
  __shared__ Pick p;
  const int tid = threadIdx.x;
  const int count = int(s.count);
  const bool whole = count <= kSelSample;  // the sample is every value
  T v[kHold];
  int held = 0;
#pragma unroll
  for (int u = 0; u < kHold; ++u) {
    const int t = tid + u * kNTB;
    v[u] = sel_at<T>(s, t < count ? t : count - 1);
    held += t < count;
  }
  if (tid < kSelSample)
    smp[tid] = (whole && tid >= count)
                   ? ~0ull
                   : sel_key(sel_at<T>(s, whole ? tid : sample_pos(tid, kSelSample, count)));
  sample_sort(smp);
  double m = 0.0;
  T med = T(0);
  for (int dev = 0; dev < (o.mad ? 2 : 1); ++dev) {
    if (dev) {
#pragma unroll
      for (int u = 0; u < kHold; ++u) v[u] = T(fabs(v[u] - med));
      if (whole) {  // the padding stays behind
        if (tid < kSelSample) smp[tid] = tid < count ? sel_key(v[0]) : ~0ull;
        sample_sort(smp);
      } else {
        sample_deviations<T>(smp, med);
      }
    }
    if (whole) {
      if (tid < 2) p.key[tid] = smp[tid == 0 ? (count - 1) / 2 : count / 2];
    } else {
      const uint64_t* edges = smp + kEdge0;
      for (int i = tid; i < kSelBuckets; i += kNTB) bins[i] = 0;
      __syncthreads();
      const uint64_t e0 = edges[0], e1 = edges[kSelEdges - 1];
      unsigned below = 0;
#pragma unroll
      for (int u = 0; u < kHold; ++u) {
        const uint64_t key = sel_key(v[u]);
        below += u < held && key < e0;
        if (u < held && key >= e0 && key <= e1)
          atomicAdd(&bins[bucket_of(edges, key)], 1u);
      }
#pragma unroll
      for (int q = 32; q > 0; q >>= 1) below += __shfl_xor(below, q, 64);
      if ((tid & 63) == 0) atomicAdd(&bins[0], below);
      __syncthreads();
      block_pick<kNTB, 1>(bins, edges, count, &p, wsum);
      block_resolve(&p, buf, hist, wsum, [&](auto fn) {
#pragma unroll
        for (int u = 0; u < kHold; ++u)
          if (u < held) fn(sel_key(v[u]));
      });
    }
    __syncthreads();
    m = middle<T>(p.key);
    med = T(m);
    __syncthreads();
  }
  deliver(m, o);
}

// ---------------------------------------------------------------- grid
// counters cleared, sample taken and sorted, first edges
template <typename T>
__global__ __launch_bounds__(kSelSample) void sel_sample_k(SelSrc s, SelState* st) {
  __shared__ uint64_t smp[kSelSample];
  const int tid = threadIdx.x;
  const T v = sel_at<T>(s, sample_pos(tid, kSelSample, s.count));
  for (int i = tid; i < 2 * kReplicas * kSelBuckets; i += kSelSample) (&st->bins[0][0])[i] = 0;
  for (int i = tid; i < 2 * kBins; i += kSelSample) (&st->hist[0][0])[i] = 0;
  if (tid < 2 * kReplicas) (&st->ncand[0][0])[tid * kSelPad] = 0;
  smp[tid] = sel_key(v);
  sample_sort(smp);
  st->sample[tid] = smp[tid];
  if (tid < kSelEdges) st->edges[0][tid] = smp[kEdge0 + tid];
}

// every value counted into the buckets of the round (0: values, 1: deviations)
template <typename T>
__global__ __launch_bounds__(kNT) void sel_count_k(SelSrc s, SelState* st, int round) {
  __shared__ uint64_t edges[kSelEdges];
  __shared__ unsigned bins[kSelBuckets];
  const int tid = threadIdx.x;
  for (int i = tid; i < kSelEdges; i += kNT) edges[i] = st->edges[round][i];
  for (int i = tid; i < kSelBuckets; i += kNT) bins[i] = 0;
  __syncthreads();
  const T med = round ? T(st->med) : T(0);
  const uint64_t e0 = edges[0], e1 = edges[kSelEdges - 1];
  unsigned below = 0;
  for_keys<T>(s, int64_t(blockIdx.x) * kNT + tid, int64_t(gridDim.x) * kNT, round, med,
              [&](uint64_t key) {
                below += key < e0;
                if (key >= e0 && key <= e1) atomicAdd(&bins[bucket_of(edges, key)], 1u);
              });
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) below += __shfl_xor(below, o, 64);
  if ((tid & 63) == 0 && below) atomicAdd(&bins[0], below);
  __syncthreads();
  for (int i = tid; i < kSelBuckets; i += kNT)
    if (bins[i])
      atomicAdd(&st->bins[round][(blockIdx.x % kReplicas) * kSelBuckets + i], u64(bins[i]));
}

// The open bucket that holds the middle ranks is 2 count / kSelSample values
// on average (a rank falls in a bucket in proportion to its size) and x times
// count / kSelSample or more with probability (1 + x) e^-x.  Up to kRefineMin values
// it outgrows half of the candidate buffer (x = 16) in two of a million calls, which
// is left to the last resort, a workgroup alone that reads every value; when the
// buffer held 2^17 keys that was the lot of one median in eleven at 2^24 values
// (cross-validated smoothing of 2^21 FP32 samples, eight levels of details: 7.0 ms
// instead of 1.0).  So beyond kRefineMin, where the bucket is that full, one more
// pass counts the leading 11 bits of its keys' offsets (half of the buffer, for the
// regions fill unevenly); beyond kRefineAll it always does, since ranking the
// bucket's 2^16 keys and more costs one workgroup longer (MAD of 3e7 sorted FP32
// values 240 us, 337 without).
__device__ __forceinline__ bool sel_refines(int refine, const Pick& p) {
  return refine == kRefineAlways || (refine == kRefineFull && p.inside > u64(kSelCandCap) / 2);
}

template <typename T>
__global__ __launch_bounds__(kNT) void sel_refine_k(SelSrc s, SelState* st, int round, int refine) {
  __shared__ unsigned hist[kBins];
  __shared__ u64 wsum[kNT / 64];
  __shared__ Pick p;
  const int tid = threadIdx.x;
  block_pick<kNT, kReplicas>(st->bins[round], st->edges[round], s.count, &p, wsum);
  if ((p.found[0] && p.found[1]) || !sel_refines(refine, p)) return;
  for (int i = tid; i < kBins; i += kNT) hist[i] = 0;
  __syncthreads();
  const T med = round ? T(st->med) : T(0);
  const uint64_t base = p.base, width = p.width;
  const int bits = width_bits(width), sh = bits > kBits ? bits - kBits : 0;
  for_keys<T>(s, int64_t(blockIdx.x) * kNT + tid, int64_t(gridDim.x) * kNT, round, med,
              [&](uint64_t key) {
                if (key - base < width) atomicAdd(&hist[(key - base) >> sh], 1u);
              });
  __syncthreads();
  for (int i = tid; i < kBins; i += kNT)
    if (hist[i]) atomicAdd(&st->hist[round][i], u64(hist[i]));
}

// the keys still in play appended to the candidate buffer, one region of it
// per replica, through a list of the workgroup's own: one atomic serves a
// workgroup
template <typename T>
__global__ __launch_bounds__(kNT) void sel_gather_k(SelSrc s, SelState* st, int round, int refine) {
  constexpr unsigned kList = 512;
  __shared__ uint64_t list[kList];
  __shared__ u64 wsum[kNT / 64];
  __shared__ Pick p;
  __shared__ unsigned nlist;
  __shared__ u64 at;
  const int tid = threadIdx.x;
  if (tid == 0) nlist = 0;
  block_pick<kNT, kReplicas>(st->bins[round], st->edges[round], s.count, &p, wsum);
  if (p.found[0] && p.found[1]) return;
  if (refine && sel_refines(refine, p)) (void)block_narrow<kNT>(st->hist[round], &p, wsum);
  if (p.inside > u64(kSelCandCap)) return;  // the last step reads the values
  const T med = round ? T(st->med) : T(0);
  const uint64_t base = p.base, width = p.width;
  const int rep = blockIdx.x % kReplicas;
  u64* count = &st->ncand[round][rep * kSelPad];
  uint64_t* region = st->cand[round] + rep * kRegion;
  for_keys<T>(s, int64_t(blockIdx.x) * kNT + tid, int64_t(gridDim.x) * kNT, round, med,
              [&](uint64_t key) {
                if (key - base >= width) return;
                const unsigned i = atomicAdd(&nlist, 1u);
                if (i < kList) {
                  list[i] = key;
                } else {
                  const u64 g = atomicAdd(count, u64(1));
                  if (g < kRegion) region[g] = key;
                }
              });
  __syncthreads();
  const unsigned n = min(nlist, kList);
  if (n == 0) return;
  if (tid == 0) at = atomicAdd(count, u64(n));
  __syncthreads();
  for (unsigned i = tid; i < n; i += kNT)
    if (at + i < kRegion) region[at + i] = list[i];
}

// ranks the gathered keys; a MAD's first round (next) leaves the median and
// the deviations' edges, the last one the result
template <typename T>
__global__ __launch_bounds__(kNTB) void sel_finish_k(SelSrc s, SelState* st, int round, int refine,
                                                     int next, SelOut o) {
  __shared__ uint64_t smp[kSelSample];
  __shared__ uint64_t buf[kDirect];
  __shared__ u64 hist[kBins];
  __shared__ u64 wsum[kNTB / 64];
  __shared__ Pick p;
  const int tid = threadIdx.x;
  if (next && tid < kSelSample) smp[tid] = st->sample[tid];
  block_pick<kNTB, kReplicas>(st->bins[round], st->edges[round], s.count, &p, wsum);
  if (refine && !(p.found[0] && p.found[1]) && sel_refines(refine, p))
    (void)block_narrow<kNTB>(st->hist[round], &p, wsum);
  const T med = round ? T(st->med) : T(0);
  // gathered unless there were too many in all, or for one region
  unsigned nc[kReplicas];
  bool kept = p.inside <= u64(kSelCandCap);
#pragma unroll
  for (int r = 0; r < kReplicas; ++r) {
    const u64 c = st->ncand[round][r * kSelPad];
    nc[r] = unsigned(c);
    kept = kept && c <= u64(kRegion);
  }
  __syncthreads();
  block_resolve(&p, buf, hist, wsum, [&](auto fn) {
    if (kept) {
      // an eighth of the workgroup per region
      constexpr int kPer = kNTB / kReplicas;
      const int r = tid / kPer;
      unsigned n = 0;
#pragma unroll
      for (int q = 0; q < kReplicas; ++q) n = q == r ? nc[q] : n;
      for (unsigned i = tid % kPer; i < n; i += kPer) fn(st->cand[round][r * kRegion + i]);
    } else {
      for_keys<T>(s, tid, kNTB, round, med, fn);
    }
  });
  const double m = middle<T>(p.key);
  if (!next) {
    deliver(m, o);
    return;
  }
  if (tid == 0) st->med = m;
  sample_deviations<T>(smp, T(m));
  if (tid < kSelEdges) st->edges[1][tid] = smp[kEdge0 + tid];
}

template <typename T>
int select_t(SelSrc s, SelState* st, const SelOut& o, hipStream_t stream) {
  if (s.count <= kOneMax) {
    hipLaunchKernelGGL(sel_one_k<T>, dim3(1), dim3(kNTB), 0, stream, s, o);
    WH_HIP_CHECK(hipGetLastError());
    return WH_OK;
  }
  const int64_t E = s.mode == 2 ? s.n : s.count;
  const unsigned blocks = unsigned(std::min<int64_t>((E + kFly * kNT - 1) / (kFly * kNT), 1024));
  const int refine = s.count > kRefineAll ? kRefineAlways : s.count > kRefineMin ? kRefineFull : 0;
  hipLaunchKernelGGL(sel_sample_k<T>, dim3(1), dim3(kSelSample), 0, stream, s, st);
  for (int round = 0; round < (o.mad ? 2 : 1); ++round) {
    hipLaunchKernelGGL(sel_count_k<T>, dim3(blocks), dim3(kNT), 0, stream, s, st, round);
    if (refine)
      hipLaunchKernelGGL(sel_refine_k<T>, dim3(blocks), dim3(kNT), 0, stream, s, st, round, refine);
    hipLaunchKernelGGL(sel_gather_k<T>, dim3(blocks), dim3(kNT), 0, stream, s, st, round, refine);
    hipLaunchKernelGGL(sel_finish_k<T>, dim3(1), dim3(kNTB), 0, stream, s, st, round, refine,
                       (o.mad && round == 0) ? 1 : 0, o);
  }
  WH_HIP_CHECK(hipGetLastError());
  return WH_OK;
}

}  // namespace

int select_median(const SelSrc& s0, int dtype, SelState* st, const SelOut& o, hipStream_t stream) {
  if (s0.count <= 0) return set_error(WH_ERR_ARG, "median of an empty selection");
  SelSrc s = s0;
  s.lgn = 0;
  while ((int64_t(1) << s.lgn) < s.n) ++s.lgn;
  return dtype == WH_F32 ? select_t<float>(s, st, o, stream) : select_t<double>(s, st, o, stream);
}

}  // namespace wh
