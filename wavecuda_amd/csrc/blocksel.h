// blocksel.h -- exact median / MAD of one signal's detail coefficients by a
// single workgroup (the batched pipeline smooths one signal per workgroup).
//
// MSB-first radix selection over order-preserving integer keys with 11-bit
// digits and an LDS histogram, tracking the two middle ranks (count-1)/2
// and count/2 at once; median = 0.5 (a + b) and MAD = 1.4826 median|v - med|
// as in reference src/utils.cpp:166-203.
//
// The values live in global memory (the workgroup's scratch).  Each pass
// over them issues kSelUnroll independent loads per thread before using
// any, so a pass costs a few memory latencies rather than one per element.
// As soon as the histogram shows that the values still matching the
// selected prefixes fit in LDS (kSelCap keys), one more pass copies their
// keys there and the remaining digits are resolved in LDS -- or, when at
// most kSelDirect keys are left (the usual case: a middle rank's bucket
// holds a few dozen values after one or two digits), every candidate's rank
// within its bucket is counted directly, one pass and one barrier instead
// of a radix digit's five barriers for each remaining digit.
//
// Two shortcuts, both exact: the deviations |v - med|, whose keys crowd a few
// exponents, are first counted into equal-width bins over [0, bound], the
// bound following from the extreme first digits the values have; and long
// inputs are read once per median, see block_median_sampled.
#pragma once

#include <type_traits>

#include "wh_common.h"

namespace wh {

constexpr int kSelBits = 11;
constexpr int kSelBins = 1 << kSelBits;
constexpr int kSelCap = 2048;   // keys kept in LDS
constexpr int kSelUnroll = 8;   // loads in flight per thread and pass
constexpr int kSelDirect = 256; // candidates ranked by direct counting

__device__ __forceinline__ double sel_val(uint64_t k, double*) {
  uint64_t u = (k >> 63) ? (k & 0x7fffffffffffffffull) : ~k;
  return __longlong_as_double(int64_t(u));
}
__device__ __forceinline__ double sel_val(uint64_t k, float*) {
  uint32_t kk = uint32_t(k);
  uint32_t u = (kk >> 31) ? (kk & 0x7fffffffu) : ~kk;
  return double(__uint_as_float(u));
}

// first radix digit of a value's key
template <typename T>
__device__ __forceinline__ unsigned sel_digit0(T v) {
  return unsigned(sel_key(v) >> (sizeof(T) * 8 - kSelBits));
}

// bin of a value y >= 0 among kSelBins equal-width bins over [0, hi] (scale =
// kSelBins / hi); monotone non-decreasing in y's key, clamped to the last bin,
// which also takes NaN: keys rank positive NaN above every number
__device__ __forceinline__ int sel_bin(double y, double scale) {
  const double u = y * scale;
  return u < double(kSelBins - 1) ? int(u) : kSelBins - 1;
}

// smallest and largest digit with a non-zero count in h[0..kSelBins), by
// all NT threads (the same in every thread; -1 and kSelBins when empty).
// wk: 8 (NT / 64) bytes of LDS scratch.
template <int NT>
__device__ __forceinline__ void sel_digit_range(const unsigned* h, int* wk, int* dmin, int* dmax) {
  constexpr int per = kSelBins / NT;
  constexpr int kWaves = NT / 64;
  int lo = kSelBins, hi = -1;
#pragma unroll
  for (int i = 0; i < per; ++i) {
    const int d = int(threadIdx.x) * per + i;
    if (h[d]) {
      lo = min(lo, d);
      hi = max(hi, d);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    lo = min(lo, __shfl_xor(lo, o, 64));
    hi = max(hi, __shfl_xor(hi, o, 64));
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    wk[wave] = lo;
    wk[kWaves + wave] = hi;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    lo = min(lo, wk[w]);
    hi = max(hi, wk[kWaves + w]);
  }
  __syncthreads();  // wk is reused by the caller
  *dmin = lo;
  *dmax = hi;
}

// LDS layout of block_median: the candidate keys (8-byte aligned) first,
// then the two histograms, the scan array (the wave totals of the bucket
// scan) and the selection state (prefixes, ranks, counts, the copy
// counter, the values' first-digit range).
template <int NT>
constexpr size_t block_sel_lds() {
  return size_t(kSelCap) * 8 + size_t(2) * kSelBins * 4 + size_t(NT) * 4 + 128;
}
// where block_median leaves the smallest and largest first digit (2 ints)
template <int NT>
__device__ __forceinline__ int* sel_range_slot(unsigned char* ws) {
  return reinterpret_cast<int*>(ws + size_t(kSelCap) * 8 + size_t(2) * kSelBins * 4 +
                                size_t(NT) * 4 + 96);
}

// f(key) for every value v[e], e < count (|v - center| when deviation).
// Values aligned to 16 bytes are read 16 bytes at a time (two FP64 or four
// FP32 values per load); kSelUnroll loads in flight per thread either way.
template <typename T, int NT, typename F>
__device__ __forceinline__ void sel_for_each(const T* __restrict__ v, int64_t count,
                                             bool deviation, T c, F f) {
  constexpr int kW = 16 / int(sizeof(T));
  typedef T TW __attribute__((ext_vector_type(kW)));
  auto key_of = [&](T y) { return sel_key(deviation ? T(fabs(y - c)) : y); };
  if (reinterpret_cast<uintptr_t>(v) % sizeof(TW) == 0) {
    const TW* __restrict__ vw = reinterpret_cast<const TW*>(v);
    const int64_t nv = count / kW;
    for (int64_t b = threadIdx.x; b < nv; b += int64_t(NT) * kSelUnroll) {
      TW x[kSelUnroll];
#pragma unroll
      for (int u = 0; u < kSelUnroll; ++u) {
        const int64_t p = b + int64_t(u) * NT;
        x[u] = vw[p < nv ? p : b];
      }
#pragma unroll
      for (int u = 0; u < kSelUnroll; ++u) {
        const int64_t p = b + int64_t(u) * NT;
        if (p < nv) {
#pragma unroll
          for (int w = 0; w < kW; ++w) f(key_of(x[u][w]));
        }
      }
    }
    const int64_t tail = nv * kW;
    if (threadIdx.x < count - tail) f(key_of(v[tail + threadIdx.x]));
    return;
  }
  for (int64_t b = threadIdx.x; b < count; b += int64_t(NT) * kSelUnroll) {
    T x[kSelUnroll];
#pragma unroll
    for (int u = 0; u < kSelUnroll; ++u) {
      const int64_t e = b + int64_t(u) * NT;
      x[u] = (e < count) ? v[e] : T(0);
    }
#pragma unroll
    for (int u = 0; u < kSelUnroll; ++u) {
      const int64_t e = b + int64_t(u) * NT;
      if (e < count) f(key_of(x[u]));
    }
  }
}

// Median of v[e], e < count (|v - center| when deviation),
// computed by all NT threads of the workgroup; returns the same value in
// every thread.  ws: block_sel_lds<NT>() bytes of LDS.  bound > 0
// (deviations only): every finite value lies in [0, bound]; one pass then counts the values into
// kSelBins equal-width bins (what lies beyond in the last), and when the middle ranks' bins hold at most
// kSelDirect values they are copied to LDS and ranked directly (otherwise
// the radix digits start from the top).  Of values, the smallest and largest
// first digit any has are left at sel_range_slot(ws).  pre (or null): the
// values' first digits, already counted.
template <typename T, int NT>
__device__ __forceinline__ double block_median(const T* __restrict__ v, int64_t count,
                                               bool deviation, double center,
                                               unsigned char* ws, double bound,
                                               const unsigned* pre) {
  uint64_t* cand = reinterpret_cast<uint64_t*>(ws);                     // [kSelCap]
  unsigned* hist = reinterpret_cast<unsigned*>(cand + kSelCap);        // [2][kSelBins]
  unsigned* part = hist + 2 * kSelBins;                                 // [NT]
  uint64_t* st = reinterpret_cast<uint64_t*>(part + NT);  // prefix0, prefix1 (+2 spare)
  long long* ks = reinterpret_cast<long long*>(st + 4);   // k0, k1
  long long* cs = ks + 2;                                  // keys under the new prefixes
  int* ncand = reinterpret_cast<int*>(cs + 2);
  const int tid = threadIdx.x;
  const T c = T(center);
  if (tid == 0) {
    st[0] = st[1] = 0;
    ks[0] = (count - 1) / 2;
    ks[1] = count / 2;
    *ncand = 0;
  }
  constexpr int kbits = int(sizeof(T)) * 8;
  constexpr int per = kSelBins / NT;
  constexpr int kWaves = NT / 64;
  bool in_lds = false;
  int nc = 0;
  if (bound > 0.0) {
    // equal-width bins over [0, bound] (monotone in the value): the middle
    // ranks fall in bins b0 <= b1, with no value between them
    const double scale = double(kSelBins) / bound;
    for (int i = tid; i < kSelBins; i += NT) hist[i] = 0;
    __syncthreads();
    sel_for_each<T, NT>(v, count, deviation, c, [&](uint64_t k) {
      atomicAdd(&hist[sel_bin(sel_val(k, (T*)nullptr), scale)], 1u);
    });
    __syncthreads();
    uint64_t* wsum = reinterpret_cast<uint64_t*>(part);  // [kWaves]
    const long long k0 = ks[0], k1 = ks[1];
    uint64_t loc = 0;
#pragma unroll
    for (int i = 0; i < per; ++i) loc += hist[tid * per + i];
    uint64_t inc = loc;
    const int lane = tid & 63, wave = tid >> 6;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint64_t t = __shfl_up(inc, o, 64);
      if (lane >= o) inc += t;
    }
    if (lane == 63) wsum[wave] = inc;
    __syncthreads();
    uint64_t base = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w)
      if (w < wave) base += wsum[w];
    const long long before = (long long)(base + inc - loc);
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const long long k = r ? k1 : k0;
      if (before <= k && k < before + (long long)loc) {
        long long acc = before;
        for (int i = 0; i < per; ++i) {
          const unsigned cnt = hist[tid * per + i];
          if (acc + cnt > k) {
            st[2 + r] = uint64_t(tid * per + i);
            ks[r] = k - acc;
            cs[r] = cnt;
            break;
          }
          acc += cnt;
        }
      }
    }
    __syncthreads();
    const int b0 = int(st[2]), b1 = int(st[3]);
    const long long total = cs[0] + (b1 != b0 ? cs[1] : 0);
    if (total <= kSelDirect) {
      const long long r0 = ks[0], r1 = (b1 != b0 ? cs[0] : 0) + ks[1];
      sel_for_each<T, NT>(v, count, deviation, c, [&](uint64_t k) {
        const int q = sel_bin(sel_val(k, (T*)nullptr), scale);
        if (q >= b0 && q <= b1) cand[atomicAdd(ncand, 1)] = k;
      });
      __syncthreads();
      nc = *ncand;
      in_lds = true;
      // every candidate is ranked among all of them (prefix 0 of 0 bits)
      if (tid == 0) {
        ks[0] = r0;
        ks[1] = r1;
      }
    } else if (tid == 0) {  // bins too full: radix digits from the top
      ks[0] = (count - 1) / 2;
      ks[1] = count / 2;
    }
    __syncthreads();
  }
  for (int hi = kbits; hi > 0;) {
    if (in_lds && nc <= kSelDirect) {
      // rank of each candidate among the candidates of its bucket: the key
      // of rank k in bucket q is the x with lt <= k < lt + eq
      const uint64_t q0 = st[0], q1 = st[1];
      const long long k0 = ks[0], k1 = ks[1];
      __syncthreads();  // every thread has read st and ks before they change
      // counts of candidate x among the candidates j in [j0, j1)
      auto count = [&](uint64_t x, int j0, int j1, int* c) {
        c[0] = c[1] = c[2] = c[3] = 0;
        for (int j = j0; j < j1; ++j) {
          const uint64_t y = cand[j], ty = hi >= 64 ? 0 : y >> hi;
          if (ty == q0) {
            c[0] += (y < x);
            c[1] += (y == x);
          }
          if (ty == q1) {
            c[2] += (y < x);
            c[3] += (y == x);
          }
        }
      };
      auto decide = [&](uint64_t x, const int* c) {
        const uint64_t tx = hi >= 64 ? 0 : x >> hi;
        if (tx == q0 && c[0] <= k0 && k0 < c[0] + c[1]) st[0] = x;
        if (tx == q1 && c[2] <= k1 && k1 < c[2] + c[3]) st[1] = x;
      };
      if (2 * nc <= NT) {
        // two threads per candidate, each counting half of the others
        // (partial counts in the histograms' space, unused here)
        int* pc = reinterpret_cast<int*>(hist);  // [4][NT]
        const int half = tid / (NT / 2), i = tid % (NT / 2);
        const int jm = nc / 2;
        if (i < nc) {
          int c[4];
          count(cand[i], half ? jm : 0, half ? nc : jm, c);
#pragma unroll
          for (int q = 0; q < 4; ++q) pc[q * NT + tid] = c[q];
        }
        __syncthreads();
        if (tid < nc) {
          int c[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) c[q] = pc[q * NT + tid] + pc[q * NT + tid + NT / 2];
          decide(cand[tid], c);
        }
      } else {
        for (int i = tid; i < nc; i += NT) {
          int c[4];
          count(cand[i], 0, nc, c);
          decide(cand[i], c);
        }
      }
      __syncthreads();
      break;
    }
    const int lo = hi > kSelBits ? hi - kSelBits : 0;
    for (int i = tid; i < 2 * kSelBins; i += NT) hist[i] = 0;
    __syncthreads();
    const uint64_t p0 = st[0], p1 = st[1];
    const bool same = (p0 == p1);
    const uint64_t dmask = (uint64_t(1) << (hi - lo)) - 1;
    auto count_key = [&](uint64_t k) {
      const uint64_t top = (hi >= 64) ? 0 : (k >> hi);
      const unsigned d = unsigned((k >> lo) & dmask);
      if (top == p0) atomicAdd(&hist[d], 1u);
      if (!same && top == p1) atomicAdd(&hist[kSelBins + d], 1u);
    };
    if (in_lds) {
      for (int i = tid; i < nc; i += NT) count_key(cand[i]);
    } else if (pre && !deviation && hi == kbits) {
      for (int i = tid; i < kSelBins; i += NT) hist[i] = pre[i];
    } else {
      sel_for_each<T, NT>(v, count, deviation, c, count_key);
    }
    __syncthreads();
    // Both ranks' bucket counts packed in one word (rank 0 in the low 32
    // bits, rank 1 in the high; each is at most count < 2^32, so the low
    // half never carries), so one scan serves both: each thread sums its
    // `per` buckets, a wave scans by shuffles, then the wave totals.
    uint64_t* wsum = reinterpret_cast<uint64_t*>(part);  // [kWaves]
    const long long k0 = ks[0], k1 = ks[1];  // the finder below updates ks
    const unsigned* h0 = hist;
    const unsigned* h1 = same ? h0 : hist + kSelBins;
    uint64_t loc = 0;
#pragma unroll
    for (int i = 0; i < per; ++i)
      loc += uint64_t(h0[tid * per + i]) | (uint64_t(h1[tid * per + i]) << 32);
    uint64_t inc = loc;
    const int lane = tid & 63, wave = tid >> 6;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint64_t t = __shfl_up(inc, o, 64);
      if (lane >= o) inc += t;
    }
    if (lane == 63) wsum[wave] = inc;
    __syncthreads();
    uint64_t base = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w)
      if (w < wave) base += wsum[w];
    const uint64_t before = base + inc - loc;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const unsigned* hr = r ? h1 : h0;
      const long long k = r ? k1 : k0;
      const long long bef = (long long)(r ? (before >> 32) : (before & 0xffffffffull));
      const long long mine = (long long)(r ? (loc >> 32) : (loc & 0xffffffffull));
      if (bef <= k && k < bef + mine) {
        long long acc = bef;
        for (int i = 0; i < per; ++i) {
          const unsigned cnt = hr[tid * per + i];
          if (acc + cnt > k) {
            // the rank's prefix grows by this digit (every thread read the
            // old prefixes before counting)
            st[r] = ((r ? p1 : p0) << (hi - lo)) | uint64_t(tid * per + i);
            ks[r] = k - acc;
            cs[r] = cnt;
            break;
          }
          acc += cnt;
        }
      }
    }
    __syncthreads();
    // the first digit's counts cover every value: their extreme digits
    // bound the values (the copy area is free until a copy pass)
    if (!deviation && hi == kbits) {
      int dmin, dmax;
      sel_digit_range<NT>(h0, reinterpret_cast<int*>(cand), &dmin, &dmax);
      if (tid == 0) {
        int* slot = sel_range_slot<NT>(ws);
        slot[0] = dmin;
        slot[1] = dmax;
      }
    }
    hi = lo;
    if (!in_lds && hi > 0) {
      const uint64_t q0 = st[0], q1 = st[1];
      const long long total = cs[0] + (q0 != q1 ? cs[1] : 0);
      if (total <= kSelCap) {
        // one more pass keeps the keys under the selected prefixes in LDS
        sel_for_each<T, NT>(v, count, deviation, c, [&](uint64_t k) {
          const uint64_t top = k >> hi;
          if (top == q0 || top == q1) cand[atomicAdd(ncand, 1)] = k;
        });
        __syncthreads();
        nc = *ncand;
        in_lds = true;
      }
    }
  }
  const double a = sel_val(st[0], (T*)nullptr), b = sel_val(st[1], (T*)nullptr);
  __syncthreads();
  return 0.5 * (a + b);
}

// ------------------------------------------------- selection from a sample
// Long inputs are read once per median instead of twice (the persistent
// kernel of 8192 mixed signals in FP64 697 -> 493 us, with 48 KB of LDS
// instead of 64): a sample of
// kSelSample values gives a bracket around the middle ranks, one pass counts
// the values below it and keeps those inside (about a fifteenth) in LDS, and
// the ranks are resolved there.  Exact: the counts tell whether the middle
// ranks lie inside; if not, or if too many values do, block_median starts
// over from the whole input.
constexpr int kSelSample = 2048;   // values sampled, in runs of kSelRun
constexpr int kSelRun = 8;
constexpr int kSelMargin = 96;     // sample ranks on either side of the middle, at most
// values kept: a 512-thread workgroup has its CU's LDS alone, of the others
// three share it
__host__ __device__ constexpr int sel_gather(int NT, size_t esz) {
  return NT == 512 ? (esz == 8 ? 16384 : 12288) : 4608;
}
// below, the passes saved are shorter than the sample's
constexpr int64_t kSelSampledMin = 16384;
// The longest input sampled, sixteen values a kept one: beyond, the bracket that
// fits is narrower than 2.2 standard deviations of the sample's middle, the middle
// ranks fall outside it too often, and then the pass was for nothing.  Batches of
// MODWT signals, J = 4 (a D_1 as long as the signal), us, read in whole / sampled:
// 512 threads FP64 2^17 one signal 238 / 119, 256 signals 671 / 531; 2^18 431 / 196
// and 1384 / 1251; FP32 2^17 364 / 351 and beyond the line, 2^18, 722 / 789; 256
// threads FP64 2^17 784 / 891.
__host__ __device__ constexpr int64_t sel_sampled_max(int NT, size_t esz) {
  return 16 * sel_gather(NT, esz);
}

// Whether block_median_sampled takes `count` values: its loop asks lane 63 of a
// wave for the wave's place, so a wave takes part with all its lanes or none (64
// loads of 16 bytes).
__host__ __device__ constexpr bool sel_sampled_takes(int NT, int64_t count, size_t esz) {
  return count >= kSelSampledMin && count <= sel_sampled_max(NT, esz) &&
         count % int64_t(64 * (16 / esz)) == 0;
}
static_assert(sel_sampled_takes(256, 1 << 14, 8) && sel_sampled_takes(256, 1 << 14, 4) &&
                  sel_sampled_takes(256, (1 << 14) + 128, 8) &&
                  !sel_sampled_takes(256, (1 << 14) + 64, 8) &&
                  !sel_sampled_takes(256, (1 << 14) + 128, 4),
              "a wave of the sampled selection must be whole");

// keys as wide as the values
template <typename T>
using SelKey = std::conditional_t<sizeof(T) == 8, uint64_t, uint32_t>;

__host__ __device__ constexpr size_t sel_sampled_lds(int NT, size_t esz) {
  return size_t(sel_gather(NT, esz) + kSelDirect) * esz + size_t(kSelBins) * 4 + 16 * 8 + 256;
}

// Bins of the ranks r0 <= r1 in h[0..kSelBins): the bin, the count before it
// and its own, for each rank, in f[0..2], f[3..5].  Ends with a barrier.
template <int NT>
__device__ __forceinline__ void sel_find(const unsigned* h, int r0, int r1, int* wsum, int* f) {
  constexpr int per = kSelBins / NT, kWaves = NT / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int loc = 0;
#pragma unroll
  for (int i = 0; i < per; ++i) loc += int(h[tid * per + i]);
  int inc = loc;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int t = __shfl_up(inc, o, 64);
    if (lane >= o) inc += t;
  }
  if (lane == 63) wsum[wave] = inc;
  __syncthreads();
  int before = inc - loc;
#pragma unroll
  for (int w = 0; w < kWaves; ++w)
    if (w < wave) before += wsum[w];
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int k = r ? r1 : r0;
    if (before <= k && k < before + loc) {
      int acc = before;
      for (int i = 0; i < per; ++i) {
        const int c = int(h[tid * per + i]);
        if (acc + c > k) {
          f[3 * r] = tid * per + i;
          f[3 * r + 1] = acc;
          f[3 * r + 2] = c;
          break;
        }
        acc += c;
      }
    }
  }
  __syncthreads();
}

// The median of v[0..count) (of |v - center| when deviation) into *res, the
// same in every thread; false: not resolved.  ws: sel_sampled_lds bytes.
template <typename T, int NT>
__device__ __forceinline__ bool block_median_sampled(const T* __restrict__ v, int64_t count,
                                                     bool deviation, double center,
                                                     unsigned char* ws, double* res) {
  constexpr int kWaves = NT / 64, K = kSelSample / NT, kGather = sel_gather(NT, sizeof(T));
  constexpr int kRuns = kSelSample / kSelRun;
  using Key = SelKey<T>;
  Key* cand = reinterpret_cast<Key*>(ws);
  Key* top = cand + kGather;                                     // [kSelDirect]
  unsigned* hist = reinterpret_cast<unsigned*>(top + kSelDirect);   // [kSelBins]
  double* red = reinterpret_cast<double*>(hist + kSelBins);         // [2 kWaves]
  int* wsum = reinterpret_cast<int*>(red + 16);                     // [kWaves]
  int* f = wsum + 8;                                                // [6]
  int* ngat = f + 6;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const T c = T(center);
  double s[K], mn = 1.0e300, mx = -1.0e300;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int i = tid + k * NT;
    const int64_t run = int64_t(i / kSelRun) * count / kRuns;
    const int64_t p = (run & ~int64_t(kSelRun - 1)) + i % kSelRun;
    const T x = v[p];
    s[k] = double(deviation ? T(fabs(x - c)) : x);
    mn = fmin(mn, s[k]);
    mx = fmax(mx, s[k]);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    mn = fmin(mn, __shfl_xor(mn, o, 64));
    mx = fmax(mx, __shfl_xor(mx, o, 64));
  }
  if (lane == 0) {
    red[wave] = mn;
    red[kWaves + wave] = mx;
  }
  for (int i = tid; i < kSelBins; i += NT) hist[i] = 0;
  if (tid == 0) *ngat = 0;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    mn = fmin(mn, red[w]);
    mx = fmax(mx, red[kWaves + w]);
  }
  const double scale = double(kSelBins) / (mx - mn);
  if (!(mx > mn && mx - mn < 1.0e300 && scale < 1.0e300)) return false;  // (uniform)
#pragma unroll
  for (int k = 0; k < K; ++k) atomicAdd(&hist[sel_bin(s[k] - mn, scale)], 1u);
  __syncthreads();
  // ranks to either side: four standard deviations of independent samples, or
  // what leaves the kept values room
  const int fit = int(0.8 * double(kGather) / double(count) * double(kSelSample / 2));
  const int margin = fit < kSelMargin ? fit : kSelMargin;
  sel_find<NT>(hist, kSelSample / 2 - margin, kSelSample / 2 + margin, wsum, f);
  const int b0 = f[0], b1 = f[3], inside = f[4] + f[5] - f[1];
  if (double(inside) * double(count) > 0.9 * double(kSelSample) * double(kGather)) return false;
  const T lo = T(mn + double(b0) / scale), hi = T(mn + double(b1 + 1) / scale);
  const Key klo = Key(sel_key(lo)), khi = Key(sel_key(hi));
  for (int i = tid; i < kSelBins; i += NT) hist[i] = 0;

  // one pass: count below, keep inside
  constexpr int kW = 16 / int(sizeof(T)), kU = 16 / kW;
  typedef T TW __attribute__((ext_vector_type(kW)));
  const TW* __restrict__ vw = reinterpret_cast<const TW*>(v);
  const int nv = int(count / kW);  // whole waves: see sel_sampled_takes
  int below = 0;
  T bad = T(0);  // NaN and infinities: left to block_median
  for (int b = tid; b < nv; b += NT * kU) {
    TW x[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int p = b + u * NT;
      x[u] = vw[p < nv ? p : b];
    }
#pragma unroll
    for (int u = 0; u < kU; ++u)
#pragma unroll
      for (int w = 0; w < kW; ++w) bad = fma(x[u][w], T(0), bad);
    asm volatile("" : "+v"(bad));  // here, not beyond the loop
    unsigned in = 0;  // bit per value
#pragma unroll
    for (int u = 0; u < kU; ++u) {
#pragma unroll
      for (int w = 0; w < kW; ++w) {
        const T y = x[u][w];
        const Key k = Key(sel_key(deviation ? T(fabs(y - c)) : y));
        const bool have = b + u * NT < nv;
        below += have && k < klo;
        in |= unsigned(have && k >= klo && k <= khi) << (u * kW + w);
      }
    }
    const int mine = __popc(in);
    int inc = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(inc, o, 64);
      if (lane >= o) inc += t;
    }
    int base = 0;
    if (lane == 63) base = atomicAdd(ngat, inc);
    int at = __shfl(base, 63, 64) + inc - mine;
#pragma unroll
    for (int u = 0; u < kU; ++u) {
#pragma unroll
      for (int w = 0; w < kW; ++w) {
        if (in >> (u * kW + w) & 1) {
          const T y = x[u][w];
          if (at < kGather) cand[at] = Key(sel_key(deviation ? T(fabs(y - c)) : y));
          ++at;
        }
      }
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) below += __shfl_xor(below, o, 64);
  if (lane == 0) wsum[wave] = below;
  if (__syncthreads_or(!(bad == T(0)))) return false;
  below = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) below += wsum[w];
  const int n = *ngat;
  const int r0 = int((count - 1) / 2) - below, r1 = int(count / 2) - below;
  const double width = double(hi) - double(lo), sc = double(kSelBins) / width;
  if (r0 < 0 || r1 >= n || n > kGather || !(width > 0.0 && sc < 1.0e300)) return false;
  __syncthreads();  // wsum and ngat have been read
  if (tid == 0) *ngat = 0;
  auto bin = [&](Key k) { return sel_bin(sel_val(k, (T*)nullptr) - double(lo), sc); };
  for (int i = tid; i < n; i += NT) atomicAdd(&hist[bin(cand[i])], 1u);
  __syncthreads();
  sel_find<NT>(hist, r0, r1, wsum, f);
  const int q0 = f[0], q1 = f[3], first = f[1], last = f[4] + f[5];
  if (last - first > kSelDirect) return false;
  for (int i = tid; i < n; i += NT) {
    const Key k = cand[i];
    const int q = bin(k);
    if (q >= q0 && q <= q1) top[atomicAdd(ngat, 1)] = k;
  }
  __syncthreads();
  const int m = last - first, k0 = r0 - first, k1 = r1 - first;
  for (int i = tid; i < m; i += NT) {
    const Key x = top[i];
    int lt = 0, eq = 0;
    for (int j = 0; j < m; ++j) {
      lt += top[j] < x;
      eq += top[j] == x;
    }
    if (lt <= k0 && k0 < lt + eq) red[0] = sel_val(x, (T*)nullptr);
    if (lt <= k1 && k1 < lt + eq) red[1] = sel_val(x, (T*)nullptr);
  }
  __syncthreads();
  *res = 0.5 * (red[0] + red[1]);
  __syncthreads();  // the workspace is free again
  return true;
}

// Short inputs stay in registers: equal-width bins between the extremes, the
// middle ranks' bins ranked directly, seven barriers a median.  Reading them
// once per digit cost 20 to 25 us of latency an item, which bounded batches of
// short signals.
constexpr int kSelSmallPer = 8;  // values a thread

// LDS: kSelDirect keys, the bins and what sel_find needs
__host__ __device__ constexpr size_t sel_small_lds(size_t esz) {
  return size_t(kSelDirect) * esz + size_t(kSelBins) * 4 + 16 * 8 + 256;
}

// 1.4826 median|v - median(v)| of count <= kSelSmallPer NT values into *res, the
// same in every thread; false: not resolved (NaN, infinities, a crowded bin)
template <typename T, int NT>
__device__ __forceinline__ bool block_mad_small(const T* __restrict__ v, int count,
                                                unsigned char* ws, double* res) {
  using Key = SelKey<T>;
  constexpr int kWaves = NT / 64, K = kSelSmallPer;
  Key* top = reinterpret_cast<Key*>(ws);                            // [kSelDirect]
  unsigned* hist = reinterpret_cast<unsigned*>(top + kSelDirect);   // [kSelBins]
  double* red = reinterpret_cast<double*>(hist + kSelBins);         // [2 kWaves]
  int* wsum = reinterpret_cast<int*>(red + 16);                     // [kWaves]
  int* f = wsum + 8;                                                // [6]
  int* ngat = f + 6;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  T x[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int e = tid + k * NT;
    x[k] = v[e < count ? e : count - 1];
  }
  double med = 0.0;
#pragma unroll 1
  for (int dev = 0; dev < 2; ++dev) {
    double mn = 1.0e300, mx = -1.0e300;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (dev) x[k] = T(fabs(x[k] - T(med)));
      mn = fmin(mn, double(x[k]));
      mx = x[k] == x[k] ? fmax(mx, double(x[k])) : double(INFINITY);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      mn = fmin(mn, __shfl_xor(mn, o, 64));
      mx = fmax(mx, __shfl_xor(mx, o, 64));
    }
    if (lane == 0) {
      red[wave] = mn;
      red[kWaves + wave] = mx;
    }
    for (int i = tid; i < kSelBins; i += NT) hist[i] = 0;
    if (tid == 0) *ngat = 0;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      mn = fmin(mn, red[w]);
      mx = fmax(mx, red[kWaves + w]);
    }
    if (!(mx < 1.0e300 && mn > -1.0e300)) return false;  // (uniform)
    const double width = mx - mn, scale = double(kSelBins) / width;
    if (width > 0.0 && !(scale < 1.0e300)) return false;
    if (width == 0.0) {
      med = mn;
      __syncthreads();  // red and hist are written again
      continue;
    }
#pragma unroll
    for (int k = 0; k < K; ++k)
      if (tid + k * NT < count) atomicAdd(&hist[sel_bin(double(x[k]) - mn, scale)], 1u);
    __syncthreads();
    const int r0 = (count - 1) / 2, r1 = count / 2;
    sel_find<NT>(hist, r0, r1, wsum, f);
    const int q0 = f[0], q1 = f[3], first = f[1], m = f[4] + f[5] - first;
    if (m > kSelDirect) return false;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (tid + k * NT < count) {
        const int q = sel_bin(double(x[k]) - mn, scale);
        if (q >= q0 && q <= q1) top[atomicAdd(ngat, 1)] = Key(sel_key(x[k]));
      }
    }
    __syncthreads();
    for (int i = tid; i < m; i += NT) {
      const Key y = top[i];
      int lt = 0, eq = 0;
      for (int j = 0; j < m; ++j) {
        lt += top[j] < y;
        eq += top[j] == y;
      }
      if (lt <= r0 - first && r0 - first < lt + eq) red[0] = sel_val(y, (T*)nullptr);
      if (lt <= r1 - first && r1 - first < lt + eq) red[1] = sel_val(y, (T*)nullptr);
    }
    __syncthreads();
    med = 0.5 * (red[0] + red[1]);
    __syncthreads();  // red, hist and top are written again
  }
  *res = 1.4826 * med;
  return true;
}

// 1.4826 median|v - median(v)|, v 16-byte aligned where it is long enough
// to be sampled.  The smallest and largest first digits present (from the
// median's own first digit) bound the values, so the deviations' median can
// start from equal-width bins.  pre: see block_median (beyond the sampled counts
// only, whose workspace may overlap it).
template <typename T, int NT>
__device__ __forceinline__ double block_mad(const T* __restrict__ v, int64_t count,
                                            unsigned char* ws, const unsigned* pre) {
  const bool sampled =
      sel_sampled_takes(NT, count, sizeof(T)) && reinterpret_cast<uintptr_t>(v) % 16 == 0;
  if (count <= kSelSmallPer * NT) {
    double mad;
    if (block_mad_small<T, NT>(v, int(count), ws, &mad)) return mad;
    __syncthreads();
  }
  double med[2] = {0.0, 0.0}, bound = 0.0;  // of the values, of the deviations
#pragma unroll 1
  for (int dev = 0; dev < 2; ++dev) {
    double m;
    if (!sampled || !block_median_sampled<T, NT>(v, count, dev, med[0], ws, &m)) {
      __syncthreads();
      m = block_median<T, NT>(v, count, dev, med[0], ws, bound, pre);
      const int* slot = sel_range_slot<NT>(ws);  // written before block_median's last barrier
      const int d0 = slot[0], d1 = slot[1];
      if (count > kSelDirect && d0 <= d1) {
        // every value lies in [vlo, vhi], the ends of those digits' key
        // ranges; |v - med| computed as the selection computes it (v - med
        // rounds monotonically in v) is then at most max(vhi - med, med - vlo).
        // An end that decodes to a NaN (infinities, NaN) is left out: what is
        // beyond the bound shares the last bin
        constexpr int sh = int(sizeof(T)) * 8 - kSelBits;
        const T vlo = T(sel_val(uint64_t(d0) << sh, (T*)nullptr));
        const T vhi = T(sel_val((uint64_t(d1) << sh) | ((uint64_t(1) << sh) - 1), (T*)nullptr));
        const T cm = T(m);
        const double b = double(fmax(vhi - cm, cm - vlo));
        if (b > 0.0 && b <= 1.0e300 && double(kSelBins) / b < 1.0e300) bound = b;
      }
      __syncthreads();
    }
    if (dev) med[1] = m;
    else med[0] = m;
  }
  return 1.4826 * med[1];
}

}  // namespace wh
