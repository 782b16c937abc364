// batch_kern.h -- device side of the batched smoothing pipeline.
//
// Thousands of independent signals of power-of-two lengths are smoothed
// (forward transform -> hard/soft universal threshold -> inverse) by a fixed
// sequence of launches, whatever their mix: the head tiles (batch_tile.h), the
// persistent kernel below, and the last passes' tiles.  The persistent
// workgroups take whole signals from a device work queue: an atomic counter
// over an item list sorted longest-first, so the large signals start first and
// the small ones fill the tail.
//
//   MODWT: the item is the exact MAD of D_1 (the reference's univ_thresh(w,
//   0, 0): src/thresh.cpp:170-201, src/rfunctions.cu:82-87), which the head
//   left in the workspace.
//   DWT: the same and the levels beyond the head's, or, of signals without
//   tiles, the whole smoothing.  Levels run on compact sequences, through the
//   workgroup's slice of scratch while they are longer than the LDS tile and
//   in LDS afterwards; the MAD is taken over the level-1 details (all of
//   x[1..n-1] when J = 1, as in the reference) and the inverse thresholds
//   the details as it reads them.
//
// Nothing of the pipeline returns to the host.
#pragma once

#include "batch_tile.h"
#include "blocksel.h"
#include "dwt_dev.h"

namespace wh {

// transform and filter of an item in one word
__host__ __device__ constexpr int batch_kind(int ttype, int filt) { return (ttype << 3) | filt; }
__host__ __device__ constexpr int kind_ttype(int kind) { return kind >> 3; }
__host__ __device__ constexpr int kind_filter(int kind) { return kind & 7; }

// One signal of the batch.
struct BatchItem {
  int64_t off;    // first sample in the packed signal buffers
  int64_t scr;    // the tiles' workspace of the signal, or -1: no tiles
  double factor;  // sqrt(2 ln n) (sqrt(2 ln(n-1)) for a one-level DWT)
  int32_t n;      // length (power of two)
  int32_t J;      // levels
  int32_t kind;   // batch_kind(ttype, filter)
  int32_t sig;    // signal index (threshold output slot)
};

struct BatchArgs {
  const BatchItem* items;
  int count;
  int* counter;  // [0] work-queue head, [1] finished workgroups
  const void* x;
  void* y;
  double* thresh_out;  // optional, one per signal
  double* thresh;      // one per signal, for the shrink passes
  void* tiles;         // the tiles' workspace
  void* scratch;
  int64_t scratch_stride;  // elements per workgroup
  int hardness;
};

__device__ __forceinline__ int batch_next(int* counter, int* sh) {
  __syncthreads();
  if (threadIdx.x == 0) *sh = atomicAdd(counter, 1);
  __syncthreads();
  return *sh;
}

// phase boundary inside a workgroup when the phases exchange data through
// global memory (the workgroup's own scratch slice).  Only this
// workgroup's waves, all on one CU, read what they wrote, so the barrier's
// workgroup-scope release/acquire is enough; a device-scope fence would
// write back and invalidate the L2 of the workgroup's XCD at every item.
__device__ __forceinline__ void batch_phase() { __syncthreads(); }

// Longest sequence in LDS.  A level's outputs (forward) or inputs (inverse) are
// half of it, so the second buffer has half the size: 48 KB in FP64, three
// workgroups a CU.
template <typename T>
constexpr int batch_lds_elems() {
  return 4096;
}

// FP64 512-thread workgroups count the first radix digit of the level-1 details
// as the forward makes them, where there are more than the selection samples:
// kSelBins counts at this LDS offset, beyond the forward's levels and
// block_median's workspace.  It saves the median's first pass over them (a DWT of
// 2^20 samples, J = 3 LA8: 1990 -> 1826 us).
constexpr size_t kBatchPreOff = size_t(48) << 10;
__host__ __device__ constexpr size_t batch_pre_lds(int NT, size_t esz) {
  return esz == 8 && NT == 512 ? kBatchPreOff + size_t(kSelBins) * 4 : 0;
}
static_assert(batch_lds_elems<double>() * 8 * 3 / 2 <= int(kBatchPreOff) &&
                  block_sel_lds<512>() <= kBatchPreOff,
              "the first-digit counts lie beyond the forward's and the selection's LDS");

// DWT item coefficients in scratch C, level by level and each level
// contiguous: d_j at C[n - n/2^{j-1} ..) (n/2^j values), then s_J; for
// J = 1, s_1[0] goes last, so that C[0 .. n-1) holds d_1 and s_1[1..]: the
// values of the reference's interleaved layout at positions 1..n-1, which
// its one-level universal threshold reads (src/thresh.cpp:170-201).
__device__ __forceinline__ int64_t batch_dwt_doff(int64_t n, int j) { return n - (n >> (j - 1)); }
__device__ __forceinline__ int64_t batch_dwt_sidx(int64_t n, int J, int64_t m) {
  if (J == 1) return m == 0 ? n - 1 : n / 2 + m - 1;
  return n - (n >> J) + m;
}

// DWT item, forward: levels run on compact sequences, through scratch while
// longer than the LDS tile and in LDS afterwards; the coefficients end in
// scratch C as above (n values, gA/gB n/2 each behind it).
template <typename T, int FILT, int NT>
__device__ __forceinline__ void batch_dwt_fwd(const T* x, int64_t n, int J, T* C,
                                              unsigned char* smem, unsigned* pre) {
  constexpr int L = Filter<FILT>::L;
  constexpr int kBatchLds = batch_lds_elems<T>();
  constexpr int kUp = 2;  // global-level output pairs of pairs per thread in flight
  typedef T T2 __attribute__((ext_vector_type(2)));
  T* lA = reinterpret_cast<T*>(smem);
  T* lB = lA + kBatchLds;
  const int tid = threadIdx.x;
  {
    T* gA = C + n;          // n/2
    T* gB = gA + n / 2;     // n/2

    // ---- forward: global levels while the input is longer than the tile
    const T* src = x;
    int64_t N = n;
    int j = 1;
    bool toA = true;
    while (j <= J && N > kBatchLds) {
      T* dst = toA ? gA : gB;
      T* dj = C + batch_dwt_doff(n, j);
      // each thread takes outputs m = 2p and 2p + 1, whose taps 4p ..
      // 4p + L + 1 come as L / 2 + 1 aligned element pairs (N is a multiple
      // of 4, so no pair straddles the wrap), and stores them as 16-byte
      // pairs; kUp such pairs per thread in flight, clamped p for
      // unconditional loads
      const int64_t np = N / 4;
      for (int64_t p0 = tid; p0 < np; p0 += int64_t(NT) * kUp) {
        T v[kUp][L + 2];
#pragma unroll
        for (int u = 0; u < kUp; ++u) {
          const int64_t p = p0 + int64_t(u) * NT;
          const int64_t pc = (p < np) ? p : p0;
#pragma unroll
          for (int k = 0; k < L + 2; k += 2) {
            const T2 pr = *reinterpret_cast<const T2*>(src + ((4 * pc + k) & (N - 1)));
            v[u][k] = pr.x;
            v[u][k + 1] = pr.y;
          }
        }
#pragma unroll
        for (int u = 0; u < kUp; ++u) {
          const int64_t p = p0 + int64_t(u) * NT;
          if (p < np) {
            T s0, d0, s1, d1;
            fwd_pair<T, FILT>(v[u], s0, d0);
            fwd_pair<T, FILT>(v[u] + 2, s1, d1);
            *reinterpret_cast<T2*>(dst + 2 * p) = T2{s0, s1};
            *reinterpret_cast<T2*>(dj + 2 * p) = T2{d0, d1};
            if (pre && j == 1) {
              atomicAdd(&pre[sel_digit0(d0)], 1u);
              atomicAdd(&pre[sel_digit0(d1)], 1u);
            }
          }
        }
      }
      batch_phase();
      src = dst;
      toA = !toA;
      N >>= 1;
      ++j;
    }
    // remaining levels in LDS (or, when every level ran above, s_J itself)
    T* cur = lA;
    T* nxt = lB;
    const bool all_global = (j > J);
    if (all_global) {
      for (int64_t m = tid; m < N; m += NT) C[batch_dwt_sidx(n, J, m)] = src[m];
    } else {
      for (int64_t i = tid; i < N; i += NT) lA[i] = src[i];
    }
    __syncthreads();
    for (; j <= J; ++j) {
      const int P = int(N / 2);
      for (int m = tid; m < P; m += NT) {
        T v[L];
#pragma unroll
        for (int k = 0; k < L; k += 2) {
          const T2 pr = *reinterpret_cast<const T2*>(cur + ((2 * m + k) & (N - 1)));
          v[k] = pr.x;
          v[k + 1] = pr.y;
        }
        T s, d;
        fwd_pair<T, FILT>(v, s, d);
        nxt[m] = s;
        C[batch_dwt_doff(n, j) + m] = d;
      }
      __syncthreads();
      T* t = cur;
      cur = nxt;
      nxt = t;
      N = P;
    }
    if (!all_global)
      for (int64_t m = tid; m < N; m += NT) C[batch_dwt_sidx(n, J, m)] = cur[m];
    batch_phase();
  }
}

// DWT item, inverse: from the interleaved coefficients in scratch C, the
// thresholding inverse into y (levels J.. in LDS while the output fits the
// tile, the long levels through gA/gB)
template <typename T, int FILT, int NT>
__device__ __forceinline__ void batch_dwt_inv(T* y, int64_t n, int J, T* C,
                                              unsigned char* smem, double t, int hardness) {
  constexpr int L = Filter<FILT>::L;
  constexpr int kBatchLds = batch_lds_elems<T>();
  constexpr int kUp = 2;  // global-level output pairs of pairs per thread in flight
  typedef T T2 __attribute__((ext_vector_type(2)));
  T* lA = reinterpret_cast<T*>(smem);
  T* lB = lA + kBatchLds;
  const int tid = threadIdx.x;
  {
    T* gA = C + n;          // n/2
    T* gB = gA + n / 2;     // n/2
    const T tt = t >= 0.0 ? T(t) : T(0);  // a NaN is no threshold, as in dwt.hip
    int64_t N;
    T* cur;
    T* nxt;
    int j;

    // ---- inverse: levels J.. in LDS while the output fits the tile
    N = n >> J;  // length of s_J
    const bool lds_tail = (2 * N <= kBatchLds);
    // levels that run in LDS: the last one's outputs need the whole buffer lA
    int steps = 0;
    while (steps < J && (N << steps) * 2 <= kBatchLds) ++steps;
    cur = (steps & 1) ? lB : lA;
    nxt = (steps & 1) ? lA : lB;
    if (lds_tail) {
      for (int64_t m = tid; m < N; m += NT) cur[m] = C[batch_dwt_sidx(n, J, m)];
    } else {
      for (int64_t m = tid; m < N; m += NT) gA[m] = C[batch_dwt_sidx(n, J, m)];
    }
    batch_phase();
    j = J;
    while (j >= 1 && 2 * N <= kBatchLds) {
      for (int m = tid; m < int(N); m += NT) {
        T sv[L / 2], dv[L / 2];
#pragma unroll
        for (int q = 0; q < L / 2; ++q) {
          const int mm = (m - q) & int(N - 1);
          sv[q] = cur[mm];
          dv[q] = thresh_coef(C[batch_dwt_doff(n, j) + mm], tt, hardness);
        }
        T e, o;
        inv_pair<T, FILT>(sv, dv, e, o);
        *reinterpret_cast<T2*>(nxt + 2 * m) = T2{e, o};
      }
      __syncthreads();
      T* tp = cur;
      cur = nxt;
      nxt = tp;
      N *= 2;
      --j;
    }
    if (j == 0) {
      for (int64_t i = tid; i < n; i += NT) y[i] = cur[i];
    } else {
      // hand s_j to global (already there when no level ran in LDS) and
      // finish the long levels there
      if (lds_tail) {
        for (int64_t i = tid; i < N; i += NT) gA[i] = cur[i];
        batch_phase();
      }
      const T* s = gA;
      bool inA = true;
      // each thread takes the outputs of m = 2p and 2p + 1: their taps
      // 2p - H + 1 .. 2p + 1 of s_j and d_j come as K aligned element pairs
      // (N is even here, so no pair straddles the wrap), and the four
      // outputs go out as two 16-byte pair stores
      constexpr int H = L / 2, K = (H + 2) / 2;
      for (; j >= 1; --j) {
        T* out = (j == 1) ? y : (inA ? gB : gA);
        const T* dj = C + batch_dwt_doff(n, j);
        const int64_t np = N / 2;
        for (int64_t p0 = tid; p0 < np; p0 += int64_t(NT) * kUp) {
          T ws[kUp][2 * K], wd[kUp][2 * K];
#pragma unroll
          for (int u = 0; u < kUp; ++u) {
            const int64_t p = p0 + int64_t(u) * NT;
            const int64_t pc = (p < np) ? p : p0;  // clamped: unconditional loads
#pragma unroll
            for (int k = 0; k < K; ++k) {
              const int64_t i = (2 * pc - 2 * K + 2 + 2 * k) & (N - 1);
              const T2 a = *reinterpret_cast<const T2*>(s + i);
              const T2 d = *reinterpret_cast<const T2*>(dj + i);
              ws[u][2 * k] = a.x;
              ws[u][2 * k + 1] = a.y;
              wd[u][2 * k] = d.x;
              wd[u][2 * k + 1] = d.y;
            }
          }
#pragma unroll
          for (int u = 0; u < kUp; ++u) {
            const int64_t p = p0 + int64_t(u) * NT;
            if (p < np) {
#pragma unroll
              for (int i = 0; i < 2 * K; ++i) wd[u][i] = thresh_coef(wd[u][i], tt, hardness);
              // output m = 2p + r reads s_j[m - q] = w[2K - 2 + r - q]
              T sv[H], dv[H], e0, o0, e1, o1;
#pragma unroll
              for (int q = 0; q < H; ++q) {
                sv[q] = ws[u][2 * K - 2 - q];
                dv[q] = wd[u][2 * K - 2 - q];
              }
              inv_pair<T, FILT>(sv, dv, e0, o0);
#pragma unroll
              for (int q = 0; q < H; ++q) {
                sv[q] = ws[u][2 * K - 1 - q];
                dv[q] = wd[u][2 * K - 1 - q];
              }
              inv_pair<T, FILT>(sv, dv, e1, o1);
              *reinterpret_cast<T2*>(out + 4 * p) = T2{e0, o0};
              *reinterpret_cast<T2*>(out + 4 * p + 2) = T2{e1, o1};
            }
          }
        }
        batch_phase();
        s = out;
        inA = !inA;
        N *= 2;
      }
    }
  }
  batch_phase();
}

// The persistent pipeline: every workgroup takes items until the queue is
// empty; the last workgroup to leave rewinds the queue, so the launch can be
// replayed (a captured graph) without a memset node.  Held to 168 registers, three
// waves a SIMD, although FP64 with 256 threads spills 14 of them (60 bytes a lane):
// with two waves and no spills 8192 mixed signals take 2208 us instead of 2120, FP32
// (no spills either way) 1405 instead of 1311.
template <typename T, int NT>
__global__ __launch_bounds__(NT, NT == 128 ? 2 : 3) void batch_smooth_k(BatchArgs b) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ int item_sh;
  T* scr = static_cast<T*>(b.scratch) + int64_t(blockIdx.x) * b.scratch_stride;
  for (;;) {
    const int it = batch_next(b.counter, &item_sh);
    if (it >= b.count) break;
    const BatchItem I = b.items[it];
    const bool dwt = kind_ttype(I.kind) == kDWT, tiled = I.scr >= 0;
    // a tiled signal's D_1 is in the tiles' workspace; the DWT's levels beyond
    // the head's run here, from s_4 to s'_4
    const int64_t n = dwt && tiled ? I.n >> kBatchHead : I.n;
    const int J = dwt && tiled ? I.J - kBatchHead : I.J;
    T* d1 = tiled ? static_cast<T*>(b.tiles) + I.scr : scr;
    T* s4 = d1 + batch_pad(I.n);
    const T* in = tiled ? s4 : static_cast<const T*>(b.x) + I.off;
    T* out = tiled ? s4 + batch_pad(n) : static_cast<T*>(b.y) + I.off;
    unsigned* pre = nullptr;
    if constexpr (batch_pre_lds(NT, sizeof(T)) > 0) {
      // (not of a one-level DWT, whose selection takes s_1[1..] too)
      if (dwt && !tiled && J > 1 && n / 2 > sel_sampled_max(NT, sizeof(T))) {
        pre = reinterpret_cast<unsigned*>(smem + kBatchPreOff);
        for (int i = threadIdx.x; i < kSelBins; i += NT) pre[i] = 0;
        __syncthreads();
      }
    }
    if (dwt) {
      switch (kind_filter(I.kind)) {
        case kHAAR: batch_dwt_fwd<T, kHAAR, NT>(in, n, J, scr, smem, pre); break;
        case kD4: batch_dwt_fwd<T, kD4, NT>(in, n, J, scr, smem, pre); break;
        case kC6: batch_dwt_fwd<T, kC6, NT>(in, n, J, scr, smem, pre); break;
        default: batch_dwt_fwd<T, kLA8, NT>(in, n, J, scr, smem, pre); break;
      }
      batch_phase();
    }
    // the universal threshold from the level-1 details: one call site for
    // every kind of item, so the selection is inlined once (a called
    // function would keep its saved registers in scratch memory)
    const int64_t mcount = !dwt ? n : tiled ? I.n / 2 : J == 1 ? n - 1 : n / 2;
    const double t = block_mad<T, NT>(d1, mcount, smem, pre) * I.factor;
    if (threadIdx.x == 0) {
      b.thresh[I.sig] = t;
      if (b.thresh_out) b.thresh_out[I.sig] = t;
    }
    if (!dwt) continue;
    switch (kind_filter(I.kind)) {
      case kHAAR: batch_dwt_inv<T, kHAAR, NT>(out, n, J, scr, smem, t, b.hardness); break;
      case kD4: batch_dwt_inv<T, kD4, NT>(out, n, J, scr, smem, t, b.hardness); break;
      case kC6: batch_dwt_inv<T, kC6, NT>(out, n, J, scr, smem, t, b.hardness); break;
      default: batch_dwt_inv<T, kLA8, NT>(out, n, J, scr, smem, t, b.hardness); break;
    }
    batch_phase();
  }
  if (threadIdx.x == 0) {
    __threadfence();
    if (atomicAdd(b.counter + 1, 1) == int(gridDim.x) - 1) {
      atomicExch(b.counter, 0);
      atomicExch(b.counter + 1, 0);
    }
  }
}

struct BatchLaunch {
  int NT;
  unsigned grid;
  size_t lds;
};
// launch of the batch kernel of element type T, and its resident
// workgroups per CU for NT threads and lds bytes of dynamic LDS; defined in
// batch_<type>.hip
template <typename T>
int batch_launch(const BatchLaunch& bl, const BatchArgs& a, hipStream_t st);
template <typename T>
int batch_occupancy(int NT, size_t lds, int* blocks);

}  // namespace wh
