// batch_tile.h -- tiles of the batched MODWT smoothing.
//
// A signal's universal threshold needs its level-1 details only, so a batch
// is smoothed in passes over tiles of all signals at once: the head writes
// D_1 and, for more than kBatchHead levels, S_4; the threshold follows from
// D_1 (batch_kern.h); then the levels beyond the fourth are computed,
// thresholded and inverted in one pass over S_4 (giving S'_4), and the first
// four in one pass over the signal and S'_4.  No detail level but the first
// is ever stored: recomputing four levels costs 40 LDS-fed FMA pairs per
// sample (LA8) where storing and reading their details costs 8 words, and
// the deeper levels are computed once, in the pass that thresholds them.
//
// Beyond the fourth level a tap's distance is a multiple of 16, so S_4 is
// kept residue by residue: 16 circular sequences of n / 16 contiguous values,
// on which levels 5..8 are levels 1..4.  Every pass is therefore the same
// tile: kBatchP consecutive values of a circular sequence, with the halo its
// levels need on both sides (W = (L-1)(2^G - 1): 105 for LA8 and 4 levels, 10
// % of a tile), or, where sequences are shorter than a tile, whole sequences
// without any.  All arithmetic is the single-signal path's, term by term.
#pragma once

#include "modwt_tile.h"

namespace wh {

constexpr int kBatchNT = 256;    // threads of a tile
constexpr int kBatchP = 2048;    // values of a tile
constexpr int kBatchHead = 4;    // levels of the head group
constexpr int kBatchMaxModwtJ = 2 * kBatchHead;  // deepest MODWT of a batch
constexpr int kBatchRes = 1 << kBatchHead;       // residues of S_4

// One tile of one signal.  The signal's workspace: D_1 (later S'_4), S_4 and
// a copy of the signal (batches smoothed in place), batch_pad(n) values each.
struct BatchTile {
  int64_t off;   // the signal's first sample
  int64_t scr;   // its workspace
  int32_t n;
  int32_t tile;  // values kBatchP tile .. of each sequence array
  int32_t kind;  // filter | J << 3
  int32_t sig;
};

__host__ __device__ constexpr int64_t batch_pad(int64_t n) { return (n + 63) / 64 * 64; }

struct BatchTileArgs {
  const BatchTile* tiles;
  const void* x;
  void* y;
  void* scratch;
  const double* thresh;  // one per signal
  int in_place;          // x and y overlap: read the copy
  int hardness;
};

// where slot e of a tile reads its tap at distance o: a fixed LDS offset with
// halos, around its own sequence without
template <bool CIRC>
__device__ __forceinline__ int batch_slot(int e, int o, int mask) {
  return CIRC ? ((e & ~mask) | ((e + o) & mask)) : e + o;
}

// Pins the computation of v here.  A slot's outputs are first used after the
// barrier, so the compiler would sink their FMAs there and keep the taps of
// all nine slots in registers instead (446 in FP64).
template <typename T>
__device__ __forceinline__ void batch_pin(T& v) {
  asm volatile("" : "+v"(v));
}

// ------------------------------------------------------------------- head
// G = 1: D_1.  G = kBatchHead: D_1 and S_G, one buffer for all levels (a
// level's outputs wait in registers until every tap has been read).
template <typename T, int FILT, int G, bool CIRC>
__device__ __forceinline__ void batch_head(const BatchTileArgs& a, const BatchTile& I, T* b) {
  constexpr int L = Filter<FILT>::L, NT = kBatchNT, W = tile_halo(L, G);
  constexpr int N0 = CIRC ? kBatchP : kBatchP + W, K = (N0 + NT - 1) / NT;
  constexpr int KO = kBatchP / NT;
  const int64_t n = I.n, m0 = int64_t(I.tile) * kBatchP;
  const int mask = int(n - 1), tid = threadIdx.x;
  const int cnt = CIRC ? int(n) : N0;  // a short signal is one tile
  const T* __restrict__ in = static_cast<const T*>(a.x) + I.off;
  T* d1 = static_cast<T*>(a.scratch) + I.scr;
  T* s4 = d1 + batch_pad(n);
  T* xc = a.in_place ? s4 + batch_pad(n) : nullptr;
  T v[K];
#pragma unroll
  for (int k = 0; k < K; ++k) v[k] = in[(m0 + tid + k * NT) & (n - 1)];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int e = tid + k * NT;
    if (e < cnt) {
      b[e] = v[k];
      if (xc && k < KO) xc[m0 + e] = v[k];
    }
  }
  __syncthreads();
  auto level = [&](auto lc) {
    constexpr int l = decltype(lc)::value, s = 1 << (l - 1);
    const int no = CIRC ? cnt : kBatchP + W - tile_halo(L, l);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int e = tid + k * NT;
      if (e < no) {
        T w[L], D;
#pragma unroll
        for (int j = 0; j < L; ++j) w[j] = b[batch_slot<CIRC>(e, j * s, mask)];
        analysis1<T, FILT>(w, v[k], D);
        if (l < G) batch_pin(v[k]);
        if (l == 1 && k < KO) d1[m0 + e] = D;
        if (l == kBatchHead && k < KO) {
          const int64_t i = m0 + e;
          s4[(i & (kBatchRes - 1)) * (n / kBatchRes) + i / kBatchRes] = v[k];
        }
      }
    }
    if constexpr (l < G) {
      __syncthreads();  // every tap of this level read before any is replaced
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int e = tid + k * NT;
        if (e < no) b[e] = v[k];
      }
      __syncthreads();
    }
  };
  level(std::integral_constant<int, 1>{});
  if constexpr (G > 1) {
    level(std::integral_constant<int, 2>{});
    level(std::integral_constant<int, 3>{});
    level(std::integral_constant<int, 4>{});
  }
}

// ------------------------------------------------------------------ shrink
// G levels of a sequence array: forward, threshold, inverse.  The smooth of
// the top level is the tile's own, or (COARSE) the already smoothed S'_4.
// A thread keeps the details of its slots in registers; slot e of every level
// is the value at m0 - W + e.
template <typename T, int FILT, int G, bool CIRC, bool COARSE>
__device__ __forceinline__ void batch_shrink(const T* __restrict__ in, T* __restrict__ out,
                                             const T* __restrict__ coarse, int64_t N,
                                             int64_t first, int cnt, T t, int hardness,
                                             unsigned char* smem) {
  using V = typename Vec2<T>::type;
  constexpr int L = Filter<FILT>::L, NT = kBatchNT, W = CIRC ? 0 : tile_halo(L, G);
  constexpr int N0 = kBatchP + 2 * W, K = (N0 + NT - 1) / NT;
  T* b = reinterpret_cast<T*>(smem);
  V* p = reinterpret_cast<V*>(smem);
  const int tid = threadIdx.x, mask = int(N - 1);
  // sequence and position of the tile (CIRC: whole sequences from `first`)
  const int64_t seq = CIRC ? first : first & ~(N - 1), m0 = CIRC ? 0 : first & (N - 1);
  auto pos = [&](int e) { return CIRC ? int64_t(e) : (m0 - W + e) & (N - 1); };
  T S[K], d[G][K], top[COARSE ? K : 1];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int e = tid + k * NT;
    const int ec = e < cnt ? e : cnt - 1;  // unconditional load, clamped
    S[k] = in[seq + pos(ec)];
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int e = tid + k * NT;
    if (e < cnt) b[e] = S[k];
  }
  __syncthreads();
  auto forward = [&](auto lc) {
    constexpr int l = decltype(lc)::value, s = 1 << (l - 1);
    if constexpr (l <= G) {
      const int no = CIRC ? cnt : N0 - tile_halo(L, l);
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int e = tid + k * NT;
        d[l - 1][k] = T(0);
        if (e < no) {
          T w[L];
#pragma unroll
          for (int j = 0; j < L; ++j) w[j] = b[batch_slot<CIRC>(e, j * s, mask)];
          T D;
          analysis1<T, FILT>(w, S[k], D);
          d[l - 1][k] = t >= T(0) ? thresh_coef(D, t, hardness) : D;
          batch_pin(d[l - 1][k]);
          if (l < G || !COARSE) batch_pin(S[k]);
        }
      }
      __syncthreads();  // every tap of this level read before any is replaced
      if constexpr (l < G) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
          const int e = tid + k * NT;
          if (e < no) b[e] = S[k];
        }
        __syncthreads();
      }
    }
  };
  forward(std::integral_constant<int, 1>{});
  forward(std::integral_constant<int, 2>{});
  forward(std::integral_constant<int, 3>{});
  forward(std::integral_constant<int, 4>{});
  if constexpr (COARSE) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int e = tid + k * NT;
      const int64_t i = pos(e < cnt ? e : cnt - 1);
      top[k] = coarse[(i & (kBatchRes - 1)) * (N / kBatchRes) + i / kBatchRes];
    }
  }
  const int hi = CIRC ? cnt : W + kBatchP;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int e = tid + k * NT;
    if (e < hi) p[e] = V{COARSE ? top[COARSE ? k : 0] : S[k], d[G - 1][k]};
  }
  __syncthreads();
  auto inverse = [&](auto lc) {
    constexpr int l = decltype(lc)::value, s = 1 << (l - 1);
    if constexpr (l <= G) {
      const int lo = CIRC ? 0 : W - tile_halo(L, l - 1);
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int e = tid + k * NT;
        if (e >= lo && e < hi) {
          T ws[L], wd[L];
#pragma unroll
          for (int j = 0; j < L; ++j) {
            const V v = p[batch_slot<CIRC>(e, (j - (L - 1)) * s, mask)];
            ws[j] = v.x;
            wd[j] = v.y;
          }
          S[k] = synthesis<T, FILT>(ws, wd, L - 1);
          batch_pin(S[k]);
          if constexpr (l == 1) out[seq + (CIRC ? e : m0 + e - W)] = S[k];
        }
      }
      if constexpr (l > 1) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < K; ++k) {
          const int e = tid + k * NT;
          if (e >= lo && e < hi) p[e] = V{S[k], d[l > 1 ? l - 2 : 0][k]};
        }
        __syncthreads();
      }
    }
  };
  inverse(std::integral_constant<int, 4>{});
  inverse(std::integral_constant<int, 3>{});
  inverse(std::integral_constant<int, 2>{});
  inverse(std::integral_constant<int, 1>{});
}

template <typename T, int FILT, int G, bool COARSE>
__device__ __forceinline__ void batch_shrink_len(const T* in, T* out, const T* coarse, int64_t N,
                                                 int64_t total, int64_t first, T t, int hardness,
                                                 unsigned char* smem) {
  constexpr int W = tile_halo(Filter<FILT>::L, G);
  if (N < kBatchP)
    batch_shrink<T, FILT, G, true, COARSE>(in, out, coarse, N, first,
                                           int(total < kBatchP ? total : kBatchP), t, hardness,
                                           smem);
  else
    batch_shrink<T, FILT, G, false, COARSE>(in, out, coarse, N, first, kBatchP + 2 * W, t,
                                            hardness, smem);
}

// SECOND: levels 5..J of S_4 into S'_4; else the first levels into y
template <typename T, int FILT, bool SECOND>
__device__ __forceinline__ void batch_shrink_f(const BatchTileArgs& a, const BatchTile& I,
                                               unsigned char* smem) {
  const int64_t n = I.n, first = int64_t(I.tile) * kBatchP;
  const int J = I.kind >> 3, h = a.hardness;
  T* scr = static_cast<T*>(a.scratch) + I.scr;
  const T* s4 = scr + batch_pad(n);
  const T t = T(a.thresh[I.sig]);
  if constexpr (SECOND) {
    const int64_t N = n / kBatchRes;
    switch (J - kBatchHead) {
      case 1: batch_shrink_len<T, FILT, 1, false>(s4, scr, nullptr, N, n, first, t, h, smem); break;
      case 2: batch_shrink_len<T, FILT, 2, false>(s4, scr, nullptr, N, n, first, t, h, smem); break;
      case 3: batch_shrink_len<T, FILT, 3, false>(s4, scr, nullptr, N, n, first, t, h, smem); break;
      default: batch_shrink_len<T, FILT, 4, false>(s4, scr, nullptr, N, n, first, t, h, smem);
    }
  } else {
    const T* x = a.in_place ? s4 + batch_pad(n) : static_cast<const T*>(a.x) + I.off;
    T* y = static_cast<T*>(a.y) + I.off;
    switch (J) {
      case 1: batch_shrink_len<T, FILT, 1, false>(x, y, nullptr, n, n, first, t, h, smem); break;
      case 2: batch_shrink_len<T, FILT, 2, false>(x, y, nullptr, n, n, first, t, h, smem); break;
      case 3: batch_shrink_len<T, FILT, 3, false>(x, y, nullptr, n, n, first, t, h, smem); break;
      case 4: batch_shrink_len<T, FILT, 4, false>(x, y, nullptr, n, n, first, t, h, smem); break;
      default: batch_shrink_len<T, FILT, 4, true>(x, y, scr, n, n, first, t, h, smem);
    }
  }
}

// LDS of a tile: (S, D) pairs of a tile and its left halo, or the head's and
// the forward's values with both halos
template <typename T>
constexpr int batch_tile_lds() {
  return (kBatchP + tile_halo(8, kBatchHead)) * 2 * int(sizeof(T));
}

template <typename T>
__global__ __launch_bounds__(kBatchNT) void batch_head_k(BatchTileArgs a) {
  __shared__ __align__(16) T b[kBatchP + tile_halo(8, kBatchHead)];
  const BatchTile I = a.tiles[blockIdx.x];
  const bool deep = (I.kind >> 3) > kBatchHead, circ = I.n < kBatchP;
#define WH_HEAD(F)                                              \
  if (deep) {                                                   \
    if (circ) batch_head<T, F, kBatchHead, true>(a, I, b);      \
    else batch_head<T, F, kBatchHead, false>(a, I, b);          \
  } else {                                                      \
    if (circ) batch_head<T, F, 1, true>(a, I, b);               \
    else batch_head<T, F, 1, false>(a, I, b);                   \
  }
  switch (I.kind & 7) {
    case kHAAR: WH_HEAD(kHAAR) break;
    case kD4: WH_HEAD(kD4) break;
    case kC6: WH_HEAD(kC6) break;
    default: WH_HEAD(kLA8) break;
  }
#undef WH_HEAD
}

template <typename T, bool SECOND>
__global__ __launch_bounds__(kBatchNT, 4) void batch_shrink_k(BatchTileArgs a) {
  __shared__ __align__(16) unsigned char smem[batch_tile_lds<T>()];
  const BatchTile I = a.tiles[blockIdx.x];
  switch (I.kind & 7) {
    case kHAAR: batch_shrink_f<T, kHAAR, SECOND>(a, I, smem); break;
    case kD4: batch_shrink_f<T, kD4, SECOND>(a, I, smem); break;
    case kC6: batch_shrink_f<T, kC6, SECOND>(a, I, smem); break;
    default: batch_shrink_f<T, kLA8, SECOND>(a, I, smem); break;
  }
}

// launches over tiles [0, count); defined in batch_tile_<type>.hip
enum class BatchPass { kHead, kSecond, kFirst };
template <typename T>
int batch_tile_launch(BatchPass pass, unsigned count, const BatchTileArgs& a, hipStream_t st);

template <typename T>
int batch_tile_launch_impl(BatchPass pass, unsigned count, const BatchTileArgs& a,
                           hipStream_t st) {
  if (!count) return WH_OK;
  const dim3 grid(count), nt(kBatchNT);
  switch (pass) {
    case BatchPass::kHead: hipLaunchKernelGGL((batch_head_k<T>), grid, nt, 0, st, a); break;
    case BatchPass::kSecond:
      hipLaunchKernelGGL((batch_shrink_k<T, true>), grid, nt, 0, st, a);
      break;
    case BatchPass::kFirst:
      hipLaunchKernelGGL((batch_shrink_k<T, false>), grid, nt, 0, st, a);
      break;
  }
  WH_HIP_CHECK(hipGetLastError());
  return WH_OK;
}

}  // namespace wh
