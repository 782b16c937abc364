// batch_tile.h -- tiles of the batched smoothing.
//
// A signal's universal threshold needs its level-1 details only, so a batch
// is smoothed in passes over tiles of all signals at once: the head writes
// D_1 and, for more than kBatchHead levels, S_4; the threshold follows from
// D_1 (batch_kern.h); then the MODWT's levels beyond the fourth are computed,
// thresholded and inverted in one pass over S_4 (giving S'_4), and the first
// four levels in one pass over the signal and S'_4.  No detail level but the
// first is ever stored: recomputing four levels costs 32 LDS-fed FMA pairs per
// sample (LA8) where storing and reading their details costs 8 words, and
// the deeper levels are computed once, in the pass that thresholds them.
//
// MODWT: beyond the fourth level a tap's distance is a multiple of 16, so S_4
// is kept residue by residue: 16 circular sequences of n / 16 contiguous
// values, on which levels 5..8 are levels 1..4.  Every pass is therefore the
// same tile: consecutive values of a circular sequence, with the halo its
// levels need (W = (L-1)(2^G - 1): 105 for LA8 and 4 levels), or, where
// sequences are shorter than a tile, whole sequences without any.
// DWT (signals longer than kBatchDwtWhole): s_4 is a sixteenth of the signal,
// and the levels beyond it run in the persistent kernel.
// All arithmetic is the single-signal path's, term by term.
#pragma once

#include "dwt_dev.h"
#include "modwt_tile.h"

namespace wh {

constexpr int kBatchNT = 256;    // threads of a tile
constexpr int kBatchP = 2048;    // values of a tile
constexpr int kBatchHead = 4;    // levels of the head group
constexpr int kBatchMaxModwtJ = 2 * kBatchHead;  // deepest MODWT of a batch
constexpr int kBatchRes = 1 << kBatchHead;       // residues of S_4

constexpr int kBatchDwtWhole = 4096;  // longest DWT signal that is no tiles

// One tile of one signal.  The signal's workspace: D_1 (later S'_4), S_4 (the
// DWT's s_4 and s'_4) and a copy of the signal (batches smoothed in place),
// batch_pad(n) values each.
struct BatchTile {
  int64_t off;   // the signal's first sample
  int64_t scr;   // its workspace
  int32_t n;
  int32_t m0;    // first value stored, of its sequence
  int32_t kind;  // filter | J << 3 | first sequence << 8 | DWT << 16
  int32_t sig;
};

__host__ __device__ constexpr int tile_levels(int kind) { return (kind >> 3) & 31; }
__host__ __device__ constexpr int tile_seq(int kind) { return (kind >> 8) & 255; }
constexpr int kTileDwt = 1 << 16;

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

// ------------------------------------------------------------------- head
// G = 1: D_1.  G = kBatchHead: D_1 and S_G, one buffer for all levels (a
// level's outputs wait in registers until every tap has been read).
template <typename T, int FILT, int G, bool CIRC>
__device__ __forceinline__ void batch_head(const BatchTileArgs& a, const BatchTile& I, T* b) {
  constexpr int L = Filter<FILT>::L, NT = kBatchNT, W = tile_halo(L, G);
  constexpr int N0 = CIRC ? kBatchP : kBatchP + W, K = (N0 + NT - 1) / NT;
  constexpr int KO = kBatchP / NT;
  const int64_t n = I.n, m0 = I.m0;
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
        if (l < G) tile_pin(v[k]);
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

// -------------------------------------------------------------------- DWT
// Tiles of kBatchP samples: level l owns kBatchP / 2^l values, computes R(l)
// more to the right for the level above it and, in the last pass, E(l) to
// the left, H(l) of which the inverse reads.  The head moves 1.6 words a
// sample, the last pass 2.1.  One buffer serves every level, a level's outputs
// waiting in registers until every tap has been read.
// Threads of the last pass: it is bound by its short levels' instructions, so
// fewer threads with more values each are faster (8192 mixed signals FP64:
// 1024 threads 720 us, 512 413, 256 308, 128 281, 64 461, whose registers
// leave one wave per SIMD).
constexpr int kDwtLastNT = 128;

template <typename T, int FILT, int NT>
struct DwtTile {
  typedef T T2 __attribute__((ext_vector_type(2)));
  static constexpr int L = Filter<FILT>::L, A = kBatchHead;
  static constexpr int R(int l) { return l == A ? 0 : 2 * R(l + 1) + L - 2; }
  static constexpr int H(int l) { return l == 0 ? 0 : (H(l - 1) + 1) / 2 + L / 2 - 1; }
  static constexpr int own(int l) { return kBatchP >> l; }
  // values computed of level l, `left` of level 0 to the left of the tile's
  static constexpr int cnt(int l, int left) { return own(l) + (left >> l) + R(l); }
  static constexpr int kLeft = H(A) << A;
  static constexpr int kElems = own(0) + kLeft + R(0);
  static constexpr int per(int n) { return (n + NT - 1) / NT; }

  // s_0 of the tile from x (and its copy to xc) into b
  template <int left>
  static __device__ __forceinline__ void load(const T* __restrict__ x, T* xc, int64_t n, int m0,
                                              T* b) {
    constexpr int np = cnt(0, left) / 2, K = per(np);
    T2 v[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int p = int(threadIdx.x) + k * NT;
      const int pc = p < np ? p : np - 1;  // unconditional load, clamped
      v[k] = *reinterpret_cast<const T2*>(x + ((m0 - left + 2 * pc) & (n - 1)));
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int p = int(threadIdx.x) + k * NT;
      if (p < np) *reinterpret_cast<T2*>(b + 2 * p) = v[k];
      if (xc && p < own(0) / 2) *reinterpret_cast<T2*>(xc + m0 + 2 * p) = v[k];
    }
    __syncthreads();
  }
  // level l of the buffer: f(slot, k, s, d); s_l replaces s_{l-1} unless l = A
  template <int l, int left, typename F>
  static __device__ __forceinline__ void level(T* b, F f) {
    constexpr int no = cnt(l, left), K = per(no);
    T s[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int m = int(threadIdx.x) + k * NT;
      if (m < no) {
        T v[L], d;
#pragma unroll
        for (int j = 0; j < L; j += 2) {
          const T2 pr = *reinterpret_cast<const T2*>(b + 2 * m + j);
          v[j] = pr.x;
          v[j + 1] = pr.y;
        }
        fwd_pair<T, FILT>(v, s[k], d);
        tile_pin(s[k]);
        f(m, k, s[k], d);
      }
    }
    __syncthreads();
    if constexpr (l < A) {
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int m = int(threadIdx.x) + k * NT;
        if (m < no) b[m] = s[k];
      }
      __syncthreads();
    }
  }

  static __device__ __forceinline__ void head(const BatchTileArgs& a, const BatchTile& I, T* b) {
    const int64_t n = I.n;
    T* d1 = static_cast<T*>(a.scratch) + I.scr + I.m0 / 2;
    T* s4 = static_cast<T*>(a.scratch) + I.scr + batch_pad(n) + (I.m0 >> A);
    T* xc = static_cast<T*>(a.scratch) + I.scr + 2 * batch_pad(n);
    load<0>(static_cast<const T*>(a.x) + I.off, a.in_place ? xc : nullptr, n, I.m0, b);
    level<1, 0>(b, [&](int m, int, T, T d) {
      if (m < own(1)) d1[m] = d;
    });
    level<2, 0>(b, [](int, int, T, T) {});
    level<3, 0>(b, [](int, int, T, T) {});
    level<A, 0>(b, [&](int m, int, T s, T) { s4[m] = s; });
  }

  // level l's (s', d) in S and D from slot of position own start - H(l) on:
  // l - 1's, whose details are d[]
  template <int l, int K>
  static __device__ __forceinline__ void up(T* S, T* D, const T (&d)[K], T* y) {
    constexpr int h = (H(l - 1) + 1) / 2, no = own(l) + h, KO = per(no), Q = L / 2;
    T e[KO], o[KO];
#pragma unroll
    for (int k = 0; k < KO; ++k) {
      const int m = int(threadIdx.x) + k * NT;
      if (m < no) {
        T sv[Q], dv[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          sv[q] = S[m + H(l) - h - q];
          dv[q] = D[m + H(l) - h - q];
        }
        inv_pair<T, FILT>(sv, dv, e[k], o[k]);
        tile_pin(e[k]);
        tile_pin(o[k]);
        if constexpr (l == 1) *reinterpret_cast<T2*>(y + 2 * m) = T2{e[k], o[k]};
      }
    }
    if constexpr (l > 1) {
      __syncthreads();
#pragma unroll
      for (int k = 0; k < KO; ++k) {
        const int m = int(threadIdx.x) + k * NT, j = 2 * (m - h) + H(l - 1);
        if (m < no) {
          if (j >= 0) S[j] = e[k];
          S[j + 1] = o[k];
        }
      }
      details<l - 1>(D, d);
      __syncthreads();
    }
  }
  template <int l, int K>
  static __device__ __forceinline__ void details(T* D, const T (&d)[K]) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int j = int(threadIdx.x) + k * NT - ((kLeft >> l) - H(l));
      if (j >= 0 && j < own(l) + H(l)) D[j] = d[k];
    }
  }

  static __device__ __forceinline__ void last(const BatchTileArgs& a, const BatchTile& I, T* b) {
    const int64_t n = I.n;
    const double t0 = a.thresh[I.sig];
    const T t = t0 >= 0.0 ? T(t0) : T(0);  // a NaN is no threshold, as in dwt.hip
    const T* s4 = static_cast<const T*>(a.scratch) + I.scr + batch_pad(n) + batch_pad(n >> A);
    const T* xc = static_cast<const T*>(a.scratch) + I.scr + 2 * batch_pad(n);
    T* y = static_cast<T*>(a.y) + I.off + I.m0;
    load<kLeft>(a.in_place ? xc : static_cast<const T*>(a.x) + I.off, nullptr, n, I.m0, b);
    T d1[per(cnt(1, kLeft))], d2[per(cnt(2, kLeft))], d3[per(cnt(3, kLeft))],
        d4[per(cnt(4, kLeft))];
    const int hard = a.hardness;
    auto cut = [&](T* d) {
      return [=](int, int k, T, T v) {
        d[k] = thresh_coef(v, t, hard);
        tile_pin(d[k]);
      };
    };
    level<1, kLeft>(b, cut(d1));
    level<2, kLeft>(b, cut(d2));
    level<3, kLeft>(b, cut(d3));
    level<A, kLeft>(b, cut(d4));
    T *S = b, *D = b + own(1) + H(1) + 1;
#pragma unroll
    for (int k = 0; k < per(own(A) + H(A)); ++k) {
      const int c = int(threadIdx.x) + k * NT;
      if (c < own(A) + H(A)) S[c] = s4[((I.m0 >> A) - H(A) + c) & ((n >> A) - 1)];
    }
    details<A>(D, d4);
    __syncthreads();
    up<4>(S, D, d3, y);
    up<3>(S, D, d2, y);
    up<2>(S, D, d1, y);
    up<1>(S, D, d1, y);
  }
};

// ------------------------------------------------------------------ shrink
// G levels of a sequence array: forward, threshold, inverse.  The smooth of
// the top level is the tile's own, or (COARSE) the already smoothed S'_4.
//
// The tile's slots hold shrink_slots values of one sequence, W of them halo
// on either side (their results are wrong towards the ends and are not
// stored), or whole sequences, on which taps wrap at `mask`; a sequence
// shorter than a quad's reach, 2^(G+1), is repeated to that length.  LDS reads bound the
// pass, so a thread computes four outputs a level's stride apart, which share
// L + 3 taps (one by one they read 4 L), and keeps its details in registers.
// Lanes being 4 slots a stride apart, those reads would fall on a quarter of the
// banks: slot e of a buffer that is read at stride s lies at e ^ (r s), r the low
// two bits of its 128-byte row, which spreads them over all.
// 8192 mixed signals in FP64 / 3001 in FP32, us: one output at a time 521 /
// 128 for levels 5..8 and 590 / 144 for levels 1..4, as quads 470 / 106 and 494
// / 127 (vector instructions then busy 70 % of the time, LDS 60 %).  A tile of
// 4096 slots holds a residue of 2^16 samples without halo; of the first
// levels, which wait for more memory, four tiles of 2048 a CU overlap better
// than two of 4096 (655 / 168).
__host__ __device__ constexpr int shrink_nt(bool second) { return second ? 512 : 256; }
__host__ __device__ constexpr int shrink_slots(bool second) { return 8 * shrink_nt(second); }

template <typename T, int FILT, int G, bool COARSE, bool SECOND, bool HARD>
struct Shrink {
  static constexpr int L = Filter<FILT>::L, NT = shrink_nt(SECOND), P0 = shrink_slots(SECOND);
  static constexpr int QN = P0 / 4 / NT, K = P0 / NT;
  static constexpr int W = tile_halo(L, G);
  static constexpr int kLog = sizeof(T) == 8 ? 3 : 2;
  // log2 of a row in a buffer read at stride 2^ls: the 128 bytes of all banks,
  // or a quad's block where that is longer
  static constexpr int row(int ls) {
    const int b = sizeof(T) == 8 ? 4 : 5;
    return b > ls + 2 ? b : ls + 2;
  }
  T S[QN][4], d[G][QN][4];
  T *A, *B;
  int mask, cnt;
  T t;

  // place of slot e in a buffer read at stride 2^ls
  static __device__ __forceinline__ int place(int e, int ls) {
    return e ^ (((e >> row(ls)) & 3) << ls);
  }
  // tap group jj of the quad whose block starts at b4 (offset o in it): its
  // place and the exclusive-or of its four taps, in bytes
  __device__ __forceinline__ int group(int b4, int o, int jj, int ls, int* x) const {
    const int s4 = 4 << ls;
    const int g = (b4 & ~mask) | ((b4 + jj * s4) & mask);
    *x = ((g >> row(ls)) & 3) << (ls + kLog);
    return (g + o) << kLog;
  }
  static __device__ __forceinline__ T at(const T* buf, int bytes) {
    return *reinterpret_cast<const T*>(reinterpret_cast<const unsigned char*>(buf) + bytes);
  }
  // thresh_coef's values (t = 0 where there is no threshold, a NaN)
  __device__ __forceinline__ T cut(T c) const {
    if constexpr (HARD) return fabs(c) < t ? T(0) : c;
    tile_pin(c);  // rounded: no product of c's is fused into the difference
    return soft_cut(c, t);
  }

  // levels l..last
  template <int l, int last>
  __device__ __forceinline__ void forward() {
    if constexpr (l <= last) {
      constexpr int ls = l - 1, s = 1 << ls;
      const T* src = (l & 1) ? A : B;
      T* dst = (l & 1) ? B : A;
#pragma unroll
      for (int q = 0; q < QN; ++q) {
        const int u = int(threadIdx.x) + q * NT;
        if (4 * u < cnt) {
          const int b4 = (u >> ls) << (ls + 2), o = u & (s - 1);
          T w[L + 3];
#pragma unroll
          for (int jj = 0; jj <= (L + 2) / 4; ++jj) {
            int x;
            const int g = group(b4, o, jj, ls, &x);
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (4 * jj + i < L + 3) w[4 * jj + i] = at(src, g + ((i << (ls + kLog)) ^ x));
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            T D;
            analysis1<T, FILT>(w + i, S[q][i], D);
            d[l - 1][q][i] = cut(D);
            tile_pin(d[l - 1][q][i]);
            if (l < G || !COARSE) tile_pin(S[q][i]);
          }
          if constexpr (l < G) {  // to be read at stride 2 s
#pragma unroll
            for (int c = 0; c < 2; ++c) {
              const int p = place(b4 + o + 2 * c * s, l);
              dst[p] = S[q][2 * c];
              dst[p + s] = S[q][2 * c + 1];
            }
          }
        }
      }
      __syncthreads();
      forward<l + 1, last>();
    }
  }
  // v[q][i], the values of quads at stride 2^ls, into a buffer read at it
  template <int ls>
  __device__ __forceinline__ void park(T* buf, const T (*v)[4]) {
#pragma unroll
    for (int q = 0; q < QN; ++q) {
      const int u = int(threadIdx.x) + q * NT;
      const int b4 = (u >> ls) << (ls + 2), o = u & ((1 << ls) - 1);
      const int x = ((b4 >> row(ls)) & 3) << ls;
      if (4 * u < cnt) {
#pragma unroll
        for (int i = 0; i < 4; ++i) buf[b4 + o + ((i << ls) ^ x)] = v[q][i];
      }
    }
  }
  template <int l>
  __device__ __forceinline__ void inverse() {
    if constexpr (l >= 1) {
      constexpr int ls = l - 1, s = 1 << ls, kBack = (L + 2) / 4;
#pragma unroll
      for (int q = 0; q < QN; ++q) {
        const int u = int(threadIdx.x) + q * NT;
        if (4 * u < cnt) {
          const int b4 = (u >> ls) << (ls + 2), o = u & (s - 1);
          T ws[L + 3], wd[L + 3];
#pragma unroll
          for (int jj = -kBack; jj <= 0; ++jj) {
            int x;
            const int g = group(b4, o, jj, ls, &x);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int j = 4 * jj + i + L - 1;
              if (j >= 0) {
                ws[j] = at(A, g + ((i << (ls + kLog)) ^ x));
                wd[j] = at(B, g + ((i << (ls + kLog)) ^ x));
              }
            }
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            S[q][i] = synthesis<T, FILT>(ws, wd, L - 1 + i);
            tile_pin(S[q][i]);
          }
        }
      }
      __syncthreads();
      // to be read at stride s / 2 (the tile's output: in order)
#pragma unroll
      for (int q = 0; q < QN; ++q) {
        const int u = int(threadIdx.x) + q * NT;
        const int b4 = (u >> ls) << (ls + 2), o = u & (s - 1);
        if (4 * u < cnt) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int e = b4 + o + i * s;
            A[l > 1 ? place(e, l > 1 ? ls - 1 : 0) : e] = S[q][i];
          }
        }
      }
      if constexpr (l > 1) park<l - 2>(B, d[l - 2]);
      __syncthreads();
      inverse<l - 1>();
    }
  }
};

// nseq sequences of N values at `in`; the tile starts at value m0 of sequence
// seq0
template <typename T, int FILT, int G, bool COARSE, bool SECOND, bool HARD>
__device__ __forceinline__ void batch_shrink(const T* __restrict__ in, T* __restrict__ out,
                                             const T* __restrict__ coarse, int N, int nseq,
                                             int seq0, int m0, T t, T* lds) {
  using C = Shrink<T, FILT, G, COARSE, SECOND, HARD>;
  constexpr int NT = C::NT, P0 = C::P0, K = C::K, W = C::W;
  const bool circ = N <= P0;
  const int lN = 31 - __builtin_clz(N);
  const int lR = circ ? (lN > G + 1 ? lN : G + 1) : 31;  // slots per sequence
  const int start = circ ? 0 : m0 - W;
  const int64_t base = int64_t(seq0) << lN;
  C c;
  c.A = lds;
  c.B = lds + P0;
  c.t = HARD || t >= T(0) ? t : T(0);
  c.mask = circ ? (1 << lR) - 1 : P0 - 1;
  c.cnt = P0;
  if (circ && (int64_t(nseq - seq0) << lR) < P0) c.cnt = (nseq - seq0) << lR;
  auto index = [&](int e) {
    return base + (int64_t(e >> lR) << lN) + ((start + e) & (N - 1));
  };
  T v[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int e = int(threadIdx.x) + k * NT;
    v[k] = in[index(e < c.cnt ? e : c.cnt - 1)];  // unconditional load, clamped
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int e = int(threadIdx.x) + k * NT;
    c.A[C::place(e, 0)] = v[k];
  }
  __syncthreads();
  c.template forward<1, G - 1>();
  if constexpr (COARSE) {  // in flight during the last level
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int e = int(threadIdx.x) + k * NT;
      const int i = int(index(e < c.cnt ? e : c.cnt - 1));
      v[k] = coarse[int64_t(i & (kBatchRes - 1)) * (N / kBatchRes) + i / kBatchRes];
    }
  }
  c.template forward<G, G>();
  if constexpr (COARSE) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int e = int(threadIdx.x) + k * NT;
      c.A[C::place(e, G - 1)] = v[k];
    }
  } else {
    c.template park<G - 1>(c.A, c.S);
  }
  c.template park<G - 1>(c.B, c.d[G - 1]);
  __syncthreads();
  c.template inverse<G>();
  // stored values: of HALO tiles those between the halos, of repeated
  // sequences the first copy
  const int lo = circ ? 0 : W, hi = circ ? c.cnt : (P0 - W < W + N - m0 ? P0 - W : W + N - m0);
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int e = int(threadIdx.x) + k * NT;
    if (e >= lo && e < hi && (!circ || (e & c.mask) < N)) out[index(e)] = c.A[e];
  }
}

// SECOND: levels 5..J of S_4 into S'_4; else the first levels into y
template <typename T, int FILT, bool SECOND, bool HARD>
__device__ __forceinline__ void batch_shrink_f(const BatchTileArgs& a, const BatchTile& I,
                                               T* lds) {
  const int n = I.n, J = tile_levels(I.kind), seq = tile_seq(I.kind);
  T* scr = static_cast<T*>(a.scratch) + I.scr;
  const T* s4 = scr + batch_pad(n);
  const T t = T(a.thresh[I.sig]);
  if constexpr (SECOND) {
    const int N = n / kBatchRes, R = kBatchRes;
    switch (J - kBatchHead) {
      case 1: batch_shrink<T, FILT, 1, false, SECOND, HARD>(s4, scr, nullptr, N, R, seq, I.m0, t, lds); break;
      case 2: batch_shrink<T, FILT, 2, false, SECOND, HARD>(s4, scr, nullptr, N, R, seq, I.m0, t, lds); break;
      case 3: batch_shrink<T, FILT, 3, false, SECOND, HARD>(s4, scr, nullptr, N, R, seq, I.m0, t, lds); break;
      default: batch_shrink<T, FILT, 4, false, SECOND, HARD>(s4, scr, nullptr, N, R, seq, I.m0, t, lds);
    }
  } else {
    const T* x = a.in_place ? s4 + batch_pad(n) : static_cast<const T*>(a.x) + I.off;
    T* y = static_cast<T*>(a.y) + I.off;
    switch (J) {
      case 1: batch_shrink<T, FILT, 1, false, SECOND, HARD>(x, y, nullptr, n, 1, 0, I.m0, t, lds); break;
      case 2: batch_shrink<T, FILT, 2, false, SECOND, HARD>(x, y, nullptr, n, 1, 0, I.m0, t, lds); break;
      case 3: batch_shrink<T, FILT, 3, false, SECOND, HARD>(x, y, nullptr, n, 1, 0, I.m0, t, lds); break;
      case 4: batch_shrink<T, FILT, 4, false, SECOND, HARD>(x, y, nullptr, n, 1, 0, I.m0, t, lds); break;
      default: batch_shrink<T, FILT, 4, true, SECOND, HARD>(x, y, scr, n, 1, 0, I.m0, t, lds);
    }
  }
}

template <typename T>
__global__ __launch_bounds__(kBatchNT) void batch_head_k(BatchTileArgs a) {
  __shared__ __align__(16) T b[kBatchP + tile_halo(8, kBatchHead)];
  const BatchTile I = a.tiles[blockIdx.x];
  if (I.kind & kTileDwt) {
    switch (I.kind & 7) {
      case kHAAR: DwtTile<T, kHAAR, kBatchNT>::head(a, I, b); break;
      case kD4: DwtTile<T, kD4, kBatchNT>::head(a, I, b); break;
      case kC6: DwtTile<T, kC6, kBatchNT>::head(a, I, b); break;
      default: DwtTile<T, kLA8, kBatchNT>::head(a, I, b); break;
    }
    return;
  }
  const bool deep = tile_levels(I.kind) > kBatchHead, circ = I.n < kBatchP;
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

template <typename T, bool SECOND, bool HARD>
__global__ __launch_bounds__(shrink_nt(SECOND), 4) void batch_shrink_k(BatchTileArgs a) {
  __shared__ __align__(16) T lds[2 * shrink_slots(SECOND)];
  const BatchTile I = a.tiles[blockIdx.x];
  switch (I.kind & 7) {
    case kHAAR: batch_shrink_f<T, kHAAR, SECOND, HARD>(a, I, lds); break;
    case kD4: batch_shrink_f<T, kD4, SECOND, HARD>(a, I, lds); break;
    case kC6: batch_shrink_f<T, kC6, SECOND, HARD>(a, I, lds); break;
    default: batch_shrink_f<T, kLA8, SECOND, HARD>(a, I, lds); break;
  }
}

// The DWT's last pass, apart from the MODWT's, whose registers and LDS would
// halve the workgroups of a CU.
template <typename T>
__global__ __launch_bounds__(kDwtLastNT) void batch_dwt_last_k(BatchTileArgs a) {
  __shared__ __align__(16) T lds[DwtTile<T, kLA8, kDwtLastNT>::kElems];
  const BatchTile I = a.tiles[blockIdx.x];
  switch (I.kind & 7) {
    case kHAAR: DwtTile<T, kHAAR, kDwtLastNT>::last(a, I, lds); break;
    case kD4: DwtTile<T, kD4, kDwtLastNT>::last(a, I, lds); break;
    case kC6: DwtTile<T, kC6, kDwtLastNT>::last(a, I, lds); break;
    default: DwtTile<T, kLA8, kDwtLastNT>::last(a, I, lds); break;
  }
}

// launches over tiles [0, count); defined in batch_tile_<type>.hip
enum class BatchPass { kHead, kSecond, kFirst, kDwtLast };
constexpr int kBatchPasses = 4;
template <typename T>
int batch_tile_launch(BatchPass pass, unsigned count, const BatchTileArgs& a, hipStream_t st);

template <typename T>
int batch_tile_launch_impl(BatchPass pass, unsigned count, const BatchTileArgs& a,
                           hipStream_t st) {
  if (!count) return WH_OK;
  const dim3 grid(count);
  const bool shrink = pass == BatchPass::kFirst || pass == BatchPass::kSecond;
  const dim3 nt(shrink ? shrink_nt(pass == BatchPass::kSecond)
                       : pass == BatchPass::kHead ? kBatchNT : kDwtLastNT);
  switch (pass) {
    case BatchPass::kHead: hipLaunchKernelGGL((batch_head_k<T>), grid, nt, 0, st, a); break;
    case BatchPass::kDwtLast:
      hipLaunchKernelGGL((batch_dwt_last_k<T>), grid, nt, 0, st, a);
      break;
    case BatchPass::kSecond:
      hipLaunchKernelGGL((a.hardness == kHARD ? batch_shrink_k<T, true, true>
                                              : batch_shrink_k<T, true, false>),
                         grid, nt, 0, st, a);
      break;
    case BatchPass::kFirst:
      hipLaunchKernelGGL((a.hardness == kHARD ? batch_shrink_k<T, false, true>
                                              : batch_shrink_k<T, false, false>),
                         grid, nt, 0, st, a);
      break;
  }
  WH_HIP_CHECK(hipGetLastError());
  return WH_OK;
}

}  // namespace wh
