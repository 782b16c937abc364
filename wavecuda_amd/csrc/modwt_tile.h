// modwt_tile.h -- tile form of the level-fused MODWT for launches too small
// to fill the chip with sliding windows (modwt_kern.h has the mathematics).
//
// A sliding-window workgroup walks its segment chunk by chunk, and every
// chunk is a chain of memory latency and G barriers; that pays when each
// workgroup has many chunks.  For a launch of up to 2^21 samples the grid
// runs out first: the planner then cut the group depth instead (five fused
// levels and one launch for each further one), and the time was the launches
// and chains, not bytes.  Here a workgroup computes one tile and ends: all
// its loads are issued at the start, the levels follow with one barrier each,
// and the halo the cascade needs, W_l = (L-1)(2^l - 1) positions at level l,
// is loaded and recomputed instead of carried.  LA8, J = 10, n = 2^18 FP64:
// forward 29.6 -> 16.5 us (42 MB stored), inverse 36.4 -> 14.2 us (23 MB
// read), in two launches each instead of six; both are bound by the tile's
// chain (load, G levels) and the launch.  The dispatch rule and its
// measurements are at default_knobs in modwt.hip.
//
// Geometry as in modwt_kern.h: inside a group that starts at level j0,
// position i = r + 2^{j0} m; a tile is P consecutive m of R residues, element
// e = q R + r, so a tap at distance k 2^{l-1} in m is k 2^{l-1} R elements
// away and consecutive lanes always touch consecutive LDS slots (no bank
// conflicts, whatever the level's stride).
#pragma once

#include "modwt_kern.h"

namespace wh {

constexpr int kTileGmax = 6;  // deepest tile group (5 beyond the first)
// Residues of a group beyond the first: consecutive in memory, so R elements
// are a run; more of them means fewer positions per tile and a larger halo
// share.  The forward's stores want the longer run (n = 2^18, J = 10 FP32:
// 11.9 -> 11.3 us from 4 to 8), the inverse the shorter halo.
__host__ __device__ constexpr int tile_r(bool inverse) { return inverse ? 4 : 8; }

constexpr int kTileAdjNT = 512;  // threads of the adjoint and gradient tiles

// What the gradient tile needs beside ModwtArgs (in: the cotangent, xmod: the
// coefficients before thresholding, out: the hand-off to the next group)
struct GradArgs {
  void* gc;         // cotangent of the coefficients, or null
  int zero_s;       // also write zeros into its S_j slots, j < J (the group's last
                    // level apart: a slot that may hold the hand-off)
  int last;         // this group ends at level J
  double* partial;  // [level][signal][per_signal], or null
  int64_t per_signal;
  int hardness, minlevel, maxlevel;  // no level: minlevel > maxlevel
  double value;
  const double* levels;
};

__host__ __device__ constexpr int tile_halo(int L, int l) { return (L - 1) * ((1 << l) - 1); }

// This workgroup's tile and signal.  Workgroups are handed to the eight XCDs in
// turn, in the order of their linear id, so each XCD gets a contiguous run of the
// launch's tiles: halos, and the residue blocks that share a line of memory, stay
// in one L2.  The run goes over the signals' ends: 256 signals of 2^13 samples
// have eight tiles each, and with the runs laid out signal by signal every tile
// of a signal was on an XCD of its own (inverse, J = 8 Haar FP64: 72 us, now 35;
// adjoint of the forward, J = 10 Haar FP32: 124, now 44).
struct TileId {
  int64_t t, sig;
};
__device__ __forceinline__ TileId tile_id() {
  const unsigned per_signal = gridDim.x, total = per_signal * gridDim.y;  // a power of two each signal
  const unsigned id = blockIdx.y * per_signal + blockIdx.x;
  const unsigned xcd = id & 7, rest = total & 7;
  const unsigned at = xcd * (total >> 3) + (xcd < rest ? xcd : rest) + (id >> 3);
  return {at & (per_signal - 1), at >> (31 - __builtin_clz(per_signal))};
}

// first residue and position of tile t of a group of 2^j0 residues, R a tile
template <int R, int P>
__device__ __forceinline__ void tile_origin(int64_t t, int j0, int64_t& r0, int64_t& m0) {
  const int lg = j0 - (31 - __builtin_clz(R));  // 2^lg residue blocks
  r0 = (t & ((int64_t(1) << lg) - 1)) * R;
  m0 = (t >> lg) * P;
}

// Pins the computation of v here: the compiler would sink it beyond the next
// barrier, where v is used, and keep its taps in registers instead.
template <typename T>
__device__ __forceinline__ void tile_pin(T& v) {
  asm volatile("" : "+v"(v));
}

// thresh_coef's soft values at t >= 0 in three operations (t = 0: c itself)
// where it takes twelve in FP64;
// maximum and minimum as instructions because the functions add one for
// signalling NaNs to each operand
template <typename T>
__device__ __forceinline__ T soft_cut(T c, T t) {
  T m;
  if constexpr (sizeof(T) == 8)
    asm("v_max_f64 %0, %1, -%2\n\tv_min_f64 %0, %0, %2" : "=&v"(m) : "v"(c), "v"(t));
  else
    asm("v_max_f32 %0, %1, -%2\n\tv_min_f32 %0, %0, %2" : "=&v"(m) : "v"(c), "v"(t));
  return c - m;
}

// thresh_coef at a threshold t that is t >= 0 or none (negative, a NaN)
template <typename T>
__device__ __forceinline__ T tile_cut(T c, T t, bool soft) {
  if (soft) return soft_cut(c, t >= T(0) ? t : T(0));
  return fabs(c) < t ? T(0) : c;
}

// ---------------------------------------------------------------- forward
// one output (S, D) of taps w[0..L-1] (the terms and order of analysis2)
template <typename T, int FILT>
__device__ __forceinline__ void analysis1(const T* w, T& s, T& d) {
  constexpr int L = Filter<FILT>::L;
  if constexpr (FILT == kHAAR) {
    s = (w[0] + w[1]) * T(kInvR2);
    d = (w[0] - w[1]) * T(kInvR2);
  } else {
    s = w[0] * T(Filter<FILT>::c(0));
    d = w[0] * T(gcoef<FILT>(0));
#pragma unroll
    for (int k = 1; k < L; ++k) {
      s = fma(w[k], T(Filter<FILT>::c(k)), s);
      d = fma(w[k], T(gcoef<FILT>(k)), d);
    }
  }
}

template <typename T, int FILT, int R, int G, int NT, int SP>
struct FwdTile {
  static constexpr int L = Filter<FILT>::L;
  static constexpr int PR = 2 * NT;           // outputs per level and tile
  static constexpr int WG = tile_halo(L, G);
  static constexpr int N0 = PR + WG * R;                       // input elements
  static constexpr int N1 = PR + (WG - tile_halo(L, 1)) * R;   // level-1 outputs
  static constexpr int kLdsElems = N0 + N1;

  // level l reads buffer (l - 1) & 1 and writes buffer l & 1
  template <int l>
  static __device__ __forceinline__ void levels(T* b0, T* b1, T* xmod, const ModwtArgs& a,
                                                int64_t base, int64_t qmax) {
    if constexpr (l <= G) {
      constexpr int s = 1 << (l - 1);
      constexpr int cnt = PR + (WG - tile_halo(L, l)) * R;
      const T* in = (l & 1) ? b0 : b1;
      T* nxt = (l & 1) ? b1 : b0;
      T* oS = xmod + 2 * a.n * int64_t(a.j0 + l - 1);
#pragma unroll
      for (int k = 0; k < (cnt + NT - 1) / NT; ++k) {
        const int o = int(threadIdx.x) + k * NT;
        if (o < cnt) {
          T w[L], S, D;
#pragma unroll
          for (int t = 0; t < L; ++t) w[t] = in[o + t * s * R];
          analysis1<T, FILT>(w, S, D);
          if constexpr (l < G) nxt[o] = S;
          if (o < PR && o / R < qmax) {
            const int64_t i = base + (o % R) + (int64_t(o / R) << a.j0);
            if constexpr (SP == kStoreAll || l == G) oS[i] = S;
            oS[a.n + i] = D;
          }
        }
      }
      if constexpr (l < G) __syncthreads();
      levels<l + 1>(b0, b1, xmod, a, base, qmax);
    }
  }
};

template <typename T, int FILT, int R, int G, int NT, int SP>
__global__ __launch_bounds__(NT) void modwt_fwd_tile_k(ModwtArgs args) {
  using C = FwdTile<T, FILT, R, G, NT, SP>;
  __shared__ __align__(16) T lds[C::kLdsElems];
  const TileId id = tile_id();
  const ModwtArgs a = batch_slice<T>(args, id.sig);
  constexpr int P = C::PR / R;
  const int64_t Nm = a.n >> a.j0;
  int64_t r0, m0;
  tile_origin<R, P>(id.t, a.j0, r0, m0);
  const T* __restrict__ in = static_cast<const T*>(a.in);
  constexpr int K = (C::N0 + NT - 1) / NT;
  T v[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int e = int(threadIdx.x) + k * NT;
    const int ec = e < C::N0 ? e : C::N0 - 1;  // unconditional load, clamped
    v[k] = in[r0 + (ec % R) + (((m0 + ec / R) & (Nm - 1)) << a.j0)];
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int e = int(threadIdx.x) + k * NT;
    if (e < C::N0) lds[e] = v[k];
  }
  __syncthreads();
  C::template levels<1>(lds, lds + C::N0, static_cast<T*>(a.xmod), a, r0 + (m0 << a.j0), Nm - m0);
}

// The adjoint of the thresholding inverse: the forward over the output's
// cotangent, level l scaled by 2^-l, and at each detail the threshold's
// gradient where the coefficient c passes it.  The coefficients are loaded
// at the start; per-level sums of dL/dt stay in registers and leave as one
// partial per workgroup, in an order that repeats.  With gc the cotangent of
// the coefficients is stored (details, S_J, and zeros in the other S slots
// if asked for); without it the kernel writes nothing but its hand-off and
// partials: 512 x 2^14 FP32, J = 8, LA8 took a pass that stored the 2nJ
// cotangents (102 us) and one that read them back beside c (108 us).
// the cotangent g of a detail through its threshold t (act: the level is
// thresholded) at coefficient v, and dL/dt added to sum
template <typename T>
__device__ __forceinline__ T grad_cut(const GradArgs& q, T g, T v, T t, bool act, double& sum) {
  if (!act) return g;
  const T m = fabs(v);
  if (q.hardness == kSOFT) {
    const bool pass = m > t;
    if (pass) sum += double(v < T(0) ? g : -g);
    return pass ? g : T(0);
  }
  return m < t ? T(0) : g;
}

// the workgroup's sums of levels j0..j0+G-1 into its partials
template <int G, int NT>
__device__ __forceinline__ void grad_partials(double* acc, double (*red)[NT / 64], int j0,
                                              const TileId& id, const GradArgs& q) {
#pragma unroll
  for (int l = 0; l < G; ++l) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) acc[l] += __shfl_xor(acc[l], o, 64);
    if ((threadIdx.x & 63) == 0) red[l][threadIdx.x >> 6] = acc[l];
  }
  __syncthreads();
  if (threadIdx.x < G) {
    double sum = 0.0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) sum += red[threadIdx.x][w];
    q.partial[((j0 + int64_t(threadIdx.x)) * gridDim.y + id.sig) * q.per_signal + id.t] = sum;
  }
}

template <typename T, int FILT, int R, int G, int NT>
struct GradTile {
  using F = FwdTile<T, FILT, R, G, NT, kStoreAll>;
  static constexpr int L = F::L;
  static constexpr int KO = F::PR / NT;  // owned outputs per thread
  static constexpr int kWaves = NT / 64;
  T c[G][KO];
  double acc[G];

  template <int l>
  __device__ __forceinline__ void levels(T* b0, T* b1, const ModwtArgs& a, const GradArgs& q,
                                         T* gc, int64_t base, int64_t qmax) {
    if constexpr (l <= G) {
      constexpr int s = 1 << (l - 1);
      constexpr int cnt = F::PR + (F::WG - tile_halo(L, l)) * R;
      constexpr T sc = T(1.0 / double(1 << l));
      const T* in = (l & 1) ? b0 : b1;
      T* nxt = (l & 1) ? b1 : b0;
      const int lev = a.j0 + l - 1;
      const bool act = lev >= q.minlevel && lev <= q.maxlevel;
      const T t = !act ? T(0) : q.levels ? T(q.levels[lev]) : T(q.value);
      T* oS = gc ? gc + 2 * a.n * int64_t(lev) : nullptr;
      const bool top = l == G && q.last;  // S_J
#pragma unroll
      for (int k = 0; k < (cnt + NT - 1) / NT; ++k) {
        const int o = int(threadIdx.x) + k * NT;
        if (o < cnt) {
          T w[L], S, D;
#pragma unroll
          for (int j = 0; j < L; ++j) w[j] = in[o + j * s * R];
          analysis1<T, FILT>(w, S, D);
          if constexpr (l < G) nxt[o] = S;
          // the owned outputs come first in every level's order
          if (k < KO && o / R < qmax) {
            const T g = grad_cut(q, D * sc, c[l - 1][k < KO ? k : 0], t, act, acc[l - 1]);
            const int64_t i = base + (o % R) + (int64_t(o / R) << a.j0);
            if (oS) {
              oS[a.n + i] = g;
              if (top) oS[i] = S * sc;
              else if (l < G && q.zero_s) oS[i] = T(0);
            }
            if (l == G && !q.last) static_cast<T*>(a.out)[i] = S * sc;
          }
        }
      }
      if constexpr (l < G) __syncthreads();
      levels<l + 1>(b0, b1, a, q, gc, base, qmax);
    }
  }
};

template <typename T, int FILT, int R, int G, int NT>
__global__ __launch_bounds__(NT) void modwt_grad_tile_k(ModwtArgs args, GradArgs q) {
  using C = GradTile<T, FILT, R, G, NT>;
  using F = typename C::F;
  __shared__ __align__(16) T lds[F::kLdsElems];
  __shared__ double red[G][C::kWaves];
  const TileId id = tile_id();
  const ModwtArgs a = batch_slice<T>(args, id.sig);
  constexpr int P = F::PR / R;
  const int64_t Nm = a.n >> a.j0;
  int64_t r0, m0;
  tile_origin<R, P>(id.t, a.j0, r0, m0);
  const T* __restrict__ in = static_cast<const T*>(a.in);
  const T* __restrict__ xm = static_cast<const T*>(a.xmod);
  constexpr int K = (F::N0 + NT - 1) / NT;
  C c;
  T v[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int e = int(threadIdx.x) + k * NT;
    const int ec = e < F::N0 ? e : F::N0 - 1;  // unconditional load, clamped
    v[k] = in[r0 + (ec % R) + (((m0 + ec / R) & (Nm - 1)) << a.j0)];
  }
#pragma unroll
  for (int l = 1; l <= G; ++l) {
    c.acc[l - 1] = 0.0;
#pragma unroll
    for (int k = 0; k < C::KO; ++k) {
      const int o = int(threadIdx.x) + k * NT, lev = a.j0 + l - 1;
      const int64_t i = r0 + (o % R) + (((m0 + o / R) & (Nm - 1)) << a.j0);
      c.c[l - 1][k] = lev >= q.minlevel && lev <= q.maxlevel
                          ? xm[2 * a.n * int64_t(lev) + a.n + i]
                          : T(0);
    }
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int e = int(threadIdx.x) + k * NT;
    if (e < F::N0) lds[e] = v[k];
  }
  __syncthreads();
  T* gc = q.gc ? static_cast<T*>(q.gc) + id.sig * a.bs_xmod : nullptr;
  c.template levels<1>(lds, lds + F::N0, a, q, gc, r0 + (m0 << a.j0), Nm - m0);
  if (q.partial) grad_partials<G, NT>(c.acc, red, a.j0, id, q);
}

// ---------------------------------------------------------------- inverse
// Slot o of level l's buffer holds (S_l, D_l) at m = m0 - W_l + o / R.  The
// details of every level are loaded to registers at the start; a level's
// threads write the pair they own -- the S just computed and that level's
// detail -- with one 16-byte store, into the buffer the level above it
// (l + 1) did not read, so a level costs one barrier.
//
// The same tile is the adjoint of the forward (Adj): u_{j-1} = Sb_{j-1} +
// H_j^T u_j + G_j^T Db_j reads positions i - k s as the inverse does, without
// the factor 1/2 and the threshold, and with each level's own S cotangent
// Sb added (kAdjFull) or known to be zero (kAdjDetails).
constexpr int kInverse = 0;
constexpr int kAdjFull = 1;
constexpr int kAdjDetails = 2;

// one output of the adjoint: acc + sum_k C_k u[tap k] + g_k Db[tap k], k
// ascending, tap k at w[L - 1 - k]
template <typename T, int FILT>
__device__ __forceinline__ T adjoint1(const T* wu, const T* wd, T acc) {
  constexpr int L = Filter<FILT>::L;
#pragma unroll
  for (int k = 0; k < L; ++k) {
    acc = fma(wu[L - 1 - k], T(Filter<FILT>::c(k)), acc);
    acc = fma(wd[L - 1 - k], T(gcoef<FILT>(k)), acc);
  }
  return acc;
}

template <typename T, int FILT, int R, int G, int NT, int MODE>
struct InvTile {
  using V = typename Vec2<T>::type;
  static constexpr int L = Filter<FILT>::L;
  static constexpr int PR = 2 * NT;
  static constexpr int cnt(int l) { return PR + tile_halo(L, l) * R; }  // slots of level l
  static constexpr int K(int l) { return (cnt(l) + NT - 1) / NT; }
  static constexpr int kSlots = G > 1 ? cnt(G) + cnt(G - 1) : cnt(G);
  T d[G + 1][K(G)];  // details of levels 1..G-1 (and the group's top level)
  T sb[MODE == kAdjFull ? G + 1 : 1][K(G)];  // Sb of the levels 0..G-1 of the group

  static __device__ __forceinline__ T thr(const ModwtArgs& a, int l) {
    const int lev = a.j0 + l - 1;
    if (!a.th_on || lev < a.minlevel || lev > a.maxlevel) return T(-1);
    return a.th_levels ? T(a.th_levels[lev]) : T(a.th_value);
  }
  // global index of slot e of level l
  template <int l>
  static __device__ __forceinline__ int64_t gidx(const ModwtArgs& a, int64_t r0, int64_t m0,
                                                 int64_t Nm, int e) {
    const int64_t m = (m0 - tile_halo(L, l) + e / R) & (Nm - 1);
    return r0 + (e % R) + (m << a.j0);
  }
  template <int l>
  __device__ __forceinline__ void load(const ModwtArgs& a, int64_t r0, int64_t m0, int64_t Nm) {
    if constexpr (l >= 1) {
      const T* D = static_cast<const T*>(a.xmod) + 2 * a.n * int64_t(a.j0 + l - 1) + a.n;
#pragma unroll
      for (int k = 0; k < K(l); ++k) {
        const int e = int(threadIdx.x) + k * NT;
        d[l][k] = D[gidx<l>(a, r0, m0, Nm, e < cnt(l) ? e : cnt(l) - 1)];
      }
      if constexpr (MODE == kAdjFull) {
        // S_{j0 + l - 1}, this level's output slots; none below level 1
        const bool have = a.j0 + l > 1;
        const T* S = static_cast<const T*>(a.xmod) + 2 * a.n * int64_t(a.j0 + l - 2);
#pragma unroll
        for (int k = 0; k < K(l - 1); ++k) {
          const int e = int(threadIdx.x) + k * NT;
          sb[l - 1][k] =
              have ? S[gidx<l - 1>(a, r0, m0, Nm, e < cnt(l - 1) ? e : cnt(l - 1) - 1)] : T(0);
        }
      }
      load<l - 1>(a, r0, m0, Nm);
    }
  }
  template <int l>
  __device__ __forceinline__ void levels(V* ba, V* bb, T* out, const ModwtArgs& a, int64_t base,
                                         int64_t qmax) {
    if constexpr (l >= 1) {
      constexpr int s = 1 << (l - 1);
      constexpr int no = cnt(l - 1);  // outputs of this level (cnt(0) = PR)
      const T t = MODE == kInverse && l > 1 ? thr(a, l - 1) : T(-1);
#pragma unroll
      for (int k = 0; k < (no + NT - 1) / NT; ++k) {
        const int o = int(threadIdx.x) + k * NT;
        if (o < no) {
          T ws[L], wd[L];
#pragma unroll
          for (int j = 0; j < L; ++j) {
            const V v = ba[o + j * s * R];
            ws[j] = v.x;
            wd[j] = v.y;
          }
          T e;
          if constexpr (MODE == kInverse) e = synthesis<T, FILT>(ws, wd, L - 1);
          else e = adjoint1<T, FILT>(ws, wd, MODE == kAdjFull ? sb[l - 1][k] : T(0));
          if constexpr (l > 1) {
            T c = d[l - 1][k];
            if (MODE == kInverse) c = tile_cut(c, t, a.hardness == kSOFT);
            bb[o] = V{e, c};
          } else if (o / R < qmax) {
            out[base + (o % R) + (int64_t(o / R) << a.j0)] = e;
          }
        }
      }
      if constexpr (l > 1) __syncthreads();
      levels<l - 1>(bb, ba, out, a, base, qmax);
    }
  }
};

template <typename T, int FILT, int R, int G, int NT, int MODE>
__global__ __launch_bounds__(NT) void modwt_inv_tile_k(ModwtArgs args) {
  using C = InvTile<T, FILT, R, G, NT, MODE>;
  using V = typename Vec2<T>::type;
  __shared__ __align__(16) V lds[C::kSlots];
  const TileId id = tile_id();
  const ModwtArgs a = batch_slice<T>(args, id.sig);
  constexpr int P = C::PR / R;
  const int64_t Nm = a.n >> a.j0;
  int64_t r0, m0;
  tile_origin<R, P>(id.t, a.j0, r0, m0);
  C c;
  const T* __restrict__ S = static_cast<const T*>(a.stop);
  T sg[C::K(G)];
#pragma unroll
  for (int k = 0; k < C::K(G); ++k) {
    const int e = int(threadIdx.x) + k * NT;
    sg[k] = S[C::template gidx<G>(a, r0, m0, Nm, e < C::cnt(G) ? e : C::cnt(G) - 1)];
  }
  c.template load<G>(a, r0, m0, Nm);
  const T t = MODE == kInverse ? C::thr(a, G) : T(-1);
#pragma unroll
  for (int k = 0; k < C::K(G); ++k) {
    const int e = int(threadIdx.x) + k * NT;
    if (e < C::cnt(G)) {
      T d = c.d[G][k];
      if (MODE == kInverse) d = tile_cut(d, t, a.hardness == kSOFT);
      lds[e] = V{sg[k], d};
    }
  }
  __syncthreads();
  c.template levels<G>(lds, lds + C::cnt(G), static_cast<T*>(a.out), a, r0 + (m0 << a.j0),
                       Nm - m0);
}

// ------------------------------------------------------------ wide tiles
// FP32 launches that fill the chip many times over: all J <= 8 levels in one
// group of one launch (no hand-off between groups, whole runs of one
// position per lane), so the halo of the whole cascade -- 1785 positions for
// LA8 at J = 8 -- is carried by tiles of 2048 (inverse) or 4096 (gradient)
// positions.  One buffer serves every level: a level's outputs are held in
// registers over a barrier and written back over its inputs, which leaves
// LDS for several workgroups per CU, and only the next kWideAhead levels'
// arrays are in flight, which leaves registers for them.  LA8, J = 8,
// 512 x 2^14: inverse 147 us as one sliding group (one 80 KB workgroup per
// CU) -> 92 (302 MB read; 256 threads x 8 outputs; 512 x 4 takes 100, 1024 x
// 2 112) -> 84 with the short soft threshold; gradient in two tile groups 148
// -> 85 -> 80.  Quads of outputs that share their taps read less LDS (thresholded
// 87 us) but leave launches of few tiles slower (2^20 samples D4 16.4 us against
// 15.6).  In FP64 the kernels need all 256 registers (252 us against 191
// sliding), so they are not built.
constexpr int kWideInvNT = 256, kWideInvPer = 8, kWideInvAhead = 3;
constexpr int kWideGradNT = 512, kWideGradPer = 8, kWideGradAhead = 2;
constexpr int kWideGmin = 3, kWideGmax = 8;
constexpr int kWideInvP = kWideInvNT * kWideInvPer;     // positions per tile
constexpr int kWideGradP = kWideGradNT * kWideGradPer;

template <typename T, int FILT, int G, int MODE>
struct InvWide {
  using V = typename Vec2<T>::type;
  static constexpr int L = Filter<FILT>::L, NT = kWideInvNT;
  static constexpr int cnt(int l) { return kWideInvP + tile_halo(L, l); }  // slots of level l
  static constexpr int K(int l) { return (cnt(l) + NT - 1) / NT; }
  T d[G + 1][K(G)];

  template <int l>
  static __device__ __forceinline__ int64_t gidx(const ModwtArgs& a, int64_t m0, int k) {
    const int e = int(threadIdx.x) + k * NT;
    return (m0 - tile_halo(L, l) + (e < cnt(l) ? e : cnt(l) - 1)) & (a.n - 1);
  }
  template <int l>
  __device__ __forceinline__ void load(const ModwtArgs& a, int64_t m0) {
    if constexpr (l >= 1) {
      const T* D = static_cast<const T*>(a.xmod) + 2 * a.n * int64_t(l - 1) + a.n;
#pragma unroll
      for (int k = 0; k < K(l); ++k) d[l][k] = __builtin_nontemporal_load(D + gidx<l>(a, m0, k));
    }
  }
  template <int l, int left>
  __device__ __forceinline__ void load_ahead(const ModwtArgs& a, int64_t m0) {
    if constexpr (left > 0) {
      load<l>(a, m0);
      load_ahead<l - 1, left - 1>(a, m0);
    }
  }
  template <int l>
  __device__ __forceinline__ void levels(V* b, const ModwtArgs& a, int64_t m0) {
    if constexpr (l >= 1) {
      load<l - kWideInvAhead>(a, m0);
      constexpr int s = 1 << (l - 1), no = cnt(l - 1), ko = K(l - 1);
      T e[ko];
#pragma unroll
      for (int k = 0; k < ko; ++k) {
        const int o = int(threadIdx.x) + k * NT;
        if (o < no) {
          T ws[L], wd[L];
#pragma unroll
          for (int j = 0; j < L; ++j) {
            const V v = b[o + j * s];
            ws[j] = v.x;
            wd[j] = v.y;
          }
          if constexpr (MODE == kInverse) e[k] = synthesis<T, FILT>(ws, wd, L - 1);
          else e[k] = adjoint1<T, FILT>(ws, wd, T(0));
        }
      }
      if constexpr (l > 1) {
        const T t = MODE == kInverse ? InvTile<T, FILT, 1, G, NT, MODE>::thr(a, l - 1) : T(-1);
        __syncthreads();  // every tap of this level read before any is replaced
#pragma unroll
        for (int k = 0; k < ko; ++k) {
          const int o = int(threadIdx.x) + k * NT;
          T c = d[l - 1][k];
          if (MODE == kInverse) c = tile_cut(c, t, a.hardness == kSOFT);
          if (o < no) b[o] = V{e[k], c};
        }
        __syncthreads();
      } else {
        T* out = static_cast<T*>(a.out);
#pragma unroll
        for (int k = 0; k < ko; ++k) out[m0 + threadIdx.x + k * NT] = e[k];
      }
      levels<l - 1>(b, a, m0);
    }
  }
};

// n is a multiple of kWideInvP
template <typename T, int FILT, int G, int MODE>
__global__ __launch_bounds__(kWideInvNT) void modwt_inv_wide_k(ModwtArgs args) {
  using C = InvWide<T, FILT, G, MODE>;
  using V = typename Vec2<T>::type;
  __shared__ __align__(16) V lds[C::cnt(G)];
  const TileId id = tile_id();
  const ModwtArgs a = batch_slice<T>(args, id.sig);
  const int64_t m0 = id.t * kWideInvP;
  C c;
  T sg[C::K(G)];
#pragma unroll
  for (int k = 0; k < C::K(G); ++k)
    sg[k] = static_cast<const T*>(a.stop)[C::template gidx<G>(a, m0, k)];
  c.template load_ahead<G, kWideInvAhead>(a, m0);
  const T t = MODE == kInverse ? InvTile<T, FILT, 1, G, kWideInvNT, MODE>::thr(a, G) : T(-1);
#pragma unroll
  for (int k = 0; k < C::K(G); ++k) {
    const int e = int(threadIdx.x) + k * kWideInvNT;
    T d = c.d[G][k];
    if (MODE == kInverse) d = tile_cut(d, t, a.hardness == kSOFT);
    if (e < C::cnt(G)) lds[e] = V{sg[k], d};
  }
  __syncthreads();
  c.template levels<G>(lds, a, m0);
}

template <typename T, int FILT, int G>
struct GradWide {
  static constexpr int L = Filter<FILT>::L, NT = kWideGradNT, KO = kWideGradPer;
  static constexpr int cnt(int l) { return kWideGradP + tile_halo(L, G) - tile_halo(L, l); }
  T c[G + 1][KO];
  double acc[G];

  template <int l>
  __device__ __forceinline__ void load(const ModwtArgs& a, const GradArgs& q, int64_t m0) {
    if constexpr (l <= G) {
      const T* D = static_cast<const T*>(a.xmod) + 2 * a.n * int64_t(l - 1) + a.n + m0;
      const bool act = l - 1 >= q.minlevel && l - 1 <= q.maxlevel;
#pragma unroll
      for (int k = 0; k < KO; ++k)
        c[l][k] = act ? __builtin_nontemporal_load(D + threadIdx.x + k * NT) : T(0);
    }
  }
  template <int l, int left>
  __device__ __forceinline__ void load_ahead(const ModwtArgs& a, const GradArgs& q, int64_t m0) {
    if constexpr (left > 0) {
      load<l>(a, q, m0);
      load_ahead<l + 1, left - 1>(a, q, m0);
    }
  }
  template <int l>
  __device__ __forceinline__ void levels(T* b, const ModwtArgs& a, const GradArgs& q, T* gc,
                                         int64_t m0) {
    if constexpr (l <= G) {
      load<l + kWideGradAhead>(a, q, m0);
      constexpr int s = 1 << (l - 1), no = cnt(l), ko = (no + NT - 1) / NT;
      constexpr T sc = T(1.0 / double(1 << l));
      const bool act = l - 1 >= q.minlevel && l - 1 <= q.maxlevel;
      const T t = !act ? T(0) : q.levels ? T(q.levels[l - 1]) : T(q.value);
      T* oS = gc ? gc + 2 * a.n * int64_t(l - 1) + m0 : nullptr;
      T S[ko];
      double sum = 0.0;
#pragma unroll
      for (int k = 0; k < ko; ++k) {
        const int o = int(threadIdx.x) + k * NT;
        if (o < no) {
          T w[L], D;
#pragma unroll
          for (int j = 0; j < L; ++j) w[j] = b[o + j * s];
          analysis1<T, FILT>(w, S[k], D);
          tile_pin(S[k]);
          if (k < KO) {  // owned
            const T g = grad_cut(q, D * sc, c[l][k < KO ? k : 0], t, act, sum);
            if (oS) {
              oS[a.n + o] = g;
              if (l == G) oS[o] = S[k] * sc;
              else if (q.zero_s) oS[o] = T(0);
            }
          }
        }
      }
      acc[l - 1] = sum;
      if constexpr (l < G) {
        __syncthreads();  // every tap of this level read before any is replaced
#pragma unroll
        for (int k = 0; k < ko; ++k) {
          const int o = int(threadIdx.x) + k * NT;
          if (o < no) b[o] = S[k];
        }
        __syncthreads();
      }
      levels<l + 1>(b, a, q, gc, m0);
    }
  }
};

// n is a multiple of kWideGradP
template <typename T, int FILT, int G>
__global__ __launch_bounds__(kWideGradNT) void modwt_grad_wide_k(ModwtArgs args, GradArgs q) {
  using C = GradWide<T, FILT, G>;
  constexpr int NT = kWideGradNT, N0 = C::cnt(0), K = (N0 + NT - 1) / NT;
  __shared__ __align__(16) T lds[N0];
  __shared__ double red[G][NT / 64];
  const TileId id = tile_id();
  const ModwtArgs a = batch_slice<T>(args, id.sig);
  const int64_t m0 = id.t * kWideGradP;
  const T* __restrict__ in = static_cast<const T*>(a.in);
  C c;
  T v[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int e = int(threadIdx.x) + k * NT;
    v[k] = in[(m0 + (e < N0 ? e : N0 - 1)) & (a.n - 1)];
  }
  c.template load_ahead<1, kWideGradAhead>(a, q, m0);
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int e = int(threadIdx.x) + k * NT;
    if (e < N0) lds[e] = v[k];
  }
  __syncthreads();
  T* gc = q.gc ? static_cast<T*>(q.gc) + id.sig * a.bs_xmod : nullptr;
  c.template levels<1>(lds, a, q, gc, m0);
  if (q.partial) grad_partials<G, NT>(c.acc, red, 0, id, q);
}

// What a tile launch computes
enum class TileOp { kForward, kForwardDetails, kInverse, kAdjFull, kAdjDetails, kGrad };

// Launch of a tile group of (element type, filter); defined per element
// type in modwt_tile_<type>.hip.
template <typename T>
int modwt_tile_launch(TileOp op, int filt, const GroupLaunch& gl, const ModwtArgs& a,
                      const GradArgs& q, hipStream_t st);

template <typename T, int FILT, bool INV, int R, int NT, int G>
int tile_launch_g(TileOp op, const GroupLaunch& gl, const ModwtArgs& a, const GradArgs& q,
                  hipStream_t st) {
  if constexpr (G > kTileGmax || (R > 1 && G > kTileGmax - 1)) {
    return set_error(WH_ERR_UNSUPPORTED, "modwt: tile group depth out of range");
  } else {
    if (gl.G != G) return tile_launch_g<T, FILT, INV, R, NT, G + 1>(op, gl, a, q, st);
    const dim3 grid(unsigned(gl.blocks), unsigned(gl.count), gl.cand);
    if constexpr (INV) {
      if (op == TileOp::kInverse)
        hipLaunchKernelGGL((modwt_inv_tile_k<T, FILT, R, G, NT, kInverse>), grid, dim3(NT), 0, st,
                           a);
      else if constexpr (NT == kTileAdjNT)
        hipLaunchKernelGGL((op == TileOp::kAdjFull
                                ? modwt_inv_tile_k<T, FILT, R, G, NT, kAdjFull>
                                : modwt_inv_tile_k<T, FILT, R, G, NT, kAdjDetails>),
                           grid, dim3(NT), 0, st, a);
    } else {
      if (op == TileOp::kForward)
        hipLaunchKernelGGL((modwt_fwd_tile_k<T, FILT, R, G, NT, kStoreAll>), grid, dim3(NT), 0,
                           st, a);
      else if (op == TileOp::kForwardDetails)
        hipLaunchKernelGGL((modwt_fwd_tile_k<T, FILT, R, G, NT, kStoreSmooth>), grid, dim3(NT), 0,
                           st, a);
      else if constexpr (NT == kTileAdjNT)
        hipLaunchKernelGGL((modwt_grad_tile_k<T, FILT, R, G, NT>), grid, dim3(NT), 0, st, a, q);
    }
    WH_HIP_CHECK(hipGetLastError());
    return WH_OK;
  }
}

template <typename T, int FILT, bool INV>
int tile_launch_f(TileOp op, const GroupLaunch& gl, const ModwtArgs& a, const GradArgs& q,
                  hipStream_t st) {
  constexpr int RD = tile_r(INV);
  if (gl.R == 1 && gl.NT == 512) return tile_launch_g<T, FILT, INV, 1, 512, 1>(op, gl, a, q, st);
  if (gl.R == 1 && gl.NT == 256) return tile_launch_g<T, FILT, INV, 1, 256, 1>(op, gl, a, q, st);
  if (gl.R == RD && gl.NT == 512) return tile_launch_g<T, FILT, INV, RD, 512, 1>(op, gl, a, q, st);
  if (gl.R == RD && gl.NT == 256) return tile_launch_g<T, FILT, INV, RD, 256, 1>(op, gl, a, q, st);
  return set_error(WH_ERR_UNSUPPORTED, "modwt: unsupported tile shape");
}

template <typename T, int FILT, int G>
int wide_launch_g(TileOp op, const GroupLaunch& gl, const ModwtArgs& a, const GradArgs& q,
                  hipStream_t st) {
  if constexpr (G > kWideGmax) {
    return set_error(WH_ERR_UNSUPPORTED, "modwt: wide tile depth out of range");
  } else {
    if (gl.G != G) return wide_launch_g<T, FILT, G + 1>(op, gl, a, q, st);
    const dim3 grid(unsigned(gl.blocks), unsigned(gl.count), gl.cand);
    if (op == TileOp::kGrad)
      hipLaunchKernelGGL((modwt_grad_wide_k<T, FILT, G>), grid, dim3(kWideGradNT), 0, st, a, q);
    else if (op == TileOp::kInverse)
      hipLaunchKernelGGL((modwt_inv_wide_k<T, FILT, G, kInverse>), grid, dim3(kWideInvNT), 0, st,
                         a);
    else if (op == TileOp::kAdjDetails)
      hipLaunchKernelGGL((modwt_inv_wide_k<T, FILT, G, kAdjDetails>), grid, dim3(kWideInvNT), 0,
                         st, a);
    else
      return set_error(WH_ERR_UNSUPPORTED, "modwt: no such wide tile");
    WH_HIP_CHECK(hipGetLastError());
    return WH_OK;
  }
}

template <typename T, int FILT>
int tile_launch(TileOp op, const GroupLaunch& gl, const ModwtArgs& a, const GradArgs& q,
                hipStream_t st) {
  if constexpr (sizeof(T) == 4) {
    if (gl.wide) return wide_launch_g<T, FILT, kWideGmin>(op, gl, a, q, st);
  }
  const bool inv = op == TileOp::kInverse || op == TileOp::kAdjFull || op == TileOp::kAdjDetails;
  return inv ? tile_launch_f<T, FILT, true>(op, gl, a, q, st)
             : tile_launch_f<T, FILT, false>(op, gl, a, q, st);
}

template <typename T>
int modwt_tile_launch_impl(TileOp op, int filt, const GroupLaunch& gl, const ModwtArgs& a,
                           const GradArgs& q, hipStream_t st) {
  switch (filt) {
    case kHAAR: return tile_launch<T, kHAAR>(op, gl, a, q, st);
    case kD4: return tile_launch<T, kD4>(op, gl, a, q, st);
    case kC6: return tile_launch<T, kC6>(op, gl, a, q, st);
    default: return tile_launch<T, kLA8>(op, gl, a, q, st);
  }
}

}  // namespace wh
