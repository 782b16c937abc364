// modwt_tile.h -- tile form of the level-fused MODWT for launches too small
// to fill the chip with sliding windows (modwt_kern.h has the mathematics).
//
// A sliding-window workgroup walks its segment chunk by chunk, and every
// chunk is a chain of memory latency and G barriers; that pays when each
// workgroup has many chunks.  For a launch of up to 2^20 samples the grid
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

__host__ __device__ constexpr int tile_halo(int L, int l) { return (L - 1) * ((1 << l) - 1); }

// workgroup id -> (signal segment, residue block): workgroups are handed to
// the eight XCDs in turn, so each XCD gets a contiguous run of tiles whose
// halos and residue blocks share its L2
__device__ __forceinline__ int64_t tile_index(int64_t id, int64_t blocks) {
  if (blocks & 7) return id;
  return (id & 7) * (blocks >> 3) + (id >> 3);
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
  const ModwtArgs a = batch_slice<T>(args);
  constexpr int P = C::PR / R;
  const int64_t Nm = a.n >> a.j0, nrb = (int64_t(1) << a.j0) / R;
  const int64_t t = tile_index(blockIdx.x, gridDim.x);
  const int64_t r0 = (t % nrb) * R, m0 = (t / nrb) * P;
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

// ---------------------------------------------------------------- inverse
// Slot o of level l's buffer holds (S_l, D_l) at m = m0 - W_l + o / R.  The
// details of every level are loaded to registers at the start; a level's
// threads write the pair they own -- the S just computed and that level's
// detail -- with one 16-byte store, into the buffer the level above it
// (l + 1) did not read, so a level costs one barrier.
template <typename T, int FILT, int R, int G, int NT>
struct InvTile {
  using V = typename Vec2<T>::type;
  static constexpr int L = Filter<FILT>::L;
  static constexpr int PR = 2 * NT;
  static constexpr int cnt(int l) { return PR + tile_halo(L, l) * R; }  // slots of level l
  static constexpr int K(int l) { return (cnt(l) + NT - 1) / NT; }
  static constexpr int kSlots = G > 1 ? cnt(G) + cnt(G - 1) : cnt(G);
  T d[G + 1][K(G)];  // details of levels 1..G-1 (and the group's top level)

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
      load<l - 1>(a, r0, m0, Nm);
    }
  }
  template <int l>
  __device__ __forceinline__ void levels(V* ba, V* bb, T* out, const ModwtArgs& a, int64_t base,
                                         int64_t qmax) {
    if constexpr (l >= 1) {
      constexpr int s = 1 << (l - 1);
      constexpr int no = cnt(l - 1);  // outputs of this level (cnt(0) = PR)
      const T t = l > 1 ? thr(a, l - 1) : T(-1);
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
          const T e = synthesis<T, FILT>(ws, wd, L - 1);
          if constexpr (l > 1) {
            T c = d[l - 1][k];
            if (t >= T(0)) c = thresh_coef(c, t, a.hardness);
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

template <typename T, int FILT, int R, int G, int NT>
__global__ __launch_bounds__(NT) void modwt_inv_tile_k(ModwtArgs args) {
  using C = InvTile<T, FILT, R, G, NT>;
  using V = typename Vec2<T>::type;
  __shared__ __align__(16) V lds[C::kSlots];
  const ModwtArgs a = batch_slice<T>(args);
  constexpr int P = C::PR / R;
  const int64_t Nm = a.n >> a.j0, nrb = (int64_t(1) << a.j0) / R;
  const int64_t ti = tile_index(blockIdx.x, gridDim.x);
  const int64_t r0 = (ti % nrb) * R, m0 = (ti / nrb) * P;
  C c;
  const T* __restrict__ S = static_cast<const T*>(a.stop);
  T sg[C::K(G)];
#pragma unroll
  for (int k = 0; k < C::K(G); ++k) {
    const int e = int(threadIdx.x) + k * NT;
    sg[k] = S[C::template gidx<G>(a, r0, m0, Nm, e < C::cnt(G) ? e : C::cnt(G) - 1)];
  }
  c.template load<G>(a, r0, m0, Nm);
  const T t = C::thr(a, G);
#pragma unroll
  for (int k = 0; k < C::K(G); ++k) {
    const int e = int(threadIdx.x) + k * NT;
    if (e < C::cnt(G)) {
      T d = c.d[G][k];
      if (t >= T(0)) d = thresh_coef(d, t, a.hardness);
      lds[e] = V{sg[k], d};
    }
  }
  __syncthreads();
  c.template levels<G>(lds, lds + C::cnt(G), static_cast<T*>(a.out), a, r0 + (m0 << a.j0),
                       Nm - m0);
}

// Launch of a tile group of (element type, filter); defined per element
// type in modwt_tile_<type>.hip.
template <typename T>
int modwt_tile_launch(bool inverse, int filt, const GroupLaunch& gl, const ModwtArgs& a,
                      hipStream_t st);

template <typename T, int FILT, bool INV, int R, int NT, int G>
int tile_launch_g(const GroupLaunch& gl, const ModwtArgs& a, hipStream_t st) {
  if constexpr (G > kTileGmax || (R > 1 && G > kTileGmax - 1)) {
    return set_error(WH_ERR_UNSUPPORTED, "modwt: tile group depth out of range");
  } else {
    if (gl.G != G) return tile_launch_g<T, FILT, INV, R, NT, G + 1>(gl, a, st);
    const dim3 grid(unsigned(gl.blocks), unsigned(gl.count));
    if constexpr (INV)
      hipLaunchKernelGGL((modwt_inv_tile_k<T, FILT, R, G, NT>), grid, dim3(NT), 0, st, a);
    else if (gl.sp == kStoreSmooth)
      hipLaunchKernelGGL((modwt_fwd_tile_k<T, FILT, R, G, NT, kStoreSmooth>), grid, dim3(NT), 0,
                         st, a);
    else
      hipLaunchKernelGGL((modwt_fwd_tile_k<T, FILT, R, G, NT, kStoreAll>), grid, dim3(NT), 0, st,
                         a);
    WH_HIP_CHECK(hipGetLastError());
    return WH_OK;
  }
}

template <typename T, int FILT, bool INV>
int tile_launch_f(const GroupLaunch& gl, const ModwtArgs& a, hipStream_t st) {
  constexpr int RD = tile_r(INV);
  if (gl.R == 1 && gl.NT == 512) return tile_launch_g<T, FILT, INV, 1, 512, 1>(gl, a, st);
  if (gl.R == 1 && gl.NT == 256) return tile_launch_g<T, FILT, INV, 1, 256, 1>(gl, a, st);
  if (gl.R == RD && gl.NT == 512) return tile_launch_g<T, FILT, INV, RD, 512, 1>(gl, a, st);
  if (gl.R == RD && gl.NT == 256) return tile_launch_g<T, FILT, INV, RD, 256, 1>(gl, a, st);
  return set_error(WH_ERR_UNSUPPORTED, "modwt: unsupported tile shape");
}

template <typename T, int FILT>
int tile_launch(bool inverse, const GroupLaunch& gl, const ModwtArgs& a, hipStream_t st) {
  return inverse ? tile_launch_f<T, FILT, true>(gl, a, st)
                 : tile_launch_f<T, FILT, false>(gl, a, st);
}

template <typename T>
int modwt_tile_launch_impl(bool inverse, int filt, const GroupLaunch& gl, const ModwtArgs& a,
                           hipStream_t st) {
  switch (filt) {
    case kHAAR: return tile_launch<T, kHAAR>(inverse, gl, a, st);
    case kD4: return tile_launch<T, kD4>(inverse, gl, a, st);
    case kC6: return tile_launch<T, kC6>(inverse, gl, a, st);
    default: return tile_launch<T, kLA8>(inverse, gl, a, st);
  }
}

}  // namespace wh
