// adjoint.hip -- gradients of the soft threshold and of the mean squared
// error (gfx950).  The transforms' adjoints: MODWT in modwt_tile.h and
// modwt.hip; the DWT is orthogonal, so its forward and inverse are each
// other's.
//
// MODWT forward F: x -> (S_1, D_1, ..., S_J, D_J) with
//   S_j = H_j S_{j-1},  D_j = G_j S_{j-1},  (H_j u)[i] = sum_k C_k u[(i + k s) mod n]
// (reference src/daub4.cpp:561-571, s = 2^{j-1}).  Its adjoint takes the
// cotangents (Sb_j, Db_j) of every output back to x:
//   u_J = Sb_J,  u_{j-1} = Sb_{j-1} + H_j^T u_j + G_j^T Db_j,  xb = u_0
// with (H_j^T u)[p] = sum_k C_k u[(p - k s) mod n].
//
// Soft threshold y = sign(c) max(|c| - t, 0) on the details of levels
// [minlevel, maxlevel] (reference src/thresh.cpp:142-157): dy/dc = 1[|c| > t],
// dy/dt = -sign(c) 1[|c| > t] (0 at |c| = t, where the rule gives 0); the
// hard rule keeps c when |c| >= t: dy/dc = 1[|c| >= t], dy/dt = 0 almost
// everywhere.  The per-level sums of dy/dt * ybar are block partials reduced
// in a fixed order, so repeated runs give identical gradients.
#include <algorithm>

#include "wh_common.h"
#include "wh_internal.h"
#include "wh_stats.h"

namespace wh {

namespace {

constexpr int kGradNT = 256;
constexpr int kGradMinPer = 4096;         // elements per workgroup, at least
constexpr int64_t kGradMaxPartials = 65536;  // partial sums per call, at most

template <typename T>
__device__ __forceinline__ void grad_one(T cv, T g, T t, int hardness, T* gcp, double& acc) {
  const T a = fabs(cv);
  if (hardness == kSOFT) {
    const bool pass = a > t;
    if (gcp) *gcp = pass ? g : T(0);
    if (pass) acc += double(cv < T(0) ? g : -g);
  } else if (gcp) {
    *gcp = (a < t) ? T(0) : g;
  }
}

// One workgroup per (chunk, level, signal).  MODWT details of a level are
// contiguous and move as element pairs; the DWT's are strided.  The
// workgroup's sum is reduced in a fixed order (lanes by shuffles, then the
// four waves), so results repeat bit for bit.
template <typename T>
__global__ __launch_bounds__(kGradNT) void thresh_grad_k(const T* __restrict__ c0,
                                                         const T* __restrict__ gy0,
                                                         T* __restrict__ gc0,
                                                         double* __restrict__ partial, int64_t n,
                                                         int J, int ttype, Thr1 th, int write_gc) {
  using V = typename Vec2<T>::type;
  const int l = th.minlevel + int(blockIdx.y);
  const int nl = int(gridDim.y);
  const int64_t sig = blockIdx.z;
  const int64_t per = (ttype == kDWT) ? n : 2 * n * J;
  const T* __restrict__ c = c0 + sig * per;
  const T* __restrict__ gy = gy0 + sig * per;
  T* __restrict__ gc = write_gc ? gc0 + sig * per : nullptr;
  const T t = th.levels ? T(th.levels[l]) : T(th.value);
  double acc = 0.0;
  if (ttype == kDWT) {
    const int64_t off = int64_t(1) << l, stride = int64_t(2) << l, cnt = n >> (l + 1);
    const int64_t chunk = (cnt + gridDim.x - 1) / gridDim.x;
    const int64_t e0 = int64_t(blockIdx.x) * chunk, e1 = std::min<int64_t>(cnt, e0 + chunk);
    for (int64_t e = e0 + threadIdx.x; e < e1; e += kGradNT) {
      const int64_t i = off + e * stride;
      grad_one(c[i], gy[i], t, th.hardness, gc ? gc + i : nullptr, acc);
    }
  } else {
    const int64_t off = 2 * n * l + n, cnt = n / 2;  // element pairs of D_{l+1}
    const int64_t chunk = (cnt + gridDim.x - 1) / gridDim.x;
    const int64_t e0 = int64_t(blockIdx.x) * chunk, e1 = std::min<int64_t>(cnt, e0 + chunk);
    for (int64_t e = e0 + threadIdx.x; e < e1; e += kGradNT) {
      const int64_t i = off + 2 * e;
      const V cv = *reinterpret_cast<const V*>(c + i);
      const V g = *reinterpret_cast<const V*>(gy + i);
      if (gc) {
        V o;
        grad_one(cv.x, g.x, t, th.hardness, &o.x, acc);
        grad_one(cv.y, g.y, t, th.hardness, &o.y, acc);
        *reinterpret_cast<V*>(gc + i) = o;
      } else {
        grad_one(cv.x, g.x, t, th.hardness, static_cast<T*>(nullptr), acc);
        grad_one(cv.y, g.y, t, th.hardness, static_cast<T*>(nullptr), acc);
      }
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  __shared__ double red[kGradNT / 64];
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0)
    partial[(sig * nl + (l - th.minlevel)) * int64_t(gridDim.x) + blockIdx.x] =
        (red[0] + red[1]) + (red[2] + red[3]);
}

// glam[l] = sum over signals and chunks of the level's partials (fixed
// order); zero outside [minlevel, maxlevel]
__global__ __launch_bounds__(kGradNT) void thresh_grad_reduce_k(const double* __restrict__ partial,
                                                                double* __restrict__ glam,
                                                                int64_t count, int nchunk,
                                                                int minlevel, int maxlevel) {
  const int l = blockIdx.x;
  __shared__ double red[kGradNT];
  double acc = 0.0;
  if (l >= minlevel && l <= maxlevel) {
    const int nl = maxlevel - minlevel + 1;
    const int64_t items = count * nchunk;
    for (int64_t k = threadIdx.x; k < items; k += kGradNT) {
      const int64_t sig = k / nchunk, ch = k % nchunk;
      acc += partial[(sig * nl + (l - minlevel)) * nchunk + ch];
    }
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int o = kGradNT / 2; o > 0; o >>= 1) {
    if (int(threadIdx.x) < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) glam[l] = red[0];
}

}  // namespace

int thresh_grad(const void* c, const void* gy, void* gc, double* glam, int64_t n, int64_t count,
                int J, int ttype, int dtype, const wh_thresh* thr, hipStream_t st) {
  if (count < 1 || count > 65535) return set_error(WH_ERR_ARG, "threshold gradient: signal count out of range");
  const size_t esz = dtype == WH_F32 ? 4 : 8;
  const int64_t per = (ttype == kDWT) ? n : 2 * n * J;
  // gc takes gy where the threshold does not act (scaling coefficients,
  // levels outside the range); without gc only glam is computed
  if (gc && gc != gy)
    WH_HIP_CHECK(hipMemcpyAsync(gc, gy, size_t(per) * size_t(count) * esz,
                                hipMemcpyDeviceToDevice, st));
  const int nl = thr->maxlevel - thr->minlevel + 1;
  // workgroups per (signal, level): at least kGradMinPer elements each, and
  // at most kGradMaxPartials partial sums in all
  const int64_t longest = ttype == kDWT ? n / 2 : n;
  const int64_t nchunk = std::max<int64_t>(
      1, std::min<int64_t>(longest / kGradMinPer, kGradMaxPartials / (count * nl)));
  void* p = nullptr;
  const size_t np = size_t(count) * size_t(nl) * size_t(nchunk);
  int rc = stats_get(np * sizeof(double), &p);
  if (rc) return rc;
  double* partial = static_cast<double*>(p);
  Thr1 th{thr->hardness, thr->minlevel, thr->maxlevel, thr->value, thr->levels};
  const dim3 grid{unsigned(nchunk), unsigned(nl), unsigned(count)};
  if (dtype == WH_F32)
    hipLaunchKernelGGL(thresh_grad_k<float>, grid, dim3(kGradNT), 0, st,
                       static_cast<const float*>(c), static_cast<const float*>(gy),
                       static_cast<float*>(gc), partial, n, J, ttype, th, gc ? 1 : 0);
  else
    hipLaunchKernelGGL(thresh_grad_k<double>, grid, dim3(kGradNT), 0, st,
                       static_cast<const double*>(c), static_cast<const double*>(gy),
                       static_cast<double*>(gc), partial, n, J, ttype, th, gc ? 1 : 0);
  WH_HIP_CHECK(hipGetLastError());
  if (glam) {
    hipLaunchKernelGGL(thresh_grad_reduce_k, dim3(unsigned(J)), dim3(kGradNT), 0, st, partial,
                       glam, count, int(nchunk), thr->minlevel, thr->maxlevel);
    WH_HIP_CHECK(hipGetLastError());
  }
  return WH_OK;
}

// ------------------------------------------------- mean squared error
namespace {

constexpr int kMsePer = 8;  // elements per thread, at least

// g = 2 (y - ref) / total (the order of operations of torch's mean of a
// square), and the workgroup's sum of (y - ref)^2 in 64 bits.  One read of
// each array and one write: bound by HBM.
template <typename T>
__global__ __launch_bounds__(256) void mse_k(const T* y, const T* __restrict__ ref, T* g,
                                             int64_t total, double* __restrict__ partial) {
  const T inv = T(1) / T(total);
  double acc = 0.0;
  const int64_t stride = int64_t(gridDim.x) * 256;
  for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < total; i += stride) {
    const T d = y[i] - ref[i];
    acc += double(d) * double(d);
    g[i] = inv * (T(2) * d);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  __shared__ double red[4];
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) partial[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

__global__ __launch_bounds__(256) void mse_sum_k(const double* __restrict__ partial, int np,
                                                 int64_t total, double* out) {
  __shared__ double red[256];
  double acc = 0.0;
  for (int i = threadIdx.x; i < np; i += 256) acc += partial[i];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (int(threadIdx.x) < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = red[0] / double(total);
}

}  // namespace

int mse_grad(const void* y, const void* ref, void* g, int64_t total, int dtype, double* out,
             hipStream_t st) {
  const unsigned np =
      unsigned(std::max<int64_t>(1, std::min<int64_t>((total + 256 * kMsePer - 1) / (256 * kMsePer), 2048)));
  void* p = nullptr;
  int rc = stats_get(np * sizeof(double), &p);
  if (rc) return rc;
  double* partial = static_cast<double*>(p);
  if (dtype == WH_F32)
    hipLaunchKernelGGL(mse_k<float>, dim3(np), dim3(256), 0, st, static_cast<const float*>(y),
                       static_cast<const float*>(ref), static_cast<float*>(g), total, partial);
  else
    hipLaunchKernelGGL(mse_k<double>, dim3(np), dim3(256), 0, st, static_cast<const double*>(y),
                       static_cast<const double*>(ref), static_cast<double*>(g), total, partial);
  hipLaunchKernelGGL(mse_sum_k, dim3(1), dim3(256), 0, st, partial, int(np), total, out);
  WH_HIP_CHECK(hipGetLastError());
  return WH_OK;
}

}  // namespace wh
