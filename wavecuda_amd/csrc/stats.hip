// stats.hip -- thresholding and the smoothing statistics (gfx950).
//
//  * in-place hard/soft thresholding of DWT / MODWT details
//    (reference src/thresh.cpp:15-83, :142-157);
//  * the CV interpolation error (reference src/thresh.cpp:344-384) as a
//    fixed-order two-stage reduction, so repeated runs are bit-identical.
#include <algorithm>
#include <cmath>
#include <mutex>

#include "wh_common.h"
#include "wh_internal.h"
#include "wh_stats.h"

namespace wh {

// ---------------------------------------------------------------- threshold
template <typename T>
__global__ void thresh_dwt_kernel(T* __restrict__ y0, int64_t n, int J, Thr1 th) {
  T* y = y0 + int64_t(blockIdx.y) * n;
  const int64_t stride = int64_t(gridDim.x) * blockDim.x;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) {
    if (i == 0) continue;
    const int l = __builtin_ctzll(uint64_t(i));  // detail of 0-based level l
    if (l >= J || l < th.minlevel || l > th.maxlevel) continue;
    const T t = th.levels ? T(th.levels[l]) : T(th.value);
    y[i] = thresh_coef(y[i], t, th.hardness);
  }
}

template <typename T>
__global__ void thresh_modwt_kernel(T* __restrict__ xmod0, int64_t n, int J, Thr1 th) {
  T* xmod = xmod0 + int64_t(blockIdx.y) * 2 * n * J;
  const int64_t cnt = int64_t(th.maxlevel - th.minlevel + 1) * n;
  const int64_t stride = int64_t(gridDim.x) * blockDim.x;
  for (int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; e < cnt; e += stride) {
    const int l = th.minlevel + int(e / n);
    const int64_t i = 2 * n * l + n + (e - int64_t(l - th.minlevel) * n);
    const T t = th.levels ? T(th.levels[l]) : T(th.value);
    xmod[i] = thresh_coef(xmod[i], t, th.hardness);
  }
}

int threshold_inplace(void* c, int64_t n, int64_t count, int J, int ttype, int dtype,
                      const wh_thresh* thr, hipStream_t st) {
  Thr1 th{thr->hardness, thr->minlevel, thr->maxlevel, thr->value, thr->levels};
  const int nt = 256;
  if (count < 1 || count > 65535) return set_error(WH_ERR_ARG, "threshold: signal count out of range");
  const int64_t work = (ttype == kDWT) ? n : int64_t(thr->maxlevel - thr->minlevel + 1) * n;
  const unsigned blocks = unsigned(std::min<int64_t>((work + nt - 1) / nt, 4096));
  const dim3 grid(blocks, unsigned(count));
  if (ttype == kDWT) {
    if (dtype == WH_F32)
      hipLaunchKernelGGL(thresh_dwt_kernel<float>, grid, dim3(nt), 0, st,
                         static_cast<float*>(c), n, J, th);
    else
      hipLaunchKernelGGL(thresh_dwt_kernel<double>, grid, dim3(nt), 0, st,
                         static_cast<double*>(c), n, J, th);
  } else {
    if (dtype == WH_F32)
      hipLaunchKernelGGL(thresh_modwt_kernel<float>, grid, dim3(nt), 0, st,
                         static_cast<float*>(c), n, J, th);
    else
      hipLaunchKernelGGL(thresh_modwt_kernel<double>, grid, dim3(nt), 0, st,
                         static_cast<double*>(c), n, J, th);
  }
  WH_HIP_CHECK(hipGetLastError());
  return WH_OK;
}

// ------------------------------------------------- cross-validation search
// The scalar steps of the reference's golden-section loop
// (src/thresh.cpp:296-330), with products and sums rounded separately as
// in its host build, so the visited thresholds are the same doubles: take
// the error m of the pending point and advance the bracket.
__device__ __forceinline__ void cv_advance(CvState* cs, double m, double tol) {
#pragma clang fp contract(off)
  if (cs->stop) return;
  const double R = 0.61803399, C = 1. - R;
  if (cs->pending == 1)
    cs->m1 = m;
  else
    cs->m2 = m;
  const int ne = ++cs->nevals;
  if (ne == 1) {  // the first two evaluations: t1, then t2
    cs->pending = 2;
    return;
  }
  if (ne > 2) cs->iter++;  // the loop body that ordered this evaluation ends
  if (!(fabs(cs->t3 - cs->t0) > tol * (cs->t1 + cs->t2)) || cs->iter > 50) {
    cs->stop = 1;
    return;
  }
  if (cs->m2 < cs->m1) {
    cs->t0 = cs->t1;
    cs->t1 = cs->t2;
    cs->t2 = R * cs->t2 + C * cs->t3;
    cs->m1 = cs->m2;
    cs->pending = 2;
  } else {
    cs->t3 = cs->t2;
    cs->t2 = cs->t1;
    cs->t1 = R * cs->t1 + C * cs->t0;
    cs->m2 = cs->m1;
    cs->pending = 1;
  }
}

// --------------------------------------------------------- interp_mse
template <typename T>
__global__ __launch_bounds__(256) void interp_mse_partial(const T* __restrict__ xn,
                                                          const T* __restrict__ ye,
                                                          const T* __restrict__ yo, int64_t len,
                                                          int64_t per_block, double* partial) {
  __shared__ double red[256];
  const int64_t lenh = len / 2;
  ye += int64_t(blockIdx.y) * len;  // a candidate's halves are adjacent
  yo += int64_t(blockIdx.y) * len;
  partial += int64_t(blockIdx.y) * kMaxPartials;
  const int64_t j0 = int64_t(blockIdx.x) * per_block;
  const int64_t j1 = std::min(lenh, j0 + per_block);
  double acc = 0.0;
  for (int64_t j = j0 + threadIdx.x; j < j1; j += blockDim.x) {
    const int64_t i = 2 * j;
    double yie, yio;
    if (i == 0) {
      yie = double(yo[0]);
      yio = 0.5 * (double(ye[0]) + double(ye[1]));
    } else if (i == len - 2) {
      yio = double(ye[lenh - 1]);
      yie = 0.5 * (double(yo[j]) + double(yo[j - 1]));
    } else {
      yio = 0.5 * (double(ye[j]) + double(ye[j + 1]));
      yie = 0.5 * (double(yo[j]) + double(yo[j - 1]));
    }
    const double a = yie - double(xn[i]), b = yio - double(xn[i + 1]);
    acc += a * a + b * b;
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if (threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// The sums of every candidate's partials (256 threads each), then the
// search's steps: the first candidate is the pending point, and with three
// the others follow it either way (cv_points), so the search takes two.  The
// state is fetched beside the partials and stepped in registers by one
// thread; the points go out in parallel (4.8 -> 3.1 us against stepping it
// in memory).
__global__ __launch_bounds__(256 * kCvCandidates) void sum_partials(const double* partial, int np,
                                                                   double scale, double* out,
                                                                   CvArgs cv) {
  __shared__ double sums[kCvCandidates][256];
  __shared__ double pts[kCvCandidates];
  const int c = threadIdx.x >> 8, t = threadIdx.x & 255;
  double* red = sums[c];
  CvState cs{};
  if (threadIdx.x == 0 && cv.cs) cs = *cv.cs;
  double acc = 0.0;
  for (int i = t; i < np; i += 256) acc += partial[c * kMaxPartials + i];
  red[t] = acc;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if (t < off) red[t] += red[t + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    if (out) *out = red[0] * scale;
    if (cv.cs) {
      cv_advance(&cs, red[0] * scale, cv.tol);
      if (cv.cand == kCvCandidates && !cs.stop)
        cv_advance(&cs, sums[cs.pending == 2 ? 1 : 2][0] * scale, cv.tol);
      *cv.cs = cs;
      cv_points(cs, pts);
    }
  }
  if (!cv.cs) return;
  __syncthreads();
  for (int i = threadIdx.x; i < cv.J * kCvCandidates; i += blockDim.x)
    cv.levels[(i / cv.J) * kCandLevels + i % cv.J] = pts[i / cv.J];
}

int interp_mse(const void* xn, const void* ye, const void* yo, int64_t len, int dtype,
               double* partial_buf, double* out, hipStream_t st, const CvArgs& cv) {
  const int64_t lenh = len / 2;
  const int64_t per_block = 512;
  const int np = int(std::min<int64_t>((lenh + per_block - 1) / per_block, kMaxPartials));
  const int64_t pb = (lenh + np - 1) / np;
  const dim3 grid{unsigned(np), unsigned(cv.cand)};
  if (dtype == WH_F32)
    hipLaunchKernelGGL(interp_mse_partial<float>, grid, dim3(256), 0, st,
                       static_cast<const float*>(xn), static_cast<const float*>(ye),
                       static_cast<const float*>(yo), len, pb, partial_buf);
  else
    hipLaunchKernelGGL(interp_mse_partial<double>, grid, dim3(256), 0, st,
                       static_cast<const double*>(xn), static_cast<const double*>(ye),
                       static_cast<const double*>(yo), len, pb, partial_buf);
  hipLaunchKernelGGL(sum_partials, dim3(1), dim3(256 * cv.cand), 0, st, partial_buf, np, 0.5, out,
                     cv);
  WH_HIP_CHECK(hipGetLastError());
  return WH_OK;
}

// ------------------------------------------------------------- helpers
template <typename T>
__global__ void split_even_odd(const T* __restrict__ x, T* __restrict__ e, T* __restrict__ o,
                               int64_t lenh) {
  const int64_t stride = int64_t(gridDim.x) * blockDim.x;
  for (int64_t j = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; j < lenh; j += stride) {
    e[j] = x[2 * j];
    o[j] = x[2 * j + 1];
  }
}

int split_halves(const void* x, void* e, void* o, int64_t len, int dtype, hipStream_t st) {
  const int64_t lenh = len / 2;
  const unsigned blocks = unsigned(std::max<int64_t>(1, std::min<int64_t>((lenh + 255) / 256, 4096)));
  if (dtype == WH_F32)
    hipLaunchKernelGGL(split_even_odd<float>, dim3(blocks), dim3(256), 0, st,
                       static_cast<const float*>(x), static_cast<float*>(e),
                       static_cast<float*>(o), lenh);
  else
    hipLaunchKernelGGL(split_even_odd<double>, dim3(blocks), dim3(256), 0, st,
                       static_cast<const double*>(x), static_cast<double*>(e),
                       static_cast<double*>(o), lenh);
  WH_HIP_CHECK(hipGetLastError());
  return WH_OK;
}

}  // namespace wh
