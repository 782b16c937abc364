// wh_stats.h -- thresholding / statistics back ends shared by stats.hip and
// smooth.cpp.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/wavehip.h"
#include "wh_common.h"

namespace wh {

// per-level (or single) threshold handed to the in-place kernels
struct Thr1 {
  int hardness, minlevel, maxlevel;
  double value;
  const double* levels;  // device, one per level, or nullptr
};

// Values taking part in a median:
//   mode 0: base[off .. off+count)
//   mode 1: MODWT detail blocks 0..(count/n - 1): base[2 n b + n + i]
//   mode 2: DWT details of 0-based levels [lmin, lmax] (positions with
//           ctz in range and < J) of an n-long interleaved vector
struct SelSrc {
  const void* base;
  int mode;
  int64_t n;
  int64_t count;
  int64_t off;
  int lmin, lmax, J;
  int lgn;  // log2 n (set by select_median)
};

// device-resident selection state (select.hip); [2]: values, deviations
constexpr int kSelCandCap = 1 << 19;  // gathered keys it keeps
constexpr int kSelSample = 512;
constexpr int kSelEdges = 104;        // +- 4.6 standard deviations of the sample's middle
constexpr int kSelReplicas = 8;       // copies of the counters
constexpr int kSelPad = 16;           // a cache line of counters
constexpr int kSelBuckets = 2 * kSelEdges + 1;

struct SelState {
  double med;
  unsigned long long ncand[2][kSelReplicas * kSelPad];
  unsigned long long bins[2][kSelReplicas * kSelBuckets];
  unsigned long long hist[2][2048];
  uint64_t edges[2][kSelEdges];
  uint64_t sample[kSelSample];
  uint64_t cand[2][kSelCandCap];
};

constexpr int kMaxPartials = 1024;  // per candidate

// Golden-section search of the cross-validated threshold, kept on the device
// (reference src/thresh.cpp:296-330): the bracket t0 <= t1 <= t2 <= t3, the
// errors m1, m2 at t1, t2, the loop count, which point the pending
// evaluation is for (1: t1, 2: t2), evaluations consumed so far, and stop.
constexpr int kCvCandidates = 3;  // points a round evaluates at once, at most
struct CvState {
  double t0, t1, t2, t3, m1, m2;
  int iter, pending, nevals, stop;
};

// The points of the next round: the pending one, then the one the search
// visits after it -- t2 after the first t1; else one for each outcome of
// the comparison, right (m2 < m1) and left.
__device__ __forceinline__ void cv_points(const CvState& cs, double* p) {
#pragma clang fp contract(off)
  const double R = 0.61803399, C = 1. - R;
  p[0] = cs.pending == 2 ? cs.t2 : cs.t1;
  p[1] = cs.nevals > 0 ? R * cs.t2 + C * cs.t3 : cs.t2;
  p[2] = cs.nevals > 0 ? R * cs.t1 + C * cs.t0 : cs.t2;
}

// bracket [0, t3] and the first round's points (one thread)
__device__ inline void cv_start(CvState* out, double t3, double* levels, int J) {
#pragma clang fp contract(off)
  const double C = 1. - 0.61803399;
  const double tb = t3 / 2.;
  CvState cs{};
  cs.t2 = tb;
  cs.t1 = tb - C * (tb - 0.);
  cs.t3 = t3;
  cs.pending = 1;
  *out = cs;
  double p[kCvCandidates];
  cv_points(cs, p);
#pragma unroll
  for (int c = 0; c < kCvCandidates; ++c)
    for (int l = 0; l < J; ++l) levels[c * kCandLevels + l] = p[c];
}

// in-place threshold of `count` transformed signals (DWT: n apart, MODWT:
// 2nJ apart)
int threshold_inplace(void* c, int64_t n, int64_t count, int J, int ttype, int dtype,
                      const wh_thresh* thr, hipStream_t st);
// Median of the selection, or with `mad` 1.4826 times the median of the
// deviations from it, times `factor` when > 0; written to *out, and to
// levels[0..J) or, with cv, as the bracket of a search whose first point
// goes there (each where not null).
struct SelOut {
  double* out = nullptr;
  int mad = 0;
  double factor = 0.0;
  double* levels = nullptr;
  int J = 0;
  CvState* cv = nullptr;
};
int select_median(const SelSrc& s, int dtype, SelState* st, const SelOut& o, hipStream_t stream);
// Universal threshold (smooth.cpp): the MAD of the levels' details times the
// reference's factor, whose sqrt(2 ln n) comes from the host's C library so
// that it rounds like the reference
int univ_thresh_dev(const void* c, int64_t n, int J, int ttype, int dtype, int minlevel,
                    int maxlevel, SelState* sel, SelOut o, hipStream_t st);
// search state the CV error reduction advances (cs == nullptr: none)
struct CvArgs {
  CvState* cs = nullptr;
  double* levels = nullptr;
  int J = 0;
  double tol = 0.0;
  int cand = 1;  // candidates (ye, yo: halves of candidate c at c len; 1 or kCvCandidates)
};
// partial_buf: kMaxPartials per candidate
int interp_mse(const void* xn, const void* ye, const void* yo, int64_t len, int dtype,
               double* partial_buf, double* out, hipStream_t st, const CvArgs& cv = CvArgs{});
int split_halves(const void* x, void* e, void* o, int64_t len, int dtype, hipStream_t st);

}  // namespace wh
