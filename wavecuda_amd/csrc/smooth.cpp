// smooth.cpp -- forward transform -> threshold -> inverse on the GPU
// (reference src/rfunctions.cu:71-136 and src/thresh.cpp:170-342).
//
// The coefficient arrays stay on the device for the whole pipeline.  The
// threshold is applied inside the inverse transform as the details are
// read, so smoothing costs one forward and one inverse pass.  Cross
// validation follows the reference's CPU algorithm (src/thresh.cpp:203-342)
// step for step: the universal threshold of the full transform brackets a
// golden-section search over the threshold of the even/odd half-length
// transforms, each round costing one fused threshold+inverse launch over
// both halves and one interpolation-error reduction.  The search's scalar
// steps run on the device with the reference's arithmetic (cv_advance), so
// rounds follow one another without the host; the host reads the search
// state back only to learn how many more evaluations the loop is certain to
// make.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>

#include "wh_common.h"
#include "wh_internal.h"
#include "wh_stats.h"

namespace wh {

namespace {

// Longest signals whose search evaluates kCvCandidates points a round: the
// extra candidates run in workgroups the chip has to spare, and a round of
// two steps costs 33 us of kernels at n = 2^18 (LA8 MODWT, J = 10) where
// two rounds of one took 40 and four more launches; at n = 2^16 (D4 DWT) 18
// against 29.  A round of three needs half again the memory traffic of two
// steps, so where the halves fill the chip one point a round stays.  Whole calls,
// us, one point -> three: LA8 MODWT J = 10 FP64 2^18 428 -> 377, 2^19 569 -> 523,
// 2^20 816 -> 1122 (FP32 410 -> 364, 493 -> 468, 675 -> 905; Haar FP32 2^19 level at
// 424); LA8 DWT FP64 2^20 496 -> 426, 2^21 619 -> 538, 2^22 815 -> 790 but Haar 630
// -> 672, 2^23 1261 -> 1475.
constexpr int64_t kCvRoundMaxModwt = int64_t(1) << 19;
constexpr int64_t kCvRoundMaxDwt = int64_t(1) << 21;

struct StatsBuf {
  SelState sel;
  double partial[kCvCandidates * kMaxPartials];
  double vals[16];
  double levels[64];
  double cvlev[kCvCandidates * kCandLevels];  // a candidate's threshold of every level
  CvState cv;
};

int stats_buf(StatsBuf** out) {
  void* p = nullptr;
  int rc = stats_get(sizeof(StatsBuf), &p);
  if (rc) return rc;
  *out = static_cast<StatsBuf*>(p);
  return WH_OK;
}

int64_t coeff_len(int ttype, int64_t n, int J) { return ttype == kDWT ? n : 2 * n * J; }

int fwd(int ttype, const void* x, void* w, int64_t n, int64_t count, int J, int filt, int dtype,
        hipStream_t st) {
  return ttype == kDWT ? dwt_forward(x, w, n, count, J, filt, dtype, st)
                       : modwt_forward_details(x, w, n, count, J, filt, dtype, st);
}

int inv(int ttype, const void* w, void* x, int64_t n, int64_t count, int J, int filt, int dtype,
        const wh_thresh* thr, hipStream_t st, const Candidates& c = Candidates{}) {
  return ttype == kDWT ? dwt_inverse(w, x, n, count, J, filt, dtype, thr, st, c)
                       : modwt_inverse(w, x, n, count, J, filt, dtype, thr, st, c);
}

// Candidates the search will certainly evaluate from state `cs` on (not
// stopped): the pending one, then one more for every loop test that must
// pass -- the bracket narrows by R per step and t1 + t2 <= 2 t3, so
// |t3 - t0| R^j > 2 tol t3 (with a margin for rounding) keeps the loop going,
// as long as the iteration cap allows.
int cv_sure_evals(const CvState& cs, double tol) {
  const double R = 0.61803399, margin = 1. - 1e-6;
  double w = std::fabs(cs.t3 - cs.t0) * margin;
  const double lim = tol * 2. * cs.t3;
  int it = cs.iter + (cs.nevals >= 2 ? 1 : 0);
  int k = 1;
  while (k < 64 && it <= 50 && w > lim) {
    ++k;
    ++it;
    w *= R * margin;
  }
  return k;
}

int d2h(double* host, const double* dev, hipStream_t st) {
  WH_HIP_CHECK(hipMemcpyAsync(host, dev, sizeof(double), hipMemcpyDeviceToHost, st));
  WH_HIP_CHECK(hipStreamSynchronize(st));
  return WH_OK;
}

}  // namespace

// src/thresh.cpp:170-201 (with the time-ordered MODWT gathering detail
// blocks from level 0 whatever minlevel is, src/wavutils.cpp:711-717)
int univ_thresh_dev(const void* c, int64_t n, int J, int ttype, int dtype, int minlevel,
                    int maxlevel, SelState* sel, SelOut o, hipStream_t st) {
  SelSrc s{};
  s.base = c;
  s.n = n;
  double factor;
  if (ttype == kDWT) {
    if (minlevel == 0 && maxlevel == J - 1) {
      s.mode = 0;
      s.off = 1;
      s.count = n - 1;
      factor = std::sqrt(2. * std::log(double(n - 1)));
    } else {
      s.mode = 2;
      s.lmin = minlevel;
      s.lmax = maxlevel;
      s.J = J;
      s.count = 0;
      for (int l = minlevel; l <= maxlevel; ++l) s.count += n >> (l + 1);
      factor = std::sqrt(2. * std::log(double(n)));
    }
  } else {
    s.mode = 1;
    s.count = int64_t(maxlevel - minlevel + 1) * n;
    factor = std::sqrt(2. * std::log(double(n)));
  }
  o.mad = 1;
  o.factor = factor;
  return select_median(s, dtype, sel, o, st);
}

int smooth(void* x, int64_t n, int J, int ttype, int filt, int dtype, int threshtype,
           double* thresh, int hardness, int minlevel, int maxlevel, double tol,
           hipStream_t st) {
  const size_t esz = dtype == WH_F32 ? 4 : 8;
  StatsBuf* sb = nullptr;
  int rc = stats_buf(&sb);
  if (rc) return rc;
  if (minlevel < 0 || minlevel > maxlevel || maxlevel >= J)
    return set_error(WH_ERR_ARG, "levels must satisfy 0 <= minlevel <= maxlevel < nlevels");
  if (hardness != kHARD && hardness != kSOFT) return set_error(WH_ERR_ARG, "hardness must be 0 or 1");

  if (threshtype == 0 || threshtype == 1) {  // MANUAL / UNIV
    void* w = nullptr;
    if ((rc = ws_get(size_t(coeff_len(ttype, n, J)) * esz, &w))) return rc;
    if ((rc = fwd(ttype, x, w, n, 1, J, filt, dtype, st))) return rc;
    wh_thresh t{};
    t.enabled = 1;
    t.hardness = hardness;
    t.minlevel = minlevel;
    t.maxlevel = maxlevel;
    if (threshtype == 0) {
      if (!thresh) return set_error(WH_ERR_ARG, "manual threshold needs a value");
      t.value = *thresh;
    } else {
      // univ_thresh(w, 0, 0) (src/rfunctions.cu:82-87)
      SelOut o;
      o.out = &sb->vals[0];
      o.levels = sb->levels;
      o.J = J;
      if ((rc = univ_thresh_dev(w, n, J, ttype, dtype, 0, 0, &sb->sel, o, st))) return rc;
      t.levels = sb->levels;
    }
    if ((rc = inv(ttype, w, x, n, 1, J, filt, dtype, &t, st))) return rc;
    if (threshtype == 1 && thresh) {
      if ((rc = d2h(thresh, &sb->vals[0], st))) return rc;
    } else {
      WH_HIP_CHECK(hipStreamSynchronize(st));
    }
    return WH_OK;
  }
  if (threshtype != 2) return set_error(WH_ERR_ARG, "threshtype must be 0 (manual), 1 (univ) or 2 (cv)");

  // ---- cross validation (src/thresh.cpp:203-342)
  if (J <= 1) return set_error(WH_ERR_ARG, "cross validation needs at least two levels");
  if (minlevel == maxlevel)
    return set_error(WH_ERR_ARG, "cross validation needs minlevel < maxlevel");
  const int64_t lenh = n / 2;
  const int Jh = J - 1;
  const int64_t cw = coeff_len(ttype, n, J), ch = coeff_len(ttype, lenh, Jh);
  void* ws = nullptr;
  // Candidates per round: a round of three (the pending point and the one
  // that follows it either way) takes two steps of the search.
  const int cand = n <= (ttype == kDWT ? kCvRoundMaxDwt : kCvRoundMaxModwt) ? kCvCandidates : 1;
  const size_t bytes = size_t(cw + 2 * ch + (2 + 2 * cand) * lenh) * esz + 256;
  if ((rc = ws_get(bytes, &ws))) return rc;
  char* p = static_cast<char*>(ws);
  void* W = p;
  p += cw * esz;
  void* We = p;
  p += 2 * ch * esz;  // and the odd half's
  void* xe = p;
  p += lenh * esz;
  void* xo = p;
  p += lenh * esz;
  void* ye = p;
  p += lenh * esz;
  void* yo = p;

  if ((rc = fwd(ttype, x, W, n, 1, J, filt, dtype, st))) return rc;
  SelOut o;
  o.levels = sb->cvlev;
  o.J = Jh;
  o.cv = &sb->cv;
  if ((rc = univ_thresh_dev(W, n, J, ttype, dtype, minlevel, maxlevel, &sb->sel, o, st))) return rc;
  if ((rc = split_halves(x, xe, xo, n, dtype, st))) return rc;
  // the two half-length transforms run as one two-signal launch (xe, xo and
  // We, Wo and ye, yo are adjacent): twice the workgroups, half the launches
  if ((rc = fwd(ttype, xe, We, lenh, 2, Jh, filt, dtype, st))) return rc;

  // one round: the halves thresholded at every candidate cv_points wrote
  wh_thresh th{};
  th.enabled = 1;
  th.hardness = hardness;
  th.minlevel = minlevel;
  th.maxlevel = maxlevel - 1;
  th.levels = sb->cvlev;
  CvArgs cva;
  cva.cs = &sb->cv;
  cva.levels = sb->cvlev;
  cva.J = Jh;
  cva.tol = tol;
  cva.cand = cand;
  Candidates points;
  points.count = cand;
  auto eval = [&]() -> int {
    const int r = inv(ttype, We, ye, lenh, 2, Jh, filt, dtype, &th, st, points);
    if (r) return r;
    // the error reduction's last block also advances the search
    return interp_mse(x, ye, yo, n, dtype, sb->partial, nullptr, st, cva);
  };
  // the tests the first bracket [0, t3] is sure to pass do not depend on t3
  CvState cs{};
  cs.t3 = 1.;
  for (;;) {
    const int sure = cv_sure_evals(cs, tol);
    for (int i = 0; i < sure; i += cand == 1 ? 1 : 2)
      if ((rc = eval())) return rc;
    WH_HIP_CHECK(hipMemcpyAsync(&cs, &sb->cv, sizeof(CvState), hipMemcpyDeviceToHost, st));
    WH_HIP_CHECK(hipStreamSynchronize(st));
    if (cs.stop) break;
  }
  const double t1 = cs.t1, t2 = cs.t2, m1 = cs.m1, m2 = cs.m2;
  double t = m1 < m2 ? t1 : t2;
  t = t / (std::sqrt(1. - std::log(2.) / std::log(double(n))));
  wh_thresh tf{};
  tf.enabled = 1;
  tf.hardness = hardness;
  tf.minlevel = minlevel;
  tf.maxlevel = maxlevel;
  tf.value = t;
  if ((rc = inv(ttype, W, x, n, 1, J, filt, dtype, &tf, st))) return rc;
  WH_HIP_CHECK(hipStreamSynchronize(st));
  if (thresh) *thresh = t;
  return WH_OK;
}

}  // namespace wh
