// prior_math.h -- log incomplete gamma functions and the analytic
// integrals of the genealogy prior over uniform priors on population size
// and migration rate (integrate_coalescent_term / integrate_migration_term,
// update_gtree_common.cpp:109-296).
//
// The incomplete gammas follow the published Numerical Recipes methods the
// reference uses (utilities.cpp:812-1122): series for x < a + 1, continued
// fraction otherwise, relative tolerance 3e-7, at most 1000 terms; E_1 by
// its series (x <= 1) or continued fraction (at most 100 terms).  The
// termination rules decide the value to ~3e-7, so they are kept as they
// are.  The functions take lga = log Gamma(a) = log((a-1)!) for their order
// a; callers read it from `lf`, a table built on the host as the running sum
// of log(i), as the reference's setlogfact builds it.  Everything is FP64.
// The batch prior kernels compile these without floating-point contraction,
// so sums round as written.
//
// Bound: latency.  In the sweep's accept step a wavefront evaluates one
// parameter's integral for 63 scenarios, three wavefronts a SIMD: about 450
// dependent FP64 instructions with the library's logarithm (60, 3 to 5 uses),
// exponential (40) and division (15, two a term of the fraction), 2.4 to 4.5
// us.  So: logarithm, exponential and division below in 32, 24 and 8
// instructions, the fraction and the series as numerator and denominator
// recurrences with one division at the end, and the logarithms of the weight
// and of the gamma's argument side by side.  The argument's could be pieced
// together from the weight's and the bound's, and the logarithm take five
// instructions less: 2.2 to 3.4 us, and 107 us for the accept launch of 64
// chains x 50 loci instead of 110, but two coalescences over [0, 20] then
// integrate with 0.52 ulp root mean square instead of 0.44.
#pragma once

#include <hip/hip_runtime.h>

#include "ima_internal.h"

namespace ima {

constexpr double kPriEps = 3.0e-7;
constexpr int kPriItmax = 1000;
constexpr double kLog2 = 0.69314718055994530941723212146;

// n / d, d in the normal range and well inside it: the reciprocal estimate,
// two Newton steps, one correction of the quotient.
__device__ __forceinline__ double pri_div(double n, double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = fma(fma(-d, r, 1.0), r, r);
  r = fma(fma(-d, r, 1.0), r, r);
  const double q = n * r;
  return fma(fma(-d, q, n), r, q);
}

// log x.  x = m 2^e with m in [sqrt(1/2), sqrt 2), f = m - 1 (exact), s = f /
// (2 + f): log m = 2 atanh(s) = f - (f^2/2 - s (f^2/2 + R)), R = 2 (atanh(s) /
// s - 1) by a polynomial in s^2 (interpolation of atanh(s) / s at Chebyshev
// nodes, 5e-18 relative), so that what is rounded is small beside f; e ln 2 +
// f is added as a sum and its rest.  Within 0.87 ulp of the logarithm, 0.295
// root mean square (the library's: 0.293; 2 atanh(s) itself, rounded in s:
// 1.98 and 0.46).  No branches and no call of the library: at the integrals'
// many uses either would fill the instruction cache.
__device__ __forceinline__ double pri_log(double x) {
#pragma clang fp contract(off)
  double m = __builtin_amdgcn_frexp_mant(x);
  int e = __builtin_amdgcn_frexp_exp(x);
  const bool lo = m < 0.70710678118654752440;
  m = lo ? m + m : m;
  e = lo ? e - 1 : e;
  const double f = m - 1.0, d = 2.0 + f, h = 0.5 * f * f;
  double q = __builtin_amdgcn_rcp(d);
  q = fma(fma(-d, q, 1.0), q, q);
  q = fma(fma(-d, q, 1.0), q, q);
  const double s = f * q, z = s * s;
  double p = 0.14616449685043406;
  p = fma(p, z, 0.15331721600556042);
  p = fma(p, z, 0.1818288912526122);
  p = fma(p, z, 0.2222221113479488);
  p = fma(p, z, 0.28571428625986754);
  p = fma(p, z, 0.39999999999899504);
  p = fma(p, z, 0.666666666666667);
  // ln 2 in two parts, the first of 32 bits: e times it is exact
  const double k = e, a = fma(k, 6.93147180369123816490e-01, f);
  const double b = fma(k, 6.93147180369123816490e-01, -a) + f;
  const double r = a + (fma(s, fma(z, p, h), fma(k, 1.90821492927058770002e-10, b)) - h);
  // 0, infinity, negative numbers and NaN
  const double odd = x == 0.0 ? -INFINITY : x > 0.0 ? x : NAN;
  return x > 0.0 && x < INFINITY ? r : odd;
}

// e^x = 2^n e^r, r = x - n ln 2 through the two parts of ln 2 with the
// rounding of the second kept, 1 + r added as a sum and its rest: within 0.75
// ulp, 0.293 root mean square (the library's: 0.86 and 0.302; r rounded once
// and 1 + r p(r) for the end: 0.93 and 0.304).  0 and infinity beyond the
// range come from the scaling, NaN passes through.
__device__ __forceinline__ double pri_exp(double x) {
#pragma clang fp contract(off)
  x = x > 1e5 ? 1e5 : x < -1e5 ? -1e5 : x;
  const double n = rint(x * 1.4426950408889634074);
  const double hi = fma(-n, 6.93147180369123816490e-01, x);
  const double r = fma(-n, 1.90821492927058770002e-10, hi);
  const double c = fma(-n, 1.90821492927058770002e-10, hi - r);
  // e^r on [-ln 2 / 2, ln 2 / 2], interpolated at the Chebyshev nodes: 2e-17
  // relative
  double p = 2.5110037605963777e-08;
  p = fma(p, r, 2.763263963904103e-07);
  p = fma(p, r, 2.755724091857897e-06);
  p = fma(p, r, 2.4801485482328494e-05);
  p = fma(p, r, 0.00019841269890047113);
  p = fma(p, r, 0.0013888888952314775);
  p = fma(p, r, 0.008333333333319601);
  p = fma(p, r, 0.0416666666664881);
  p = fma(p, r, 0.1666666666666668);
  p = fma(p, r, 0.5000000000000019);
  const double a = 1.0 + r, b = (1.0 - a) + r;
  return ldexp(a + (b + fma(r * r, p, c)), (int)n);
}

// The continued fraction h = 1 / (b_0 + a_1 / (b_1 + a_2 / ...)) with b_i =
// b_0 + 2 i as q / p by the forward recurrences.  All quantities are
// positive here (for the upper gamma of whole order a and x > a the partial
// numerators i (a - i) are positive until the one that ends it; E_1's
// convergents are positive).  They are scaled down together by a power of
// two, exactly.  The convergent is the one Lentz's method stops at: |del -
// 1| < EPS, tested on the products.  Beyond b_0 = 2^100 the first term ends
// the fraction (its partial numerator is below 2^31).
constexpr double kPriBig = 0x1p250, kPriDown = 0x1p-250;
__device__ inline double pri_fraction(double a, double b, int itmax) {
  if (!(b < 0x1p100)) return 1.0 / b;
  double p1 = 1.0, q1 = 0.0, p = b, q = 1.0;
  for (int i = 1; i <= itmax; i++) {
    const double an = -i * (i - a);
    b += 2.0;
    const double pn = fma(b, p, an * p1), qn = fma(b, q, an * q1);
    const double s = qn * p, t = pn * q;
    p1 = p;
    q1 = q;
    p = pn;
    q = qn;
    if (fabs(s - t) < kPriEps * t) break;  // del = s / t
    if (p > kPriBig) {
      p *= kPriDown;
      q *= kPriDown;
      p1 *= kPriDown;
      q1 *= kPriDown;
    }
  }
  return pri_div(q, p);
}

// lx = log x throughout
__device__ inline double pri_gcf(double a, double x, double lx, double lga, double *gln,
                                 double *h_out) {
  *gln = lga;
  *h_out = pri_fraction(a, x + 1.0 - a, kPriItmax);
  return -x + a * lx - (*gln);
}

// series: returns the sum and the log prefactor -x + a log x - log Gamma(a)
__device__ inline double pri_gser(int a, double x, double lx, double lga, double *gln,
                                  double *pre) {
  *gln = lga;
  *pre = 0.0;
  if (x <= 0.0) return 0.0;
  // sum = s / d after n terms, d = a (a + 1) .. (a + n), the last x^n / d
  double ap = a, d = a, s = 1.0, xn = 1.0;
  for (int n = 1; n <= kPriItmax; n++) {
    ++ap;
    xn *= x;
    d *= ap;
    s = fma(s, ap, xn);
    if (xn < s * kPriEps) break;
    if (d > kPriBig || s > kPriBig) {
      xn *= kPriDown;
      d *= kPriDown;
      s *= kPriDown;
    }
  }
  *pre = -x + a * lx - (*gln);
  return pri_div(s, d);
}

// E_1(x) or its log (*islog)
__device__ inline double pri_expint1(double x, int *islog) {
  const double euler = 0.5772156649;
  *islog = 0;
  if (x > 1.0) {
    *islog = 1;
    return pri_log(pri_fraction(0.0, x + 1.0, 100)) - x;
  }
  double ans = -pri_log(x) - euler, fact = 1.0;
  for (int i = 1; i <= 100; i++) {
    fact *= -x / i;
    const double del = -fact / (i - 0);
    ans += del;
    if (fabs(del) < fabs(ans) * kPriEps) break;
  }
  return ans;
}

__device__ inline double pri_uppergamma(int a, double x, double lga) {
  double gln, p;
  if (a == 0) {
    int islog;
    const double t = pri_expint1(x, &islog);
    p = islog ? t : pri_log(t);
  } else if (x < (a + 1.0)) {
    double pre;
    const double s = pri_gser(a, x, pri_log(x), lga, &gln, &pre);
    const double g = (x <= 0.0) ? 0.0 : s * pri_exp(pre);
    p = gln + pri_log(1.0 - g);
  } else {
    double h;
    const double pre = pri_gcf((double)a, x, pri_log(x), lga, &gln, &h);
    p = gln + (pre + pri_log(h));
  }
  if (p < -1e200) p = -1e200;
  return p;
}

__device__ inline double pri_lowergamma(int a, double x, double lga) {
  double gln, p;
  if (x < (a + 1.0)) {
    double pre;
    const double s = pri_gser(a, x, pri_log(x), lga, &gln, &pre);
    const double g = (x <= 0.0) ? 0.0 : pri_log(s) + pre;
    p = gln + g;
  } else {
    double h;
    const double pre = pri_gcf((double)a, x, pri_log(x), lga, &gln, &h);
    p = gln + pri_log(1 - pri_exp(pre) * h);
  }
  if (p < -1e200) p = -1e200;
  return p;
}

// Both log incomplete gammas of one (a, x) share their series or continued
// fraction: run it once, then pri_upper_of / pri_lower_of give exactly the
// values pri_uppergamma / pri_lowergamma would (a >= 1).
struct GammaPrep {
  bool series;
  double sum_or_h, pre, gln, x;
};
__device__ inline GammaPrep pri_gamma_prep(int a, double x, double lx, double lga) {
  GammaPrep g;
  g.x = x;
  g.series = x < (a + 1.0);
  if (g.series)
    g.sum_or_h = pri_gser(a, x, lx, lga, &g.gln, &g.pre);
  else
    g.pre = pri_gcf((double)a, x, lx, lga, &g.gln, &g.sum_or_h);
  return g;
}
__device__ inline double pri_upper_of(const GammaPrep &g) {
  double p;
  if (g.series) {
    const double gg = (g.x <= 0.0) ? 0.0 : g.sum_or_h * pri_exp(g.pre);
    p = g.gln + pri_log(1.0 - gg);
  } else {
    p = g.gln + (g.pre + pri_log(g.sum_or_h));
  }
  return p < -1e200 ? -1e200 : p;
}
__device__ inline double pri_lower_of(const GammaPrep &g) {
  double p;
  if (g.series) {
    const double gg = (g.x <= 0.0) ? 0.0 : pri_log(g.sum_or_h) + g.pre;
    p = g.gln + gg;
  } else {
    p = g.gln + pri_log(1 - pri_exp(g.pre) * g.sum_or_h);
  }
  return p < -1e200 ? -1e200 : p;
}

// log(e^a - e^b) for a > b (LogDiff, imamp.hpp:257-263)
__device__ inline double pri_logdiff(double a, double b) {
  if (a - b < 7.0978271289338397e+02) return b + pri_log(pri_exp(a - b) - 1.0);
  return a;
}

// log int_min^max (2/t)^cc e^(-2 fc/t - hcc) dt; lga = log((cc-2)!), lmax =
// log max
__device__ inline double pri_coalescent_term(int cc, double fc, double hcc, double max,
                                             double min, double lga, double lmax) {
  double p;
  if (cc > 0) {
    if (min == 0) {
      // cc = 1: order 0, the exponential integral; else one series serves
      // both gammas
      GammaPrep gp{};
      const double x = 2 * fc / max, lfc = pri_log(fc), lx = pri_log(x);
      if (cc > 1) gp = pri_gamma_prep(cc - 1, x, lx, lga);
      double ug = cc > 1 ? pri_upper_of(gp) : pri_uppergamma(0, 2 * fc / max, lga);
      if (cc > 1) {
        const double fullg = lga;
        if (fullg - ug < 1e-15 || fullg - ug > 7.0978271289338397e+02) {
          const double lg = pri_lower_of(gp);
          if (fullg > lg) {
            const double ugalt = pri_logdiff(fullg, lg);
            if (fabs(ugalt - ug) > 1e-10) ug = ugalt;
          }
        }
      }
      p = ug + kLog2 - hcc + (1 - cc) * lfc;
    } else {
      const double a = pri_uppergamma(cc - 1, 2 * fc / max, lga);
      const double b = pri_uppergamma(cc - 1, 2 * fc / min, lga);
      p = pri_logdiff(a, b) + (kLog2 - hcc + (1 - cc) * pri_log(fc));
    }
  } else if (2 * fc / max > 0) {
    if (min == 0) {
      const double a = lmax - 2.0 * fc / max;
      const double b = kLog2 + pri_log(fc) + pri_uppergamma(0, 2.0 * fc / max, 0.0);
      p = pri_logdiff(a, b);
    } else {
      double a = pri_uppergamma(0, 2 * fc / max, 0.0), b = pri_uppergamma(0, 2 * fc / min, 0.0);
      const double c = pri_logdiff(a, b) + kLog2 + log(fc);
      a = log(max) - 2.0 * fc / max;
      b = log(min) - 2.0 * fc / min;
      p = pri_logdiff(pri_logdiff(a, b), c);
    }
  } else {
    p = log(max - min);
  }
  return p;
}

// log int_min^max m^cm e^(-fm m) dm; lga = log(cm!)
__device__ inline double pri_migration_term(int cm, double fm, double max, double min,
                                            double lga) {
  const double mpriormin = 0.000001;  // MPRIORMIN, imamp.hpp:141
  double p;
  if (cm > 0) {
    if (min == 0) {
      const double lfm = pri_log(fm), lx = pri_log(fm * max);
      const GammaPrep gp = pri_gamma_prep(cm + 1, fm * max, lx, lga);
      double lg = pri_lower_of(gp);
      const double fullg = lga;
      if (fullg - lg < 1e-15 || fullg - lg > 7.0978271289338397e+02) {
        const double ug = pri_upper_of(gp);
        if (fullg > ug) {
          const double lgalt = pri_logdiff(fullg, ug);
          if (fabs(lgalt - lg) > 1e-12) lg = lgalt;
        }
      }
      p = (-1 - cm) * lfm + lg;
    } else {
      const double a = pri_uppergamma(cm + 1, fm * min, lga);
      const double b = pri_uppergamma(cm + 1, fm * max, lga);
      p = (-1 - cm) * pri_log(fm) + pri_logdiff(a, b);
    }
  } else if (fm > mpriormin) {
    if (min == 0)
      p = (max == mpriormin) ? 0.0 : pri_logdiff(0.0, -fm * max) - pri_log(fm);
    else
      p = pri_logdiff(-fm * min, -fm * max) - log(fm);
  } else {
    p = log(max - min);
  }
  return p;
}

// Count, weight and hcc sums of parameter t (population sizes first, then
// migration rates) over its (period, position) entries of a weight record,
// in parameter-map order (integrate_tree_prob's loops).
// get(r) returns record entry r.
template <typename Get>
__device__ inline void prior_param_sums_of(const ModelView &md, int P, int npsize, int t,
                                           const Get &get, int *c, double *f, double *h) {
  int cc = 0;
  double ff = 0.0, hh = 0.0;
  if (t < npsize) {
    for (int w = md.theta_off[t]; w < md.theta_off[t + 1]; ++w) {
      const int kk = md.theta_wp[2 * w], ii = md.theta_wp[2 * w + 1];
      cc += (int)get(kk * P + ii);
      ff += get(P * P + kk * P + ii);
      hh += get(2 * P * P + kk * P + ii);
    }
  } else {
    const int m = t - npsize;
    for (int w = md.mig_off[m]; w < md.mig_off[m + 1]; ++w) {
      const int kk = md.mig_wp[3 * w], ii = md.mig_wp[3 * w + 1], jj = md.mig_wp[3 * w + 2];
      cc += (int)get(3 * P * P + (kk * P + ii) * P + jj);
      ff += get(3 * P * P + P * P * P + (kk * P + ii) * P + jj);
    }
  }
  *c = cc;
  *f = ff;
  *h = hh;
}

__device__ inline void prior_param_sums(const ModelView &md, int P, int npsize, int t,
                                        const double *rec, int *c, double *f, double *h) {
  prior_param_sums_of(md, P, npsize, t, [rec](int r) { return rec[r]; }, c, f, h);
}

// log Gamma of the incomplete gamma order parameter t's integral uses at
// count c: log((c-2)!) for a population size (no gamma below c = 2),
// log(c!) for a migration rate.
__device__ inline double prior_param_lga(int npsize, int t, int c, const double *lf) {
  return t < npsize ? (c >= 2 ? lf[c - 2] : 0.0) : lf[c];
}

// The analytic integral of parameter t at those sums (uniform prior on
// [0, qmax] / [0, mmax]), given prior_param_lga and the log of its bound.
__device__ inline double prior_param_bound(const ModelView &md, int npsize, int t) {
  return t < npsize ? md.qmax[t] : md.mmax[t - npsize];
}
// A function of its own: about 900 instructions that the accept step calls
// from two places.
static __device__ __attribute__((noinline)) double prior_param_term_lga(int npsize, int t, int c, double f, double h,
                                              double lga, double max, double lmax) {
  return t < npsize ? pri_coalescent_term(c, f, h, max, 0.0, lga, lmax)
                    : pri_migration_term(c, f, max, 0.0, lga);
}

__device__ inline double prior_param_term(const ModelView &md, int npsize, int t, int c,
                                          double f, double h, const double *lf) {
  const double max = prior_param_bound(md, npsize, t);
  return prior_param_term_lga(npsize, t, c, f, h, prior_param_lga(npsize, t, c, lf), max,
                              pri_log(max));
}

// sum_{i < n} rec[i * stride + r] in order, with eight loads in flight
__device__ inline double ordered_rec_sum(const double *rec, int64_t stride, int n, int r) {
  double s = 0.0;
  int i = 0;
  for (; i + 8 <= n; i += 8) {
    double v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = rec[(int64_t)(i + k) * stride + r];
#pragma unroll
    for (int k = 0; k < 8; ++k) s += v[k];
  }
  for (; i < n; ++i) s += rec[(int64_t)i * stride + r];
  return s;
}

}  // namespace ima
