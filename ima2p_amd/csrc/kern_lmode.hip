// kern_lmode.hip -- L-mode surfaces over stored genealogy tables.
//
//   jointp      jointfind.cpp:885-1047   joint -log posterior at a point
//   margincalc  surface_call_functions.cpp:120-173   marginal for one param
//
// Tables hold one row of K floats per saved genealogy in the savegsampinf
// layout (ginfo.cpp:288-316): cc | fc | hcc (npsize each), mc | fm (nmig
// each), qintegrate (npsize), mintegrate (nmig), pdg, probg, split times.
//
// jointp is a matrix product on the FP64 matrix unit, genealogies times
// points, with an exp and a sum over the genealogies behind it (see below).
// Chunk partials are merged by a second kernel in a fixed order, and the
// rows a lane works on depend on the table only, never on how many points
// share a launch, so a point's result is the same alone and batched with
// others.  margincalc and the 2NM density have rows on the lanes, the 2NM
// density of many points has points; a point's value is the same in any batch
// there too.
#include <float.h>
#include <limits.h>

#include <algorithm>

#include "ima_internal.h"
#include "prior_math.h"

namespace ima {

struct JointLayout {
  int ccp, fcp, hccp, mcp, fmp, qip, mip, pdgp, probgp;
};

__host__ __device__ inline JointLayout joint_layout(int npsize, int nmig) {
  JointLayout L;
  L.ccp = 0;
  L.fcp = L.ccp + npsize;
  L.hccp = L.fcp + npsize;
  L.mcp = L.hccp + npsize;
  L.fmp = L.mcp + nmig;
  L.qip = L.fmp + nmig;
  L.mip = L.qip + npsize;
  L.pdgp = L.mip + nmig;
  L.probgp = L.pdgp + 1;
  return L;
}

struct LArgs {
  const float *rows;
  int G, K, npsize, nmig, npops, modeltype, r0, r1;
  const double *x;  // [npoints][np]
  int npoints, nchunks, chunk_rows;
};

constexpr int kXLanes = 256;


// ------------------------------------------------------------- jointp --
// A point's term for a genealogy is
//   p = c0 + sum_k count_k * A_k + weight_k * F_k
// with c0 = (the row's base term) minus the hcc of the parameters in range,
// A = log 2 - log x (theta, models 0/1; else 0) or log x (migration), F =
// -2/x (theta: 2 fc / x) or -x (migration); (2/x) fc equals (2 fc)/x
// exactly, the remaining differences from the reference's order are the
// fused multiply-adds and the summation order (about 1e-16 relative).  A
// batch of points against a table is therefore a matrix product, genealogies
// x (1 + 2 parameters) x points, followed by an exp and a sum over the
// genealogies.  It runs on the FP64 matrix unit.  (In logarithms to base 2 a
// term's exponential takes one operation less, 4.01 ms for the surface below
// instead of 4.15, but the base terms and coefficients are then rounded once
// more, the result is 1.1 to 1.4 times as far from 64 bits, and terms overflow
// from 1.25e308 on.)
//
// One workgroup of four wavefronts takes one chunk of rows and up to
// 16 * T points.  It stages kRows rows at a time in LDS as FP64 records
// [c0, count_0, weight_0, ...]; each wavefront multiplies its quarter of
// them, 16 rows a tile, with every tile of 16 points.  A lane of the product
// holds one point and four consecutive rows of a tile; it keeps that point's
// running maximum and sums over its own rows, so no lane talks to another
// until the end of the chunk, where the 16 partials of a point (4 wavefronts
// x 4 lanes) are merged in a fixed order.  The rows a lane sees depend on
// the table and the parameter range alone: a point's value is the same
// alone and batched with others.
//
// Bound: FP64 issue, 20 vector operations per (point, genealogy) pair
// (subtract, scale, round, 12 multiply-adds, conversion and ldexp, the maximum
// and two sums; 2.2 ns per 64 lanes) and the product (48 ns per 16 x 16 x 4 on a SIMD).  The two
// share their issue here: a loop of half of each takes the sum of both.
// Multiply-adds in place of the product would cost 22 ns instead of 36 per
// 64 pairs at five parameters, but the row values then pass through LDS once
// per lane: 4.5 ms where this took 3.9 (4096 points on 1e6 genealogies).
// With one lane per point (rows in order, the library's exp and a branch on
// every new maximum) that surface took 6.45 ms, 500 points on 1e5 in
// REF_COMPAT 277 us, and one point on 1e5 171 us (one lane of 256 working);
// here 4.15 ms, 111 us and 13 us.
typedef double dvec4 __attribute__((ext_vector_type(4)));

constexpr double kLog2E = 1.4426950408889634074;
constexpr double kLn10 = 2.3025850929940456840;
// Coefficients, and counts and weights (a row's base term: their product),
// beyond this take the careful path: below it a term's size is under 1e24.
constexpr double kBadSize = 1e11;
constexpr double kPadRow = -1e25;  // c0 of the rows past the end: e^(p - M) = 0

template <int NR>
struct XShape {
  static constexpr int kRows = NR <= 8 ? 256 : 128;    // staged at a time
  static constexpr int kRT = kRows / 64;               // row tiles per wavefront
  // matrix steps of 4: the parameters' counts and weights, and c0 as one
  // more operand where they leave room, else as the product's addend
  static constexpr bool kAdd = (2 * NR) % 4 == 0;
  static constexpr int kSteps = (2 * NR + 3) / 4;
  static constexpr int kKP = 4 * kSteps;  // record length, zero padded
  // distance of records: 24, 40, 56 or (padded) 4 mod 8 dwords, so that the
  // rows of a fragment load spread over the banks
  static constexpr int kStride = kKP + (kKP % 8 == 0 ? 2 : 0);
  static constexpr int kLds = kRows * kStride + (kAdd ? kRows : 0);
  // place of parameter k's count in a record (its weight follows)
  static __device__ __forceinline__ constexpr int at(int k) { return (kAdd ? 0 : 1) + 2 * k; }
  static constexpr int kEnd = (kAdd ? 0 : 1) + 2 * NR;
};

// e^t, |t| < 1e26 and e^t in range: 2^n e^r with r = t - n ln 2, |r| <= ln 2 /
// 2, by a polynomial of degree 11 (interpolation at the Chebyshev nodes, 2e-17
// relative), exactly 1 at t = 0.  ln 2 is one constant: r is off by n 2.3e-17,
// which counts for terms near the largest only, where n is small.  Far below
// the range r is anything to 1e10, and the scaling gives 0 all the same.
__device__ __forceinline__ double exp_fast(double t) {
  const double n = rint(t * kLog2E), r = fma(-n, kLn2, t);
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
  p = fma(p, r, 1.0);
  p = fma(p, r, 1.0);
  return ldexp(p, (int)n);
}
// e^t for any t <= 0, infinite or NaN too
__device__ __forceinline__ double exp_any(double t) { return t < -800.0 ? 0.0 : exp_fast(t); }

// Rows [g0, g0 + cnt) as records in sh, rows cnt .. kRows - 1 as padding.
// Returns whether this thread met a value that is not finite, or large.
template <int NR>
__device__ inline bool stage_rows(const LArgs &a, double *sh, int g0, int cnt) {
  using X = XShape<NR>;
  const JointLayout L = joint_layout(a.npsize, a.nmig);
  bool bad = false;
  for (int r = threadIdx.x; r < X::kRows; r += kXLanes) {
    double *o = sh + r * X::kStride;
    double *c0 = X::kAdd ? sh + X::kRows * X::kStride + r : o;
    if (r >= cnt) {
#pragma unroll
      for (int k = 0; k < X::kKP; ++k) o[k] = 0.0;
      *c0 = kPadRow;
      continue;
    }
    const float *g = a.rows + (size_t)(g0 + r) * a.K;
    double base;
    if (a.npops == 2) {
      base = -(double)g[L.probgp];
    } else {
      double t = 0.0;
      if (a.modeltype == 1)
        for (int i = 0; i < a.npsize; ++i) t += (double)g[L.qip + i];
      else
        for (int i = 0; i < a.nmig; ++i) t += (double)g[L.mip + i];
      base = -t;
    }
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      const int i = a.r0 + k;
      double c, w;
      if (i < a.npsize) {
        base -= (double)g[L.hccp + i];
        c = (double)g[L.ccp + i];
        w = (double)g[L.fcp + i];
      } else {
        c = (double)g[L.mcp + i - a.npsize];
        w = (double)g[L.fmp + i - a.npsize];
      }
      o[X::at(k)] = c;
      o[X::at(k) + 1] = w;
      bad = bad || !(fabs(c) < kBadSize) || !(fabs(w) < kBadSize);
    }
    bad = bad || !(fabs(base) < kBadSize * kBadSize);
#pragma unroll
    for (int k = X::kEnd; k < X::kKP; ++k) o[k] = 0.0;
    *c0 = base;
  }
  return bad;
}

// The points' coefficients, [tile][k][16], from point pt0 on (points past
// the end repeat the last one); ptbad[tile * 16 + j] flags a point whose
// terms might overflow.
template <int NR, int T>
__device__ inline void stage_points(const LArgs &a, double *sh, int *ptbad, int pt0) {
  using X = XShape<NR>;
  const int np = a.npsize + a.nmig;
  for (int x = threadIdx.x; x < T * 16; x += kXLanes) ptbad[x] = 0;
  __syncthreads();
  for (int x = threadIdx.x; x < T * 16 * NR; x += kXLanes) {
    const int p = x / NR, k = x % NR, i = a.r0 + k;
    const double v = a.x[(size_t)min(pt0 + p, a.npoints - 1) * np + i];
    double A, F;
    if (i < a.npsize) {
      A = (a.modeltype == 0 || a.modeltype == 1) ? kLn2 - log(v) : 0.0;
      F = -2.0 * (1.0 / v);
    } else {
      A = log(v);
      F = -v;
    }
    if (!(fabs(A) < kBadSize) || !(fabs(F) < kBadSize)) ptbad[p] = 1;
    double *o = sh + ((size_t)(p / 16) * X::kKP) * 16 + p % 16;
    o[X::at(k) * 16] = A;
    o[(X::at(k) + 1) * 16] = F;
  }
  for (int p = threadIdx.x; p < T * 16; p += kXLanes) {
    double *o = sh + ((size_t)(p / 16) * X::kKP) * 16 + p % 16;
    if (!X::kAdd) o[0] = 1.0;
    for (int k = X::kEnd; k < X::kKP; ++k) o[k * 16] = 0.0;
  }
  __syncthreads();
}

// Operand fragments.  The matrix unit gives lane l the rows l / 16 + 4 i of
// the product (i = 0..3) and column l % 16; operand row i of a tile is
// loaded from staged row 4 (i % 4) + i / 4, so the lane's four values are
// the consecutive rows 4 (l / 16) .. + 3.
template <int NR>
struct RowFrag {
  double v[XShape<NR>::kRT][XShape<NR>::kSteps];
  dvec4 c0[XShape<NR>::kRT];  // the lane's rows' c0, or zero
  __device__ __forceinline__ void load(const double *sh, int wave, int lane) {
    using X = XShape<NR>;
    const int i = lane & 15, row = 4 * (i & 3) + (i >> 2);
#pragma unroll
    for (int t = 0; t < X::kRT; ++t) {
      const double *o = sh + (size_t)((wave * X::kRT + t) * 16 + row) * X::kStride + (lane >> 4);
#pragma unroll
      for (int s = 0; s < X::kSteps; ++s) v[t][s] = o[4 * s];
      const double *c = sh + X::kRows * X::kStride + (wave * X::kRT + t) * 16 + 4 * (lane >> 4);
      c0[t] = X::kAdd ? dvec4{c[0], c[1], c[2], c[3]} : dvec4{0.0, 0.0, 0.0, 0.0};
    }
  }
};

template <int NR>
struct PointFrag {
  double v[XShape<NR>::kSteps];
  __device__ __forceinline__ void load(const double *sh, int tile, int lane) {
    using X = XShape<NR>;
    const double *o = sh + ((size_t)tile * X::kKP + (lane >> 4)) * 16 + (lane & 15);
#pragma unroll
    for (int s = 0; s < X::kSteps; ++s) v[s] = o[s * 64];
  }
};

// terms (logs) of the lane's point for rows 4 (lane / 16) + i of row tile t
template <int NR>
__device__ __forceinline__ void terms(const RowFrag<NR> &a, const PointFrag<NR> &b,
                                      dvec4 (&p)[XShape<NR>::kRT]) {
  using X = XShape<NR>;
#pragma unroll
  for (int t = 0; t < X::kRT; ++t) p[t] = a.c0[t];
#pragma unroll
  for (int s = 0; s < X::kSteps; ++s)
#pragma unroll
    for (int t = 0; t < X::kRT; ++t)
      p[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.v[t][s], b.v[s], p[t], 0, 0, 0);
}

// The largest, and the x-th, of a lane's values.
template <int NR>
__device__ __forceinline__ double largest(const dvec4 (&p)[XShape<NR>::kRT]) {
  double m = fmax(fmax(p[0][0], p[0][1]), fmax(p[0][2], p[0][3]));
#pragma unroll
  for (int t = 1; t < XShape<NR>::kRT; ++t)
    m = fmax(m, fmax(fmax(p[t][0], p[t][1]), fmax(p[t][2], p[t][3])));
  return m;
}
template <int NR>
__device__ __forceinline__ double pick(const dvec4 (&p)[XShape<NR>::kRT], int x) {
  double v = p[0][0];
#pragma unroll
  for (int k = 1; k < 4 * XShape<NR>::kRT; ++k) v = x == k ? p[k / 4][k % 4] : v;
  return v;
}

// Chunk and first point of this workgroup.
struct XPlace {
  int pt0, chunk, gbeg, gend, wave, lane;
  int part;  // wavefront * 4 + lane group
  int row0;  // the lane's first row of a stage (16 on per row tile)
};
template <int NR, int T>
__device__ __forceinline__ XPlace x_place(const LArgs &a) {
  XPlace w;
  w.pt0 = blockIdx.x * (16 * T);
  w.chunk = blockIdx.y;
  w.gbeg = w.chunk * a.chunk_rows;
  w.gend = min(a.G, w.gbeg + a.chunk_rows);
  w.wave = threadIdx.x / kWave;
  w.lane = threadIdx.x & (kWave - 1);
  w.part = threadIdx.x / 16;
  w.row0 = w.wave * XShape<NR>::kRT * 16 + 4 * (w.lane >> 4);
  return w;
}

// --------------------------------------------------------------- EXACT --
// Per (point, chunk): a reference M and s = sum e^(p - M), s2 = sum
// e^(2(p - M)) for the effective sample number.  M is a value the lane met
// and at most kSlack below its largest: FP64's range takes the difference,
// so sums are rescaled when a term leaves it, not on every new maximum.
struct XPart {
  double M, s, s2;
};
constexpr double kSlack = 50.0;

template <int NR, int T>
__global__ __launch_bounds__(kXLanes, 2) void jointp_exact(LArgs a, XPart *work) {
  using X = XShape<NR>;
  extern __shared__ double sh[];
  double *shp = sh + X::kLds;
  __shared__ int ptbad[T * 16];
  const XPlace w = x_place<NR, T>(a);
  stage_points<NR, T>(a, shp, ptbad, w.pt0);
  PointFrag<NR> b[T];
  double M[T], s[T], s2[T];
  bool pbad[T];
#pragma unroll
  for (int j = 0; j < T; ++j) {
    b[j].load(shp, j, w.lane);
    pbad[j] = ptbad[j * 16 + (w.lane & 15)] != 0;
    M[j] = -DBL_MAX;
    s[j] = s2[j] = 0.0;
  }
  // rbad: the careful path from the first stage with such a row on, so that
  // padding (behind the last row) is only added to references above it
  bool rbad = false;
  for (int g0 = w.gbeg; g0 < w.gend; g0 += X::kRows) {
    const int cnt = min(X::kRows, w.gend - g0);
    __syncthreads();
    const bool bad = stage_rows<NR>(a, sh, g0, cnt);
    rbad = __syncthreads_or(bad || rbad) != 0;
    if (w.wave * (X::kRows / 4) >= cnt) continue;  // only padding in this quarter
    RowFrag<NR> r;
    r.load(sh, w.wave, w.lane);
#pragma unroll
    for (int j = 0; j < T; ++j) {
      dvec4 p[X::kRT];
      terms<NR>(r, b[j], p);
      if (rbad || pbad[j]) {
        // infinities and NaN: one value after another, as they come
#pragma unroll 1
        for (int x = 0; x < 4 * X::kRT; ++x) {
          if (w.row0 + x / 4 * 16 + x % 4 >= cnt) continue;
          const double v = pick<NR>(p, x);
          const bool up = v > M[j];
          const double e = exp_any(up ? M[j] - v : v - M[j]);
          s[j] = up ? s[j] * e + 1.0 : s[j] + e;
          s2[j] = up ? s2[j] * e * e + 1.0 : fma(e, e, s2[j]);
          M[j] = up ? v : M[j];
        }
        continue;
      }
      const double m = largest<NR>(p);
      if (__any(m - M[j] > kSlack)) {
        // the reference moves up to the largest of these (the first rows'
        // way in, too: M is below everything)
        const double to = m - M[j] > kSlack ? m : M[j], sc = exp_any(M[j] - to);
        s[j] *= sc;
        s2[j] *= sc * sc;
        M[j] = to;
      }
#pragma unroll
      for (int t = 0; t < X::kRT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const double e = exp_fast(p[t][i] - M[j]);
          s[j] += e;
          s2[j] = fma(e, e, s2[j]);
        }
    }
  }
  // merge: 16 partials per point in LDS (over the rows' buffer), wavefront by
  // wavefront and lane group by lane group
  __syncthreads();
  XPart *part = reinterpret_cast<XPart *>(sh);
#pragma unroll
  for (int j = 0; j < T; ++j) {
    const bool none = !rbad && !pbad[j] && M[j] < 0.1 * kPadRow;  // padding alone
    part[w.part * (T * 16) + j * 16 + (w.lane & 15)] =
        none ? XPart{-DBL_MAX, 0.0, 0.0} : XPart{M[j], s[j], s2[j]};
  }
  __syncthreads();
  const int pt = w.pt0 + (int)threadIdx.x;
  if (threadIdx.x < T * 16 && pt < a.npoints) {
    XPart o{-DBL_MAX, 0.0, 0.0};
#pragma unroll 2
    for (int k = 0; k < 16; ++k) o.M = fmax(o.M, part[k * (T * 16) + threadIdx.x].M);
#pragma unroll 2
    for (int k = 0; k < 16; ++k) {
      const XPart q = part[k * (T * 16) + threadIdx.x];
      if (q.s == 0.0) continue;
      const double sc = exp_any(q.M - o.M);
      o.s += q.s * sc;
      o.s2 += q.s2 * sc * sc;
    }
    work[(size_t)pt * a.nchunks + w.chunk] = o;
  }
}

// over the W lanes of a point
template <int W>
__device__ inline double group_max(double v) {
  for (int off = W / 2; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, W));
  return v;
}
template <int W>
__device__ inline double group_add(double v) {
  for (int off = W / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, W);
  return v;
}

// W lanes per point take the chunks in turn, then a butterfly (a thread per
// point walking its chunks took 63 us for one point on 1e5 genealogies and
// 160 us for 4096 on 1e6).  A wavefront, or four lanes on the few chunks of a
// small table (20000 points on 30 genealogies in REF_COMPAT: 202 us a call and
// 167).  How many depends on the table alone, as the sums' order does.
constexpr int kFewChunks = 16;
template <int W>
__global__ __launch_bounds__(256) void jointp_exact_final(LArgs a, const XPart *work, double *out,
                                                          double *ess) {
  const int pt = blockIdx.x * (256 / W) + threadIdx.x / W;
  const int lane = threadIdx.x % W;
  if (pt >= a.npoints) return;
  const XPart *w = work + (size_t)pt * a.nchunks;
  double M = -DBL_MAX;
  for (int c = lane; c < a.nchunks; c += W) M = fmax(M, w[c].M);
  M = group_max<W>(M);
  double s = 0.0, s2 = 0.0;
  for (int c = lane; c < a.nchunks; c += W) {
    if (w[c].s == 0.0) continue;
    const double sc = exp_any(w[c].M - M);
    s += w[c].s * sc;
    s2 += w[c].s2 * sc * sc;
  }
  s = group_add<W>(s);
  s2 = group_add<W>(s2);
  if (lane == 0) {
    out[pt] = log((double)a.G) - (M + log(s));
    if (ess) ess[pt] = s * s / s2;
  }
}

// ---------------------------------------------------------- REF_COMPAT --
// The reference keeps only values within PRANGELOG = 10 nats of the running
// maximum (the first value always), then sums at most (kept - 1) of them
// from the top while they stay within 10 nats of the final maximum, as
// eexp mantissa/exponent pairs scaled to 10^(z - (z_max - 10)).  Every
// value within the final window is always kept, so the sum covers the
// whole final window, minus its smallest member when nothing outside the
// window was kept and the window holds more than one value.
//
// pass 1: chunk maxima; then, per point, the maxima of the chunks before
// each one; pass 2: per chunk, the window sums, and whether a kept value
// lies outside the window; final: the chunks merged and the list cap.
//
// A kept value's term is e^p / 10^maxz (the mantissa m 10^(z - maxz) of the
// reference's eexp, utilities.cpp:1507-1539), taken here as exp(p - maxz ln
// 10): the window, the list cap and the ordering of the running maximum are the reference's, the term
// itself differs from the degree-10 Taylor series of eexp by at most its
// truncation, ~4e-10 relative, which moves the result by less than 1e-12
// relative.
constexpr double kWindow = 10.0;

// Per (point, chunk) record of pass 2: sums of the window's terms and of
// their squares, its smallest value, its size, and whether a kept value
// lies outside.
struct RefPart {
  double sum, sum2, minp;
  int32_t cnt, outside;
};

// maxz: eexp's exponent of the largest term (10^z <= e^p < 10^(z + 1)) less 10
__device__ inline int ref_maxz(double Mfin) {
  return (int)floor(Mfin * 0.43429448190325182765) - 10;
}

template <int NR, int T>
__global__ __launch_bounds__(kXLanes, 2) void jointp_ref_max(LArgs a, double *cmax) {
  using X = XShape<NR>;
  extern __shared__ double sh[];
  double *shp = sh + X::kLds;
  __shared__ int ptbad[T * 16];
  const XPlace w = x_place<NR, T>(a);
  stage_points<NR, T>(a, shp, ptbad, w.pt0);
  PointFrag<NR> b[T];
  double M[T];
#pragma unroll
  for (int j = 0; j < T; ++j) {
    b[j].load(shp, j, w.lane);
    M[j] = -DBL_MAX;
  }
  for (int g0 = w.gbeg; g0 < w.gend; g0 += X::kRows) {
    const int cnt = min(X::kRows, w.gend - g0);
    __syncthreads();
    stage_rows<NR>(a, sh, g0, cnt);
    __syncthreads();
    RowFrag<NR> r;
    r.load(sh, w.wave, w.lane);
#pragma unroll
    for (int j = 0; j < T; ++j) {
      dvec4 p[X::kRT];
      terms<NR>(r, b[j], p);
      if (cnt == X::kRows) {
        M[j] = fmax(M[j], largest<NR>(p));
      } else {
#pragma unroll
        for (int t = 0; t < X::kRT; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            M[j] = fmax(M[j], w.row0 + t * 16 + i < cnt ? p[t][i] : -DBL_MAX);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < T; ++j) sh[w.part * (T * 16) + j * 16 + (w.lane & 15)] = M[j];
  __syncthreads();
  const int pt = w.pt0 + (int)threadIdx.x;
  if (threadIdx.x < T * 16 && pt < a.npoints) {
    double m = -DBL_MAX;
#pragma unroll 2
    for (int k = 0; k < 16; ++k) m = fmax(m, sh[k * (T * 16) + threadIdx.x]);
    cmax[(size_t)pt * a.nchunks + w.chunk] = m;
  }
}

// The term (log) of one point (its parameters x) for one table row.
__device__ inline double one_term(const LArgs &a, const float *g, const double *x) {
  const JointLayout L = joint_layout(a.npsize, a.nmig);
  double p;
  if (a.npops == 2) {
    p = -(double)g[L.probgp];
  } else {
    double t = 0.0;
    if (a.modeltype == 1)
      for (int i = 0; i < a.npsize; ++i) t += (double)g[L.qip + i];
    else
      for (int i = 0; i < a.nmig; ++i) t += (double)g[L.mip + i];
    p = -t;
  }
  for (int i = a.r0; i < a.r1; ++i) {
    if (i < a.npsize) {
      const double A = (a.modeltype == 0 || a.modeltype == 1) ? kLn2 - log(x[i]) : 0.0;
      p += (double)g[L.ccp + i] * A - (double)g[L.hccp + i] - 2.0 * (double)g[L.fcp + i] / x[i];
    } else {
      p += (double)g[L.mcp + i - a.npsize] * log(x[i]) - (double)g[L.fmp + i - a.npsize] * x[i];
    }
  }
  return p;
}

// Per point, cmax[c] becomes the maximum over the chunks before c, and mfin
// the maximum over all: W lanes per point, W chunks at a time.  A
// point whose first value (always kept) lies outside the final window needs
// no further search for one: its cmax[c] are the final maximum.
template <int W>
__global__ __launch_bounds__(256) void jointp_ref_prefix(LArgs a, double *cmax, double *mfin) {
  const int pt = blockIdx.x * (256 / W) + threadIdx.x / W;
  const int lane = threadIdx.x % W;
  if (pt >= a.npoints) return;
  double *cm = cmax + (size_t)pt * a.nchunks;
  const double first = one_term(a, a.rows, a.x + (size_t)pt * (a.npsize + a.nmig));
  double before = -DBL_MAX;
  for (int c0 = 0; c0 < a.nchunks; c0 += W) {
    const int c = c0 + lane;
    double v = c < a.nchunks ? cm[c] : -DBL_MAX;
    for (int off = 1; off < W; off <<= 1) {
      const double o = __shfl_up(v, off, W);
      if (lane >= off) v = fmax(v, o);
    }
    const double up = __shfl_up(v, 1, W);
    if (c < a.nchunks) cm[c] = lane ? fmax(before, up) : before;
    before = fmax(before, __shfl(v, W - 1, W));
  }
  if (lane == 0) mfin[pt] = before;
  if (before - first >= kWindow + 1.0)  // clear of rounding: the kernel takes its own first value
    for (int c = lane; c < a.nchunks; c += W) cm[c] = before;
}

template <int NR, int T>
__global__ __launch_bounds__(kXLanes, 2) void jointp_ref_sum(LArgs a, const double *before,
                                                             const double *mfin, RefPart *part) {
  using X = XShape<NR>;
  extern __shared__ double sh[];
  double *shp = sh + X::kLds;
  __shared__ int ptbad[T * 16];
  __shared__ double smax[16][16], wmax[4][16];
  const XPlace w = x_place<NR, T>(a);
  stage_points<NR, T>(a, shp, ptbad, w.pt0);
  PointFrag<NR> b[T];
  double run[T], Mf[T], sc[T], seen[T];
  RefPart o[T];
  bool open = false;
#pragma unroll
  for (int j = 0; j < T; ++j) {
    b[j].load(shp, j, w.lane);
    const int pt = min(w.pt0 + j * 16 + (w.lane & 15), a.npoints - 1);
    run[j] = before[(size_t)pt * a.nchunks + w.chunk];
    Mf[j] = mfin[pt];
    sc[j] = (double)ref_maxz(Mf[j]) * kLn10;
    seen[j] = -DBL_MAX;
    o[j] = RefPart{0.0, 0.0, DBL_MAX, 0, 0};
    open = open || run[j] < Mf[j];
  }
  // A kept value outside the final window lies within the window of a
  // running maximum below the final one: once that is the final one (run =
  // Mf, also set for points whose first value lies outside) there is none.
  const bool look = __syncthreads_or(open) != 0;
  for (int g0 = w.gbeg; g0 < w.gend; g0 += X::kRows) {
    const int cnt = min(X::kRows, w.gend - g0);
    __syncthreads();
    stage_rows<NR>(a, sh, g0, cnt);
    __syncthreads();
    RowFrag<NR> r;
    r.load(sh, w.wave, w.lane);
#pragma unroll
    for (int j = 0; j < T; ++j) {
      dvec4 p[X::kRT];
      terms<NR>(r, b[j], p);
      if (g0 == 0 && w.part == 0 && !(Mf[j] - p[0][0] < kWindow)) o[j].outside = 1;
      if (look) {
        // candidates: within the window of the maximum before the chunk
        bool cand = false;
#pragma unroll
        for (int t = 0; t < X::kRT; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            cand = cand || (w.row0 + t * 16 + i < cnt && run[j] - p[t][i] < kWindow &&
                            !(Mf[j] - p[t][i] < kWindow));
        if (__syncthreads_or(cand && !o[j].outside)) {
          // with the running maximum before each value: the earlier chunks
          // (run), the earlier stages (seen), the earlier wavefronts of this
          // stage, the earlier tiles and lane groups of this wavefront
          double m = -DBL_MAX;
#pragma unroll 1
          for (int x = 0; x < 4 * X::kRT; ++x)
            if (w.row0 + x / 4 * 16 + x % 4 < cnt) m = fmax(m, pick<NR>(p, x));
          m = fmax(m, __shfl_xor(m, 16, kWave));
          m = fmax(m, __shfl_xor(m, 32, kWave));
          if (w.lane < 16) wmax[w.wave][w.lane] = m;
          smax[w.part][w.lane & 15] = seen[j];
          __syncthreads();
          double ru = run[j];
#pragma unroll 1
          for (int k = 0; k < 16; ++k) ru = fmax(ru, smax[k][w.lane & 15]);
#pragma unroll 1
          for (int k = 0; k < w.wave; ++k) ru = fmax(ru, wmax[k][w.lane & 15]);
#pragma unroll 1
          for (int t = 0; t < X::kRT; ++t) {
            const int row = w.row0 + t * 16;
            double m4 = -DBL_MAX;
#pragma unroll 1
            for (int i = 0; i < 4; ++i)
              if (row + i < cnt) m4 = fmax(m4, pick<NR>(p, 4 * t + i));
            double st = ru;  // with the lane groups before this one
#pragma unroll 1
            for (int q = 0; q < 4; ++q) {
              const double mq = __shfl(m4, q * 16 + (w.lane & 15), kWave);
              if (q < (w.lane >> 4)) st = fmax(st, mq);
              ru = fmax(ru, mq);
            }
#pragma unroll 1
            for (int i = 0; i < 4; ++i) {
              if (row + i >= cnt) continue;
              const double v = pick<NR>(p, 4 * t + i);
              const bool kept = st - v < kWindow;
              if (kept && !(Mf[j] - v < kWindow)) o[j].outside = 1;
              if (kept && v > st) st = v;
            }
          }
          __syncthreads();  // smax and wmax are written again for the next tile
        }
#pragma unroll
        for (int t = 0; t < X::kRT; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            seen[j] = fmax(seen[j], w.row0 + t * 16 + i < cnt ? p[t][i] : -DBL_MAX);
      }
      // most values lie outside the window and cost no exp
#pragma unroll
      for (int t = 0; t < X::kRT; ++t) {
        const int row = w.row0 + t * 16;
        const double lo = Mf[j] - fmax(fmax(p[t][0], p[t][1]), fmax(p[t][2], p[t][3]));
        if (!__any(lo < kWindow)) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const double v = p[t][i];
          const bool in = row + i < cnt && Mf[j] - v < kWindow;
          const double e = in ? exp_fast(v - sc[j]) : 0.0;
          o[j].sum += e;
          o[j].sum2 = fma(e, e, o[j].sum2);
          o[j].cnt += in ? 1 : 0;
          o[j].minp = fmin(o[j].minp, in ? v : DBL_MAX);
        }
      }
    }
  }
  __syncthreads();
  RefPart *lp = reinterpret_cast<RefPart *>(sh);
#pragma unroll
  for (int j = 0; j < T; ++j)
    lp[w.part * (T * 16) + j * 16 + (w.lane & 15)] = o[j];
  __syncthreads();
  const int pt = w.pt0 + (int)threadIdx.x;
  if (threadIdx.x < T * 16 && pt < a.npoints) {
    RefPart s{0.0, 0.0, DBL_MAX, 0, 0};
#pragma unroll 2
    for (int k = 0; k < 16; ++k) {
      const RefPart q = lp[k * (T * 16) + threadIdx.x];
      s.sum += q.sum;
      s.sum2 += q.sum2;
      s.minp = fmin(s.minp, q.minp);
      s.cnt += q.cnt;
      s.outside |= q.outside;
    }
    part[(size_t)pt * a.nchunks + w.chunk] = s;
  }
}

// W lanes per point.
template <int W>
__global__ __launch_bounds__(256) void jointp_ref_final(LArgs a, const double *mfin,
                                                        const RefPart *part, double *out,
                                                        double *ess) {
  const int pt = blockIdx.x * (256 / W) + threadIdx.x / W;
  const int lane = threadIdx.x % W;
  if (pt >= a.npoints) return;
  const RefPart *P = part + (size_t)pt * a.nchunks;
  const int maxz = ref_maxz(mfin[pt]);
  double sum = 0.0, sum2 = 0.0, minp = DBL_MAX;
  int cnt = 0, outside = 0;
  for (int c = lane; c < a.nchunks; c += W) {
    sum += P[c].sum;
    sum2 += P[c].sum2;
    minp = fmin(minp, P[c].minp);
    cnt += P[c].cnt;
    outside |= P[c].outside;
  }
  sum = group_add<W>(sum);
  sum2 = group_add<W>(sum2);
  minp = -group_max<W>(-minp);
  for (int off = W / 2; off > 0; off >>= 1) {
    cnt += __shfl_xor(cnt, off, W);
    outside |= __shfl_xor(outside, off, W);
  }
  if (lane != 0) return;
  if (!outside && cnt > 1) {  // the list cap drops the smallest kept value
    const double e = exp_fast(minp - maxz * kLn10);
    sum -= e;
    sum2 -= e * e;
  }
  out[pt] = log((double)a.G) - (log(sum) + maxz * kLn10);
  if (ess) ess[pt] = sum * sum / sum2;
}

// jointp's rows per chunk, a function of the table alone: about 256 chunks, in
// steps of 128 rows (fewer where 128 rows of FP64 exceed 32 KB).  The work
// area's size, and with it the calls that are refused, follows from these; the
// kernels round them up to whole stages (launch_nr), so they make no more
// chunks than it has room for.
static void chunking(const LTable &t, int *nchunks, int *chunk_rows) {
  const int step = std::max(8, std::min(128, 32768 / (8 * t.K) / 8 * 8));
  int rows = (t.G + 255) / 256;
  rows = std::max(step, (rows + step - 1) / step * step);
  *chunk_rows = rows;
  *nchunks = (t.G + rows - 1) / rows;
}

// Work area: per point and chunk of the table a maximum and a partial, as
// many chunks as `chunking` makes (the kernels' own chunks are no smaller).
size_t jointp_work_bytes(const LTable &t, int npoints) {
  int nc, cr;
  chunking(t, &nc, &cr);
  return (size_t)npoints * nc * 48 + 64;
}

// Dynamic LDS of a kernel with T tiles: rows and points, later the partials
// (part bytes each) over them.  With the kernel's own (stat bytes) it stays
// within the 64 KiB that every launch keeps to.
template <int NR, int T>
constexpr size_t x_lds(size_t part) {
  using X = XShape<NR>;
  return std::max((size_t)(X::kLds + T * 16 * X::kKP) * 8, (size_t)16 * T * 16 * part);
}
template <int NR, int T>
constexpr bool x_fits(size_t part, size_t stat) {
  return x_lds<NR, T>(part) + stat <= 65536;
}

// T tiles of points per workgroup, TS in the window sums (more registers a
// tile).
template <int NR, int T, int TS>
static void launch_tiles(const LArgs &a, int mode, double *work, double *out, double *ess,
                         hipStream_t st) {
  static_assert(x_fits<NR, T>(sizeof(XPart), T * 16 * 4), "jointp_exact's LDS");
  static_assert(x_fits<NR, T>(sizeof(double), T * 16 * 4), "jointp_ref_max's LDS");
  static_assert(x_fits<NR, TS>(sizeof(RefPart), TS * 16 * 4 + 20 * 16 * 8), "jointp_ref_sum's LDS");
  const bool few = a.nchunks <= kFewChunks;
  const dim3 per_point(few ? (a.npoints + 63) / 64 : (a.npoints + 3) / 4);
  auto grid = [&](int tiles) { return dim3((a.npoints + 16 * tiles - 1) / (16 * tiles), a.nchunks); };
  if (mode == IMA_LMODE_EXACT) {
    XPart *part = reinterpret_cast<XPart *>(work);
    hipLaunchKernelGGL((jointp_exact<NR, T>), grid(T), dim3(kXLanes),
                       (x_lds<NR, T>(sizeof(XPart))), st, a, part);
    hipLaunchKernelGGL(few ? jointp_exact_final<4> : jointp_exact_final<kWave>, per_point,
                       dim3(256), 0, st, a, part, out, ess);
  } else {
    double *cmax = work, *mfin = cmax + (size_t)a.npoints * a.nchunks;
    RefPart *part = reinterpret_cast<RefPart *>(mfin + a.npoints);
    hipLaunchKernelGGL((jointp_ref_max<NR, T>), grid(T), dim3(kXLanes),
                       (x_lds<NR, T>(sizeof(double))), st, a, cmax);
    hipLaunchKernelGGL(few ? jointp_ref_prefix<4> : jointp_ref_prefix<kWave>, per_point,
                       dim3(256), 0, st, a, cmax, mfin);
    hipLaunchKernelGGL((jointp_ref_sum<NR, TS>), grid(TS), dim3(kXLanes),
                       (x_lds<NR, TS>(sizeof(RefPart))), st, a, cmax, mfin, part);
    hipLaunchKernelGGL(few ? jointp_ref_final<4> : jointp_ref_final<kWave>, per_point,
                       dim3(256), 0, st, a, mfin, part, out, ess);
  }
}

// Rows per chunk: chunking's, in whole stages.  Points per workgroup: a
// workgroup stages each row once for all its tiles, so four tiles (two above
// 8 parameters, for registers) as soon as they leave about a workgroup per
// CU (256 points on 1e6 genealogies: 432 us with one tile, 317 with four;
// 64 points: 134 and 112), and twice as many, at two workgroups a CU, once
// there are several rounds of them (4096 points, 8 parameters: 6.5 and 5.1
// ms; 500 points: 0.59 and 0.83 ms).  The values do not depend on it.
constexpr int kMidGrid = 200, kWideGrid = 1024;

template <int NR>
static void launch_nr(LArgs a, int mode, double *work, double *out, double *ess, hipStream_t st) {
  constexpr int kRows = XShape<NR>::kRows, kMid = NR <= 8 ? 4 : 2, kWide = 2 * kMid;
  a.chunk_rows = (a.chunk_rows + kRows - 1) / kRows * kRows;
  a.nchunks = (a.G + a.chunk_rows - 1) / a.chunk_rows;
  auto groups = [&](int tiles) {
    return (int64_t)((a.npoints + 16 * tiles - 1) / (16 * tiles)) * a.nchunks;
  };
  if (groups(kWide) >= kWideGrid)
    launch_tiles<NR, kWide, kMid>(a, mode, work, out, ess, st);
  else if (a.npoints > 16 * (kMid - 1) && groups(kMid) >= kMidGrid)
    launch_tiles<NR, kMid, kMid>(a, mode, work, out, ess, st);
  else
    launch_tiles<NR, 1, 1>(a, mode, work, out, ess, st);
}

hipError_t launch_jointp(const LTable &t, const double *x, int npoints, int modeltype,
                         int r0, int r1, int mode, double *work, size_t work_bytes,
                         double *out, double *ess, hipStream_t st) {
  if (npoints == 0) return hipSuccess;
  LArgs a{t.rows, t.G, t.K, t.npsize, t.nmig, t.npops, modeltype, r0, r1, x, npoints, 0, 0};
  chunking(t, &a.nchunks, &a.chunk_rows);
  if (jointp_work_bytes(t, npoints) > work_bytes) return hipErrorInvalidValue;
  switch (r1 - r0) {
#define IMA_NR(N) \
  case N:         \
    launch_nr<N>(a, mode, work, out, ess, st); \
    break;
    IMA_NR(1) IMA_NR(2) IMA_NR(3) IMA_NR(4) IMA_NR(5) IMA_NR(6) IMA_NR(7) IMA_NR(8)
    IMA_NR(9) IMA_NR(10) IMA_NR(11) IMA_NR(12) IMA_NR(13) IMA_NR(14) IMA_NR(15) IMA_NR(16)
#undef IMA_NR
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// ---------------------------------------------------------- margincalc --

// The mean over genealogies of one parameter's marginal density at x
// (:120-173).  The lanes of a workgroup hold rows and go over up to T points,
// so a search that asks for one point at a time has the whole table spread
// over the chip: one lane a point left a lone point to 256 lanes in all, 80
// dependent exponentials each (20000 genealogies: 39 us, and 16 us for one
// lane to add the chunks).  A lane adds its rows of a chunk in order, then
// the lanes, the wavefronts and the chunks are added in a fixed tree: a
// point's value does not depend on the points beside it.  Bound: latency for
// a few points, FP64 exponentials for many (a row's four floats are reread
// for every T points, from L2).

// Rows across workgroups: a function of the table alone, a row or more a
// lane and at most 256 chunks.
constexpr int kRowLanes = 256;
static void row_chunks(int G, int *nchunks, int *chunk_rows) {
  int rows = (G + 255) / 256;
  rows = std::max(1, (rows + kRowLanes - 1) / kRowLanes) * kRowLanes;
  *chunk_rows = rows;
  *nchunks = (G + rows - 1) / rows;
}

__device__ inline double lanes_sum(double s) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, kWave);
  return s;
}

// lanes_sum of T sums, the one of s[lane T / 64] in each lane.  The lanes of a
// pair split the sums between them as long as there are several: 10 exchanges
// for eight sums instead of 48, the same additions.
template <int T, int H>
__device__ __forceinline__ void split_sums(double (&s)[T], int lane) {
  if constexpr (H > 0) {
    constexpr int off = kWave * H / T;
    const bool up = (lane & off) != 0;
#pragma unroll
    for (int t = 0; t < H; ++t) {
      const double keep = up ? s[t + H] : s[t], give = up ? s[t] : s[t + H];
      s[t] = keep + __shfl_xor(give, off, kWave);
    }
    split_sums<T, H / 2>(s, lane);
  }
}
template <int T>
__device__ __forceinline__ double lanes_sums(double (&s)[T], int lane) {
  split_sums<T, T / 2>(s, lane);
#pragma unroll
  for (int off = kWave / T / 2; off > 0; off >>= 1) s[0] += __shfl_xor(s[0], off, kWave);
  return s[0];
}

struct MArgs {
  const float *rows;
  int G, K, npsize, nmig, param, expo;
  double meani;
  const double *x;
  int nx, nchunks, chunk_rows;
};

template <int T, int Q>
__global__ __launch_bounds__(kRowLanes) void margin_partial(MArgs a, double *work) {
  constexpr int N = T * Q;  // a workgroup's points, T at a time
  __shared__ double sx[N], slx[N], part[kRowLanes / kWave][N];
  const int p0 = blockIdx.x * N, np = min(N, a.nx - p0);
  const int chunk = blockIdx.y, tid = threadIdx.x;
  if (tid < N) {
    sx[tid] = a.x[p0 + min(tid, np - 1)];
    slx[tid] = log(sx[tid]);
  }
  __syncthreads();
  const JointLayout L = joint_layout(a.npsize, a.nmig);
  const bool size = a.param < a.npsize;
  const int p = size ? a.param : a.param - a.npsize;
  const double lmean = log(a.meani);
  const int gend = min(a.G, (chunk + 1) * a.chunk_rows);
#pragma unroll 1
  for (int q0 = 0; q0 < np; q0 += T) {
    double s[T] = {};
    for (int r = chunk * a.chunk_rows + tid; r < gend; r += kRowLanes) {
      const float *g = a.rows + (size_t)r * a.K;
      const float c = g[(size ? L.ccp : L.mcp) + p];
      const double cnt = (double)(c >= 0 ? (long)(c + 0.5) : (long)(c - 0.5));  // INTEGERROUND
      // (fused where written so, whatever T; the last points' neighbours are
      // copies of them)
      const double w = g[(size ? L.fcp : L.fmp) + p], q = g[(size ? L.qip : L.mip) + p];
      if (size) {
        const double h = g[L.hccp + p], w2 = 2 * w;
#pragma unroll
        for (int t = 0; t < T; ++t)
          s[t] += exp(fma(cnt, kLn2 - slx[q0 + t], -q) - h - w2 / sx[q0 + t]);
      } else if (a.expo) {
#pragma unroll
        for (int t = 0; t < T; ++t)
          s[t] += exp(fma(-w, sx[q0 + t],
                          fma(cnt, slx[q0 + t], fma(-sx[q0 + t], a.meani, -q + lmean))));
      } else {
#pragma unroll
        for (int t = 0; t < T; ++t)
          s[t] += exp(fma(-w, sx[q0 + t], fma(cnt, slx[q0 + t], -q)));
      }
    }
    const double sum = lanes_sums(s, tid % kWave);
    if (tid % (kWave / T) == 0) part[tid / kWave][q0 + tid % kWave / (kWave / T)] = sum;
  }
  __syncthreads();
  if (tid >= np) return;
  double v = 0.0;
#pragma unroll
  for (int w = 0; w < kRowLanes / kWave; ++w) v += part[w][tid];
  work[(size_t)(p0 + tid) * a.nchunks + chunk] = v;
}

// one wavefront a point
__global__ __launch_bounds__(256) void margin_final(MArgs a, int logi, double yadjust,
                                                    const double *work, double *out) {
  const int pt = blockIdx.x * 4 + threadIdx.x / kWave, lane = threadIdx.x % kWave;
  if (pt >= a.nx) return;
  double s = 0.0;
  for (int c = lane; c < a.nchunks; c += kWave) s += work[(size_t)pt * a.nchunks + c];
  s = lanes_sum(s);
  if (lane != 0) return;
  s /= a.G;
  if (logi) s = (s <= 0) ? -1e200 : log(s);
  out[pt] = s - yadjust;
}

size_t margincalc_work_bytes(const LTable &t, int nx) {
  int nc, cr;
  row_chunks(t.G, &nc, &cr);
  return (size_t)nx * nc * sizeof(double) + 64;
}

hipError_t launch_margincalc(const LTable &t, int param, const double *x, int nx, int logi,
                             double yadjust, int expo, double prior_mean, double *work,
                             double *out, hipStream_t st) {
  if (nx == 0) return hipSuccess;
  MArgs a{t.rows, t.G, t.K, t.npsize, t.nmig, param, expo,
          expo ? 1.0 / prior_mean : 1.0, x, nx, 0, 0};
  row_chunks(t.G, &a.nchunks, &a.chunk_rows);
  // A workgroup takes 8 points where that leaves 8 workgroups a CU, else 2 (64
  // points on 1e6 rows: 179 us with 2).  It takes 32, 8 at a time, where a lane
  // has no more than two rows, whose loads and sums of lanes these share, and 4
  // workgroups a CU are left: 20000 points on 30000 rows 1.01 ms, with 8 a
  // workgroup 1.30 (with 16 in a loop the compiler did not unroll, 1.40); but
  // 350 points on 1e6 rows 539 us, with 8 485.
  const int64_t pairs = (int64_t)nx * a.nchunks;
  if (pairs >= 32 * 1024 && a.chunk_rows <= 2 * kRowLanes)
    hipLaunchKernelGGL((margin_partial<8, 4>), dim3((nx + 31) / 32, a.nchunks), dim3(kRowLanes), 0,
                       st, a, work);
  else if (pairs >= 8 * 2048)
    hipLaunchKernelGGL((margin_partial<8, 1>), dim3((nx + 7) / 8, a.nchunks), dim3(kRowLanes), 0,
                       st, a, work);
  else
    hipLaunchKernelGGL((margin_partial<2, 1>), dim3((nx + 1) / 2, a.nchunks), dim3(kRowLanes), 0,
                       st, a, work);
  hipLaunchKernelGGL(margin_final, dim3((nx + 3) / 4), dim3(256), 0, st, a, logi, yadjust, work,
                     out);
  return hipGetLastError();
}

// -------------------------------------------------------------- popmig --
//
// The density of 2NM = theta_i m_i / 2 at x, per genealogy the closed form
// of integrating the coalescent and migration likelihoods over the priors
// of theta_i and m_i along x = theta m / 2 (popmig.cpp:9-351):
//   uniform priors: 2 x^mc (fc + fm x)^-(cc+mc) [G(cc+mc, 2(fc+fm x)/qmax)
//     - G(cc+mc, mmax(fm + fc/x))] e^(-hc - qint - mint), with the
//     reference's special cases when the counts or sums vanish;
//   exponential migration prior (mean mmean): its own closed form with one
//     upper incomplete gamma.
// For a few points the lanes hold rows, for many they hold points.  Uniform
// terms are summed (terms whose log lies outside (-700, 700) are skipped, as
// the reference does); exponential-prior terms are summed relative to their
// maximum (log-sum-exp), the reference's eexp sum to rounding.
//
// Both layouts add the same tree, so a point's value has the same bits in any
// batch: a chunk has 64 leaves, rows l, l + 64, ... of it, added in order; the
// leaves are joined two by two, and the chunks as popmig_final does.  What
// rounds is written out (no contraction: the compiler may fuse the two
// kernels' products differently), and joining is commutative.

struct PArgs {
  const float *rows;
  int K, g0;               // rows [g0, g0 + n)
  int n, cc, fc, hc, mc, fm, qi, mi;  // column offsets
  double qmax, mmax, mmean;
  int expo, kind, prob_or_like;
  double xmax;             // MARGIN: 1.0 outside [0, xmax]
  double denom;            // rows averaged over (MARGIN: the reference's divisor)
  const double *x;
  int nx, nchunks, chunk_rows;
  const double *lf;        // log(k!) for k < nlf
  int nlf;
};

// A function of its own: inlined at its uses the gammas (and lgamma, for
// counts beyond the table) took 235 registers, two wavefronts a SIMD.
__device__ __attribute__((noinline)) double pm_gamma(const double *lf, int nlf, int k, double x,
                                                     bool upper) {
  const double lga = (k >= 1 && k - 1 < nlf) ? lf[k - 1] : lgamma((double)k);  // log((k-1)!)
  return upper ? pri_uppergamma(k, x, lga) : pri_lowergamma(k, x, lga);
}
__device__ inline double pm_upper(const PArgs &a, int k, double x) {
  return pm_gamma(a.lf, a.nlf, k, x, true);
}
__device__ inline double pm_lower(const PArgs &a, int k, double x) {
  return pm_gamma(a.lf, a.nlf, k, x, false);
}

// log of the term of one genealogy, or flags a skipped term (uniform: the
// reference adds exp(t) only for -700 < t < 700).
__device__ inline double popmig_term(const PArgs &a, const float *g, double x, bool *use) {
#pragma clang fp contract(off)
  const int cc = (int)g[a.cc], mc = (int)g[a.mc];
  const double fc = g[a.fc], hc = g[a.hc], fm = g[a.fm], qintg = g[a.qi], mintg = g[a.mi];
  *use = true;
  if (!a.expo) {
    double t1, t2;
    if (fc == 0 && cc == 0 && fm > 0) {
      t1 = fma(-mc, log(fm), kLog2) - hc - qintg - mintg;
      t2 = log(exp(pm_upper(a, mc, 2 * fm * x / a.qmax)) - exp(pm_upper(a, mc, a.mmax * fm)));
    } else if (fm == 0 && mc == 0 && fc > 0) {
      t1 = fma(-cc, log(fc), kLog2) - hc - qintg - mintg;
      t2 = log(exp(pm_upper(a, cc, 2 * fc / a.qmax)) - exp(pm_upper(a, cc, fc * a.mmax / x)));
    } else if (fc == 0 && cc == 0 && mc == 0 && fm == 0) {
      t1 = log(2 * log(a.mmax * a.qmax / (2 * x))) - hc - qintg - mintg;
      t2 = 0;
    } else {
      const double w = fma(fm, x, fc), lo = 2 * w / a.qmax, hi = a.mmax * (fm + fc / x);
      t1 = fma(-(cc + mc), log(w), fma(mc, log(x), kLog2)) - hc - qintg - mintg;
      double ua = pm_upper(a, cc + mc, lo), ub = pm_upper(a, cc + mc, hi);
      if (ua == ub) {  // both gammas saturate: the lower ones differ instead
        ub = pm_lower(a, cc + mc, lo);
        ua = pm_lower(a, cc + mc, hi);
      }
      if (ua > ub) {
        t2 = pri_logdiff(ua, ub);
      } else {
        t1 = t2 = 0.0;  // the reference then adds exp(0)
      }
    }
    const double t = t1 + t2;
    *use = (t < 700) && (t > -700);
    return t;
  }
  const double mmean = a.mmean;
  const double u1 = fma(fm * mmean, x, fma(fc, mmean, x));
  double t2 = kLog2 - hc - log(mmean) - qintg - mintg;
  const double t3 = 2 * u1 / (mmean * a.qmax);
  if (mc == 0 && cc == 0) {
    t2 += pm_upper(a, 0, t3);
  } else if (cc == 0) {
    t2 += fma(-mc, log(fm + 1 / mmean), pm_upper(a, mc, t3));
  } else if (mc == 0) {
    t2 += fma(-cc, log(fma(x, fm + 1 / mmean, fc)), pm_upper(a, cc, t3));
  } else {
    t2 = fma(cc + mc, log(mmean * x / u1), fma(-cc, log(x), t2 + pm_upper(a, mc + cc, t3)));
  }
  return t2;
}

// Terms added: s under uniform priors, s e^m under the exponential one (no
// terms: s = 0 and m = -inf; a NaN among them is in s).
struct PmSum {
  double m, s;
};
constexpr PmSum kPmNone{-INFINITY, 0.0};

__device__ inline PmSum pm_join(const PArgs &a, PmSum u, PmSum v) {
#pragma clang fp contract(off)
  if (!a.expo) return PmSum{u.m, u.s + v.s};
  const bool up = v.m > u.m;
  const PmSum hi = up ? v : u, lo = up ? u : v;
  if (lo.m == -INFINITY && lo.s == 0.0) return hi;
  return PmSum{hi.m, fma(lo.s, exp(lo.m - hi.m), hi.s)};
}

// sum with row r's term at x joined
__device__ inline PmSum pm_add(const PArgs &a, int r, double x, PmSum sum) {
  bool use;
  const double t = popmig_term(a, a.rows + (size_t)(a.g0 + r) * a.K, x, &use);
  PmSum v = kPmNone;
  if (!a.expo)
    v.s = use ? exp(t) : 0.0;
  else if (t > -INFINITY)
    v = PmSum{t, 1.0};
  else if (t != t)
    v.s = t;
  return pm_join(a, sum, v);
}

// work[pt][chunk]
__device__ inline void popmig_put(const PArgs &a, int pt, int chunk, PmSum v, double *work) {
  const size_t o = (size_t)pt * a.nchunks + chunk;
  if (!a.expo) {
    work[o] = v.s;
  } else {
    work[2 * o] = v.m;
    work[2 * o + 1] = v.s;
  }
}

__device__ inline bool popmig_inside(const PArgs &a, double x) {
  return !(a.kind == IMA_POPMIG_MARGIN && (x < 0 || x > a.xmax));
}

// The lanes hold a chunk's leaves; a wavefront takes a chunk, a workgroup one
// point.
__global__ __launch_bounds__(kRowLanes, 4) void popmig_rows(PArgs a, double *work) {
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int pt = blockIdx.x, chunk = blockIdx.y * (kRowLanes / kWave) + wave;
  if (chunk >= a.nchunks) return;
  const double x = a.x[pt];
  const int beg = chunk * a.chunk_rows, end = min(a.n, beg + a.chunk_rows);
  PmSum v = kPmNone;
  if (popmig_inside(a, x))
    for (int r = beg + lane; r < end; r += kWave) v = pm_add(a, r, x, v);
#pragma unroll 1
  for (int off = 1; off < kWave; off <<= 1)
    v = pm_join(a, v, PmSum{__shfl_xor(v.m, off, kWave), __shfl_xor(v.s, off, kWave)});
  if (lane == 0) popmig_put(a, pt, chunk, v, work);
}

// The lanes hold points; a workgroup takes a chunk, each wavefront RUN of its
// leaves.
template <int RUN>
__global__ __launch_bounds__(kWave / RUN *kWave, 4) void popmig_points(PArgs a, double *work) {
  constexpr int kWaves = kWave / RUN, kTop = RUN == 16 ? 4 : 2;  // RUN = 2^kTop
  static_assert(RUN == 1 << kTop, "whole subtrees");
  // a lane's joined leaves that wait for others: 1, 2, 4, ... of them
  __shared__ PmSum part[kWaves][kTop + 1][kWave];
  const int chunk = blockIdx.y, lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int pt = blockIdx.x * kWave + lane;
  const double x = a.x[min(pt, a.nx - 1)];
  const bool inside = popmig_inside(a, x);
  const int beg = chunk * a.chunk_rows, end = min(a.n, beg + a.chunk_rows);
#pragma unroll 1
  for (int j = 0; j < RUN; ++j) {
    PmSum v = kPmNone;
    if (inside)
      for (int r = beg + wave * RUN + j; r < end; r += kWave) v = pm_add(a, r, x, v);
    int k = 0;  // v: 2^k leaves
    for (; (j >> k) & 1; ++k) v = pm_join(a, part[wave][k][lane], v);
    part[wave][k][lane] = v;
  }
  __syncthreads();
  if (wave != 0 || pt >= a.nx) return;
#pragma unroll 1
  for (int step = 1; step < kWaves; step *= 2)
    for (int w = 0; w < kWaves; w += 2 * step)
      part[w][kTop][lane] = pm_join(a, part[w][kTop][lane], part[w + step][kTop][lane]);
  popmig_put(a, pt, chunk, part[0][kTop][lane], work);
}

// one wavefront a point
__global__ __launch_bounds__(256) void popmig_final(PArgs a, const double *work, double *out) {
  const int pt = blockIdx.x * 4 + threadIdx.x / kWave, lane = threadIdx.x % kWave;
  if (pt >= a.nx) return;
  const double x = a.x[pt];
  if (a.kind == IMA_POPMIG_MARGIN && (x < 0 || x > a.xmax)) {
    if (lane == 0) out[pt] = 1.0;  // OFFSCALEVAL
    return;
  }
  double v;
  if (!a.expo) {
    double s = 0.0;
    for (int c = lane; c < a.nchunks; c += kWave) s += work[(size_t)pt * a.nchunks + c];
    v = lanes_sum(s) / a.denom;
  } else {
    PmSum t = kPmNone;
    for (int c = lane; c < a.nchunks; c += kWave)
      t = pm_join(a, t, PmSum{work[2 * ((size_t)pt * a.nchunks + c)],
                              work[2 * ((size_t)pt * a.nchunks + c) + 1]});
    for (int off = 32; off > 0; off >>= 1)
      t = pm_join(a, t, PmSum{__shfl_xor(t.m, off, kWave), __shfl_xor(t.s, off, kWave)});
    v = exp(t.m + log(t.s) - log(a.denom));
  }
  if (lane != 0) return;
  if (a.kind == IMA_POPMIG_MARGIN) {
    out[pt] = -v;
    return;
  }
  if (a.prob_or_like) {
    const double prior = a.expo ? 2 * exp(pri_uppergamma(0, 2 * x / (a.mmean * a.qmax), 0.0)) /
                                      (a.qmax * a.mmean)
                                : 2 * (log(a.qmax) + log(a.mmax) - log(2 * x)) / (a.qmax * a.mmax);
    v /= prior;
  }
  out[pt] = v;
}

// How nx points over n rows are laid out, and the work area that takes.  The
// chunks follow from n alone, the rows of the call: whole leaves, at most
// 1024 chunks.  A launch takes as many points as leave the area within 64 MiB
// (4096 or more); a call with more of them makes several.
//
// A wavefront runs as long as its longest series or fraction.  Lanes that
// hold points are at one row, and alike where many points lie close; lanes
// that hold rows have a lone point's rows side by side, but take about 1.5 times
// as long a term.  So points once the rows' wavefronts are more than twice
// what the chip holds (4096) and 64 points are not mostly padding; then 16
// leaves a wavefront where those fill the chip, else four.  Calls in us (25
// of them copies and waiting), uniform prior:
//   20000 rows, 1 point:     42 with rows, 122 with points (16 leaves)
//   20000 rows, 100 points:  163, 182
//   20000 rows, 256 points:  342, 258 (four leaves: 283)
//   20000 rows, 500 points:  602, 409
//   2000 rows, 256 points:   77, 118 (84)
//   2000 rows, 500 points:   107, 119 (85)
//   2000 rows, 2000 points:  290, 206 (228)
PopmigPlan popmig_plan(int n, int nx, int expo) {
  PopmigPlan p;
  const int leaf = (n - 1) / (1024 * kWave) + 1;
  p.chunk_rows = leaf * kWave;
  p.nchunks = (n - 1) / p.chunk_rows + 1;
  const size_t point = (size_t)p.nchunks * (expo ? 2 : 1) * sizeof(double);
  nx = p.points = (int)std::min((size_t)nx, ((size_t)64 << 20) / point);
  constexpr int64_t kFull = 4096;
  const int64_t groups = ((int64_t)nx + kWave - 1) / kWave;
  p.run = nx < 2 * kWave || (int64_t)nx * p.nchunks <= 2 * kFull ? 0
          : groups * p.nchunks * 4 < kFull                       ? 4
                                                                 : 16;
  p.bytes = nx * point;
  return p;
}

hipError_t launch_popmig(const LTable &t, int theta_i, int mig_i, double qmax, double mprior,
                         int expo, int kind, int prob_or_like, int first, int last,
                         const double *x, int nx, const double *lf, int nlf,
                         const PopmigPlan &plan, double *work, size_t work_bytes, double *out,
                         hipStream_t st) {
  if (nx == 0) return hipSuccess;
  const JointLayout L = joint_layout(t.npsize, t.nmig);
  PArgs a{};
  a.rows = t.rows;
  a.K = t.K;
  a.g0 = kind == IMA_POPMIG_MARGIN ? first : 0;
  a.n = kind == IMA_POPMIG_MARGIN ? last - first : t.G;
  a.cc = L.ccp + theta_i;
  a.fc = L.fcp + theta_i;
  a.hc = L.hccp + theta_i;
  a.mc = L.mcp + mig_i;
  a.fm = L.fmp + mig_i;
  a.qi = L.qip + theta_i;
  a.mi = L.mip + mig_i;
  a.qmax = qmax;
  a.mmax = expo ? 0.0 : mprior;
  a.mmean = expo ? mprior : 0.0;
  a.expo = expo;
  a.kind = kind;
  a.prob_or_like = prob_or_like;
  a.xmax = expo ? 20.0 * mprior : qmax * mprior / 2.0;  // EXPOMIGPLOTSCALE x mean
  a.denom = kind == IMA_POPMIG_MARGIN ? (double)(last - first + (first == 0)) : (double)t.G;
  a.x = x;
  a.nx = nx;
  a.lf = lf;
  a.nlf = nlf;
  a.nchunks = plan.nchunks;
  a.chunk_rows = plan.chunk_rows;
  // every row in one chunk, every partial in the work area
  if ((int64_t)a.nchunks * a.chunk_rows < a.n ||
      (size_t)nx * a.nchunks * (expo ? 2 : 1) * sizeof(double) > work_bytes)
    return hipErrorInvalidValue;
  const dim3 points((nx + kWave - 1) / kWave, a.nchunks);
  if (plan.run == 16)
    hipLaunchKernelGGL(popmig_points<16>, points, dim3(4 * kWave), 0, st, a, work);
  else if (plan.run == 4)
    hipLaunchKernelGGL(popmig_points<4>, points, dim3(16 * kWave), 0, st, a, work);
  else
    hipLaunchKernelGGL(popmig_rows,
                       dim3(nx, (a.nchunks + kRowLanes / kWave - 1) / (kRowLanes / kWave)),
                       dim3(kRowLanes), 0, st, a, work);
  hipLaunchKernelGGL(popmig_final, dim3((nx + 3) / 4), dim3(256), 0, st, a, work, out);
  return hipGetLastError();
}

// ------------------------------------------------------- greater-than --
//
// P(parameter i > parameter j) per genealogy (gtint.cpp:1-331): closed
// forms where the reference has them, else the reference's trapezoid
// refinement (qtrap: relative change below 1e-4, tested from the sixth
// refinement, at most 20) of the integrand over (MINPARAMVAL, prior max).
// One lane per genealogy: each runs the reference's sequence of points and
// sums them in the same order.  A second launch averages the terms of each
// ordered pair.

struct GArgs {
  const float *rows;
  int K, treeinc, ntrees, kind;
  int ccp, fcp, hccp, mcp, fmp, qip, mip;
  const int2 *pairs;  // [npairs] (i, j)
  const double *pmax; // [npairs] prior maximum of the pair
  const double *lf;
  int nlf;
};

struct GtOne {
  int cci, ccj, wi, wj;
  double fci, fcj, hval, denom, fmi, fmj;
};

__device__ inline double gt_lf(const GArgs &a, int k) {  // log(k!)
  return k < a.nlf ? a.lf[k] : lgamma((double)k + 1.0);
}
__device__ inline double gt_upper(const GArgs &a, int k, double x) {
  return pri_uppergamma(k, x, k >= 1 ? gt_lf(a, k - 1) : 0.0);
}
__device__ inline double gt_lower(const GArgs &a, int k, double x) {
  return pri_lowergamma(k, x, gt_lf(a, k - 1));
}

constexpr double kGtSwitch = 1e-15;  // SWITCH_TO_LOWERGAMMA_CRIT
constexpr double kGtMinParam = 1e-7; // MINPARAMVAL

__device__ inline double gt_mgt(const GArgs &a, const GtOne &s, double mi) {  // mgt_wj_gt_0
  if (mi < kGtMinParam) return 0.0;
  const double la = gt_lf(a, s.wj), lb = gt_upper(a, s.wj + 1, s.fmj * mi);
  if (la <= lb) return 0.0;
  const double t1 = (la - lb) < kGtSwitch ? gt_lower(a, s.wj + 1, s.fmj * mi) : pri_logdiff(la, lb);
  double t2 = s.wi * log(mi) - s.fmi * mi - (s.wj + 1) * log(s.fmj) + t1;
  t2 -= s.denom;
  return exp(t2);
}

__device__ inline double gt_pgt(const GArgs &a, const GtOne &s, double qi) {  // pgt_fcj_gt_0
  if (qi < kGtMinParam) return 0.0;
  const double fcj2 = 2 * s.fcj, fci2 = 2 * s.fci;
  if (s.ccj == 0) {
    const double la = log(qi) - fcj2 / qi;
    const double lb = log(fcj2) + gt_upper(a, 0, fcj2 / qi);
    if (la > lb) {
      const double t1 = pri_logdiff(la, lb);
      const double t2 = -fci2 / qi + s.cci * log(2 / qi);
      return exp(t1 + t2 - s.hval - s.denom);
    }
    return 0.0;
  }
  const double t1 = gt_upper(a, s.ccj - 1, fcj2 / qi);
  const double t2 = kLog2 + s.cci * log(2 / qi) + (1 - s.ccj) * log(s.fcj) - fci2 / qi;
  return exp(t2 + t1 - s.hval - s.denom);
}

__device__ inline double gt_f(const GArgs &a, const GtOne &s, bool mig, double x) {
  return mig ? gt_mgt(a, s, x) : gt_pgt(a, s, x);
}

__device__ double gt_qtrap(const GArgs &a, const GtOne &s, bool mig, double lo, double hi) {
  double st = 0.0, olds = -1.0e100;
  for (int j = 1; j <= 20; ++j) {
    if (j == 1) {
      st = 0.5 * (hi - lo) * (gt_f(a, s, mig, lo) + gt_f(a, s, mig, hi));
    } else {
      const int it = 1 << (j - 2);
      const double tnm = it, del = (hi - lo) / tnm;
      double x = lo + 0.5 * del, sum = 0.0;
      for (int k = 1; k <= it; ++k, x += del) sum += gt_f(a, s, mig, x);
      st = 0.5 * (st + (hi - lo) * sum / tnm);
    }
    if (j > 5 && (fabs(st - olds) < 1.0e-4 * fabs(olds) || (st == 0.0 && olds == 0.0)))
      return st;
    olds = st;
  }
  return st;
}

__device__ double gtmig_one(const GArgs &a, const float *g, int mi, int mj, double mmax) {
  GtOne s{};
  s.fmi = g[a.fmp + mi];
  s.fmj = g[a.fmp + mj];
  s.wi = (int)g[a.mcp + mi];
  s.wj = (int)g[a.mcp + mj];
  s.denom = (double)g[a.mip + mi] + (double)g[a.mip + mj];
  double temp;
  if (s.wj == 0) {
    if (s.fmj > 0.0) {
      if (s.wi > 0) {
        const double la = gt_lf(a, s.wi);
        const double lb = gt_upper(a, s.wi + 1, (s.fmi + s.fmj) * mmax);
        const double lc = gt_upper(a, s.wi + 1, s.fmi * mmax);
        if (la <= lb || la <= lc) {
          temp = 0.0;
        } else {
          double t1 = (la - lb) < kGtSwitch ? gt_lower(a, s.wi + 1, (s.fmi + s.fmj) * mmax)
                                             : pri_logdiff(la, lb);
          t1 += -(s.wi + 1) * log(s.fmi + s.fmj);
          double t2 = (la - lc) < kGtSwitch ? gt_lower(a, s.wi + 1, s.fmi * mmax)
                                             : pri_logdiff(la, lc);
          t2 += -(s.wi + 1) * log(s.fmi);
          temp = t2 <= t1 ? 0.0 : exp(pri_logdiff(t2, t1) - log(s.fmj) - s.denom);
        }
      } else if (s.fmi > 0.0) {
        const double t1 = s.fmi * (exp(-(s.fmi + s.fmj) * mmax) - exp(-s.fmi * mmax));
        const double t2 = s.fmj * (1 - exp(-s.fmi * mmax));
        const double t3 = (t1 + t2) / (s.fmi * s.fmj * (s.fmi + s.fmj));
        temp = exp(log(t3) - s.denom);
      } else {
        const double t1 = (s.fmj * mmax - 1.0 + exp(-s.fmj * mmax)) / (s.fmj * s.fmj);
        temp = exp(log(t1) - s.denom);
      }
    } else {
      if (s.wi > 0) {
        const double la = gt_lf(a, s.wi + 1), lb = gt_upper(a, s.wi + 2, s.fmi * mmax);
        if (la <= lb) {
          temp = 0.0;
        } else {
          const double t1 = (la - lb) < kGtSwitch ? gt_lower(a, s.wi + 2, s.fmi * mmax)
                                                   : pri_logdiff(la, lb);
          temp = exp(-(s.wi + 2) * log(s.fmi) + t1 - s.denom);
        }
      } else if (s.fmi > 0.0) {
        const double t1 = (1.0 - exp(-s.fmi * mmax) * (s.fmi * mmax + 1.0)) / (s.fmi * s.fmi);
        temp = exp(log(t1) - s.denom);
      } else {
        temp = exp(log(mmax * mmax / 2.0) - s.denom);
      }
    }
  } else {
    temp = gt_qtrap(a, s, true, kGtMinParam, mmax);
  }
  return fmin(1.0, temp);
}

__device__ double gtpops_one(const GArgs &a, const float *g, int pi, int pj, double qmax) {
  GtOne s{};
  s.cci = (int)g[a.ccp + pi];
  s.ccj = (int)g[a.ccp + pj];
  s.fci = g[a.fcp + pi];
  s.fcj = g[a.fcp + pj];
  s.hval = (double)g[a.hccp + pi] + (double)g[a.hccp + pj];
  s.denom = (double)g[a.qip + pi] + (double)g[a.qip + pj];
  double temp;
  if (s.ccj == 0 && s.fcj == 0) {
    if (s.fci == 0) {
      temp = exp(2.0 * log(qmax) - kLog2 - s.hval - s.denom);
    } else if (s.cci >= 2) {
      const double t1 = 2 * kLog2 + (2 - s.cci) * log(s.fci);
      const double t2 = gt_upper(a, s.cci - 2, 2 * s.fci / qmax);
      temp = exp(t1 + t2 - s.hval - s.denom);
    } else if (s.cci == 1) {
      const double t1 = 4 * s.fci * exp(gt_upper(a, 0, 2 * s.fci / qmax));
      const double t2 = 2 * qmax * exp(-2 * s.fci / qmax) - t1;
      temp = exp(log(t2) - s.hval - s.denom);
    } else {
      const double t1 = exp(gt_upper(a, 0, 2 * s.fci / qmax));
      const double t2 = (qmax / 2) * (qmax - 2 * s.fci) * exp(-2 * s.fci / qmax) +
                        2 * s.fci * s.fci * t1;
      temp = exp(log(t2) - s.hval - s.denom);
    }
  } else {
    temp = gt_qtrap(a, s, false, kGtMinParam, qmax);
  }
  return fmin(1.0, temp);
}

// per[pair][tree]
__global__ __launch_bounds__(64) void gt_terms(GArgs a, double *per) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int p = blockIdx.y;
  if (t >= a.ntrees) return;
  const float *g = a.rows + (size_t)t * a.treeinc * a.K;
  const int2 ij = a.pairs[p];
  per[(size_t)p * a.ntrees + t] =
      a.kind ? gtmig_one(a, g, ij.x, ij.y, a.pmax[p]) : gtpops_one(a, g, ij.x, ij.y, a.pmax[p]);
}

// one wavefront per pair: lane-strided partial sums in a fixed order
__global__ __launch_bounds__(64) void gt_mean(GArgs a, const double *per, double *out) {
  const int p = blockIdx.x, lane = threadIdx.x;
  double s = 0.0;
  for (int t = lane; t < a.ntrees; t += 64) s += per[(size_t)p * a.ntrees + t];
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if (lane == 0) out[p] = s / a.ntrees;
}

hipError_t launch_greater_than(const LTable &t, int kind, const int2 *pairs, const double *pmax,
                               int npairs, const double *lf, int nlf, double *per, double *out,
                               hipStream_t st) {
  if (npairs == 0) return hipSuccess;
  const JointLayout L = joint_layout(t.npsize, t.nmig);
  GArgs a{};
  a.rows = t.rows;
  a.K = t.K;
  // print_greater_than_tests (gtint.cpp:337-349): at most USETREESMAX = 20000
  if (t.G > 20000) {
    a.treeinc = t.G / 20000;
    a.ntrees = 20000;
  } else {
    a.treeinc = 1;
    a.ntrees = t.G;
  }
  a.kind = kind;
  a.ccp = L.ccp;
  a.fcp = L.fcp;
  a.hccp = L.hccp;
  a.mcp = L.mcp;
  a.fmp = L.fmp;
  a.qip = L.qip;
  a.mip = L.mip;
  a.pairs = pairs;
  a.pmax = pmax;
  a.lf = lf;
  a.nlf = nlf;
  hipLaunchKernelGGL(gt_terms, dim3((a.ntrees + 63) / 64, npairs), dim3(64), 0, st, a, per);
  hipLaunchKernelGGL(gt_mean, dim3(npairs), dim3(64), 0, st, a, per, out);
  return hipGetLastError();
}

}  // namespace ima
