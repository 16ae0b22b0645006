// WENO5-JS reconstruction of split fluxes at one face.
// Follows solver_2D/reconstruction/WENO5_JS.py:10-117 of the reference:
// smoothness IS_k = 1/4(.)^2 + 13/12(.)^2, alpha_k = C_k/(eps+IS_k)^2 with
// eps = 1e-6, C = (0.1, 0.6, 0.3), candidate stencils (1/3,-7/6,11/6),
// (-1/6,5/6,1/3), (1/3,5/6,-1/6).  The right-biased form is the same formula
// with the stencil mirrored, so one routine serves both.
#pragma once
#include <math.h>

#include "fastmath.hpp"
#include "janc_types.hpp"

namespace jh {

// With the first differences around f0, dA = f-1 - f-2, dB = f0 - f-1, dC =
// f+1 - f0, dD = f+2 - f+1, the smoothness indicators of WENO5_JS.py:17-33 are
// quadratic forms that complete to
//   IS_1 = 4/3 [(dA - 11/8 dB)^2 + 39/64 dB^2]
//   IS_2 = 4/3 [(dB -  5/8 dC)^2 + 39/64 dC^2]
//   IS_3 = 4/3 [(dD - 11/8 dC)^2 + 39/64 dC^2]
// (the constants are exact in binary), and the candidates are
//   q_1 - f0 = (5 dB - 2 dA)/6, q_2 - f0 = (dB + 2 dC)/6, q_3 - f0 = (4 dC - dD)/6.
// So one square per difference, t(d) = 39/64 d^2 + eps', serves two
// indicators (three along a line), the common factor 4/3 goes into eps' = 3/4
// eps, and the weights' 1 : 6 : 3 into the candidates:
//   value = f0 + [a_1 (5/2 dB - dA) + a_2 (3 dB + 6 dC) + a_3 (6 dC - 3/2 dD)] /
//           [3 (a_1 + 6 a_2 + 3 a_3)],   a_k = 1 / e_k^2,  e_k = 3/4 (eps + IS_k).
// A right-biased value is the same with the stencil reversed.
constexpr double kWenoEps = 0.75e-6;

// The FP64 Lax-Friedrichs kernels hold their split fluxes scaled by 2^-20
// (exact, undone in the divergence), which centres the shared reciprocal's e_k^8
// in FP64's range: 5e-144 at eps, so that increments down to 1e-140 keep their
// precision (trace species reach 1e-80), and finite up to jumps of 5e23.
template <typename W>
struct LfScale { static constexpr double value = 1.0 / 1048576.0; };
template <>
struct LfScale<float> { static constexpr double value = 1.0; };
constexpr double kLfEps = kWenoEps * LfScale<double>::value * LfScale<double>::value;

// Three times the numerator and the denominator above with a_k = e_i^2 e_j^2 (the
// same ratio), so the weights take no reciprocal.
__host__ __device__ __forceinline__ void weno5_parts(double dA, double dB, double dC, double dD,
                                                     double eps, double& num, double& den) {
  const double tB = fma((39.0 / 64.0) * dB, dB, eps), tC = fma((39.0 / 64.0) * dC, dC, eps);
  const double m1 = fma(-1.375, dB, dA), m2 = fma(-0.625, dC, dB), m3 = fma(-1.375, dC, dD);
  const double e1 = fma(m1, m1, tB), e2 = fma(m2, m2, tC), e3 = fma(m3, m3, tC);
  const double s1 = e1 * e1, s2 = e2 * e2, s3 = e3 * e3;
  const double P1 = s2 * s3, P2 = s1 * s3, P3 = s1 * s2;
  const double h = 6.0 * dC;
  const double c1 = fma(2.5, dB, -dA), c2 = fma(3.0, dB, h), c3 = fma(-1.5, dD, h);
  num = fma(P1, c1, fma(P2, c2, P3 * c3));
  den = fma(6.0, P2, fma(3.0, P3, P1));
}

// FP64 face value: 35 operations and one reciprocal.
__host__ __device__ __forceinline__ double weno5(double fm2, double fm1, double f0,
                                                 double fp1, double fp2) {
  double num, den;
  weno5_parts(fm1 - fm2, f0 - fm1, fp1 - f0, fp2 - fp1, kWenoEps, num, den);
  return fma(num * (1.0 / 3.0), rcp(den), f0);
}

// FP64 face flux of the Lax-Friedrichs split: left-biased value of H+ (p0..p4)
// plus right-biased value of H- (m1..m5), both scaled by LfScale.  The two
// quotients are taken over one reciprocal: 67 operations and one reciprocal, 87
// and two as separate values in the b^2 form.  Range: fluxes that alternate
// between -2e23 and 2e23 (a detonation's energy flux jumps by 1e11; separate
// values reach 3e33, and a branch to them past the range costs the tube of 4000 x
// 500 1.5 %).
__host__ __device__ __forceinline__ double weno5_lf(double p0, double p1, double p2, double p3,
                                                    double p4, double m1, double m2, double m3,
                                                    double m4, double m5) {
  double nL, dL, nR, dR;
  weno5_parts(p1 - p0, p2 - p1, p3 - p2, p4 - p3, kLfEps, nL, dL);
  weno5_parts(m4 - m5, m3 - m4, m2 - m3, m1 - m2, kLfEps, nR, dR);
  return fma(fma(nL, dR, nR * dL) * (1.0 / 3.0), rcp(dL * dR), p2 + m3);
}

// Left- and right-biased FP64 values of one face from its six-cell stencil, over one
// reciprocal: 74 operations and one reciprocal instead of 70 and two, which an FP64
// reciprocal's seven issue slots outweigh.  The stencil is unscaled, and dL dR ~
// jump^16 and the crossed products leave FP64 from jumps of about 5e17 on, so past
// kPairMax the quotients are taken one by one (finite up to jumps of 6e33).  Below
// it nothing overflows: |nL| <= 4 d dL with d the largest difference, and dL dR >=
// 1e-37 d^4, so d < 1e60.  The branch also keeps the compiler from working on several
// variables at once: 154 -> 118 registers, four waves per SIMD instead of three (HLLC
// stage of 1500 x 300 cells: 119 us with two reciprocals, 111 with one, 105 with the
// branch; the step 399 -> 377).
constexpr double kPairMax = 1e200;
__host__ __device__ __forceinline__ void weno5_LR(double v0, double v1, double v2, double v3,
                                                  double v4, double v5, double& L, double& R) {
  double nL, dL, nR, dR;
  const double d0 = v1 - v0, d1 = v2 - v1, d2 = v3 - v2, d3 = v4 - v3, d4 = v5 - v4;
  weno5_parts(d0, d1, d2, d3, kWenoEps, nL, dL);
  weno5_parts(-d4, -d3, -d2, -d1, kWenoEps, nR, dR);
  const double D = dL * dR;
  if (__builtin_expect(D < kPairMax, 1)) {
    const double X = rcp(D) * (1.0 / 3.0);
    L = fma(nL * dR, X, v2);
    R = fma(nR * dL, X, v3);
  } else {
    L = fma(nL * (1.0 / 3.0), rcp(dL), v2);
    R = fma(nR * (1.0 / 3.0), rcp(dR), v3);
  }
}

// FP32 form for the mixed-precision step: first and second
// differences b around f0 (IS_1 = (b_-1/2 + d0)^2 + 13/12 b_-1^2 and alike),
// with the weights normalised by the smallest e_k = eps + IS_k,
// alpha_k = C_k (e_min / e_k)^2 (ratios <= 1, the smallest weight's ratio 1).
// e_k itself is never squared: in SI units the split energy flux jumps by
// ~1e11 across a detonation front, so e_k reaches ~1e23 and e_k^2 would
// overflow FP32, while a ratio that underflows belongs to a weight that is
// zero at FP32 precision anyway.  ~45 FP32 operations per face.
__host__ __device__ __forceinline__ float weno5(float fm2, float fm1, float f0, float fp1,
                                                float fp2) {
  const float dA = fm1 - fm2, dB = f0 - fm1, dC = fp1 - f0, dD = fp2 - fp1;
  const float bA = dB - dA, bB = dC - dB, bC = dD - dC;
  const float hB = 0.5f * dB, hC = 0.5f * dC;
  const float A1 = fmaf(0.5f, bA, dB), A2 = hB + hC, A3 = fmaf(0.5f, bC, -dC);
  const float e1 = fmaf(A1, A1, fmaf((13.0f / 12.0f) * bA, bA, 1e-6f));
  const float e2 = fmaf(A2, A2, fmaf((13.0f / 12.0f) * bB, bB, 1e-6f));
  const float e3 = fmaf(A3, A3, fmaf((13.0f / 12.0f) * bC, bC, 1e-6f));
  const float em = fminf(e1, fminf(e2, e3));
  const float r1 = em * rcp(e1), r2 = em * rcp(e2), r3 = em * rcp(e3);
  const float a1 = 0.1f * (r1 * r1), a2 = 0.6f * (r2 * r2), a3 = 0.3f * (r3 * r3);
  const float c1 = fmaf(1.0f / 3.0f, bA, hB);
  const float c2 = fmaf(-1.0f / 6.0f, bB, hC);
  const float c3 = fmaf(-1.0f / 6.0f, bC, hC);
  return fmaf(fmaf(a1, c1, fmaf(a2, c2, a3 * c3)), rcp(a1 + a2 + a3), f0);
}

// The FP32 values at K consecutive faces of one line, read from memory (LDS)
// one value per face (f(j) = p[j * s]) and written to (ACC: added into)
// q[i * qs].  Neighbouring faces share the first and second differences and
// the 13/12 b^2 + eps terms, which the run carries; every operation is the
// one the FP32 weno5 performs for that face, so the values equal per-face
// calls bit for bit.  MIRROR = false: out_i = weno5(f(i), .., f(i+4)) (the
// face between f(i+2) and f(i+3)); MIRROR = true: out_i = weno5(f(i+4), ..,
// f(i)) (the face between f(i+1) and f(i+2)).
template <int K, bool MIRROR, bool ACC>
__host__ __device__ __forceinline__ void weno5_run(const float* p, int s, float* q, int qs) {
  // forward differences d_j = f(j+1) - f(j) and b_j = d_j - d_(j-1); the
  // mirrored stencil's differences are their exact negations
  float dB = p[2 * s] - p[s], dC = p[3 * s] - p[2 * s];
  float bA = dB - (p[s] - p[0]), bB = dC - dB;
  float tA = fmaf((13.0f / 12.0f) * bA, bA, 1e-6f), tB = fmaf((13.0f / 12.0f) * bB, bB, 1e-6f);
#pragma unroll
  for (int i = 0; i < K; ++i) {
    const float dD = p[(i + 4) * s] - p[(i + 3) * s];
    const float bC = dD - dC, tC = fmaf((13.0f / 12.0f) * bC, bC, 1e-6f);
    float A1, A2, A3, c1, c2, c3, t1, t3, f0;
    if (!MIRROR) {   // f0 = f(i+2): d0 = dB, d1 = dC; b_-1, b_0, b_+1 = bA, bB, bC
      const float hB = 0.5f * dB, hC = 0.5f * dC;
      A1 = fmaf(0.5f, bA, dB); A2 = hB + hC; A3 = fmaf(0.5f, bC, -dC);
      c1 = fmaf(1.0f / 3.0f, bA, hB); c2 = fmaf(-1.0f / 6.0f, bB, hC);
      c3 = fmaf(-1.0f / 6.0f, bC, hC);
      t1 = tA; t3 = tC;
      f0 = p[(i + 2) * s];
    } else {         // f0 = f(i+2): d0 = -dC, d1 = -dB; b_-1, b_0, b_+1 = bC, bB, bA
      const float hB = 0.5f * -dC, hC = 0.5f * -dB;
      A1 = fmaf(0.5f, bC, -dC); A2 = hB + hC; A3 = fmaf(0.5f, bA, dB);
      c1 = fmaf(1.0f / 3.0f, bC, hB); c2 = fmaf(-1.0f / 6.0f, bB, hC);
      c3 = fmaf(-1.0f / 6.0f, bA, hC);
      t1 = tC; t3 = tA;
      f0 = p[(i + 2) * s];
    }
    const float e1 = fmaf(A1, A1, t1), e2 = fmaf(A2, A2, tB), e3 = fmaf(A3, A3, t3);
    const float em = fminf(e1, fminf(e2, e3));
    const float r1 = em * rcp(e1), r2 = em * rcp(e2), r3 = em * rcp(e3);
    const float a1 = 0.1f * (r1 * r1), a2 = 0.6f * (r2 * r2), a3 = 0.3f * (r3 * r3);
    const float v = fmaf(fmaf(a1, c1, fmaf(a2, c2, a3 * c3)), rcp(a1 + a2 + a3), f0);
    if (ACC) q[i * qs] += v;
    else q[i * qs] = v;
    dB = dC; dC = dD;
    bA = bB; tA = tB; bB = bC; tB = tC;
  }
}

// FP32 face flux of the Lax-Friedrichs split, unscaled.
__host__ __device__ __forceinline__ float weno5_lf(float p0, float p1, float p2, float p3,
                                                   float p4, float m1, float m2, float m3,
                                                   float m4, float m5) {
  return weno5(p0, p1, p2, p3, p4) + weno5(m5, m4, m3, m2, m1);
}

}  // namespace jh

namespace jh {

// Value and gradient of the FP64 weno5 with respect to its five arguments
// (the reverse mode of WENO5_JS.py:17-33 as JAX differentiates it):
//   dq/dv_j = sum_k w_k dq_k/dv_j + sum_k kappa_k de_k/dv_j,
//   kappa_k = -2 w_k (q_k - q) / e_k,  e_k = eps + IS_k,
// in the first and second differences of the FP32 weno5 above (q_k - q = c_k - sum_m
// w_m c_m; the FP64 value itself is taken from completed squares), with the three
// 1/e_k from 1/(e_1 e_2 e_3) and the weights' normaliser from the same
// reciprocal (e^7 stays in FP64 range for any e = eps + IS_k the split
// fluxes produce: 1e-42 at eps, 1e154 at IS = 1e22).  With A_k the halved first-
// derivative terms (IS_k = A_k^2 + 13/12 b_k^2), de_k/dv = 2 A_k dA_k/dv +
// 13/6 b_k db_k/dv, where dA_1 = (1/2, -2, 3/2, 0, 0), dA_2 = (0, -1/2, 0,
// 1/2, 0), dA_3 = (0, 0, 3/2, -2, 1/2) and db_1 = (1, -2, 1, 0, 0), db_2 =
// (0, 1, -2, 1, 0), db_3 = (0, 0, 1, -2, 1).
__host__ __device__ __forceinline__ double weno5_grad(double v0, double v1, double v2, double v3,
                                                      double v4, double (&g)[5]) {
  const double dA = v1 - v0, dB = v2 - v1, dC = v3 - v2, dD = v4 - v3;
  const double bA = dB - dA, bB = dC - dB, bC = dD - dC;
  const double hB = 0.5 * dB, hC = 0.5 * dC;
  const double A1 = fma(0.5, bA, dB), A2 = hB + hC, A3 = fma(0.5, bC, -dC);
  const double e1 = fma(A1, A1, fma((13.0 / 12.0) * bA, bA, 1e-6));
  const double e2 = fma(A2, A2, fma((13.0 / 12.0) * bB, bB, 1e-6));
  const double e3 = fma(A3, A3, fma((13.0 / 12.0) * bC, bC, 1e-6));
  const double E12 = e1 * e2, E13 = e1 * e3, E23 = e2 * e3;
  const double P1 = 0.1 * (E23 * E23), P2 = 0.6 * (E13 * E13), P3 = 0.3 * (E12 * E12);
  // R = 1 / sum(P) and iE = 1 / (e1 e2 e3) from one reciprocal
  const double S = P1 + P2 + P3, E = E12 * e3, X = rcp(E * S);
  const double R = E * X, iE = S * X;
  const double w1 = P1 * R, w2 = P2 * R, w3 = P3 * R;
  const double c1 = fma(1.0 / 3.0, bA, hB);
  const double c2 = fma(-1.0 / 6.0, bB, hC);
  const double c3 = fma(-1.0 / 6.0, bC, hC);
  const double cb = fma(w1, c1, fma(w2, c2, w3 * c3));
  // 2 kappa_k A_k and 13/6 kappa_k b_k
  const double m1 = -2.0 * (w1 * (E23 * iE)) * (c1 - cb);
  const double m2 = -2.0 * (w2 * (E13 * iE)) * (c2 - cb);
  const double m3 = -2.0 * (w3 * (E12 * iE)) * (c3 - cb);
  const double a1 = 2.0 * m1 * A1, a2 = 2.0 * m2 * A2, a3 = 2.0 * m3 * A3;
  const double b1 = (13.0 / 6.0) * m1 * bA, b2 = (13.0 / 6.0) * m2 * bB;
  const double b3 = (13.0 / 6.0) * m3 * bC;
  g[0] = w1 * (1.0 / 3.0) + 0.5 * a1 + b1;
  g[1] = w1 * (-7.0 / 6.0) + w2 * (-1.0 / 6.0) - 2.0 * (a1 + b1) - 0.5 * a2 + b2;
  g[2] = w1 * (11.0 / 6.0) + w2 * (5.0 / 6.0) + w3 * (1.0 / 3.0) + 1.5 * (a1 + a3) + b1 -
         2.0 * b2 + b3;
  g[3] = w2 * (1.0 / 3.0) + w3 * (5.0 / 6.0) + 0.5 * a2 + b2 - 2.0 * (a3 + b3);
  g[4] = w3 * (-1.0 / 6.0) + 0.5 * a3 + b3;
  return v2 + cb;
}

}  // namespace jh
