// pda_physics.hpp -- device-side numerics of the finite-volume hot path:
// WENO3/WENO5 reconstruction (values and stencil gradients) and the face
// fluxes with their exact Jacobians for every family.
//
// Formulas follow the reference files cited per function; evaluation order
// is kept close to them, and FP64 throughout.
#pragma once
#include <hip/hip_runtime.h>

namespace pda {
namespace phys {

constexpr double kEs = 1.e-30;

// 1 / d from the hardware estimate (2^-24) and one third-order step: within an
// ulp for d and 1 / d in the normal range
__device__ __forceinline__ double frcp(double d) {
  const double r = __builtin_amdgcn_rcp(d);
  const double e = __fma_rn(-d, r, 1.);
  return __fma_rn(r, __fma_rn(e, e, e), r);
}

// n / d from that and one residual correction: within an ulp of the rounded
// quotient for d and n / d in the normal range (the densities and the Roe
// factors of the velocity's fluxes), without the IEEE division sequence's
// scaling for denormal and infinite operands.
__device__ __forceinline__ double fdiv(double n, double d) {
  const double r = frcp(d);
  const double q = n * r;
  return __fma_rn(r, __fma_rn(-d, q, n), q);
}

// sqrt(x) by Goldschmidt's iteration from the hardware reciprocal root: one step
// and two residual corrections.  The addend keeps 0 (a state at rest) from giving
// 0 * inf; it is lost in every x above 1e-284, and below 1e-300, where the root
// is lost beside the speed of sound it is added to, the result is too small.
// x < 0 gives NaN, and so does an infinite x: where a finite state's enthalpy
// overflows, its flux is not finite either way (choosing the argument for 0 and
// infinity by its class instead cost 0.8 % of the velocities and the 1D steps).
__device__ __forceinline__ double fsqrt(double x) {
  const double y = __builtin_amdgcn_rsq(x + 1e-300);
  double g = x * y, h = 0.5 * y;
  const double r = __fma_rn(-h, g, 0.5);
  g = __fma_rn(g, r, g);
  h = __fma_rn(h, r, h);
  g = __fma_rn(__fma_rn(-g, g, x), h, g);
  return __fma_rn(__fma_rn(-g, g, x), h, g);
}

// 1 / sqrt(x) from the hardware estimate and one third-order step: within an ulp
// or two for x in the normal range
__device__ __forceinline__ double frsqrt(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = __fma_rn(-x * y, y, 1.);
  return __fma_rn(y * e, __fma_rn(0.375, e, 0.5), y);
}

// ---------------------------------------------------------------- WENO3
// impl/weno3.hpp:134-246: values plus d(face)/d(q_j), j = 0..3, in the
// reference's expression forms without FMA contraction: its terms cancel where
// the smoothness indicators are small, and only their own roundings follow it
// to 1e-12 (differentiated as WENO5 below, the gradients are a thousand times
// nearer to extended precision and up to 3e-12 from the reference's).  The
// quotients are fdiv's, rounded as the IEEE sequence rounds them but for rare
// last places.  S and the numerators over S^2 carry powers of two (exact, no
// other bits), as S^2 is 1 / B^4 and would leave the normal range at cell
// differences of 1e38; with them the gradients hold to 2e41.
__device__ __forceinline__ void weno3_grad(const double *q, double &un, double &up,
                                           double *gn, double *gp) {
#pragma clang fp contract(off)
  constexpr double eps = 1.e-6, c13 = 1. / 3., c23 = 2. / 3., KS = 0x1p46, KS2 = 0x1p92;
  {
    const double qim1 = q[0], qi = q[1], qip1 = q[2];
    const double p0 = (-qim1 + 3. * qi) * 0.5, p1 = (qi + qip1) * 0.5;
    const double d0 = qim1 - qi, d1 = qi - qip1;
    const double B0 = d0 * d0, B1 = d1 * d1;
    const double a0 = fdiv(c13, eps * eps + 2. * eps * B0 + B0 * B0);
    const double a1 = fdiv(c23, eps * eps + 2. * eps * B1 + B1 * B1);
    const double s = fdiv(1., a0 + a1);
    const double e0 = B0 + eps, e1 = B1 + eps;
    const double e03 = e0 * e0 * e0, e13 = e1 * e1 * e1;
    const double S = fdiv(2. * KS, 3. * (e1 * e1)) + fdiv(KS, 3. * (e0 * e0));
    const double S2 = S * S;
    const double x0 = fdiv(4. * d0, 3. * e03), x1 = fdiv(8. * d1, 3. * e13);
    const double da0[3] = {-x0, x0, 0.};
    const double da1[3] = {0., -x1, x1};
    const double ds[3] = {fdiv((4. * KS2) * d0, 3. * e03 * S2), -fdiv(KS2 * (x0 - x1), S2),
                          -fdiv((8. * KS2) * d1, 3. * S2 * e13)};
    const double dp0[3] = {-0.5, 1.5, 0.}, dp1[3] = {0., 0.5, 0.5};
    const double w0 = a0 * s, w1 = a1 * s;
    for (int i = 0; i < 3; ++i) {
      double v = (da0[i] * s + ds[i] * a0) * p0 + dp0[i] * w0;
      v += (da1[i] * s + ds[i] * a1) * p1 + dp1[i] * w1;
      gn[i] = v;
    }
    gn[3] = 0.;
    un = w0 * p0 + w1 * p1;
  }
  {
    const double qi = q[1], qip1 = q[2], qip2 = q[3];
    const double p0 = (qi + qip1) * 0.5, p1 = (3. * qip1 - qip2) * 0.5;
    const double d0 = qi - qip1, d1 = qip1 - qip2;
    const double B0 = d0 * d0, B1 = d1 * d1;
    const double a0 = fdiv(c23, eps * eps + 2. * eps * B0 + B0 * B0);
    const double a1 = fdiv(c13, eps * eps + 2. * eps * B1 + B1 * B1);
    const double s = fdiv(1., a0 + a1);
    const double w0 = a0 * s, w1 = a1 * s;
    const double e0 = B0 + eps, e1 = B1 + eps;
    const double e03 = e0 * e0 * e0, e13 = e1 * e1 * e1;
    const double S = fdiv(KS, 3. * (e1 * e1)) + fdiv(2. * KS, 3. * (e0 * e0));
    const double S2 = S * S;
    const double x0 = fdiv(8. * d0, 3. * e03), x1 = fdiv(4. * d1, 3. * e13);
    const double da0[3] = {-x0, x0, 0.};
    const double da1[3] = {0., -x1, x1};
    const double ds[3] = {fdiv((8. * KS2) * d0, 3. * e03 * S2), -fdiv(KS2 * (x0 - x1), S2),
                          -fdiv((4. * KS2) * d1, 3. * S2 * e13)};
    const double dp0[3] = {0.5, 0.5, 0.}, dp1[3] = {0., 1.5, -0.5};
    for (int i = 0; i < 3; ++i) {
      double v = (da0[i] * s + ds[i] * a0) * p0 + dp0[i] * w0;
      v += (da1[i] * s + ds[i] * a1) * p1 + dp1[i] * w1;
      gp[i + 1] = v;
    }
    gp[0] = 0.;
    up = w0 * p0 + w1 * p1;
  }
}

// ---------------------------------------------------------------- WENO5
// Reconstruction (impl/weno5.hpp:56-178) as a correction to the cell's value.
// With the differences e_k = q_k - q_{k-1} of the cells q_0 .. q_4 about cell
// q_2, the candidates at the face towards q_3 are
//   p_0 = q_2 + (5 e_2 - 2 e_1) / 6, p_1 = q_2 + (e_2 + 2 e_3) / 6,
//   p_2 = q_2 + (4 e_3 - e_4) / 6,
// and with E_k = 4 (eps + B_k) the weights d_k / (eps + B_k)^2 are as
// d_k Prod_{j != k} E_j^2: one division per value, of the correction only, so
// that its rounding (a few ulps) counts in the correction's size, not the
// value's.  4 B = 13/3 t^2 + s^2 with t the second difference of the window
// and s its first (centred or one-sided).  Equal to the reference's weighted
// sum in exact arithmetic.  The operations are fixed (explicit FMAs) and the
// same for a window read from either side, so a face value does not depend on
// which of the forms below gives it.  58 operations for the two values of a cell
// (85 as weighted candidates with the B's and their squares formed apart).
// The products of the E's are of the eighth degree in the differences, and with
// the differences they multiply they overflow, which gives NaN, where those
// reach about 2e33.  WIDE: the products carry 2^-350 (two multiplications, exact:
// no other bits), which moves that to 6e56 and keeps every term normal for
// differences down to 1e-75.  The general row kernels and the 1D steps take it (the
// form with a division per weight held to 1e77 there); the box kernels, bound by
// FP64 issue, do not (their earlier weights, of the same degree, held to 6e33).
struct W5 {
  double e1, e2, e3, e4; // the differences
  double s0, s1, s2;     // Prod E^2 without window 0, 6 times without 1, without 2
};
template <bool WIDE = false>
__device__ __forceinline__ W5 w5_window(double q0, double q1, double q2, double q3, double q4) {
  constexpr double eps4 = 4.e-6, c133 = 13. / 3.;
  W5 w;
  w.e1 = q1 - q0;
  w.e2 = q2 - q1;
  w.e3 = q3 - q2;
  w.e4 = q4 - q3;
  const double t0 = w.e2 - w.e1, t1 = w.e3 - w.e2, t2 = w.e4 - w.e3;
  const double a0 = __fma_rn(2., w.e2, t0), a1 = w.e2 + w.e3, a2 = __fma_rn(-2., w.e3, t2);
  const double E0 = __fma_rn(c133 * t0, t0, __fma_rn(a0, a0, eps4));
  const double E1 = __fma_rn(c133 * t1, t1, __fma_rn(a1, a1, eps4));
  const double E2 = __fma_rn(c133 * t2, t2, __fma_rn(a2, a2, eps4));
  constexpr double scale = WIDE ? 0x1p-350 : 1.;
  const double E0s = scale * E0, E2s = scale * E2;
  const double p0 = E1 * E2s, p1 = E0 * E2s, p2 = E0s * E1;
  w.s0 = p0 * p0;
  w.s1 = 6. * (p1 * p1);
  w.s2 = p2 * p2;
  return w;
}
// n / d for the correction: within two ulps
__device__ __forceinline__ double w_quot(double n, double d) { return n * frcp(d); }
// value of cell q2 at the face towards q3
__device__ __forceinline__ double w5_hi(const W5 &w, double q2) {
  constexpr double c16 = 1. / 6.;
  const double m2 = 3. * w.s2;
  const double n = __fma_rn(m2, __fma_rn(4., w.e3, -w.e4),
                            __fma_rn(w.s1, __fma_rn(2., w.e3, w.e2), w.s0 * __fma_rn(5., w.e2, -2. * w.e1)));
  return __fma_rn(c16, w_quot(n, (w.s0 + w.s1) + m2), q2);
}
// value of cell q2 at the face towards q1: w5_hi of the reversed cells
__device__ __forceinline__ double w5_lo(const W5 &w, double q2) {
  constexpr double c16 = 1. / 6.;
  const double m0 = 3. * w.s0;
  const double n = __fma_rn(m0, __fma_rn(4., w.e2, -w.e1),
                            __fma_rn(w.s1, __fma_rn(2., w.e2, w.e3), w.s2 * __fma_rn(5., w.e3, -2. * w.e4)));
  return __fma_rn(-c16, w_quot(n, (w.s2 + w.s1) + m0), q2);
}
// the left-biased value: of cell q2 at the face towards q3
template <bool WIDE = false>
__device__ __forceinline__ double weno5_side_1div(double q0, double q1, double q2, double q3,
                                                  double q4) {
  return w5_hi(w5_window<WIDE>(q0, q1, q2, q3, q4), q2);
}

// Both face values of one cell from q = cells i-2 .. i+2: hi = the left
// state of face i+1/2, lo = the right state of face i-1/2 (the left-biased value
// of the reversed cells).  Bit-identical to the two weno5_side_1div calls at
// those faces; the windows are formed once.
template <bool WIDE = false>
__device__ __forceinline__ void weno5_cell_1div(double q0, double q1, double q2, double q3,
                                                double q4, double &hi, double &lo) {
  const W5 w = w5_window<WIDE>(q0, q1, q2, q3, q4);
  hi = w5_hi(w, q2);
  lo = w5_lo(w, q2);
}

// WENO3 counterparts (impl/weno3.hpp:56-132): D = (eps + B)^2 of the two-cell
// window (a, b) with B = (a - b)^2, the same in either direction, and the
// values as corrections: the candidates at the face of b towards c are
// b + (b - a) / 2 and b + (c - b) / 2 with weights 1/3 and 2/3.  WIDE: D carries
// 2^-300, and the values hold over the whole range of D (differences of 1e77;
// 1e61 without).
template <bool WIDE = false>
__device__ __forceinline__ double w3_d(double a, double b) {
  constexpr double eps = 1.e-6, scale = WIDE ? 0x1p-300 : 1.;
  const double d = a - b, E = __fma_rn(d, d, eps);
  return E * (scale * E);
}
// the face values of cell b (neighbours a below, c above) from the windows'
// D: hi at the face towards c, lo at the face towards a
__device__ __forceinline__ double w3_hi(double a, double b, double c, double Dab, double Dbc) {
  const double m = 2. * Dab;
  return __fma_rn(0.5, w_quot(__fma_rn(m, c - b, Dbc * (b - a)), Dbc + m), b);
}
__device__ __forceinline__ double w3_lo(double a, double b, double c, double Dab, double Dbc) {
  return w3_hi(c, b, a, Dbc, Dab);
}
// the left-biased value: of cell b at the face towards c
template <bool WIDE = false>
__device__ __forceinline__ double weno3_side_1div(double a, double b, double c) {
  return w3_hi(a, b, c, w3_d<WIDE>(a, b), w3_d<WIDE>(b, c));
}
// both face values of cell b, bit-identical to weno3_side_1div's at its faces
template <bool WIDE = false>
__device__ __forceinline__ void weno3_cell_1div(double a, double b, double c, double &hi, double &lo) {
  const double Dab = w3_d<WIDE>(a, b), Dbc = w3_d<WIDE>(b, c);
  hi = w3_hi(a, b, c, Dab, Dbc);
  lo = w3_lo(a, b, c, Dab, Dbc);
}

// Values with their gradients (impl/weno5.hpp:180-434).
// With weights w_k, candidate corrections c_k and their weighted sum c,
//   d value / d e = Sum w_k d c_k / d e - 2 w_k (c_k - c) / E_k d E_k / d e
// over the cell differences e, of which a window's E_k holds two; the
// gradient by the cells is the difference of that by their differences, plus 1
// at the value's own cell.  The reference differentiates weighted cell values:
// its terms are as large as value / sqrt(eps) and cancel.  Here c_k - c is of
// the size of the differences: on states of 1 % noise the largest error against
// extended precision is 3e-15 where the reference's form has 5e-12, with two
// reciprocals and about 90 operations a value instead of eight divisions and
// about 260.  The 2D Euler WENO5 Jacobian with velocity of 509 x 387 cells is
// bound by FP64 issue: 109 us (138 in the reference's form).
// The products of the E_k carry 2^-250 (two multiplications, no other bits): of
// the eighth degree in the differences, they would overflow at 2e33 to 1e38,
// where the reference's form holds to 1e39; with it the gradients hold to 8e49.

// q = cells i-2 .. i+2: the value of cell i at the face towards i+1 (w5_hi's,
// bit for bit) and its gradient by the five cells
__device__ __forceinline__ double weno5_side_grad(double q0, double q1, double q2, double q3, double q4,
                                                  double &g0, double &g1, double &g2, double &g3, double &g4) {
  constexpr double eps4 = 4.e-6, c133 = 13. / 3., c16 = 1. / 6.;
  const double e1 = q1 - q0, e2 = q2 - q1, e3 = q3 - q2, e4 = q4 - q3;
  const double t0 = e2 - e1, t1 = e3 - e2, t2 = e4 - e3;
  const double a0 = __fma_rn(2., e2, t0), a1 = e2 + e3, a2 = __fma_rn(-2., e3, t2);
  const double k0 = c133 * t0, k1 = c133 * t1, k2 = c133 * t2;
  const double E0 = __fma_rn(k0, t0, __fma_rn(a0, a0, eps4));
  const double E1 = __fma_rn(k1, t1, __fma_rn(a1, a1, eps4));
  const double E2 = __fma_rn(k2, t2, __fma_rn(a2, a2, eps4));
  const double E0s = 0x1p-250 * E0, E2s = 0x1p-250 * E2;
  const double p0 = E1 * E2s, p1 = E0 * E2s, p2 = E0s * E1;
  const double s0 = p0 * p0, s1 = 6. * (p1 * p1), m2 = 3. * (p2 * p2);
  const double iD = frcp((s0 + s1) + m2), iE = -4. * frcp(p0 * E0);
  const double c0 = __fma_rn(5., e2, -2. * e1), c1 = __fma_rn(2., e3, e2), c2 = __fma_rn(4., e3, -e4);
  const double c = __fma_rn(m2, c2, __fma_rn(s1, c1, s0 * c0)) * iD;
  // weights and, as the candidates are six times the corrections, a sixth of them
  const double iD6 = c16 * iD;
  const double w0 = s0 * iD6, w1 = s1 * iD6, w2 = m2 * iD6;
  // a window's E is 4 (eps + B): d E_0 = -2 (k0 + a0) d e1 + 2 (k0 + 3 a0) d e2 and so on
  const double f0 = (w0 * (c0 - c)) * (p0 * iE), f1 = (w1 * (c1 - c)) * (p1 * iE), f2 = (w2 * (c2 - c)) * (p2 * iE);
  const double G1 = -__fma_rn(f0, k0 + a0, 2. * w0);
  const double G2 = __fma_rn(f0, __fma_rn(3., a0, k0), __fma_rn(f1, a1 - k1, __fma_rn(5., w0, w1)));
  const double G3 = __fma_rn(-f2, __fma_rn(3., a2, k2), __fma_rn(f1, a1 + k1, __fma_rn(4., w2, 2. * w1)));
  const double G4 = __fma_rn(f2, k2 + a2, -w2);
  g0 = -G1;
  g1 = G1 - G2;
  g2 = 1. + (G2 - G3);
  g3 = G3 - G4;
  g4 = G4;
  return __fma_rn(c16, c, q2);
}

// q = {q_{i-2}, ..., q_{i+3}}: values plus d(face)/d(q_j), j = 0..5
// (gn[5] = gp[0] = 0); the right state is the reversed cells' left state
__device__ __forceinline__ void weno5_grad(const double *q, double &un, double &up,
                                           double *gn, double *gp) {
  un = weno5_side_grad(q[0], q[1], q[2], q[3], q[4], gn[0], gn[1], gn[2], gn[3], gn[4]);
  up = weno5_side_grad(q[5], q[4], q[3], q[2], q[1], gp[5], gp[4], gp[3], gp[2], gp[1]);
  gn[5] = gp[0] = 0.;
}

// ------------------------------------------------------------ Euler
// Rusanov flux for 1, 2, 3 dimensions (M = DIM+2 conserved variables),
// impl/euler_rusanov_flux_values_function.hpp:54-208.  A = face normal axis.
template <int DIM, int A>
__device__ __forceinline__ void euler_flux(const double *qL, const double *qR, double g,
                                           double *F) {
  constexpr int M = DIM + 2;
  const double half = 0.5;
  double velL[DIM], velR[DIM];
  const double rL = qL[0], rR = qR[0];
  // one reciprocal per side (the reference divides per component)
  const double iL = fdiv(1., rL + kEs), iR = fdiv(1., rR + kEs);
  double v2L = 0., v2R = 0.;
  for (int d = 0; d < DIM; ++d) {
    velL[d] = qL[1 + d] * iL;
    velR[d] = qR[1 + d] * iR;
    v2L += velL[d] * velL[d];
    v2R += velR[d] * velR[d];
  }
  const double unL = velL[A], unR = velR[A];
  const double pL = (g - 1.) * (qL[M - 1] - half * rL * v2L);
  const double pR = (g - 1.) * (qR[M - 1] - half * rR * v2R);
  const double HL = (qL[M - 1] + pL) * iL, HR = (qR[M - 1] + pR) * iR;
  double FL[M], FR[M];
  FL[0] = rL * unL;
  FR[0] = rR * unR;
  for (int d = 0; d < DIM; ++d) {
    FL[1 + d] = rL * unL * velL[d] + (d == A ? pL : 0.);
    FR[1 + d] = rR * unR * velR[d] + (d == A ? pR : 0.);
  }
  FL[M - 1] = rL * unL * HL;
  FR[M - 1] = rR * unR * HR;
  const double RT = fsqrt(rR * iL);
  const double inv = frcp(1. + RT);
  double vr2 = 0.;
  for (int d = 0; d < DIM; ++d) {
    const double v = (velL[d] + RT * velR[d]) * inv;
    vr2 += v * v;
  }
  const double H = (HL + RT * HR) * inv;
  const double a = fsqrt((g - 1.) * (H - half * vr2));
  const double smax = (DIM == 1 ? fabs((velL[0] + RT * velR[0]) * inv) : fsqrt(vr2)) + a;
  for (int i = 0; i < M; ++i) F[i] = half * (FL[i] + FR[i] + smax * (qL[i] - qR[i]));
}

// exact Jacobians of the Rusanov flux w.r.t. the left and right states,
// including the derivative of the Roe-averaged wave speed,
// impl/euler_rusanov_flux_jacobian_function.hpp:54-406.
//
// Each side's M x M block has the form
//   J_s = 1/2 A(q_s) +- 1/2 smax I + 1/2 grad_s (qL - qR)^T-outer,
// i.e. J_s(i,j) = 1/2 A_s(i,j) + [i==j] dsm + 1/2 grad_s[j] dq[i], where A_s
// is the physical flux Jacobian along axis A at the side's state.  EulerSide
// keeps the factors (side velocity, |v|^2, total enthalpy, gradient of smax,
// dq and the signed diagonal term); entries are formed on demand, so a
// kernel can stream a block to memory without holding all M*M values.  The
// reciprocals and roots are the hardware's refined to an ulp or so, and the Roe
// factors come from them by products: about 50 operations where nine divisions
// and five roots of the library took 170.  2D WENO5 Jacobian with velocity of
// 509 x 387 cells 101 -> 93 us, first-order Jacobian of 48 x 40 cells 8.8 -> 7.7 us.
template <int DIM> struct EulerSide {
  double vel[DIM], V2, H, grad[DIM + 2], dq[DIM + 2], dsm;
};

template <int DIM, int A>
__device__ __forceinline__ void euler_sides(const double *qL, const double *qR, double gamma,
                                            EulerSide<DIM> &L, EulerSide<DIM> &R) {
  constexpr int M = DIM + 2;
  const double half = 0.5, gm1 = gamma - 1.;
  const double igm1 = frcp(gm1);
  const double iL = frcp(qL[0] + kEs), iR = frcp(qR[0] + kEs);
  double aa[2];
  {
    L.V2 = 0.;
    R.V2 = 0.;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      L.vel[d] = qL[1 + d] * iL;
      R.vel[d] = qR[1 + d] * iR;
      L.V2 += L.vel[d] * L.vel[d];
      R.V2 += R.vel[d] * R.vel[d];
    }
    const double pL = gm1 * (qL[M - 1] - half * qL[0] * L.V2);
    const double pR = gm1 * (qR[M - 1] - half * qR[0] * R.V2);
    L.H = (qL[M - 1] + pL) * iL;
    R.H = (qR[M - 1] + pR) * iR;
    aa[0] = gm1 * (L.H - half * L.V2);
    aa[1] = gm1 * (R.H - half * R.V2);
  }
  const double RT = fsqrt(qR[0] * iL), inv = frcp(1. + RT);
  double vR[DIM];
  double vr2 = 0.;
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    vR[d] = (L.vel[d] + RT * R.vel[d]) * inv;
    vr2 += vR[d] * vR[d];
  }
  const double Hr = (L.H + RT * R.H) * inv;
  const double a2 = gm1 * (Hr - half * vr2), ia = frsqrt(a2), a1 = a2 * ia;
  const double a = __fma_rn(__fma_rn(-a1, a1, a2), half * ia, a1);
  const double VMagSqrRoe = vr2 + kEs;
  const double rs = frsqrt(VMagSqrRoe);
  const double smax = (DIM == 1 ? fabs(vR[0]) : vr2 * rs) + a; // vr2 rs = 0 at rest
  double rel[DIM];
#pragma unroll
  for (int d = 0; d < DIM; ++d) rel[d] = vR[d] * rs;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    EulerSide<DIM> &S = s ? R : L;
    double VV = 0.;
#pragma unroll
    for (int d = 0; d < DIM; ++d) VV += S.vel[d] * vR[d];
    const double f = s ? iR * RT * inv : iL * inv; // 1 / (rho_s + sqrt(rhoL rhoR))
    double g0 = 0.;
#pragma unroll
    for (int d = 0; d < DIM; ++d) g0 -= half * (S.vel[d] + vR[d]) * rel[d];
    g0 += half * gm1 * ia *
          (half * (VMagSqrRoe + VV) + half * (S.H - Hr) - aa[s] * igm1 + half * (gamma - 2.) * S.V2);
    S.grad[0] = f * g0;
#pragma unroll
    for (int d = 0; d < DIM; ++d) S.grad[1 + d] = f * (rel[d] - half * (gm1 * (vR[d] + gm1 * S.vel[d])) * ia);
    S.grad[M - 1] = half * f * gamma * gm1 * ia;
#pragma unroll
    for (int i = 0; i < M; ++i) S.dq[i] = qL[i] - qR[i];
    S.dsm = s ? -half * smax : half * smax;
  }
}

// entry (i, j) of one side's block; i and j are compile-time after unrolling
template <int DIM, int A>
__device__ __forceinline__ double euler_side_entry(const EulerSide<DIM> &S, double gamma, int i,
                                                   int j) {
  constexpr int M = DIM + 2;
  const double half = 0.5, gm1 = gamma - 1.;
  const double uX = S.vel[A];
  double v;
  if (i == 0) {
    v = (j == 1 + A) ? half : 0.;
  } else if (i <= DIM) {
    const int ii = i - 1;
    if (j == 0) {
      v = half * ((ii == A ? half * gm1 * S.V2 : 0.) - S.vel[ii] * uX);
    } else if (j <= DIM) {
      const int d = j - 1;
      double w = (d == A ? S.vel[ii] : 0.) - (ii == A ? gm1 * S.vel[d] : 0.);
      if (d == ii) w += uX;
      v = half * w;
    } else {
      v = (ii == A ? half * gm1 : 0.);
    }
  } else {
    if (j == 0) v = half * ((half * gm1 * S.V2 - S.H) * uX);
    else if (j <= DIM) v = half * ((j - 1 == A ? S.H : 0.) - gm1 * S.vel[j - 1] * uX);
    else v = half * gamma * uX;
  }
  if (i == j) v += S.dsm;
  return v + half * S.grad[j] * S.dq[i];
}

// JL, JR row-major M x M
template <int DIM, int A>
__device__ __forceinline__ void euler_fjac(const double *qL, const double *qR, double gamma,
                                           double *JL, double *JR) {
  constexpr int M = DIM + 2;
  EulerSide<DIM> L, R;
  euler_sides<DIM, A>(qL, qR, gamma, L, R);
#pragma unroll
  for (int i = 0; i < M; ++i)
#pragma unroll
    for (int j = 0; j < M; ++j) {
      JL[i * M + j] = euler_side_entry<DIM, A>(L, gamma, i, j);
      JR[i * M + j] = euler_side_entry<DIM, A>(R, gamma, i, j);
    }
}

// ------------------------------------------------------- shallow water
// impl/swe_rusanov_flux_values_function.hpp:54-97
template <int A>
__device__ __forceinline__ void swe_flux(const double *qL, const double *qR, double g, double *F) {
  // one reciprocal per side (the reference divides per component)
  const double hL = qL[0], iL = fdiv(1., hL + kEs), uL = qL[1] * iL, vL = qL[2] * iL;
  const double hR = qR[0], iR = fdiv(1., hR + kEs), uR = qR[1] * iR, vR = qR[2] * iR;
  const double unL = A == 0 ? uL : vL, unR = A == 0 ? uR : vR;
  const double pL = 0.5 * g * hL * hL, pR = 0.5 * g * hR * hR;
  double FL[3], FR[3];
  FL[0] = hL * unL; FL[1] = hL * unL * uL + (A == 0 ? pL : 0.); FL[2] = hL * unL * vL + (A == 1 ? pL : 0.);
  FR[0] = hR * unR; FR[1] = hR * unR * uR + (A == 0 ? pR : 0.); FR[2] = hR * unR * vR + (A == 1 ? pR : 0.);
  const double hm = 0.5 * (hL + hR);
  // the Roe average's weights sqrt(h), both divided by sqrt(hL)
  const double RT = fsqrt(hR * iL);
  const double um = fdiv(unL + RT * unR, 1. + RT);
  const double c = fsqrt(g * hm);
  // sqrt(x * x) is |x| exactly in IEEE arithmetic (no overflow here)
  const double smax = fabs(um) + fabs(c);
  for (int i = 0; i < 3; ++i) F[i] = 0.5 * (FL[i] + FR[i] + smax * (qL[i] - qR[i]));
}

// impl/swe_rusanov_flux_jacobian_function.hpp:54-137
template <int A>
__device__ __forceinline__ void swe_fjac(const double *qL, const double *qR, double g,
                                         double *JL, double *JR) {
  const double n0 = A == 0 ? 1. : 0., n1 = A == 1 ? 1. : 0.;
  const double hL = qL[0], uL = qL[1] / (hL + kEs), vL = qL[2] / (hL + kEs);
  const double hR = qR[0], uR = qR[1] / (hR + kEs), vR = qR[2] / (hR + kEs);
  const double unL = A == 0 ? uL : vL, unR = A == 0 ? uR : vR;
  const double hm = 0.5 * (hL + hR);
  const double sL = sqrt(hL), sR = sqrt(hR);
  const double um = (unL * sL + unR * sR) / (sL + sR + kEs);
  const double smax = fabs(um) + fabs(sqrt(g * hm));
  const double termL = (n0 * qL[1] + n1 * qL[2]) / (qL[0] * qL[0]);
  const double termR = (n0 * qR[1] + n1 * qR[2]) / (qR[0] * qR[0]);
  const double hsun = sL * unL + sR * unR + kEs;
  const double ahs = fabs(hsun), ssum = sL + sR;
  const double gterm = g / (2.8284271247461903 * sqrt(g * (hL + hR)));
  double dL[3], dR[3];
  dL[0] = -ahs / (2. * sL * (ssum * ssum)) + (0.5 * unL / sL - sL * termL) * hsun / (ssum * ahs) + gterm;
  dL[1] = n0 * hsun / (sL * ssum * ahs);
  dL[2] = n1 * hsun / (sL * ssum * ahs);
  dR[0] = -ahs / (2. * sR * (ssum * ssum)) + (0.5 * unR / sR - sR * termR) * hsun / (ssum * ahs) + gterm;
  dR[1] = n0 * hsun / (sR * ssum * ahs);
  dR[2] = n1 * hsun / (sR * ssum * ahs);
  const double dq0 = qR[0] - qL[0], dq1 = qR[1] - qL[1], dq2 = qR[2] - qL[2];
  JL[0] = -0.5 * dL[0] * dq0 + 0.5 * (n0 * uL + n1 * vL - qL[0] * termL) + 0.5 * smax;
  JL[1] = 0.5 * n0 - 0.5 * dL[1] * dq0;
  JL[2] = 0.5 * n1 - 0.5 * dL[2] * dq0;
  JL[3] = 0.5 * (g * n0 * qL[0] - qL[1] * termL) - 0.5 * dL[0] * dq1;
  JL[4] = n0 * uL + 0.5 * n1 * vL + 0.5 * smax - 0.5 * dL[1] * dq1;
  JL[5] = 0.5 * n1 * uL - 0.5 * dL[2] * dq1;
  JL[6] = 0.5 * (g * n1 * qL[0] - qL[2] * termL) - 0.5 * dL[0] * dq2;
  JL[7] = 0.5 * n0 * vL - 0.5 * dL[1] * dq2;
  JL[8] = n1 * vL + 0.5 * n0 * uL + 0.5 * smax - 0.5 * dL[2] * dq2;
  JR[0] = -0.5 * dR[0] * dq0 + 0.5 * (n0 * uR + n1 * vR - qR[0] * termR) - 0.5 * smax;
  JR[1] = 0.5 * n0 - 0.5 * dR[1] * dq0;
  JR[2] = 0.5 * n1 - 0.5 * dR[2] * dq0;
  JR[3] = 0.5 * (g * n0 * qR[0] - qR[1] * termR) - 0.5 * dR[0] * dq1;
  JR[4] = n0 * uR + 0.5 * n1 * vR - 0.5 * smax - 0.5 * dR[1] * dq1;
  JR[5] = 0.5 * n1 * uR - 0.5 * dR[2] * dq1;
  JR[6] = 0.5 * (g * n1 * qR[0] - qR[2] * termR) - 0.5 * dR[0] * dq2;
  JR[7] = 0.5 * n0 * vR - 0.5 * dR[1] * dq2;
  JR[8] = n1 * vR + 0.5 * n0 * uR - 0.5 * smax - 0.5 * dR[2] * dq2;
}

// ------------------------------------------------------------ Burgers
// impl/advection_diffusion_2d_flux_functions.hpp:54-114
template <int A>
__device__ __forceinline__ void burgers_flux(const double *qL, const double *qR, double *F) {
  const double a0 = fmax(fabs(qL[0]), fabs(qR[0]));
  const double a1 = fmax(fabs(qL[1]), fabs(qR[1]));
  const double cross = qL[0] * qL[1] + qR[0] * qR[1];
  double f0 = a0 * (qL[0] - qR[0]);
  double f1 = a1 * (qL[1] - qR[1]);
  if (A == 0) {
    f0 += qL[0] * qL[0] + qR[0] * qR[0];
    f1 += cross;
  } else {
    f0 += cross;
    f1 += qL[1] * qL[1] + qR[1] * qR[1];
  }
  F[0] = f0 * 0.25;
  F[1] = f1 * 0.25;
}

template <int A>
__device__ __forceinline__ void burgers_fjac(const double *qL, const double *qR, double *JL,
                                             double *JR) {
  const double n0 = A == 0 ? 1. : 0., n1 = A == 1 ? 1. : 0.;
  if (fabs(qL[0]) > fabs(qR[0])) {
    JL[0] = (2. * qL[0] - qR[0]) * copysign(1., qL[0]) + n0 * 2. * qL[0] + n1 * qL[1];
    JR[0] = n0 * 2. * qR[0] + n1 * qR[1] - fabs(qL[0]);
  } else {
    JL[0] = n0 * 2. * qL[0] + n1 * qL[1] + fabs(qR[0]);
    JR[0] = (qL[0] - 2. * qR[0]) * copysign(1., qR[0]) + n0 * 2. * qR[0] + n1 * qR[1];
  }
  if (fabs(qL[1]) > fabs(qR[1])) {
    JL[3] = (2. * qL[1] - qR[1]) * copysign(1., qL[1]) + n0 * qL[0] + n1 * 2. * qL[1];
    JR[3] = n0 * qR[0] + n1 * 2. * qR[1] - fabs(qL[1]);
  } else {
    JL[3] = n0 * qL[0] + n1 * 2. * qL[1] + fabs(qR[1]);
    JR[3] = (qL[1] - 2. * qR[1]) * copysign(1., qR[1]) + n0 * qR[0] + n1 * 2. * qR[1];
  }
  JL[0] *= 0.25; JR[0] *= 0.25; JL[3] *= 0.25; JR[3] *= 0.25;
  JL[1] = n1 * qL[0] * 0.25;
  JL[2] = n0 * qL[1] * 0.25;
  JR[1] = n1 * qR[0] * 0.25;
  JR[2] = n0 * qR[1] * 0.25;
}

}  // namespace phys
}  // namespace pda
