// bond_fast64.h -- FP64 bond arithmetic of the LDS-staged step kernels.
//
// The step kernels of the FP64 modes are bound by FP64 instructions, so the
// operations that the compiler expands into long sequences (IEEE division
// and square root with their range scaling, exp) are written here for the
// range that a bond's quantities have:
//
//  sqrt and quotients of the exact mode are the bits of the IEEE operations
//  (measured, not proven: of 6.3e9 random operands of each, none differs):
//  Goldschmidt's iteration from the hardware's reciprocal square root, then
//  Markstein's final step q' = q + (a - b q) y with the residual taken by a
//  fused multiply-add (P. Markstein, "Software division and square root using
//  Goldschmidt's algorithms", RNC6, 2004).  One iteration gives the length,
//  its reciprocal and the square's reciprocal together, so the quotients
//  S = dx.du / |dx|^2 and dx / |dx|
//  take three operations each.  No range scaling: the lengths of a mesh lie
//  far inside the exponent range (checked at setup, kStagedLenMin/Max).
//
//  exp of the softening factor: the exponent x = -beta r S^2 of a bond that
//  does not break lies in [-0.5 f^2 (1 + 2e-5), 0], f the critical-stretch
//  factor; with f <= 1 one polynomial covers it with no range reduction
//  (0.88 ulp against high-precision arithmetic; the general form 0.89 ulp; the
//  library's exp 0.5).
//  The coefficients interpolate (exp(x) - 1)/x at Chebyshev points.
//
// Every decision keeps the rule of bond_rnp.h: a bond inside a guard band is
// decided by the exact evaluation after the chunk.  The break test's
// comparisons here are written so that a NaN counts as inside the band.
#pragma once

#include "bond_rnp.h"

namespace nlm {

// Range of the horizon and lower bound of the mesh size that the sequences
// below take without range scaling.
constexpr double kStagedLenMin = 1e-100;
constexpr double kStagedLenMax = 1e100;

// Largest magnitude of x = -beta r S^2 that exp_short covers.
constexpr double kExpShortMax = 0.5002;

// exp(x) for x in [-kExpShortMax, 0].
__device__ __forceinline__ double exp_short(double x) {
  double p = 0x1.56a791f54e36fp-26;
  p = __builtin_fma(p, x, 0x1.21a336bd8a5b8p-22);
  p = __builtin_fma(p, x, 0x1.715a79339fcd5p-19);
  p = __builtin_fma(p, x, 0x1.a01338a37b710p-16);
  p = __builtin_fma(p, x, 0x1.a019c7ecb4a3fp-13);
  p = __builtin_fma(p, x, 0x1.6c16c03036706p-10);
  p = __builtin_fma(p, x, 0x1.1111110cd967ap-7);
  p = __builtin_fma(p, x, 0x1.55555555447f4p-5);
  p = __builtin_fma(p, x, 0x1.555555555532dp-3);
  p = __builtin_fma(p, x, 0x1.ffffffffffffdp-2);
  p = __builtin_fma(p, x, 1.0);
  return __builtin_fma(p, x, 1.0);
}

// exp(x) for x <= 0: x = n ln 2 + r with |r| <= 0.3467, n from the low word
// of x log2(e) + 1.5 2^52; results below 2^-1074 come out 0.
__device__ __forceinline__ double exp_nonpos(double x) {
  x = fmax(x, -800.0);
  const double t = __builtin_fma(x, 0x1.71547652b82fep+0, 0x1.8p+52);
  const double n = t - 0x1.8p+52;
  // ln 2 in two parts, the first with 21 trailing zero bits
  double r = __builtin_fma(n, -0x1.62e42fee00000p-1, x);
  r = __builtin_fma(n, -0x1.a39ef35793c76p-33, r);
  double p = 0x1.af4e8219983dfp-26;
  p = __builtin_fma(p, r, 0x1.28a2dd284e1dep-22);
  p = __builtin_fma(p, r, 0x1.71de01e0707e7p-19);
  p = __builtin_fma(p, r, 0x1.a019a64f100c1p-16);
  p = __builtin_fma(p, r, 0x1.a01a01ac05af2p-13);
  p = __builtin_fma(p, r, 0x1.6c16c17f4c498p-10);
  p = __builtin_fma(p, r, 0x1.1111111110096p-7);
  p = __builtin_fma(p, r, 0x1.555555555208fp-5);
  p = __builtin_fma(p, r, 0x1.5555555555557p-3);
  p = __builtin_fma(p, r, 0x1.0000000000005p-1);
  p = __builtin_fma(p, r, 1.0);
  p = __builtin_fma(p, r, 1.0);
  return __builtin_ldexp(p, __double2loint(t));
}

template <bool SHORT>
__device__ __forceinline__ double exp_bond(double x) {
  if constexpr (SHORT) return exp_short(x);
  return exp_nonpos(x);
}

// Reciprocal square root: the hardware's estimate (relative error below
// 2^-22) and one step of third order, error below an ulp.
__device__ __forceinline__ double rsqrt_f64_o3(double a) {
  const double y = __builtin_amdgcn_rsq(a);
  const double e = __builtin_fma(-(a * y), y, 1.0);
  const double p = __builtin_fma(0.375, e, 0.5);
  return __builtin_fma(y * e, p, y);
}

// sqrt(a), RN(1 / sqrt(a)) and RN(1 / a) (see above).
struct RootRcp {
  double r, yr, ya;
};
__device__ __forceinline__ RootRcp root_rcp(double a) {
  const double y = __builtin_amdgcn_rsq(a);
  double g = a * y, h = 0.5 * y;
  const double e = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, e, g);
  h = __builtin_fma(h, e, h);
  double d = __builtin_fma(-g, g, a);
  g = __builtin_fma(d, h, g);
  d = __builtin_fma(-g, g, a);
  g = __builtin_fma(d, h, g);
  RootRcp o;
  o.r = g;
  const double y0 = h + h;
  o.yr = __builtin_fma(__builtin_fma(-g, y0, 1.0), y0, y0);
  const double z0 = o.yr * o.yr;
  o.ya = __builtin_fma(__builtin_fma(-a, z0, 1.0), z0, z0);
  return o;
}

// RN(a / b) given y = RN(1 / b).
__device__ __forceinline__ double quot(double a, double b, double y) {
  const double q = a * y;
  return __builtin_fma(__builtin_fma(-b, q, a), y, q);
}

// a / b to about an ulp (b well inside the exponent range).
__device__ __forceinline__ double quot_near(double a, double b) {
  double y = __builtin_amdgcn_rcp(b);
  y = __builtin_fma(__builtin_fma(-b, y, 1.0), y, y);
  const double q = a * y;
  return __builtin_fma(__builtin_fma(-b, q, a), y, q);
}

// Influence function as the exact mode evaluates it (r / horizon rounded
// like the IEEE quotient).
template <int INF>
__device__ __forceinline__ double influence_rn(const RnpDev& m, double r) {
  if constexpr (INF == 0) return m.inf_a;
  const double q = quot(r, m.horizon, m.rcp_horizon);
  if constexpr (INF == 1) return m.inf_a + m.inf_b * q;
  return m.inf_a * exp(-q * q / m.inf_b);
}

// Exact mode, common path: the operations of bond_exact in its order, bit
// for bit except exp, which the deferred evaluations still call (81 instead of
// about 170 vector instructions a slot in 2D).
// F is 0 for broken bonds, bonds left to the exact evaluation (ex) and the
// zero-volume record of padded slots.  band: breakable bonds at or past the
// break test's lower bound.
template <int DIM, int INF, bool NOFAIL, bool SHORT>
__device__ __forceinline__ void bond_exact_fast(
    const RnpDev& m, const double* dx, const double* du, double volj,
    const SlotMasks& k, unsigned long long& band, unsigned long long& ex,
    double* F) {
  double dd = dx[0] * dx[0] + dx[1] * dx[1];
  double num = dx[0] * du[0] + dx[1] * du[1];
  if (DIM == 3) {
    dd = dd + dx[2] * dx[2];
    num = num + dx[2] * du[2];
  }
  const RootRcp o = root_rcp(dd);
  const double S = quot(num, dd, o.ya);
  const double x = -m.beta * o.r * S * S;
  const unsigned long long v_lo =
      __builtin_amdgcn_ballot_w64(!(x > -m.x_break_lo));
  band = k.brk & ~k.w & v_lo;
  const unsigned long long fsb = k.w & k.brk;
  ex = k.vex | band | (fsb & m.contact_mask);
  const unsigned long long keep = ~fsb & ~ex;
  // (lengths at the correction's edge are in k.vex)
  const double fac = quot(m.check_up - o.r, m.h, m.rcp_h);
  const double vj = volj * (o.r > m.low_band ? fac : 1.0);
  double ex_ = exp_bond<SHORT>(x);
  if (NOFAIL) ex_ = __builtin_amdgcn_inverse_ballot_w64(k.brk) ? ex_ : 1.0;
  double s = influence_rn<INF>(m, o.r) * 4. * S * m.C * m.beta * ex_;
  s = quot(s, m.inv_factor, m.rcp_inv_factor) * vj;
  s = __builtin_amdgcn_inverse_ballot_w64(keep) ? s : 0.0;
  for (int d = 0; d < DIM; d++) F[d] = s * quot(dx[d], o.r, o.yr);
}

// FP64 mode, common path (49 instead of 71 vector instructions a slot in
// 2D).  cvj = vol_j c4 (J when constant).  The volume-correction factor
// enters as fac / r = min((check_up/h) / r - 1/h, 1/r).
template <int DIM, int INF, bool NOFAIL, bool SHORT, bool ACC>
__device__ __forceinline__ void bond_fp64_staged(
    const RnpDev& m, const double* dx, const double* du, double cvj,
    const SlotMasks& k, unsigned long long& band, unsigned long long& ex,
    double* F) {
  double dd = __builtin_fma(dx[1], dx[1], dx[0] * dx[0]);
  double num = __builtin_fma(dx[1], du[1], dx[0] * du[0]);
  if (DIM == 3) {
    dd = __builtin_fma(dx[2], dx[2], dd);
    num = __builtin_fma(dx[2], du[2], num);
  }
  const double rinv = rsqrt_f64_o3(dd);
  const double q = num * rinv;  // S r
  const double S = q * rinv;
  const double x = (q * S) * -m.beta;
  const unsigned long long v_lo =
      __builtin_amdgcn_ballot_w64(!(x > -m.x_break_lo));
  band = k.brk & ~k.w & v_lo;
  const unsigned long long fsb = k.w & k.brk;
  ex = k.vex | band | (fsb & m.contact_mask);
  const unsigned long long keep = ~fsb & ~ex;
  const double facr =
      fmin(__builtin_fma(m.up_rcp_h, rinv, -m.rcp_h), rinv);
  double ex_ = exp_bond<SHORT>(x);
  if (NOFAIL) ex_ = __builtin_amdgcn_inverse_ballot_w64(k.brk) ? ex_ : 1.0;
  double sr = (S * ex_) * (cvj * facr);
  if constexpr (INF != 0) sr *= influence_f64<INF>(m, dd * rinv);
  sr = __builtin_amdgcn_inverse_ballot_w64(keep) ? sr : 0.0;
  for (int d = 0; d < DIM; d++) {
    if constexpr (ACC) F[d] = __builtin_fma(sr, dx[d], F[d]);
    else F[d] = sr * dx[d];
  }
}

}  // namespace nlm
