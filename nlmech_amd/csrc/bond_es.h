// bond_es.h -- per-bond arithmetic of the linear state-based material
// (material::pd::ElasticState) on the device.
//
// A force evaluation has two passes over the bonds:
//   pass 1  extension e_ij = |Y| - |X| (StateBasedHelperFunctions::dilatation,
//           stateBasedHelperFunctions.cpp:26-83), the critical-stretch break
//           test, and the dilatation
//             theta_i = sum_j (3/m_i) |X| e_ij c_ij V_j          (3D)
//             theta_i = sum_j (2/m_i) factor2D |X| e_ij c_ij V_j (2D)
//           with the volume correction c_ij (VolumeCorrection::correctVolume,
//           volumeCorrection.cpp:25-49) and the weighted volume m_i;
//   pass 2  the force: ElasticState::getBondEF (ElasticState.cpp:160-271)
//           gives T_ij = t_ij M_ij c_ij with M = Y/|Y| and the scalar state
//             3D  t_ij = (9 K / m_i) theta_i |X| / 3        (e_d stays 0)
//             2D  t_ij = C_i (theta_i |X| / 3) / 3 + alpha_d,i (e_ij - theta_i|X|/3)
//               C_i = 2 factor2D alpha_s,i - (3 - 2 factor2D) alpha_d,i,
//               alpha_s,i = (9/m_i) Kc, alpha_d,i = (8/m_i) mu;
//           QuasiStaticModel::computeForces (QuasiStaticModel.cpp:169-239)
//           adds T_ij V_j to f_i and subtracts it, times V_i, from f_j, so
//           node i collects f_i = sum_j V_j (T_ij - T_ji) with T_ji =
//           -t_ji M_ij c_ij.
//
// Arithmetic variants (as for the bond-based material):
//   EXACT  the reference's expressions and order, IEEE sqrt/division;
//   FP64   e from the cancellation-free form e = du.(2 dx + du) / (|Y| + |X|),
//          rsqrt with Newton steps, fused multiply-adds;
//   FP32F  differences dx, du formed in FP64, then the same cancellation-free
//          extension and the force in FP32; sums in FP64.
// The break decision definitelyGreaterThan(e/|X|, sc) and the volume
// correction test definitelyGreaterThan(|X|, horizon - h/2) are taken
// directly outside a guard band around their switching points and by the
// EXACT expression inside it, so they equal the reference's on the same
// displacement field.
#pragma once

#include <hip/hip_runtime.h>

#include "bond_rnp.h"
#include "device_common.h"
#include "nlm_internal.h"

namespace nlm {

constexpr double kEsGuard64 = 1e-9;
constexpr float kEsGuard32 = 2e-5f;

// Y = (xj + uj) - (xi + ui), X = xj - xi (Point3 operators, point.h), their
// lengths sqrt(x*x + y*y + z*z) (point.h:119) and the extension.
__device__ __forceinline__ void es_geom_exact(const double* xi,
                                              const double* ui,
                                              const double* xj,
                                              const double* uj, double* Y,
                                              double& lx, double& ly,
                                              double& ext) {
  double X[3];
  for (int d = 0; d < 3; d++) {
    Y[d] = (xj[d] + uj[d]) - (xi[d] + ui[d]);
    X[d] = xj[d] - xi[d];
  }
  ly = sqrt(Y[0] * Y[0] + Y[1] * Y[1] + Y[2] * Y[2]);
  lx = sqrt(X[0] * X[0] + X[1] * X[1] + X[2] * X[2]);
  ext = ly - lx;
}

// VolumeCorrection::correctVolume, volumeCorrection.cpp:40-44
__device__ __forceinline__ double es_corr_exact(const EsDev& m, double lx) {
  double c = 1.;
  if (def_greater(lx, m.check_low)) c = (m.check_up - lx) / m.h;
  return c;
}

// Pass 1, EXACT: break test (fs in/out) and the dilatation term
// ((((c3 * |X|) * e) * c) * V_j), c3 = 3/m_i (3D) or (2/m_i) factor2D (2D).
__device__ __forceinline__ double es_dil_exact(const EsDev& m,
                                               const double* xi,
                                               const double* ui,
                                               const double* xj,
                                               const double* uj, double volj,
                                               double c3, bool& fs) {
  double Y[3], lx, ly, ext;
  es_geom_exact(xi, ui, xj, uj, Y, lx, ly, ext);
  if (m.breaking && !fs && def_greater(ext / lx, m.sc)) fs = true;
  double c = es_corr_exact(m, lx);
  return c3 * lx * ext * c * volj;
}

// Pass 2, EXACT: V_j T_ij and V_j T_ji of getBondEF for the two directions
// of one bond, given the per-node coefficients (3D: P = (9/m) K; 2D: P = C,
// Q = alpha_d) and dilatations of both ends.
template <int DIM>
__device__ __forceinline__ void es_force_exact(
    const EsDev& m, const double* xi, const double* ui, const double* xj,
    const double* uj, double volj, double Pi, double Qi, double thi, double Pj,
    double Qj, double thj, double* own, double* oth) {
  double Y[3], lx, ly, ext;
  es_geom_exact(xi, ui, xj, uj, Y, lx, ly, ext);
  double M[3] = {Y[0] / ly, Y[1] / ly, Y[2] / ly};
  double c = es_corr_exact(m, lx);
  const double w = 1.;
  double tij, tji;
  if constexpr (DIM == 3) {
    double es_i = thi * lx / 3.;
    double es_j = thj * lx / 3.;
    tij = Pi * w * es_i;
    tji = Pj * w * es_j;
  } else {
    double es_i = thi * lx / 3.;
    double ed_i = ext - es_i;
    tij = Pi * w * es_i / 3. + Qi * w * ed_i;
    double es_j = thj * lx / 3.;
    double ed_j = ext - es_j;
    tji = Pj * w * es_j / 3. + Qj * w * ed_j;
  }
  for (int d = 0; d < 3; d++) {
    own[d] = volj * ((M[d] * tij) * c);
    oth[d] = volj * ((-M[d] * tji) * c);
  }
}

}  // namespace nlm
