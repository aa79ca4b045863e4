// es_staged.h -- the LDS-staged passes of the state-based material with rows
// shared by several wavefronts (k_es_dil_st, k_es_force_st): the FP64 modes
// in 2D and 3D and the FP32-force mode in 2D.  (3D FP32-force: k_es_dil,
// k_es_force with their fixed-point records.)
//
// A workgroup stages its tile's halo in LDS and reads neighbors through
// 16-bit indices; record 0 is a zero-volume record far from every node that
// padded slots and fetches past a slice address.  In the FP64 modes their terms
// are exact zeros (a node without neighbors takes coefficients of 0 for its
// infinite 1/m); the FP32-force mode, whose range the products with the far
// record leave on fine meshes, masks them by the row's length.  (The mask in
// every mode: 6.64 instead of 6.55 ms for 100 steps of the 47 x 39 x 33 block,
// exact mode.)  `parts` wavefronts share a slice (split_rows.h): in the FP64 modes with the sums of one wavefront
// walking the row, so their bits depend on neither the tile nor the split.
//
// The exact mode takes its square roots and quotients from one Goldschmidt
// iteration each (bond_fast64.h: the bits of the IEEE operations) and the
// deformed position x + u of a node once instead of once a bond.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "bond_es.h"
#include "bond_fast64.h"
#include "fd_common.h"
#include "nlm_internal.h"
#include "split_rows.h"

namespace nlm {

template <int DIM>
struct EsArgs {
  FdArgs<DIM> f;
  const double* __restrict__ mw;
  double* __restrict__ theta;
  double* __restrict__ P;
  double* __restrict__ Q;
  EsDev m;
  int stride;  // bytes from halo record to halo record (staged passes)
};

// Halo records.  First pass: position, displacement (exact mode: deformed
// position x + u), volume.  Force pass: also the force coefficients (3D: P;
// 2D: P, Q) and the exact mode's dilatation.  14- and 18-dword strides spread
// record starts over 32 of the 64 LDS banks.
template <int DIM, int MODE, bool FORCE>
struct alignas(8) EsStRec {
  static constexpr int kVals =
      2 * DIM + 1 + (FORCE ? (DIM == 2 ? 2 : 1) + (MODE == kModeExact) : 0);
  double v[kVals];
};
// Bytes from record to record: an odd number of doubles (an even one is a
// stride of a multiple of 4 dwords), unless only the unpadded records fit the
// LDS (8 doubles in the 3D FP64 force pass).
inline size_t es_st_stride(int dim, int precision, bool force,
                           int64_t halo_max, size_t behind, size_t lds_max) {
  const int vals =
      2 * dim + 1 +
      (force ? (dim == 2 ? 2 : 1) + (precision == NLM_PREC_FP64_EXACT) : 0);
  const size_t padded = size_t(vals | 1) * 8;
  return size_t(halo_max + 1) * padded + behind <= lds_max ? padded
                                                           : size_t(vals) * 8;
}

// A bond's neighbor as its record holds it.
template <int DIM, int MODE, bool FORCE>
__device__ __forceinline__ void es_st_fill(
    EsStRec<DIM, MODE, FORCE>& r, const double* x, const double* u, double vol,
    double P, double Q, double theta) {
  for (int d = 0; d < DIM; d++) {
    r.v[d] = x[d];
    r.v[DIM + d] = MODE == kModeExact ? x[d] + u[d] : u[d];
  }
  r.v[2 * DIM] = vol;
  if constexpr (FORCE) {
    r.v[2 * DIM + 1] = P;
    if constexpr (DIM == 2) r.v[2 * DIM + 2] = Q;
    if constexpr (MODE == kModeExact) r.v[DIM == 2 ? 7 : 8] = theta;
  }
}

// Stages the halo of layout block lb behind record 0 (hid: the thread's first
// halo entry, fetched by the caller ahead of other loads).
template <int DIM, int MODE, bool FORCE>
__device__ __forceinline__ void es_st_stage(
    const EsArgs<DIM>& e, int64_t hb, int hn, uint32_t hid,
    char* lds) {
  const FdArgs<DIM>& a = e.f;
  auto halo_id = [&](int t) -> uint32_t {
    return t >= 0 && t < hn ? uint32_t(a.halo[hb + t]) : 0u;
  };
  for (int t = int(threadIdx.x) - 1; t < hn; t += int(blockDim.x)) {
    EsStRec<DIM, MODE, FORCE> r;
    const uint32_t g = hid;
    hid = halo_id(t + int(blockDim.x));
    if (t < 0) {
      const double far[3] = {a.far, a.far, a.far}, zero[3] = {0., 0., 0.};
      es_st_fill<DIM, MODE, FORCE>(r, far, zero, 0., 0., 0., 0.);
    } else {
      double x[3], u[3];
      load3<DIM>(ld32(a.x, g), x);
      load3<DIM>(ld32(a.u, g), u);
      const double P = FORCE ? ld32(e.P, g) : 0.;
      const double Q = FORCE && DIM == 2 ? ld32(e.Q, g) : 0.;
      const double th =
          FORCE && MODE == kModeExact && !e.m.one_d ? ld32(e.theta, g) : 0.;
      es_st_fill<DIM, MODE, FORCE>(r, x, u, ld32(a.vol, g), P, Q, th);
    }
    *reinterpret_cast<EsStRec<DIM, MODE, FORCE>*>(lds + (t + 1) * e.stride) = r;
  }
  __syncthreads();
}

// The wavefront's slice and its slot entries.
template <int DIM>
struct EsRow {
  SplitPos p;
  int64_t lb, hb, s, i, cb, bb;
  int hn, width, len;
  bool valid;
};
template <int DIM, bool SPLIT>
__device__ __forceinline__ EsRow<DIM> es_row(const FdArgs<DIM>& a, int64_t lb,
                                             uint32_t& hid) {
  EsRow<DIM> r;
  const int bn = SPLIT ? a.tile : int(blockDim.x);
  r.p.parts = SPLIT ? a.parts : 1;
  r.p.nsl = bn >> 6;
  r.lb = lb;
  r.hb = a.halo_ptr[lb];
  r.hn = int(a.halo_ptr[lb + 1] - r.hb);
  const int t = int(threadIdx.x) - 1;
  hid = t >= 0 && t < r.hn ? uint32_t(a.halo[r.hb + t]) : 0u;
  r.p.lane = threadIdx.x & 63;
  r.p.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  r.p.sl = SPLIT ? r.p.wave % r.p.nsl : r.p.wave;
  r.p.part = SPLIT ? r.p.wave / r.p.nsl : 0;
  r.s = lb * r.p.nsl + r.p.sl;
  const bool ok = r.s < a.nslices;
  r.i = r.s * 64 + r.p.lane;
  r.valid = ok && r.i < a.n;
  r.cb = ok ? a.sl_ptr[r.s] : 0;
  r.width = ok ? int((a.sl_ptr[r.s + 1] - r.cb) >> 6) : 0;
  r.bb = r.cb >> 6;
  r.len = r.valid ? int(a.rowlen[r.i]) : 0;
  return r;
}

// Sums the chunks' summands over the row: list order (FP64 modes) or, split
// in the FP32-force mode, the parts' FP64 sums.
template <int MODE, int NC, int NF, int U, bool SPLIT, class Chunk, int DIM>
__device__ __forceinline__ void es_sum(Chunk&& chunk, double* buf,
                                       const FdArgs<DIM>& a,
                                       const EsRow<DIM>& r,
                                       double (&out)[NC]) {
  typedef
      typename std::conditional<MODE == kModeFp32, float, double>::type Real;
  if constexpr (SPLIT && MODE != kModeFp32) {
    const int64_t s0 = r.lb * r.p.nsl;
    split_ordered<NC, NF, U>(chunk, buf, r.p, a.sl_ptr + s0,
                             int(min(int64_t(r.p.nsl), a.nslices - s0)),
                             r.width, out);
  } else {
    const int stride = U * r.p.parts;
    for (int k0 = U * r.p.part; k0 < r.width; k0 += stride) {
      Real F[NF][NC];
      chunk(k0, k0 + stride, F);
#pragma unroll
      for (int m = 0; m < NF; ++m)
        for (int d = 0; d < NC; d++) out[d] += double(F[m][d]);
    }
    if constexpr (SPLIT) split_parts<NC>(buf, r.p, out);
  }
}

// The dilatation and the force coefficients of node i.
template <int DIM, int MODE>
__device__ __forceinline__ void es_coefficients(const EsArgs<DIM>& e,
                                                int64_t i, double th,
                                                double mwi) {
  e.theta[i] = th;
  if constexpr (DIM == 3) {
    // EXACT keeps alpha_s = (9/m) K (ElasticState.cpp:230-233); the fast
    // modes fold t_ij = alpha_s theta_i |X| / 3 into P_i |X|.
    e.P[i] = MODE == kModeExact ? (9. / mwi) * e.m.K : 3. * e.m.K * th / mwi;
  } else if (e.m.one_d) {
    // 1D: t_ij = (E/m_i) e_ij (ElasticState.cpp:187-193)
    e.P[i] = 0.;
    e.Q[i] = e.m.E / mwi;
  } else {
    const double as = (9. / mwi) * e.m.Kc;
    const double ad = (8. / mwi) * e.m.mu;
    const double C = 2. * e.m.f2d * as - (3. - 2. * e.m.f2d) * ad;
    // fast modes: t_ij = theta_i (C/9 - alpha_d/3) |X| + alpha_d e_ij
    e.P[i] = MODE == kModeExact ? C : th * (C / 9. - ad / 3.);
    e.Q[i] = ad;
  }
}

// Pass 1: break test, dilatation, force coefficients.
template <int DIM, int MODE, int U, bool SPLIT>
__global__ __launch_bounds__(512) void k_es_dil_st(
    EsArgs<DIM> e, const unsigned long long* __restrict__ bits_ro) {
  constexpr bool EXACT = MODE == kModeExact;
  constexpr bool F32 = MODE == kModeFp32;
  typedef typename std::conditional<F32, float, double>::type Real;
  typedef EsStRec<DIM, MODE, false> Rec;
  const FdArgs<DIM>& a = e.f;
  const int bn = SPLIT ? a.tile : int(blockDim.x);
  const int64_t nblk = (a.nslices * 64 + bn - 1) / bn;
  const int64_t lb = xcd_block(nblk);
  if (lb >= nblk) return;
  extern __shared__ double es_st_smem[];
  char* const lds = reinterpret_cast<char*>(es_st_smem);
  uint32_t hid;
  const EsRow<DIM> r = es_row<DIM, SPLIT>(a, lb, hid);
  const int lane = r.p.lane, len = r.len;
  double xi[3] = {0., 0., 0.}, ui[3] = {0., 0., 0.}, mwi = 1.;
  if (r.valid) {
    load3<DIM>(a.x[r.i], xi);
    load3<DIM>(a.u[r.i], ui);
    mwi = e.mw[r.i];
  }
  double yi[3];
  for (int d = 0; d < 3; d++) yi[d] = xi[d] + ui[d];
  const unsigned long long* __restrict__ bits_in = bits_ro + r.bb;
  const __amdgpu_buffer_rsrc_t col_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(a.colL + r.cb), 0, r.width * 64 * int(sizeof(uint16_t)),
      kBufferRsrcWord3);
  auto entry = [&](int k) -> uint32_t {
    return uint32_t(__builtin_amdgcn_raw_buffer_load_b16(
        col_rsrc, lane * int(sizeof(uint16_t)), k * 64 * int(sizeof(uint16_t)),
        0));
  };
  uint32_t jn[U];
#pragma unroll
  for (int q = 0; q < U; ++q) jn[q] = entry(U * r.p.part + q);
  es_st_stage<DIM, MODE, false>(e, r.hb, r.hn, hid, lds);
  if (!SPLIT && r.s >= a.nslices) return;  // (split tiles meet at barriers)
  // (3/m_i) in 3D, (2/m_i) factor2D in 2D: leading factors of the reference
  // product; the fast modes apply it once to the row's sum
  // (a row without bonds: m_i = 0, its sum is 0)
  const double c3 =
      len == 0 ? 0. : DIM == 3 ? 3. / mwi : (2. / mwi) * e.m.f2d;
  constexpr int NF = EXACT ? U : U / 2;
  const Real vtol = F32 ? Real(e.m.vex_tol_f) : Real(e.m.vex_tol);
  const Real lowb = F32 ? Real(e.m.low_band_f) : Real(e.m.low_band);
  const Real blo = F32 ? Real(e.m.brk_lo_f) : Real(e.m.brk_lo);
  auto fmaR = [](Real x, Real y, Real z) -> Real {
    if constexpr (F32) return __builtin_fmaf(x, y, z);
    else return __builtin_fma(x, y, z);
  };
  auto chunk = [&](int k0, int k_next, Real (&F)[NF][1]) {
    uint32_t jc[U];
#pragma unroll
    for (int q = 0; q < U; ++q) {
      jc[q] = jn[q];
      jn[q] = entry(k_next + q);
    }
    unsigned long long w[U], band[U], ex[U];
    unsigned long long ex_any = 0ull;
#pragma unroll
    for (int q = 0; q < U; ++q) w[q] = bits_in[k0 + q];
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const Rec& n = *reinterpret_cast<const Rec*>(
          lds + jc[q] * uint32_t(e.stride));
      Real term;
      unsigned long long v_vex, v_lo;
      if constexpr (EXACT) {
        // es_dil_exact's operations in its order
        double yy = 0., dd = 0.;
        for (int d = 0; d < DIM; d++) {
          const double Y = n.v[DIM + d] - yi[d], X = n.v[d] - xi[d];
          yy = d == 0 ? Y * Y : yy + Y * Y;
          dd = d == 0 ? X * X : dd + X * X;
        }
        const double ly = root_rcp(yy).r;
        const RootRcp o = root_rcp(dd);
        const double ext = ly - o.r;
        v_vex = __builtin_amdgcn_ballot_w64(fabs(o.r - lowb) <= vtol);
        v_lo = __builtin_amdgcn_ballot_w64(!(ext * o.yr < blo));
        const double c =
            o.r > lowb ? quot(e.m.check_up - o.r, e.m.h, e.m.rcp_h) : 1.;
        term = c3 * o.r * ext * c * n.v[2 * DIM];
      } else {
        Real dx[DIM], du[DIM];
        for (int d = 0; d < DIM; d++) {
          dx[d] = Real(n.v[d] - xi[d]);
          du[d] = Real(n.v[DIM + d] - ui[d]);
        }
        Real dd = fmaR(dx[1], dx[1], dx[0] * dx[0]);
        Real g = fmaR(du[1], fmaR(Real(2), dx[1], du[1]),
                      du[0] * fmaR(Real(2), dx[0], du[0]));
        if constexpr (DIM == 3) {
          dd = fmaR(dx[2], dx[2], dd);
          g = fmaR(du[2], fmaR(Real(2), dx[2], du[2]), g);
        }
        const Real yy = dd + g;
        Real rx, ly, ext, c;
        if constexpr (F32) {
          rx = __builtin_amdgcn_rsqf(dd);
          ly = yy * __builtin_amdgcn_rsqf(yy);
        } else {
          rx = rsqrt_f64_o3(dd);
          ly = yy * rsqrt_f64_o3(yy);
        }
        const Real lx = dd * rx;
        if constexpr (F32) {
          ext = g * __builtin_amdgcn_rcpf(ly + lx);
          c = __builtin_amdgcn_fmed3f(
              __builtin_fmaf(lx, -e.m.rcp_h_f, e.m.up_rcp_h_qf), 0.f, 1.f);
        } else {
          ext = quot_near(g, ly + lx);
          c = fmin((e.m.check_up - lx) * e.m.rcp_h, 1.);
        }
        v_vex = __builtin_amdgcn_ballot_w64(fabs(lx - lowb) <= vtol);
        v_lo = __builtin_amdgcn_ballot_w64(ext * rx >= blo);
        term = lx * ext * c * Real(n.v[2 * DIM]);
      }
      // one vote on the guard band's lower bound: a bond that may break is
      // decided, and its term taken, by the exact evaluation after the chunk
      const unsigned long long act =
          F32 ? __builtin_amdgcn_ballot_w64(k0 + q < len) : ~0ull;
      band[q] = act & ~w[q] & v_lo;
      ex[q] = (act & v_vex) | band[q];
      const unsigned long long keep = act & ~w[q] & ~ex[q];
      term = __builtin_amdgcn_inverse_ballot_w64(keep) ? term : Real(0);
      if constexpr (EXACT) F[q][0] = term;
      else if (q % 2 == 0) F[q / 2][0] = term;
      else F[q / 2][0] += term;
      ex_any |= ex[q];
    }
    if (ex_any != 0ull) {  // rare: whole wavefronts skip it
#pragma unroll
      for (int q = 0; q < U; ++q) {
        if (ex[q] == 0ull) continue;
        bool fsn = false;
        if (__builtin_amdgcn_inverse_ballot_w64(ex[q]) && k0 + q < len) {
          const uint32_t g = uint32_t(a.halo[r.hb + jc[q] - 1]);
          const bool fs0 = __builtin_amdgcn_inverse_ballot_w64(w[q]);
          bool fs = fs0;
          double xs[3], us[3];
          load3<DIM>(ld32(a.x, g), xs);
          load3<DIM>(ld32(a.u, g), us);
          const double d =
              es_dil_exact(e.m, xi, ui, xs, us, ld32(a.vol, g), c3, fs);
          fsn = fs && !fs0;
          if (!fs) {
            if constexpr (EXACT) F[q][0] = d;
            else F[q / 2][0] += Real(d / c3);
          }
        }
        const unsigned long long nb =
            band[q] & __builtin_amdgcn_ballot_w64(fsn);
        if (nb != 0ull && k0 + q < r.width) a.bits[r.bb + k0 + q] = w[q] | nb;
      }
    }
  };
  double sum[1] = {0.};
  es_sum<MODE, 1, NF, U, SPLIT>(
      chunk,
      reinterpret_cast<double*>(reinterpret_cast<char*>(es_st_smem) +
                                a.halo_bytes),
      a, r, sum);
  if (!r.valid || r.p.part != 0) return;
  const double th = EXACT ? sum[0] : c3 * sum[0];
  es_coefficients<DIM, MODE>(e, r.i, th, mwi);
}

// Pass 2: bond forces of both directions gathered at node i, force BCs,
// central-difference update (a.kind: KIND_*).
template <int DIM, int MODE, int U, bool SPLIT>
__global__ __launch_bounds__(512) void k_es_force_st(
    EsArgs<DIM> e, const unsigned long long* __restrict__ bits_ro,
    double t_force, double t_next) {
  constexpr bool EXACT = MODE == kModeExact;
  constexpr bool F32 = MODE == kModeFp32;
  typedef typename std::conditional<F32, float, double>::type Real;
  typedef EsStRec<DIM, MODE, true> Rec;
  if (e.f.tdev) {
    t_force = e.f.tdev[0];
    t_next = e.f.tdev[1];
  }
  const FdArgs<DIM>& a = e.f;
  const int bn = SPLIT ? a.tile : int(blockDim.x);
  const int64_t nblk = (a.nslices * 64 + bn - 1) / bn;
  const int64_t lb = xcd_block(nblk);
  if (lb >= nblk) return;
  extern __shared__ double es_st_smem[];
  char* const lds = reinterpret_cast<char*>(es_st_smem);
  uint32_t hid;
  const EsRow<DIM> r = es_row<DIM, SPLIT>(a, lb, hid);
  const int lane = r.p.lane, len = r.len;
  double xi[3] = {0., 0., 0.}, ui[3] = {0., 0., 0.};
  double Pi = 0., Qi = 0., thi = 0.;
  uint32_t fl = 0;
  if (r.valid) {
    load3<DIM>(a.x[r.i], xi);
    load3<DIM>(a.u[r.i], ui);
    Pi = e.P[r.i];
    if (DIM == 2) Qi = e.Q[r.i];
    // (1D: no dilatation term, t = Q e)
    if (EXACT) thi = e.m.one_d ? 0. : e.theta[r.i];
    fl = a.flags[r.i];
    // (a row without bonds: infinite or NaN, 1/m_i)
    if (len == 0) Pi = Qi = thi = 0.;
  }
  double yi[3];
  for (int d = 0; d < 3; d++) yi[d] = xi[d] + ui[d];
  const unsigned long long* __restrict__ bits_in = bits_ro + r.bb;
  const __amdgpu_buffer_rsrc_t col_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(a.colL + r.cb), 0, r.width * 64 * int(sizeof(uint16_t)),
      kBufferRsrcWord3);
  auto entry = [&](int k) -> uint32_t {
    return uint32_t(__builtin_amdgcn_raw_buffer_load_b16(
        col_rsrc, lane * int(sizeof(uint16_t)), k * 64 * int(sizeof(uint16_t)),
        0));
  };
  uint32_t jn[U];
#pragma unroll
  for (int q = 0; q < U; ++q) jn[q] = entry(U * r.p.part + q);
  es_st_stage<DIM, MODE, true>(e, r.hb, r.hn, hid, lds);
  if (!SPLIT && r.s >= a.nslices) return;
  constexpr int NF = EXACT ? U : U / 2;
  constexpr int NC = EXACT ? 2 * DIM : DIM;  // exact: own and other direction
  constexpr double kThird = 1.0 / 3.0;
  const Real vtol = F32 ? Real(e.m.vex_tol_f) : Real(e.m.vex_tol);
  const Real lowb = F32 ? Real(e.m.low_band_f) : Real(e.m.low_band);
  auto fmaR = [](Real x, Real y, Real z) -> Real {
    if constexpr (F32) return __builtin_fmaf(x, y, z);
    else return __builtin_fma(x, y, z);
  };
  auto chunk = [&](int k0, int k_next, Real (&F)[NF][NC]) {
    uint32_t jc[U];
#pragma unroll
    for (int q = 0; q < U; ++q) {
      jc[q] = jn[q];
      jn[q] = entry(k_next + q);
    }
    unsigned long long w[U];
#pragma unroll
    for (int q = 0; q < U; ++q) w[q] = bits_in[k0 + q];
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const Rec& n = *reinterpret_cast<const Rec*>(
          lds + jc[q] * uint32_t(e.stride));
      const double volj = n.v[2 * DIM], Pj = n.v[2 * DIM + 1];
      const double Qj = DIM == 2 ? n.v[2 * DIM + 2] : 0.;
      // the volume correction at its edge is decided exactly (rare)
      auto corr_exact = [&]() -> double {
        const uint32_t g = uint32_t(a.halo[r.hb + jc[q] - 1]);
        double xs[3];
        load3<DIM>(ld32(a.x, g), xs);
        const double X0 = xs[0] - xi[0], X1 = xs[1] - xi[1],
                     X2 = xs[2] - xi[2];
        return es_corr_exact(e.m, sqrt(X0 * X0 + X1 * X1 + X2 * X2));
      };
      // (FP32-force: against record 0 the product (P_i + P_j) |X| overflows on
      // fine meshes, P going with h^-4)
      bool live = !__builtin_amdgcn_inverse_ballot_w64(w[q]);
      if constexpr (F32) live = live && k0 + q < len;
      if constexpr (EXACT) {
        // es_force_exact's operations in its order
        double Y[DIM], yy = 0., dd = 0.;
        for (int d = 0; d < DIM; d++) {
          const double X = n.v[d] - xi[d];
          Y[d] = n.v[DIM + d] - yi[d];
          yy = d == 0 ? Y[d] * Y[d] : yy + Y[d] * Y[d];
          dd = d == 0 ? X * X : dd + X * X;
        }
        const RootRcp oy = root_rcp(yy);
        double lx = root_rcp(dd).r;
        double c = lx > lowb ? quot(e.m.check_up - lx, e.m.h, e.m.rcp_h) : 1.;
        // (inside the band: the root of 0, a NaN, too)
        if (__builtin_amdgcn_ballot_w64(!(fabs(lx - lowb) > vtol)) != 0ull)
          if (!(fabs(lx - lowb) > vtol) && k0 + q < len) {
            c = corr_exact();
            lx = dd == 0. ? 0. : lx;
          }
        const double thj = n.v[DIM == 2 ? 7 : 8];
        const double es_i = quot(thi * lx, 3., kThird);
        const double es_j = quot(thj * lx, 3., kThird);
        double tij, tji;
        if constexpr (DIM == 3) {
          tij = Pi * es_i;
          tji = Pj * es_j;
        } else {
          const double ext = oy.r - lx;
          tij = quot(Pi * es_i, 3., kThird) + Qi * (ext - es_i);
          tji = quot(Pj * es_j, 3., kThird) + Qj * (ext - es_j);
        }
        for (int d = 0; d < DIM; d++) {
          const double M = quot(Y[d], oy.r, oy.yr);
          F[q][d] = live ? volj * ((M * tij) * c) : 0.;
          F[q][DIM + d] = live ? volj * ((-M * tji) * c) : 0.;
        }
      } else {
        Real Y[DIM], dx[DIM], du[DIM];
        for (int d = 0; d < DIM; d++) {
          dx[d] = Real(n.v[d] - xi[d]);
          du[d] = Real(n.v[DIM + d] - ui[d]);
          Y[d] = dx[d] + du[d];
        }
        Real yy = fmaR(Y[1], Y[1], Y[0] * Y[0]);
        Real dd = fmaR(dx[1], dx[1], dx[0] * dx[0]);
        if constexpr (DIM == 3) {
          yy = fmaR(Y[2], Y[2], yy);
          dd = fmaR(dx[2], dx[2], dd);
        }
        Real ry, lx, c;
        if constexpr (F32) {
          ry = __builtin_amdgcn_rsqf(yy);
          lx = dd * __builtin_amdgcn_rsqf(dd);
          c = __builtin_amdgcn_fmed3f(
              __builtin_fmaf(lx, -e.m.rcp_h_f, e.m.up_rcp_h_qf), 0.f, 1.f);
        } else {
          ry = rsqrt_f64_o3(yy);
          lx = dd * rsqrt_f64_o3(dd);
          c = fmin((e.m.check_up - lx) * e.m.rcp_h, 1.);
        }
        if (__builtin_amdgcn_ballot_w64(fabs(lx - lowb) <= vtol) != 0ull)
          if (fabs(lx - lowb) <= vtol && k0 + q < len) c = Real(corr_exact());
        Real t = Real(Pi + Pj) * lx;
        if constexpr (DIM == 2) {
          const Real g = fmaR(du[1], fmaR(Real(2), dx[1], du[1]),
                              du[0] * fmaR(Real(2), dx[0], du[0]));
          Real ext;
          if constexpr (F32) ext = g * __builtin_amdgcn_rcpf(yy * ry + lx);
          else ext = quot_near(g, yy * ry + lx);
          t = fmaR(Real(Qi + Qj), ext, t);
        }
        Real sr = t * c * Real(volj) * ry;
        sr = live ? sr : Real(0);
        for (int d = 0; d < DIM; d++) {
          if (q % 2 == 0) F[q / 2][d] = sr * Y[d];
          else F[q / 2][d] = fmaR(sr, Y[d], F[q / 2][d]);
        }
      }
    }
  };
  double sum[NC] = {};
  es_sum<MODE, NC, NF, U, SPLIT>(
      chunk,
      reinterpret_cast<double*>(reinterpret_cast<char*>(es_st_smem) +
                                a.halo_bytes),
      a, r, sum);
  if (!r.valid || r.p.part != 0) return;
  double f[3] = {0., 0., 0.};
  if (a.kind == KIND_FORCE_ADD) {
    load3<DIM>(a.f_in[r.i], f);
  } else if (a.has_fbc) {
    fext_node<DIM>(a.bc, fl, xi, t_force, f);
  }
  for (int d = 0; d < DIM; d++)
    f[d] += EXACT ? sum[d] - sum[(DIM + d) % NC] : sum[d];
  if (a.kind == KIND_CD)
    node_tail<DIM, KIND_CD>(a, r.i, fl, xi, ui, f, t_next);
  else
    node_tail<DIM, KIND_FORCE>(a, r.i, fl, xi, ui, f, t_next);
}

// Launches of the two passes (es_st.hip); SPLIT by the configured parts.
template <int DIM>
void es_st_dil(nlm_ctx* c, EsArgs<DIM> e);
template <int DIM>
void es_st_force(nlm_ctx* c, EsArgs<DIM> e, double tf, double tn);

// LDS bytes behind the halo records.
inline size_t es_st_behind(int dim, int precision, int tile, int parts,
                           bool force) {
  if (parts <= 1) return 0;
  const int nc =
      force ? (precision == NLM_PREC_FP64_EXACT ? 2 * dim : dim) : 1;
  if (precision == NLM_PREC_FP32_FORCE)
    return split_parts_bytes(tile, parts, nc);
  return split_ordered_bytes(
      tile, parts, nc,
      precision == NLM_PREC_FP64_EXACT ? kStSplitU : kStSplitU / 2);
}

// A pass's LDS: record stride and bytes.
struct EsStLds {
  size_t stride, records, bytes;
};
inline EsStLds es_st_lds(int dim, int precision, int64_t halo_max, int tile,
                         int parts, bool force, size_t lds_max) {
  const size_t behind = es_st_behind(dim, precision, tile, parts, force);
  EsStLds l;
  l.stride = es_st_stride(dim, precision, force, halo_max, behind, lds_max);
  l.records = size_t(halo_max + 1) * l.stride;
  l.bytes = l.records + behind;
  return l;
}

}  // namespace nlm
