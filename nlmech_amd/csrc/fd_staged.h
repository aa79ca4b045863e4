// fd_staged.h -- the LDS-staged bond-based step kernel of the FP64 modes
// and of every mode in 3D (k_fd_st).
//
// A workgroup owns a tile of the layout's internal order (64 to 512
// nodes): it stages the tile's halo -- every node its rows reference -- in
// LDS once (one record a node) and reads neighbors through 16-bit LDS byte
// offsets.  Record 0 is a zero-volume record far from every node; padded
// slots and fetches past a slice address it and come out as exact zeros, so
// the common path carries no row-length mask.  The kernel is bound by FP64
// instructions; bond_fast64.h says what a bond costs.  Per step, before and
// after that arithmetic (and the records without the row-length mask):
// 400 x 397 nodes, horizon 4 h, exact mode 57 -> 27 us; 619 x 451 nodes,
// FP64 mode, four slots a chunk 48 -> 32 us; 1000 x 1000, 103 -> 82 us (FP64),
// 256 -> 119 us (exact).
//
// Split rows.  One wavefront per 64-node slice leaves a small model a few
// wavefronts per CU that walk their rows serially (100 x 100 nodes: 157
// slices on 1024 SIMDs), and the 3D halos leave a CU two tiles.  With SPLIT,
// `parts` wavefronts share a slice (split_rows.h): in the FP64 modes with the
// sums of one wavefront walking the row, so their bits depend on neither the
// split nor the tile.
//
// Launch kinds (a.kind, wavefront-uniform): force, force added to f, the
// fused central-difference step and the fused velocity-Verlet step.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "bond_fast64.h"
#include "bond_rnp.h"
#include "device_common.h"
#include "fd_common.h"
#include "nlm_internal.h"
#include "split_rows.h"

namespace nlm {

// Halo record of the FP64 modes: position, displacement and the volume (FP64
// mode: times c4, and J when constant).  10- and 14-dword strides spread
// record starts over 32 of the 64 LDS banks; with flags 12 and 18 dwords over
// 16 and 32 (3D without padding, 16 dwords, over 4: 56 x 57 x 60 nodes with a
// no-fail region, FP64 146 instead of 69 us a step, exact 157 instead of 140).
template <int DIM, bool NOFAIL>
struct alignas(8) StRec64 {
  double x[DIM];
  double u[DIM];
  double c;
};
template <int DIM>
struct alignas(8) StRec64<DIM, true> {
  double x[DIM];
  double u[DIM];
  double c;
  uint32_t flags, pad[DIM == 3 ? 3 : 1];
};

// FP32-force mode, 2D: the scaled displacement in FP64, the scaled
// block-relative position in FP32 (bond_fp32_scaled), the force constant.
template <int DIM, bool NOFAIL>
struct alignas(8) StRec32 {
  double u[2];
  float xq[2];
  float c;
  uint32_t flags;
  uint32_t pad[2];
};
// 3D: the position as a fixed-point offset from the tile's origin, an even
// number of quanta 1/sigma modulo 2^32.  A bond's components stay below 2^31
// quanta, so its position difference is an exact integer difference whatever
// the tile's extent (a tile of the Morton order may span a gap between two
// bodies), rounded once to FP32.  Record 0's position is odd: it coincides
// with no node.
template <bool NOFAIL>
struct alignas(8) StRec32<3, NOFAIL> {
  double u[3];
  int32_t xq[3];
  float c;
};
template <>
struct alignas(8) StRec32<3, true> {
  double u[3];
  int32_t xq[3];
  float c;
  uint32_t flags, pad;
};

template <int DIM, int MODE, bool NOFAIL>
using StRec = typename std::conditional<MODE == kModeFp32,
                                        StRec32<DIM, NOFAIL>,
                                        StRec64<DIM, NOFAIL>>::type;

// The end of a launch for node i with force density f = base + sum.
template <int DIM>
__device__ __forceinline__ void st_tail(const FdArgs<DIM>& a, int64_t i,
                                        uint32_t fl, const double* xi,
                                        const double* ui, const double* vi,
                                        double* acc, double t_force,
                                        double t_next) {
  double f[3] = {0., 0., 0.};
  if (a.kind == KIND_FORCE_ADD) {
    load3<DIM>(a.f_in[i], f);
  } else if (a.has_fbc) {
    fext_node<DIM>(a.bc, fl, xi, t_force, f);
  }
  for (int d = 0; d < DIM; d++) f[d] += acc[d];
  if (a.kind == KIND_FORCE || a.kind == KIND_FORCE_ADD) {
    a.f_out[i] = make_v<DIM>(f);
    return;
  }
  double un[3] = {0., 0., 0.}, vn[3] = {0., 0., 0.};
  for (int d = 0; d < DIM; d++) {
    const uint32_t id = (fl >> (kFlagUbcShift + 4 * d)) & 0xfu;
    if (id == 0) {
      const double uo = ui[d];
      if (a.kind == KIND_VERLET) {
        verlet_dof(a, f[d], uo, vi[d], un[d], vn[d]);
      } else {
        // u += fact*f + dt*v; v = (u - u_old)/dt  (fDModel.cpp:386-394)
        un[d] = uo + (a.fact * f[d] + a.dt * vi[d]);
        vn[d] = (un[d] - uo) / a.dt;
      }
    } else {
      double du, dv;
      ubc_dof(a, id, i, d, xi, t_next, du, dv);
      un[d] = du;
      vn[d] = dv;
    }
  }
  a.u_out[i] = make_v<DIM>(un);
  a.v_out[i] = make_v<DIM>(vn);
}

// Exact evaluation of a deferred bond from the neighbor's global arrays.
template <int DIM, int MODE, int INF>
__device__ __forceinline__ void st_deferred(const FdArgs<DIM>& a, uint32_t g,
                                            const double* xi,
                                            const double* ui, double voli,
                                            bool brk, bool& fs, double* F) {
  double xs[3], us[3];
  load3<DIM>(ld32(a.x, g), xs);
  load3<DIM>(ld32(a.u, g), us);
  const double vs = ld32(a.vol, g);
  if constexpr (MODE == kModeExact)
    bond_exact<DIM, false>(a.m, xi, ui, xs, us, voli, vs, brk, fs, F, nullptr);
  else if constexpr (MODE == kModeFp64)
    bond_fp64<DIM, INF>(a.m, xi, ui, xs, us, voli, vs, brk, fs, F);
  else
    bond_fp32<DIM, INF>(a.m, xi, ui, xs, us, voli, vs, brk, fs, F);
}

// A coordinate as the FP32-force records hold it: its offset from the tile's
// origin times sigma, in fixed point (3D: the low word of 1.5 2^52 + half of
// it is that half, rounded, modulo 2^32) or FP32 (2D).
__device__ __forceinline__ void st_pos(double x, double o, double sigma,
                                       int32_t& q) {
  const double t = __builtin_fma(x - o, 0.5 * sigma, 0x1.8p+52);
  q = int32_t(uint32_t(__double2loint(t)) << 1);
}
__device__ __forceinline__ void st_pos(double x, double o, double sigma,
                                       float& q) {
  q = float((x - o) * sigma);
}
__device__ __forceinline__ float st_diff(int32_t a, int32_t b) {
  return float(int32_t(uint32_t(a) - uint32_t(b)));
}
__device__ __forceinline__ float st_diff(float a, float b) { return a - b; }

template <int DIM, int MODE, int INF, int U, bool NOFAIL, bool SHORT,
          bool SPLIT>
__global__ __launch_bounds__(512) void k_fd_st(
    FdArgs<DIM> a, const unsigned long long* __restrict__ bits_ro,
    const unsigned long long* __restrict__ vex_ro, double t_force,
    double t_next) {
  if (a.tdev) {  // graph-captured steps read the step's times
    t_force = a.tdev[0];
    t_next = a.tdev[1];
  }
  constexpr bool F32 = MODE == kModeFp32;
  constexpr bool EXACT = MODE == kModeExact;
  static_assert(!F32 || DIM == 3 || SPLIT, "2D: k_fd_t, k_fd_w6");
  typedef typename std::conditional<F32, float, double>::type Real;
  typedef StRec<DIM, MODE, NOFAIL> Rec;
  const int bn = SPLIT ? a.tile : int(blockDim.x);
  const int parts = SPLIT ? a.parts : 1;
  const int nsl = bn >> 6;  // slices of the tile
  const int64_t nblk = (a.nslices * 64 + bn - 1) / bn;
  const int64_t lb = xcd_block(nblk);
  if (lb >= nblk) return;
  extern __shared__ double st_smem[];
  Rec* const halo_lds = reinterpret_cast<Rec*>(st_smem);
  double org[3] = {0., 0., 0.};
  if constexpr (F32)
    load3<DIM>(reinterpret_cast<const typename VT<DIM>::T*>(a.blk_org)[lb],
               org);
  const int64_t hb = a.halo_ptr[lb];
  const int hn = int(a.halo_ptr[lb + 1] - hb);
  // Loads are issued ahead of their first use: the first halo entry, the
  // slice's bounds, the node's values and the first slot entries before the
  // staging (a launch on a small model is a chain of memory latencies).
  auto halo_id = [&](int t) -> uint32_t {
    return t >= 0 && t < hn ? uint32_t(a.halo[hb + t]) : 0u;
  };
  const int ht = int(threadIdx.x) - 1;
  uint32_t hg = halo_id(ht);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sl = SPLIT ? wave % nsl : wave;  // slice of the tile
  const int part = SPLIT ? wave / nsl : 0;
  const int64_t s = lb * nsl + sl;
  const bool slice_ok = s < a.nslices;
  const int64_t i = s * 64 + lane;
  const bool valid = slice_ok && i < a.n;
  const int64_t cb = slice_ok ? a.sl_ptr[s] : 0;
  const int width = slice_ok ? int((a.sl_ptr[s + 1] - cb) >> 6) : 0;
  const int64_t bb = cb >> 6;
  const int len = valid ? int(a.rowlen[i]) : 0;
  double xi[3] = {0., 0., 0.}, ui[3] = {0., 0., 0.};
  double vi[3] = {0., 0., 0.};  // (few wavefronts a CU: fetched early)
  double voli = 1.;
  uint32_t fl = 0;
  if (valid) {
    load3<DIM>(a.x[i], xi);
    load3<DIM>(a.u[i], ui);
    voli = a.vol[i];
    fl = a.flags[i];
    if constexpr (SPLIT)
      if (part == 0) load3<DIM>(a.v[i], vi);
  }
  const bool int_i = !(fl & kFlagNonInterior);
  // FP32-force: the node's fixed-point position and scaled displacement
  typename std::conditional<DIM == 3, int32_t, float>::type xqi[3] = {0, 0,
                                                                      0};
  double uis[3] = {0., 0., 0.};
  if constexpr (F32)
    for (int d = 0; d < DIM; d++) {
      st_pos(xi[d], org[d], a.m.sigma, xqi[d]);
      uis[d] = ui[d] * a.m.tau;
    }
  const unsigned long long* __restrict__ bits_in = bits_ro + bb;
  const unsigned long long* __restrict__ vex_in = vex_ro + bb;
  // slot entries through a buffer resource over the slice (fetches past it
  // return 0: record 0)
  const __amdgpu_buffer_rsrc_t col_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(a.colL + cb), 0, width * 64 * int(sizeof(uint16_t)),
      kBufferRsrcWord3);
  auto slot_entry = [&](int k) -> uint32_t {
    return uint32_t(__builtin_amdgcn_raw_buffer_load_b16(
        col_rsrc, lane * int(sizeof(uint16_t)), k * 64 * int(sizeof(uint16_t)),
        0));
  };
  const int stride = U * parts;
  int k0 = U * part;
  uint32_t jn[U];
#pragma unroll
  for (int q = 0; q < U; ++q) jn[q] = slot_entry(k0 + q);
  // the halo
  for (int t = ht; t < hn; t += int(blockDim.x)) {
    Rec r;
    if (t < 0) {  // record 0
      for (int d = 0; d < DIM; d++) r.u[d] = 0.;
      r.c = 0;
      for (int d = 0; d < DIM; d++) {
        if constexpr (F32 && DIM == 3) r.xq[d] = 0x7fffffff;
        else if constexpr (F32) r.xq[d] = 1e15f;
        else r.x[d] = a.far;
      }
      if constexpr (NOFAIL) r.flags = 0u;
      halo_lds[0] = r;
      hg = halo_id(t + int(blockDim.x));
      continue;
    }
    // (the next halo entry is fetched before this one's node values)
    const uint32_t g = hg;
    hg = halo_id(t + int(blockDim.x));
    double xg[3], ug[3];
    load3<DIM>(ld32(a.x, g), xg);
    load3<DIM>(ld32(a.u, g), ug);
    const double vg = ld32(a.vol, g);
    for (int d = 0; d < DIM; d++) {
      if constexpr (F32) {
        st_pos(xg[d], org[d], a.m.sigma, r.xq[d]);
        r.u[d] = ug[d] * a.m.tau;
      } else {
        r.x[d] = xg[d];
        r.u[d] = ug[d];
      }
    }
    // (FP32-force 3D: rounded once; 2D: the product k_fd_t forms)
    if constexpr (F32 && DIM == 3) r.c = float(vg * a.m.c4_infl_s);
    else if constexpr (F32) r.c = float(vg) * a.m.c4f_infl_s;
    else r.c = EXACT ? vg : vg * a.m.c4_infl;
    if constexpr (NOFAIL) r.flags = ld32(a.flags, g);
    halo_lds[t + 1] = r;
  }
  __syncthreads();
  if (!SPLIT && !slice_ok) return;  // (split tiles meet at barriers)
  const unsigned long long int_m =
      NOFAIL ? __builtin_amdgcn_ballot_w64(int_i) : ~0ull;
  // one chunk of U slots from slot k0: the bonds' forces (exact mode: F[q])
  // or the slot pairs' sums (fast modes: F[m])
  constexpr int NF = EXACT ? U : U / 2;
  auto chunk = [&](int k0, int k_next, Real (&F)[NF][DIM]) {
    uint32_t jc[U];
#pragma unroll
    for (int q = 0; q < U; ++q) {
      jc[q] = jn[q];
      jn[q] = slot_entry(k_next + q);
    }
    unsigned long long w[U], vx[U], brk[U], band[U], ex[U];
    unsigned long long ex_any = 0ull;
#pragma unroll
    for (int q = 0; q < U; ++q) {
      w[q] = bits_in[k0 + q];
      vx[q] = F32 ? 0ull : vex_in[k0 + q];
    }
#pragma unroll
    for (int q = 0; q < U; ++q) {
      // the slot entry is the record's LDS address (the kernel has no
      // static LDS, checked by the host)
      typedef const __attribute__((address_space(3))) Rec LdsRec;
      LdsRec* r = (LdsRec*)jc[q];
      SlotMasks km;
      km.act = ~0ull;
      km.w = w[q];
      km.vex = vx[q];
      if constexpr (NOFAIL)
        km.brk = int_m & __builtin_amdgcn_ballot_w64(
                             (r->flags & kFlagNonInterior) == 0u);
      else
        km.brk = ~0ull;
      brk[q] = km.brk;
      if constexpr (F32) {
        float dx[3] = {0.f, 0.f, 0.f}, dv[3] = {0.f, 0.f, 0.f};
        float G[3] = {0.f, 0.f, 0.f};
        for (int d = 0; d < DIM; d++) {
          dx[d] = st_diff(r->xq[d], xqi[d]);
          dv[d] = float(r->u[d] - uis[d]);
          if (q % 2 == 1) G[d] = F[q / 2][d];
        }
        unsigned long long nb;
        if (q % 2 == 1)
          bond_fp32_scaled<DIM, INF, NOFAIL, true>(
              a.m, dx[0], dx[1], dx[2], dv[0], dv[1], dv[2], r->c, km, nb,
              band[q], ex[q], G);
        else
          bond_fp32_scaled<DIM, INF, NOFAIL, false>(
              a.m, dx[0], dx[1], dx[2], dv[0], dv[1], dv[2], r->c, km, nb,
              band[q], ex[q], G);
        for (int d = 0; d < DIM; d++) F[q / 2][d] = G[d];
      } else {
        double dx[DIM], du[DIM];
        for (int d = 0; d < DIM; d++) {
          dx[d] = r->x[d] - xi[d];
          du[d] = r->u[d] - ui[d];
        }
        if constexpr (EXACT)
          bond_exact_fast<DIM, INF, NOFAIL, SHORT>(a.m, dx, du, r->c, km,
                                                   band[q], ex[q], F[q]);
        else if (q % 2 == 1)
          bond_fp64_staged<DIM, INF, NOFAIL, SHORT, true>(
              a.m, dx, du, r->c, km, band[q], ex[q], F[q / 2]);
        else
          bond_fp64_staged<DIM, INF, NOFAIL, SHORT, false>(
              a.m, dx, du, r->c, km, band[q], ex[q], F[q / 2]);
      }
      ex_any |= ex[q];
    }
    if (ex_any != 0ull) {  // rare: whole wavefronts skip it
#pragma unroll
      for (int q = 0; q < U; ++q) {
        if (ex[q] == 0ull) continue;
        bool fsn = false;
        if (__builtin_amdgcn_inverse_ballot_w64(ex[q]) && k0 + q < len) {
          const uint32_t g = uint32_t(
              a.halo[hb + jc[q] / uint32_t(sizeof(Rec)) - 1]);
          const bool fs0 = __builtin_amdgcn_inverse_ballot_w64(w[q]);
          bool fs = fs0;
          double Fd[3];
          st_deferred<DIM, MODE, INF>(
              a, g, xi, ui, voli,
              __builtin_amdgcn_inverse_ballot_w64(brk[q]), fs, Fd);
          fsn = fs && !fs0;
          // (FP32-force: a bond force is an FP32 value; a contact force is
          // rounded to FP32 here like every force of that mode)
          for (int d = 0; d < DIM; d++) {
            if constexpr (EXACT) F[q][d] = Fd[d];
            else F[q / 2][d] += Real(Fd[d]);
          }
        }
        // new broken bits: every lane stores the same word
        const unsigned long long nb =
            band[q] & __builtin_amdgcn_ballot_w64(fsn);
        if (nb != 0ull && k0 + q < width) a.bits[bb + k0 + q] = w[q] | nb;
      }
    }
  };
  double acc[DIM] = {};
  double* const buf = reinterpret_cast<double*>(
      reinterpret_cast<char*>(st_smem) + a.halo_bytes);
  const SplitPos sp{sl, part, parts, nsl, wave, lane};
  if constexpr (SPLIT && !F32) {
    const int64_t s0 = lb * nsl;
    split_ordered<DIM, NF, U>(chunk, buf, sp, a.sl_ptr + s0,
                              int(min(int64_t(nsl), a.nslices - s0)), width,
                              acc);
  } else {
    for (; k0 < width; k0 += stride) {
      Real F[NF][DIM];
      chunk(k0, k0 + stride, F);
#pragma unroll
      for (int m = 0; m < NF; ++m)
        for (int d = 0; d < DIM; d++) acc[d] += double(F[m][d]);
    }
    if constexpr (SPLIT) split_parts<DIM>(buf, sp, acc);
  }
  if (!valid || part != 0) return;
  if constexpr (!SPLIT) load3<DIM>(a.v[i], vi);
  st_tail<DIM>(a, i, fl, xi, ui, vi, acc, t_force, t_next);
}

// LDS bytes behind the halo records of a split launch.
inline size_t st_round_bytes(int dim, int precision, int tile, int parts) {
  if (precision == kModeFp32) return split_parts_bytes(tile, parts, dim);
  return split_ordered_bytes(tile, parts, dim,
                             precision == kModeExact ? kStSplitU
                                                     : kStSplitU / 2);
}

// Bytes of a halo record.
inline size_t st_rec_bytes(int dim, int precision, bool nofail) {
  const bool f32 = precision == kModeFp32;
  if (dim == 2)
    return f32 ? sizeof(StRec32<2, false>)
               : nofail ? sizeof(StRec64<2, true>) : sizeof(StRec64<2, false>);
  if (f32)
    return nofail ? sizeof(StRec32<3, true>) : sizeof(StRec32<3, false>);
  return nofail ? sizeof(StRec64<3, true>) : sizeof(StRec64<3, false>);
}

// Launch of the staged kernel for the configured tile (fd_st2.hip,
// fd_st3.hip).
void st_launch2(nlm_ctx* c, const FdArgs<2>& a, double tf, double tn, int U);
void st_launch3(nlm_ctx* c, const FdArgs<3>& a, double tf, double tn, int U);
// Whether the kernels' static LDS size is 0, as their addressing needs.
bool st_lds_base_zero();

// Instances of one dimension and mode.
template <int DIM, int MODE, int INF, int U, bool NOFAIL, bool SHORT,
          bool SPLIT>
void st_go(nlm_ctx* c, const FdArgs<DIM>& a, double tf, double tn) {
  static_assert(sizeof(StRec<DIM, MODE, NOFAIL>) % 8 == 0, "record");
  const unsigned g = grid_xcd(c->fd.sell.nslices * 64, a.tile);
  size_t lds = size_t(a.halo_bytes);
  if constexpr (SPLIT) lds += st_round_bytes(DIM, MODE, a.tile, a.parts);
  allow_lds(reinterpret_cast<const void*>(
                &k_fd_st<DIM, MODE, INF, U, NOFAIL, SHORT, SPLIT>),
            lds);
  hipLaunchKernelGGL((k_fd_st<DIM, MODE, INF, U, NOFAIL, SHORT, SPLIT>),
                     dim3(g), dim3(unsigned(a.tile * a.parts)), lds,
                     c->stream, a, a.bits, a.vexw, tf, tn);
}

template <int DIM, int MODE, int U, bool SPLIT, bool SHORT, bool NOFAIL>
void st_inf(nlm_ctx* c, const FdArgs<DIM>& a, double tf, double tn) {
  const int inf = c->fd.rnp.inf_type;
  if (inf == 0)
    st_go<DIM, MODE, 0, U, NOFAIL, SHORT, SPLIT>(c, a, tf, tn);
  else if (inf == 1)
    st_go<DIM, MODE, 1, U, NOFAIL, SHORT, SPLIT>(c, a, tf, tn);
  else
    st_go<DIM, MODE, 2, U, NOFAIL, SHORT, SPLIT>(c, a, tf, tn);
}

template <int DIM, int MODE, int U, bool SPLIT>
void st_opt(nlm_ctx* c, const FdArgs<DIM>& a, double tf, double tn) {
  // the exponent's range form is chosen where the break test bounds it
  // (exp_short); models with no-fail regions keep the general form
  if (a.has_nofail)
    st_inf<DIM, MODE, U, SPLIT, false, true>(c, a, tf, tn);
  else if (MODE != kModeFp32 && a.m.x_break_lo <= kExpShortMax)
    st_inf<DIM, MODE, U, SPLIT, MODE != kModeFp32, false>(c, a, tf, tn);
  else
    st_inf<DIM, MODE, U, SPLIT, false, false>(c, a, tf, tn);
}

}  // namespace nlm
