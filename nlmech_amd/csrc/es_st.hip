// es_st.hip -- instances and launches of the state-based staged passes
// (es_staged.h).

#include "es_staged.h"

namespace nlm {
namespace {

// Slots a chunk of whole rows: 4 in 3D (80^3 nodes, exact mode: 317 against
// 323 us per step with 2), 2 in 2D (600 x 500, FP64: 47.9 against 48.8).
template <int DIM>
constexpr int kWholeU = DIM == 3 ? 4 : 2;

template <int DIM, int MODE, int U, bool SPLIT>
void go_dil(nlm_ctx* c, const EsArgs<DIM>& e, size_t lds) {
  allow_lds(reinterpret_cast<const void*>(&k_es_dil_st<DIM, MODE, U, SPLIT>),
            lds);
  hipLaunchKernelGGL((k_es_dil_st<DIM, MODE, U, SPLIT>),
                     dim3(grid_xcd(c->fd.sell.nslices * 64, e.f.tile)),
                     dim3(unsigned(e.f.tile * e.f.parts)), lds, c->stream, e,
                     e.f.bits);
}

template <int DIM, int MODE, int U, bool SPLIT>
void go_force(nlm_ctx* c, const EsArgs<DIM>& e, size_t lds, double tf,
              double tn) {
  allow_lds(
      reinterpret_cast<const void*>(&k_es_force_st<DIM, MODE, U, SPLIT>), lds);
  hipLaunchKernelGGL((k_es_force_st<DIM, MODE, U, SPLIT>),
                     dim3(grid_xcd(c->fd.sell.nslices * 64, e.f.tile)),
                     dim3(unsigned(e.f.tile * e.f.parts)), lds, c->stream, e,
                     e.f.bits, tf, tn);
}

// The pass's record stride and LDS, set in e.
template <int DIM>
size_t place(nlm_ctx* c, EsArgs<DIM>& e, bool force) {
  const EsStLds l = es_st_lds(DIM, c->fd.precision, c->fd.halo_max, e.f.tile,
                              e.f.parts, force, size_t(c->fd.es_lds_max));
  e.stride = int(l.stride);
  e.f.halo_bytes = int64_t(l.records);
  return l.bytes;
}

template <int DIM, int MODE>
void dil_mode(nlm_ctx* c, const EsArgs<DIM>& e, size_t lds) {
  if (e.f.parts > 1) go_dil<DIM, MODE, kStSplitU, true>(c, e, lds);
  else go_dil<DIM, MODE, kWholeU<DIM>, false>(c, e, lds);
}

template <int DIM, int MODE>
void force_mode(nlm_ctx* c, const EsArgs<DIM>& e, size_t lds, double tf,
                double tn) {
  if (e.f.parts > 1) go_force<DIM, MODE, kStSplitU, true>(c, e, lds, tf, tn);
  else go_force<DIM, MODE, kWholeU<DIM>, false>(c, e, lds, tf, tn);
}

}  // namespace

template <int DIM>
void es_st_dil(nlm_ctx* c, EsArgs<DIM> e) {
  const int mode = c->fd.precision;
  const size_t lds = place<DIM>(c, e, false);
  if (mode == kModeExact) return dil_mode<DIM, kModeExact>(c, e, lds);
  if (mode == kModeFp64) return dil_mode<DIM, kModeFp64>(c, e, lds);
  if constexpr (DIM == 2) dil_mode<DIM, kModeFp32>(c, e, lds);
}

template <int DIM>
void es_st_force(nlm_ctx* c, EsArgs<DIM> e, double tf, double tn) {
  const int mode = c->fd.precision;
  const size_t lds = place<DIM>(c, e, true);
  if (mode == kModeExact) return force_mode<DIM, kModeExact>(c, e, lds, tf, tn);
  if (mode == kModeFp64) return force_mode<DIM, kModeFp64>(c, e, lds, tf, tn);
  if constexpr (DIM == 2) force_mode<DIM, kModeFp32>(c, e, lds, tf, tn);
}

template void es_st_dil<2>(nlm_ctx*, EsArgs<2>);
template void es_st_dil<3>(nlm_ctx*, EsArgs<3>);
template void es_st_force<2>(nlm_ctx*, EsArgs<2>, double, double);
template void es_st_force<3>(nlm_ctx*, EsArgs<3>, double, double);

}  // namespace nlm
