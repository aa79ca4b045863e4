// fd_st2.hip -- 2D instances of the staged step kernel (fd_staged.h).

#include "fd_staged.h"

namespace nlm {

// The chunk width U trades instruction-level parallelism for registers: the
// FP64 mode takes the tuned width; the exact mode and split rows have one.
void st_launch2(nlm_ctx* c, const FdArgs<2>& a, double tf, double tn, int U) {
  const int mode = c->fd.precision;
  if (a.parts > 1) {
    if (mode == kModeExact)
      return st_opt<2, kModeExact, kStSplitU, true>(c, a, tf, tn);
    if (mode == kModeFp64)
      return st_opt<2, kModeFp64, kStSplitU, true>(c, a, tf, tn);
    return st_opt<2, kModeFp32, kStSplitU, true>(c, a, tf, tn);
  }
  if (mode == kModeExact)
    return st_opt<2, kModeExact, 2, false>(c, a, tf, tn);
  if (U == 2) return st_opt<2, kModeFp64, 2, false>(c, a, tf, tn);
  if (U == 8) return st_opt<2, kModeFp64, 8, false>(c, a, tf, tn);
  st_opt<2, kModeFp64, 4, false>(c, a, tf, tn);
}

bool st_lds_base_zero() {
  hipFuncAttributes fa;
  return hipFuncGetAttributes(
             &fa, reinterpret_cast<const void*>(
                      &k_fd_st<2, kModeFp64, 0, 2, false, true, false>)) ==
             hipSuccess &&
         fa.sharedSizeBytes == 0;
}

}  // namespace nlm
