// fd_st3.hip -- 3D instances of the staged step kernel (fd_staged.h).

#include "fd_staged.h"

namespace nlm {

void st_launch3(nlm_ctx* c, const FdArgs<3>& a, double tf, double tn, int U) {
  const int mode = c->fd.precision;
  if (a.parts > 1) {
    if (mode == kModeExact)
      return st_opt<3, kModeExact, kStSplitU, true>(c, a, tf, tn);
    if (mode == kModeFp64)
      return st_opt<3, kModeFp64, kStSplitU, true>(c, a, tf, tn);
    return st_opt<3, kModeFp32, kStSplitU, true>(c, a, tf, tn);
  }
  if (mode == kModeExact) return st_opt<3, kModeExact, 2, false>(c, a, tf, tn);
  if (mode == kModeFp64) {
    if (U == 2) return st_opt<3, kModeFp64, 2, false>(c, a, tf, tn);
    return st_opt<3, kModeFp64, 4, false>(c, a, tf, tn);
  }
  if (U == 2) return st_opt<3, kModeFp32, 2, false>(c, a, tf, tn);
  st_opt<3, kModeFp32, 4, false>(c, a, tf, tn);
}

}  // namespace nlm
