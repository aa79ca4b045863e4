// split_rows.h -- rows shared by several wavefronts of a workgroup.
//
// `parts` wavefronts share the 64 rows of a slice: part p takes the slot
// chunks p, p + parts, ... of U slots.  split_ordered passes the summands of
// every chunk (NF values of NC components a lane) through LDS in rounds of
// one chunk a part and adds them in list order, so the sums have the bits of
// one wavefront walking the row; split_parts adds the parts' own sums in the
// order of the parts.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace nlm {

// The wavefront's place: slice of the tile, part, and the tile's slices.
struct SplitPos {
  int sl, part, parts, nsl, wave, lane;
};

// LDS bytes of split_ordered's buffer.
inline size_t split_ordered_bytes(int tile, int parts, int nc, int nf) {
  return size_t(tile / 64) * size_t(nc * nf * parts) * 64 * sizeof(double);
}
// LDS bytes of split_parts' buffer.
inline size_t split_parts_bytes(int tile, int parts, int nc) {
  return size_t(tile / 64) * size_t(nc * (parts - 1)) * 64 * sizeof(double);
}

// chunk(k0, k_next, F) computes the summands of slots k0 .. k0 + U - 1 and
// fetches ahead for k_next.  sl_ptr: slice bounds (64 entries a slot) from the
// tile's first slice; nslices of them exist.  Every wavefront of the
// workgroup calls this; part 0 of each slice receives the sums in out.
template <int NC, int NF, int U, class Chunk>
__device__ __forceinline__ void split_ordered(
    Chunk&& chunk, double* buf, const SplitPos& p,
    const int64_t* __restrict__ sl_ptr, int nslices, int width,
    double (&out)[NC]) {
  const int stride = U * p.parts;
  const int nv = NF * p.parts;  // summands of a lane's component in a round
  const int nw = p.nsl * p.parts;
  const int ntask = p.nsl * NC;
  constexpr int MT = (NC + 1) / 2;  // tasks a wavefront (parts >= 2)
  auto width_of = [&](int q) {
    return q < nslices ? int((sl_ptr[q + 1] - sl_ptr[q]) >> 6) : 0;
  };
  int wmax = 0;
  for (int q = 0; q < p.nsl; q++) wmax = max(wmax, width_of(q));
  double sum[MT];
  int tw[MT];
#pragma unroll
  for (int t = 0; t < MT; t++) {
    const int task = p.wave + t * nw;
    sum[t] = 0.;
    tw[t] = task < ntask ? width_of(task / NC) : 0;
  }
  int k0 = U * p.part;
  for (int base = 0; base < wmax; base += stride, k0 += stride) {
    if (k0 < width) {
      double F[NF][NC];
      chunk(k0, k0 + stride, F);
#pragma unroll
      for (int m = 0; m < NF; ++m)
        for (int d = 0; d < NC; d++)
          buf[((p.sl * NC + d) * nv + p.part * NF + m) * 64 + p.lane] =
              F[m][d];
    }
    __syncthreads();
    // (slots past a row are exact zeros; chunks past a slice were not
    // written)
#pragma unroll
    for (int t = 0; t < MT; t++) {
      const int cnt = min(nv, (tw[t] - base + U - 1) / U * NF);
      const double* const v = buf + (p.wave + t * nw) * nv * 64 + p.lane;
      for (int m = 0; m < cnt; m++) sum[t] += v[m * 64];
    }
    __syncthreads();
  }
#pragma unroll
  for (int t = 0; t < MT; t++) {
    const int task = p.wave + t * nw;
    if (task < ntask) buf[task * 64 + p.lane] = sum[t];
  }
  __syncthreads();
  if (p.part == 0)
    for (int d = 0; d < NC; d++) out[d] = buf[(p.sl * NC + d) * 64 + p.lane];
}

// Adds the sums of parts 1.. to part 0's, in the order of the parts.
template <int NC>
__device__ __forceinline__ void split_parts(double* buf, const SplitPos& p,
                                            double (&acc)[NC]) {
  if (p.part > 0)
    for (int d = 0; d < NC; d++)
      buf[((p.sl * (p.parts - 1) + p.part - 1) * NC + d) * 64 + p.lane] =
          acc[d];
  __syncthreads();
  if (p.part == 0)
    for (int q = 0; q < p.parts - 1; q++)
      for (int d = 0; d < NC; d++)
        acc[d] += buf[((p.sl * (p.parts - 1) + q) * NC + d) * 64 + p.lane];
}

}  // namespace nlm
