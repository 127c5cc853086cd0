// The kernels of tppx_wide.h on MXFP4 weights, and the sums over K slices.
#include "tppx_wide.h"

namespace tppx {

hipError_t launch_wide_mxfp4(const BigParams& P, int form, int wgs, bool dual, hipStream_t stream) {
  return wide_launch<false>(P, form, wgs, dual, stream);
}

template <int F = 0>
static hipError_t wide_sum_launch(const BigParams& P, int form, int wgs, hipStream_t stream) {
  if constexpr (F < N_WIDE) {
    constexpr WideForm f = WIDE_FORMS[F];
    if constexpr (f.split)
      if (form == F) {
        const dim3 grid(wgs * f.w);
        switch (P.S) {
        case 2: return wide_go(wide_sum_kernel<f.mt, f.nt, f.w, 2>, P, grid, 64, 0, stream);
        case 3: return wide_go(wide_sum_kernel<f.mt, f.nt, f.w, 3>, P, grid, 64, 0, stream);
        case 4: return wide_go(wide_sum_kernel<f.mt, f.nt, f.w, 4>, P, grid, 64, 0, stream);
        case 6: return wide_go(wide_sum_kernel<f.mt, f.nt, f.w, 6>, P, grid, 64, 0, stream);
        }
      }
    return wide_sum_launch<F + 1>(P, form, wgs, stream);
  } else {
    return hipErrorInvalidValue;
  }
}

hipError_t launch_wide_sum(const BigParams& P, int form, int wgs, hipStream_t stream) {
  return wide_sum_launch(P, form, wgs, stream);
}

} // namespace tppx
