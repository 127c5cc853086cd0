// The kernels of tppx_wide.h on bf16 weights.
#include "tppx_wide.h"

namespace tppx {

hipError_t launch_wide_bf16(const BigParams& P, int form, int wgs, bool dual, hipStream_t stream) {
  return wide_launch<true>(P, form, wgs, dual, stream);
}

} // namespace tppx
