// What the kernels that normalise rows share.
#pragma once
#include <hip/hip_runtime.h>

#include "tppx_common.h"

namespace tppx {

template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
// sum / max over the 16 lanes of a DPP row; every lane of the row gets the result
__device__ __forceinline__ float row16_sum(float v) {
  v += dpp_mov<0xB1>(v);  // quad_perm [1,0,3,2]
  v += dpp_mov<0x4E>(v);  // quad_perm [2,3,0,1]
  v += dpp_mov<0x141>(v); // row_half_mirror
  v += dpp_mov<0x140>(v); // row_mirror
  return v;
}
__device__ __forceinline__ float wave_sum(float v) {
  v = row16_sum(v);
  float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0));
  float b = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16));
  float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
  float d = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 48));
  return (a + b) + (c + d);
}

__device__ __forceinline__ void unpack8(const uint4& w, float (&f)[8]) {
  const uint32_t d[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
  for (int i = 0; i < 4; i++) {
    f[2 * i] = bf16_bits_to_f32(d[i] & 0xffffu);
    f[2 * i + 1] = bf16_bits_to_f32(d[i] >> 16);
  }
}

// 1 / sqrt(mean square + eps) of a row from its threads' sums of squares, for a workgroup of 256; red: four floats of LDS.  In one
// place, as the launches that normalise on the way to something else promise the bits of the one that writes the rows.  (The
// whole row in one place, as a struct of registers with load() and values(): up to 4 % slower, 2048 rows of 4096 5.6 -> 5.9 us.)
__device__ __forceinline__ float rms_scale(float ss, float* red, int K, float eps) {
  const int tid = threadIdx.x;
  ss = wave_sum(ss);
  if ((tid & 63) == 0)
    red[tid >> 6] = ss;
  __syncthreads();
  const float v = ((red[0] + red[1]) + (red[2] + red[3])) * (1.0f / (float)K);
  return 1.0f / sqrtf(v + eps);
}

} // namespace tppx
