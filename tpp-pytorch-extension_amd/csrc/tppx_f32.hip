// Linears whose compute type is float or half: TppBlockedQInt8LinearW<float / half, uint8_t, float / half>
// (src/csrc/fused_gemm.h:1076-1341) and TppBlockedLinearW<float / half, uint8_t / bfloat16, float / half>
// (:785-1073), the element-type switch of fc_plain_wrap (src/csrc/llm/fused_llm_infer.cpp:1526-1545).  Everything after
// the products stays in fp32 up to the one rounding to the output type.
#include <hip/hip_runtime.h>

#include "tppx.h"
#include "tppx_common.h"
#include "tppx_launch.h"

namespace tppx {

// Where one output goes: bias, post-op and rounding on the fp32 sum, in the output type.
struct WideOut {
  const void* bias; // [N] of bias_dtype, or null
  const void* in1;  // [M][N] of the output type, or null
  const void* in2;
  void* y;          // [M][N]
  float scale;
  int bias_dtype, half, post, M, N, K;
};

__device__ __forceinline__ float load_elem(const void* p, int dtype, int64_t i) {
  if (dtype == TPPX_DT_F32)
    return reinterpret_cast<const float*>(p)[i];
  if (dtype == TPPX_DT_F16)
    return (float)reinterpret_cast<const _Float16*>(p)[i];
  return bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(p)[i]);
}

// The post-op on the fp32 tile rounded to the activations' type, re-rounding where the CPU path stores its tile
// (src/csrc/fused_gemm.h:1343-1488 on Tout = float or half): for float nothing is rounded.
template <bool HALF>
__device__ __forceinline__ float wide_round(float v) {
  return HALF ? (float)(_Float16)v : v;
}
template <bool HALF>
__device__ __forceinline__ float wide_post(float v, int post, const void* in1, const void* in2, float scale, int64_t i) {
  auto ld = [&](const void* p) {
    return HALF ? (float)reinterpret_cast<const _Float16*>(p)[i] : reinterpret_cast<const float*>(p)[i];
  };
  const float y = wide_round<HALF>(v);
  switch (post) {
    case TPPX_POST_SILU:
      return wide_round<HALF>(y * wide_round<HALF>(1.0f / (1.0f + __expf(-y))));
    case TPPX_POST_MUL:
      return wide_round<HALF>(ld(in1) * y);
    case TPPX_POST_ADD_SCALE:
      return wide_round<HALF>(fmaf(ld(in1), scale, y));
    case TPPX_POST_ADD2_SCALE:
      return wide_round<HALF>(fmaf(ld(in2), scale, wide_round<HALF>(y + ld(in1))));
    case TPPX_POST_GELU:
      return wide_round<HALF>(0.5f * y * (1.0f + erff(y * 0.70710678118654752f)));
    case TPPX_POST_RELU:
      return y < 0.f ? 0.f : y;
    default:
      return y;
  }
}
__device__ __forceinline__ void wide_store(const WideOut& o, int m, int n, float v) {
  const int64_t i = (int64_t)m * o.N + n;
  if (o.half)
    reinterpret_cast<_Float16*>(o.y)[i] = (_Float16)wide_post<true>(v, o.post, o.in1, o.in2, o.scale, i);
  else
    reinterpret_cast<float*>(o.y)[i] = wide_post<false>(v, o.post, o.in1, o.in2, o.scale, i);
}

// ---------------------------------------------------------------------------
// QINT8-family weights on int8 rows:
//   y[m][n] = bias[n] + sum_b float(sum_{k in b} xq[m][k] * wq[n][k]) * (sa[m][b] * sw[n][b])
// one fused multiply-add per K block in ascending block order.
// ---------------------------------------------------------------------------
struct F32OutParams {
  WideOut o;
  const int8_t* xq; // [M][K]
  const float* sa;  // [M][K/qbs]
  const void* qw;   // native tiles [N/16][K/64][64 lanes][16 B]
  const float* sw;  // native scales [N/16][K/qbs][16]
  int qbs, split;   // split: parts a K block is cut into
};

// Few rows: MT row tiles x NT channel tiles per workgroup, its eight waves on eight K blocks at a time.  The float chain
// of an output has to run in block order, but a block's integer sum does not depend on any other: every wave leaves its
// sums and scale products in LDS and the threads then take the chain of their outputs one round further.  (One wave
// walking all of K, one load in flight, took 38 us for 2 x 1088 x 9984 and 46 for 61 x 3264 x 8704.)  Where K has fewer
// than eight blocks (per-channel scales) a block is cut into `split` parts, summed as integers before the conversion.
// QUAD: parts of 256 channels, whose loads are requested a round ahead.
template <int MT, int NT, bool QUAD>
__global__ void __launch_bounds__(512)
linear_qint8_wide_kernel(const F32OutParams p) {
  constexpr int W = 8, T = MT * NT, OPT = (T * 256 + 511) / 512; // outputs per thread
  __shared__ int sums[W][T * 256];
  __shared__ float prods[W][T * 256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tiles = p.o.N / 16, tile0 = blockIdx.x * NT, m0 = blockIdx.y * MT * 16;
  const int KT = p.o.K / 64, NB = p.o.K / p.qbs, TPU = p.qbs / 64 / p.split, U = NB * p.split;
  const i32x4* wq[NT];
  const float* swp[NT];
#pragma unroll
  for (int ni = 0; ni < NT; ni++) { // tiles past N re-read the last one, never stored
    const int tile = min(tile0 + ni, tiles - 1);
    wq[ni] = reinterpret_cast<const i32x4*>(p.qw) + (int64_t)tile * KT * 64 + lane;
    swp[ni] = p.sw + (int64_t)tile * NB * 16 + (lane & 15);
  }
  // A operand: row lane & 15 (rows past M re-read the last one, never stored), K group lane >> 4
  const int8_t* xr[MT];
  const float* sar[MT][4];
#pragma unroll
  for (int mi = 0; mi < MT; mi++) {
    xr[mi] = p.xq + (int64_t)min(m0 + mi * 16 + (lane & 15), p.o.M - 1) * p.o.K + (lane >> 4) * 16;
#pragma unroll
    for (int r = 0; r < 4; r++)
      sar[mi][r] = p.sa + (int64_t)min(m0 + mi * 16 + (lane >> 4) * 4 + r, p.o.M - 1) * NB;
  }
  float f[OPT];
  int a[OPT];
#pragma unroll
  for (int i = 0; i < OPT; i++) {
    const int o = threadIdx.x + i * 512, n = (tile0 + (o >> 8) % NT) * 16 + ((o & 255) >> 2 & 15);
    f[i] = p.o.bias && n < p.o.N ? load_elem(p.o.bias, p.o.bias_dtype, n) : 0.f;
    a[i] = 0;
  }
  i32x4 xa[QUAD ? 4 : 1][MT], wb[QUAD ? 4 : 1][NT];
  auto request = [&](int u) {
#pragma unroll
    for (int t = 0; t < 4; t++) {
#pragma unroll
      for (int ni = 0; ni < NT; ni++)
        wb[t][ni] = __builtin_nontemporal_load(wq[ni] + (int64_t)(u * 4 + t) * 64);
#pragma unroll
      for (int mi = 0; mi < MT; mi++)
        xa[t][mi] = *reinterpret_cast<const i32x4*>(xr[mi] + (int64_t)(u * 4 + t) * 64);
    }
  };
  if (QUAD && wave < U)
    request(wave);
  for (int u0 = 0; u0 < U; u0 += W) {
    const int u = u0 + wave;
    if (u < U) {
      i32x4 acc[MT][NT];
#pragma unroll
      for (int mi = 0; mi < MT; mi++)
#pragma unroll
        for (int ni = 0; ni < NT; ni++)
          acc[mi][ni] = i32x4{0, 0, 0, 0};
      const int b = u / p.split;
      float swv[NT], sav[MT][4];
#pragma unroll
      for (int ni = 0; ni < NT; ni++)
        swv[ni] = swp[ni][(int64_t)b * 16];
#pragma unroll
      for (int mi = 0; mi < MT; mi++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          sav[mi][r] = sar[mi][r][b];
      if constexpr (QUAD) {
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
          for (int mi = 0; mi < MT; mi++)
#pragma unroll
            for (int ni = 0; ni < NT; ni++)
              acc[mi][ni] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[t][mi], wb[t][ni], acc[mi][ni], 0, 0, 0);
        if (u + W < U)
          request(u + W);
      } else {
        for (int t = u * TPU; t < (u + 1) * TPU; t++) {
#pragma unroll
          for (int ni = 0; ni < NT; ni++)
            wb[0][ni] = wq[ni][(int64_t)t * 64];
#pragma unroll
          for (int mi = 0; mi < MT; mi++)
            xa[0][mi] = *reinterpret_cast<const i32x4*>(xr[mi] + (int64_t)t * 64);
#pragma unroll
          for (int mi = 0; mi < MT; mi++)
#pragma unroll
            for (int ni = 0; ni < NT; ni++)
              acc[mi][ni] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[0][mi], wb[0][ni], acc[mi][ni], 0, 0, 0);
        }
      }
#pragma unroll
      for (int mi = 0; mi < MT; mi++)
#pragma unroll
        for (int ni = 0; ni < NT; ni++) {
          const int at = (mi * NT + ni) * 256 + lane * 4; // result rows (lane >> 4) * 4 + r, column lane & 15
          *reinterpret_cast<i32x4*>(&sums[wave][at]) = acc[mi][ni];
          *reinterpret_cast<f32x4*>(&prods[wave][at]) =
              f32x4{sav[mi][0] * swv[ni], sav[mi][1] * swv[ni], sav[mi][2] * swv[ni], sav[mi][3] * swv[ni]};
        }
    }
    __syncthreads();
    const int n = min(W, U - u0);
#pragma unroll
    for (int i = 0; i < OPT; i++) {
      const int o = threadIdx.x + i * 512;
      if (o < T * 256) {
        for (int w = 0; w < n; w++) {
          a[i] += sums[w][o];
          if (p.split == 1 || (u0 + w + 1) % p.split == 0) {
            f[i] = fmaf((float)a[i], prods[w][o], f[i]);
            a[i] = 0;
          }
        }
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < OPT; i++) {
    const int o = threadIdx.x + i * 512, t = o >> 8, l = (o & 255) >> 2;
    const int m = m0 + (t / NT) * 16 + (l >> 4) * 4 + (o & 3), n = (tile0 + t % NT) * 16 + (l & 15);
    if (o < T * 256 && m < p.o.M && n < p.o.N)
      wide_store(p.o, m, n, f[i]);
  }
}

// Many rows: enough tiles to fill the chip without cutting K, so a wave keeps the chains of its 32 x 64 outputs in
// registers; four waves = 64 rows x 128 channels.
template <bool QUAD>
__global__ void __launch_bounds__(256)
linear_qint8_wide_rows_kernel(const F32OutParams p) {
  constexpr int MT = 2, NT = 4;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tiles = p.o.N / 16, tile0 = blockIdx.x * 8 + (wave & 1) * NT, m0 = blockIdx.y * 64 + (wave >> 1) * 32;
  if (m0 >= p.o.M || tile0 >= tiles) // whole waves only; no barrier below
    return;
  const int KT = p.o.K / 64, NB = p.o.K / p.qbs, TPB = p.qbs / 64;
  const i32x4* wq[NT];
  const float* swp[NT];
  float f[MT][NT][4];
#pragma unroll
  for (int ni = 0; ni < NT; ni++) {
    const int tile = min(tile0 + ni, tiles - 1);
    wq[ni] = reinterpret_cast<const i32x4*>(p.qw) + (int64_t)tile * KT * 64 + lane;
    swp[ni] = p.sw + (int64_t)tile * NB * 16 + (lane & 15);
    const float bv = p.o.bias ? load_elem(p.o.bias, p.o.bias_dtype, tile * 16 + (lane & 15)) : 0.f;
#pragma unroll
    for (int mi = 0; mi < MT; mi++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        f[mi][ni][r] = bv;
  }
  const int8_t* xr[MT];
  const float* sar[MT][4];
#pragma unroll
  for (int mi = 0; mi < MT; mi++) {
    xr[mi] = p.xq + (int64_t)min(m0 + mi * 16 + (lane & 15), p.o.M - 1) * p.o.K + (lane >> 4) * 16;
#pragma unroll
    for (int r = 0; r < 4; r++)
      sar[mi][r] = p.sa + (int64_t)min(m0 + mi * 16 + (lane >> 4) * 4 + r, p.o.M - 1) * NB;
  }
  // QUAD (blocks in whole runs of 256 channels): every K tile is requested four tiles ahead
  constexpr int R = QUAD ? 4 : 1;
  i32x4 xa[R][MT], wb[R][NT];
  auto request = [&](int t, int at) {
#pragma unroll
    for (int ni = 0; ni < NT; ni++)
      wb[at][ni] = wq[ni][(int64_t)t * 64];
#pragma unroll
    for (int mi = 0; mi < MT; mi++)
      xa[at][mi] = *reinterpret_cast<const i32x4*>(xr[mi] + (int64_t)t * 64);
  };
  if (QUAD) {
#pragma unroll
    for (int t = 0; t < R; t++)
      request(t, t);
  }
  for (int b = 0; b < NB; b++) {
    i32x4 acc[MT][NT];
#pragma unroll
    for (int mi = 0; mi < MT; mi++)
#pragma unroll
      for (int ni = 0; ni < NT; ni++)
        acc[mi][ni] = i32x4{0, 0, 0, 0};
    for (int t0 = b * TPB; t0 < (b + 1) * TPB; t0 += R) {
#pragma unroll
      for (int at = 0; at < R; at++) {
        if (!QUAD)
          request(t0, 0);
#pragma unroll
        for (int mi = 0; mi < MT; mi++)
#pragma unroll
          for (int ni = 0; ni < NT; ni++)
            acc[mi][ni] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[at][mi], wb[at][ni], acc[mi][ni], 0, 0, 0);
        if (QUAD)
          request(min(t0 + at + R, KT - 1), at);
      }
    }
    float swv[NT];
#pragma unroll
    for (int ni = 0; ni < NT; ni++)
      swv[ni] = swp[ni][(int64_t)b * 16];
#pragma unroll
    for (int mi = 0; mi < MT; mi++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const float sav = sar[mi][r][b];
#pragma unroll
        for (int ni = 0; ni < NT; ni++)
          f[mi][ni][r] = fmaf((float)acc[mi][ni][r], sav * swv[ni], f[mi][ni][r]);
      }
  }
#pragma unroll
  for (int mi = 0; mi < MT; mi++)
#pragma unroll
    for (int ni = 0; ni < NT; ni++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int m = m0 + mi * 16 + (lane >> 4) * 4 + r, n = (tile0 + ni) * 16 + (lane & 15);
        if (m < p.o.M && n < p.o.N)
          wide_store(p.o, m, n, f[mi][ni][r]);
      }
}

// ---------------------------------------------------------------------------
// float / half activations on MXFP4 or unquantized bf16 weights: the activations keep their own precision,
//   y[m][n] = bias[n] + sum_k x[m][k] * w[n][k]          (products exact, fp32 sums)
// Every weight value is a bf16.  An activation is cut into bf16 terms that add up to it exactly -- its leading 8
// significant bits, the next 8, and for fp32 the last 8 -- so two (half) or three (float) bf16 MFMAs form the products
// that an fp32 MFMA would, at 16 times its rate each; terms are cut off, not rounded, so none is larger than the value.
// Two kinds of activations have no such terms.  Below 2^-110 the last ones would lie under the smallest bf16, 2^-133: what the
// three terms of a value leave over shows in the lower half of the third one's float.  And an infinity or NaN gives Inf - Inf:
// outputs that come out non-finite.  Rows and outputs with either are formed again by the workgroup on the fp32 MFMA, from the
// values as they are; the others keep the sums they have, so a row does not depend on its neighbours.
// Native layouts: lane (g, n) of a 128-channel K tile holds the 32 weights k = g*32 .. g*32 + 31 of channel n; MFMA j
// multiplies channels g*32 + j*8 .. + 7 of each group g.
// ---------------------------------------------------------------------------
struct WideParams {
  WideOut o;
  const void* x;     // [M][K] fp32 or fp16
  const void* qw;    // native tiles
  const uint8_t* sw; // MXFP4: native scale bytes [N/16][K/128][64]
};

// high halves of two dwords: {a[31:16], b[31:16]} as (low, high)
__device__ __forceinline__ uint32_t high_halves(uint32_t a, uint32_t b) {
  return __builtin_amdgcn_perm(b, a, 0x07060302u);
}

// eight activations -> TERMS bf16 operands; over: its low half collects what they leave over
template <bool XHALF>
__device__ __forceinline__ void split_terms(const i32x4* raw, bf16x8* out, uint32_t& over) {
  constexpr int TERMS = XHALF ? 2 : 3;
  uint32_t part[TERMS][4];
#pragma unroll
  for (int d = 0; d < 4; d++) {
    float v[2];
    if (XHALF) {
      const uint32_t u = (uint32_t)raw[0][d];
      v[0] = (float)__builtin_bit_cast(_Float16, (uint16_t)(u & 0xffffu));
      v[1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(u >> 16));
    } else {
      v[0] = __int_as_float(raw[d >> 1][(d & 1) * 2]);
      v[1] = __int_as_float(raw[d >> 1][(d & 1) * 2 + 1]);
    }
#pragma unroll
    for (int t = 0; t < TERMS; t++) {
      part[t][d] = high_halves(__float_as_uint(v[0]), __float_as_uint(v[1]));
      if (t + 1 < TERMS) {
        v[0] -= __uint_as_float(__float_as_uint(v[0]) & 0xffff0000u);
        v[1] -= __uint_as_float(__float_as_uint(v[1]) & 0xffff0000u);
      } else if (!XHALF) {
        asm("v_or3_b32 %0, %1, %2, %0" : "+v"(over) : "v"(v[0]), "v"(v[1]));
      }
    }
  }
#pragma unroll
  for (int t = 0; t < TERMS; t++)
    out[t] = __builtin_bit_cast(bf16x8, i32x4{(int)part[t][0], (int)part[t][1], (int)part[t][2], (int)part[t][3]});
}

// the weights of eight channels of K: dword of codes -> one bf16 operand
__device__ __forceinline__ bf16x8 expand_codes(uint32_t c, float sc) {
  const bf16x2 p0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(c, sc, 0), p1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(c, sc, 1);
  const bf16x2 p2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(c, sc, 2), p3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(c, sc, 3);
  return bf16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}

// MT row tiles x NT channel tiles per workgroup, its eight waves on every eighth K tile, partial tiles summed through
// LDS in wave order.  Bound by the chain of a wave's K tiles with few rows (16 x 4096 x 4096 12.2 us in half, 12.5 in
// float), by cutting the activations and by the LDS sums with many.  Its error against float64 is a fifth of that of
// one wave per 16 x 16 outputs on the fp32 MFMA (61 x 3264 x 8704 in float: 3.1e-7 relative against 1.6e-6), as eight
// partial sums of 32 products at a time round less often than one of four.  A workgroup that forms its outputs again takes the
// time of the fp32 MFMA on top (one infinity in 61 x 3264 x 8704 in half 21 -> 67 us, a row of 2^-118 in float 38 -> 90;
// all on the fp32 MFMA 64 and 104).
template <bool XHALF, bool WBF16, int MT, int NT>
__global__ void __launch_bounds__(512, MT * NT <= 2 ? 4 : 2) // two workgroups to a CU while their tiles are small
linear_wide_kernel(const WideParams p) {
  constexpr int W = 8, T = MT * NT, TERMS = XHALF ? 2 : 3, XV = XHALF ? 1 : 2, BV = WBF16 ? 4 : 1;
  __shared__ __align__(16) float part[W][T * 256];
  __shared__ __align__(16) uint16_t rows_over[MT][W]; // bit r: row r of the tile has activations beyond three terms
  __shared__ int again;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4;
  const int tiles = p.o.N / 16, tile0 = blockIdx.x * NT, m0 = blockIdx.y * MT * 16, KT = p.o.K / 128;
  const i32x4* wq[NT];
  const uint8_t* swp[NT];
#pragma unroll
  for (int ni = 0; ni < NT; ni++) { // tiles past N re-read the last one, never stored
    const int64_t tile = min(tile0 + ni, tiles - 1);
    wq[ni] = reinterpret_cast<const i32x4*>(p.qw) + tile * KT * (BV * 64) + lane;
    swp[ni] = WBF16 ? nullptr : p.sw + tile * KT * 64 + lane;
  }
  const i32x4* xr[MT];
#pragma unroll
  for (int mi = 0; mi < MT; mi++) // rows past M re-read the last one, never stored
    xr[mi] = reinterpret_cast<const i32x4*>(reinterpret_cast<const char*>(p.x) +
                                            ((int64_t)min(m0 + mi * 16 + (lane & 15), p.o.M - 1) * p.o.K + g * 32) * (XHALF ? 2 : 4));
  f32x4 acc[MT][NT];
#pragma unroll
  for (int mi = 0; mi < MT; mi++)
#pragma unroll
    for (int ni = 0; ni < NT; ni++)
      acc[mi][ni] = f32x4{0.f, 0.f, 0.f, 0.f};
  uint32_t over[MT] = {};
  i32x4 wb[NT][BV];
  uint32_t sb[NT];
  auto request = [&](int kt) {
#pragma unroll
    for (int ni = 0; ni < NT; ni++) {
#pragma unroll
      for (int j = 0; j < BV; j++)
        wb[ni][j] = wq[ni][(int64_t)kt * (BV * 64) + j * 64];
      sb[ni] = WBF16 ? 0 : swp[ni][(int64_t)kt * 64];
    }
  };
  if (wave < KT)
    request(wave);
  for (int kt = wave; kt < KT; kt += W) {
    i32x4 xv[4][MT][XV];
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int mi = 0; mi < MT; mi++)
#pragma unroll
        for (int v = 0; v < XV; v++)
          xv[j][mi][v] = xr[mi][(int64_t)kt * (16 * XV) + j * XV + v];
    i32x4 wc[NT][BV];
    float sc[NT];
#pragma unroll
    for (int ni = 0; ni < NT; ni++) {
#pragma unroll
      for (int j = 0; j < BV; j++)
        wc[ni][j] = wb[ni][j];
      sc[ni] = e8m0_to_f32(sb[ni]);
    }
    if (kt + W < KT)
      request(kt + W);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      bf16x8 w[NT];
#pragma unroll
      for (int ni = 0; ni < NT; ni++)
        w[ni] = WBF16 ? __builtin_bit_cast(bf16x8, wc[ni][WBF16 ? j : 0]) : expand_codes((uint32_t)wc[ni][0][j], sc[ni]);
#pragma unroll
      for (int mi = 0; mi < MT; mi++) {
        bf16x8 x[TERMS];
        split_terms<XHALF>(xv[j][mi], x, over[mi]);
#pragma unroll
        for (int t = TERMS - 1; t >= 0; t--)
#pragma unroll
          for (int ni = 0; ni < NT; ni++)
            acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[t], w[ni], acc[mi][ni], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int mi = 0; mi < MT; mi++)
#pragma unroll
    for (int ni = 0; ni < NT; ni++)
      *reinterpret_cast<f32x4*>(&part[wave][(mi * NT + ni) * 256 + lane * 4]) = acc[mi][ni];
  if (!XHALF) {
#pragma unroll
    for (int mi = 0; mi < MT; mi++) {
      uint64_t rows = __builtin_amdgcn_ballot_w64((over[mi] & 0xffffu) != 0); // lane (g, row)
      rows |= rows >> 32;
      rows |= rows >> 16;
      if (lane == 0)
        rows_over[mi][wave] = (uint16_t)rows;
    }
  }
  if (threadIdx.x == 0)
    again = 0;
  __syncthreads();
  uint32_t overs[MT] = {}, any_over = 0; // per row tile, of all waves
  if (!XHALF) {
#pragma unroll
    for (int mi = 0; mi < MT; mi++) {
      const i32x4 r = *reinterpret_cast<const i32x4*>(rows_over[mi]);
      const uint32_t u = (uint32_t)(r[0] | r[1] | r[2] | r[3]);
      overs[mi] = (u | u >> 16) & 0xffffu;
      any_over |= overs[mi];
    }
  }
  constexpr int OPT = (T * 256 + 511) / 512; // outputs per thread
  auto each = [&](auto&& f) {
#pragma unroll
    for (int i = 0; i < OPT; i++) {
      const int o = threadIdx.x + i * 512, t = o >> 8, l = (o & 255) >> 2, r = (l >> 4) * 4 + (o & 3);
      const int m = m0 + (t / NT) * 16 + r, n = (tile0 + t % NT) * 16 + (l & 15);
      if (o >= T * 256 || m >= p.o.M || n >= p.o.N)
        continue;
      float s = part[0][o];
#pragma unroll
      for (int w = 1; w < W; w++)
        s += part[w][o];
      f(i, t / NT, r, m, n, s);
    }
  };
  auto store = [&](int m, int n, float s) { wide_store(p.o, m, n, p.o.bias ? load_elem(p.o.bias, p.o.bias_dtype, n) + s : s); };
  uint32_t redo = 0; // bit i: this thread's i-th output
  each([&](int i, int mi, int r, int m, int n, float s) {
    bool over_row = false;
    if (any_over) {
#pragma unroll
      for (int k = 0; k < MT; k++)
        over_row |= k == mi && (overs[k] >> r & 1u);
    }
    if (over_row || !(fabsf(s) <= 3.4028234663852886e38f))
      redo |= 1u << i;
    else
      store(m, n, s);
  });
  if (redo)
    again = 1;
  __syncthreads();
  if (!again) // the same for the whole workgroup
    return;
#pragma unroll
  for (int mi = 0; mi < MT; mi++)
#pragma unroll
    for (int ni = 0; ni < NT; ni++)
      acc[mi][ni] = f32x4{0.f, 0.f, 0.f, 0.f};
  int ln = lane; // (hidden from the compiler, which would keep the operands' addresses in registers through the loop above)
  asm volatile("" : "+v"(ln));
#pragma unroll 1
  for (int kt = wave; kt < KT; kt += W) {
#pragma unroll 1
    for (int j = 0; j < 4; j++) { // MFMA e: channels g * 32 + j * 8 + e of the four groups
      float x[MT][8], w[NT][8];
#pragma unroll
      for (int mi = 0; mi < MT; mi++) {
        const i32x4* src = reinterpret_cast<const i32x4*>(reinterpret_cast<const char*>(p.x) +
            ((int64_t)min(m0 + mi * 16 + (ln & 15), p.o.M - 1) * p.o.K + kt * 128 + (ln >> 4) * 32 + j * 8) * (XHALF ? 2 : 4));
        i32x4 v[XV];
#pragma unroll
        for (int k = 0; k < XV; k++)
          v[k] = src[k];
#pragma unroll
        for (int e = 0; e < 8; e++)
          x[mi][e] = XHALF ? (float)__builtin_bit_cast(_Float16, (uint16_t)((uint32_t)v[0][e >> 1] >> (16 * (e & 1))))
                           : __int_as_float(v[XHALF ? 0 : e >> 2][e & 3]);
      }
#pragma unroll
      for (int ni = 0; ni < NT; ni++) {
        const int64_t slot = (int64_t)min(tile0 + ni, tiles - 1) * KT + kt;
        bf16x8 b;
        if constexpr (WBF16)
          b = __builtin_bit_cast(bf16x8, reinterpret_cast<const i32x4*>(p.qw)[(slot * 4 + j) * 64 + ln]);
        else
          b = expand_codes(reinterpret_cast<const uint32_t*>(p.qw)[(slot * 64 + ln) * 4 + j], e8m0_to_f32(p.sw[slot * 64 + ln]));
#pragma unroll
        for (int e = 0; e < 8; e++)
          w[ni][e] = (float)b[e];
      }
#pragma unroll
      for (int e = 0; e < 8; e++)
#pragma unroll
        for (int mi = 0; mi < MT; mi++)
#pragma unroll
          for (int ni = 0; ni < NT; ni++)
            acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[mi][e], w[ni][e], acc[mi][ni], 0, 0, 0);
    }
  }
#pragma unroll
  for (int mi = 0; mi < MT; mi++)
#pragma unroll
    for (int ni = 0; ni < NT; ni++)
      *reinterpret_cast<f32x4*>(&part[wave][(mi * NT + ni) * 256 + lane * 4]) = acc[mi][ni];
  __syncthreads();
  each([&](int i, int, int, int m, int n, float s) {
    if (redo >> i & 1u)
      store(m, n, s);
  });
}

template <bool HALF>
__global__ void __launch_bounds__(256)
post_op_wide_kernel(const float* __restrict__ acc, const void* __restrict__ in1, const void* __restrict__ in2,
                    void* __restrict__ out, int64_t n, int post, float scale) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n)
    return;
  const float o = wide_post<HALF>(acc[i], post, in1, in2, scale, i);
  if (HALF)
    reinterpret_cast<_Float16*>(out)[i] = (_Float16)o;
  else
    reinterpret_cast<float*>(out)[i] = o;
}

static int check_out(const char* who, const WideOut& o) {
  TPPX_REQUIRE(o.post >= TPPX_POST_NONE && o.post <= TPPX_POST_RELU, TPPX_EINVAL, "%s: unknown post-op id %d", who, o.post);
  const bool need1 = o.post == TPPX_POST_MUL || o.post == TPPX_POST_ADD_SCALE || o.post == TPPX_POST_ADD2_SCALE;
  TPPX_REQUIRE(!need1 || o.in1, TPPX_EINVAL, "%s: post-op %d needs post_in", who, o.post);
  TPPX_REQUIRE(o.post != TPPX_POST_ADD2_SCALE || o.in2, TPPX_EINVAL, "%s: post-op %d needs post_in2", who, o.post);
  TPPX_REQUIRE(!o.bias || o.bias_dtype == TPPX_DT_F32 || o.bias_dtype == TPPX_DT_F16 || o.bias_dtype == TPPX_DT_BF16, TPPX_EINVAL,
               "%s: bias must be fp32, fp16 or bf16 (dtype id %d)", who, o.bias_dtype);
  return TPPX_OK;
}

static int run_linear_wide(const char* who, const void* x, int x_dtype, const void* w, const void* sw, int w_kind,
                           const WideOut& o, int64_t M, int64_t N, int64_t K, hipStream_t st) {
  TPPX_REQUIRE(x && w && o.y, TPPX_EINVAL, "%s: null pointer", who);
  TPPX_REQUIRE(x_dtype == TPPX_DT_F32 || x_dtype == TPPX_DT_F16, TPPX_EINVAL, "%s: activations must be fp32 or fp16 (dtype id %d)", who, x_dtype);
  TPPX_REQUIRE(w_kind == TPPX_W_MXFP4 || w_kind == TPPX_W_BF16, TPPX_EINVAL, "%s: weight kind %d is neither MXFP4 nor bf16", who, w_kind);
  TPPX_REQUIRE(w_kind == TPPX_W_BF16 || sw, TPPX_EINVAL, "%s: MXFP4 weights need their scale bytes", who);
  TPPX_REQUIRE(aligned16(x) && aligned16(w), TPPX_EINVAL, "%s: activation / weight pointer not 16-byte aligned", who);
  TPPX_REQUIRE(M >= 0 && M < (1 << 22), TPPX_ESHAPE, "%s: M=%ld out of range", who, (long)M);
  TPPX_REQUIRE(N > 0 && N % (w_kind == TPPX_W_MXFP4 ? 32 : 16) == 0, TPPX_ESHAPE, "%s: N=%ld must be a positive multiple of %d", who, (long)N, w_kind == TPPX_W_MXFP4 ? 32 : 16);
  TPPX_REQUIRE(K > 0 && K % 128 == 0, TPPX_ESHAPE, "%s: K=%ld must be a positive multiple of 128 (native tiles span 128 input channels)", who, (long)K);
  TPPX_REQUIRE(N / 16 < (1 << 30), TPPX_ESHAPE, "%s: N=%ld too large", who, (long)N);
  if (int rc = check_out(who, o))
    return rc;
  if (M == 0)
    return TPPX_OK;
  WideParams p;
  p.o = o;
  p.o.M = (int)M;
  p.o.N = (int)N;
  p.o.K = (int)K;
  p.x = x;
  p.qw = w;
  p.sw = (const uint8_t*)sw;
  const int64_t tiles = N / 16;
  auto go = [&](auto XH, auto WB) {
    constexpr bool xh = decltype(XH)::value, wb = decltype(WB)::value;
    auto launch = [&](auto MT, auto NT) {
      constexpr int mt = decltype(MT)::value, nt = decltype(NT)::value;
      linear_wide_kernel<xh, wb, mt, nt><<<dim3((unsigned)((tiles + nt - 1) / nt), (unsigned)((M + mt * 16 - 1) / (mt * 16))), 512, 0, st>>>(p);
    };
    // One row tile: two channel tiles once one each would be more than two rounds of workgroups.  Otherwise 32 rows x 16
    // channels while those fit one round, else x 32, and from a few rounds of those the largest tile whose operands and
    // partial sums still leave two waves per SIMD (64 x 64 with 4-bit weights, 64 x 32 with the four times wider bf16
    // ones).  MXFP4 x half: 64 rows of 1088 x 9984 21.3 us on 32 x 16, 22.4 on 32 x 32, 53.9 on 64 x 64; 128 rows of
    // 11008 x 4096 51.2 on 32 x 32, 50.5 on 64 x 64; float, with three terms to cut, at 128 rows 105 and 112, at 512 rows 379
    // and 327; bf16 weights x half at 128 rows 79.6 on 32 x 32, 65.6 on 64 x 32.
    typedef std::integral_constant<int, 1> one;
    typedef std::integral_constant<int, 2> two;
    typedef std::integral_constant<int, 4> four;
    const int64_t rows32 = (M + 31) / 32;
    if (M <= 16)
      tiles < 512 ? launch(one{}, one{}) : launch(one{}, two{});
    else if (rows32 * tiles <= 256)
      launch(two{}, one{});
    else if (rows32 * ((tiles + 1) / 2) <= (wb ? 1000 : xh ? 450 : 1200))
      launch(two{}, two{});
    else
      launch(four{}, std::conditional_t<wb, two, four>{});
  };
  if (x_dtype == TPPX_DT_F16) {
    if (w_kind == TPPX_W_BF16)
      go(std::true_type{}, std::true_type{});
    else
      go(std::true_type{}, std::false_type{});
  } else {
    if (w_kind == TPPX_W_BF16)
      go(std::false_type{}, std::true_type{});
    else
      go(std::false_type{}, std::false_type{});
  }
  return check_hip(hipGetLastError(), who);
}

static int run_linear_qint8(const char* who, const void* xq, const void* sa, const void* qw, const void* sw, const WideOut& o,
                            int64_t M, int64_t N, int64_t K, int64_t qbs, hipStream_t st) {
  F32OutParams p;
  p.o = o;
  p.o.M = (int)M;
  p.o.N = (int)N;
  p.o.K = (int)K;
  p.xq = (const int8_t*)xq;
  p.sa = (const float*)sa;
  p.qw = qw;
  p.sw = (const float*)sw;
  p.qbs = (int)qbs;
  const int64_t tiles = N / 16, NB = K / qbs, TPB = qbs / 64;
  int split = 1;
  while (NB * split < 8 && TPB % (split * 2) == 0)
    split *= 2;
  p.split = split;
  // 16 channels a workgroup up to 32 rows and while 32 x 16 fits one round of the chip.  Beyond, by estimates in us
  // (measured at 48 .. 512 rows of 1088 x 9984 .. 11008 x 11008): 32 x 32 with K cut over the waves takes
  // 5 + 0.0027 K a round of 256 workgroups, 64 x 128 with whole chains per wave 15 + 0.0073 K.  11008 x 4096: 64 rows
  // 40 against 42, 128 rows 72 against 43; 1088 x 9984: 128 rows 36 against 90.
  const int64_t rows32 = (M + 31) / 32, small = (rows32 * ((tiles + 1) / 2) + 255) / 256,
                large = ((M + 63) / 64 * ((tiles + 7) / 8) + 255) / 256;
  const bool quad = TPB / split == 4;
  auto launch = [&](auto MT, auto NT) {
    constexpr int mt = decltype(MT)::value, nt = decltype(NT)::value;
    const dim3 grid((unsigned)((tiles + nt - 1) / nt), (unsigned)((M + mt * 16 - 1) / (mt * 16)));
    if (quad)
      linear_qint8_wide_kernel<mt, nt, true><<<grid, 512, 0, st>>>(p);
    else
      linear_qint8_wide_kernel<mt, nt, false><<<grid, 512, 0, st>>>(p);
  };
  typedef std::integral_constant<int, 1> one;
  typedef std::integral_constant<int, 2> two;
  if (M <= 16)
    launch(one{}, one{});
  else if (M <= 32 || rows32 * tiles <= 256)
    launch(two{}, one{});
  else if (rows32 <= 65535 && 5.0 + 0.0027 * K * small < 15.0 + 0.0073 * K * large) // (the grid: rows come in twice as many blocks)
    launch(two{}, two{});
  else {
    const dim3 grid((unsigned)((tiles + 7) / 8), (unsigned)((M + 63) / 64));
    if (TPB % 4 == 0)
      linear_qint8_wide_rows_kernel<true><<<grid, 256, 0, st>>>(p);
    else
      linear_qint8_wide_rows_kernel<false><<<grid, 256, 0, st>>>(p);
  }
  return check_hip(hipGetLastError(), who);
}

static int check_linear_qint8(const char* who, const void* xq, const void* sa, const void* qw, const void* sw, const void* y,
                              int64_t M, int64_t N, int64_t K, int64_t qbs) {
  TPPX_REQUIRE(xq && sa && qw && sw && y, TPPX_EINVAL, "%s: null pointer", who);
  TPPX_REQUIRE(aligned16(xq) && aligned16(qw), TPPX_EINVAL, "%s: activation / weight pointer not 16-byte aligned", who);
  TPPX_REQUIRE(M >= 0 && M < (1 << 30), TPPX_ESHAPE, "%s: M=%ld out of range", who, (long)M);
  TPPX_REQUIRE(N > 0 && N % 16 == 0, TPPX_ESHAPE, "%s: N=%ld must be a positive multiple of 16", who, (long)N);
  TPPX_REQUIRE(qbs >= 64 && qbs % 64 == 0, TPPX_ESHAPE, "%s: block size %ld must be a multiple of 64", who, (long)qbs);
  TPPX_REQUIRE(K > 0 && K % qbs == 0, TPPX_ESHAPE, "%s: K=%ld must be a positive multiple of the block size %ld", who, (long)K, (long)qbs);
  TPPX_REQUIRE(M * N < ((int64_t)1 << 40) && N / 16 < 65536 * 32768ll, TPPX_ESHAPE, "%s: problem too large", who);
  TPPX_REQUIRE((M + 63) / 64 <= 65535, TPPX_ESHAPE, "%s: M=%ld exceeds the grid (at most 65535 blocks of 64 rows)", who, (long)M);
  return TPPX_OK;
}

} // namespace tppx

using namespace tppx;

extern "C" int tppx_linear_wide(const void* x, int x_dtype, const void* w, const void* sw, int w_kind, const void* bias_f32,
                                void* y_f32, int64_t M, int64_t N, int64_t K, tppx_stream_t stream) {
  const WideOut o = {bias_f32, nullptr, nullptr, y_f32, 1.0f, TPPX_DT_F32, 0, TPPX_POST_NONE, 0, 0, 0};
  return run_linear_wide("tppx_linear_wide", x, x_dtype, w, sw, w_kind, o, M, N, K, (hipStream_t)stream);
}

extern "C" int tppx_linear_wide_post(const void* x, int x_dtype, const void* w, const void* sw, int w_kind, const void* bias,
                                     int bias_dtype, const void* post_in, const void* post_in2, void* y, int64_t M, int64_t N,
                                     int64_t K, int post_op, float post_scale, tppx_stream_t stream) {
  const WideOut o = {bias, post_in, post_in2, y, post_scale, bias_dtype, x_dtype == TPPX_DT_F16, post_op, 0, 0, 0};
  return run_linear_wide("tppx_linear_wide_post", x, x_dtype, w, sw, w_kind, o, M, N, K, (hipStream_t)stream);
}

extern "C" int tppx_post_op_wide(const void* acc_f32, int out_dtype, int post_op, const void* post_in, const void* post_in2,
                                 float post_scale, void* out, int64_t count, tppx_stream_t stream) {
  const char* who = "tppx_post_op_wide";
  TPPX_REQUIRE(acc_f32 && out, TPPX_EINVAL, "%s: null pointer", who);
  TPPX_REQUIRE(out_dtype == TPPX_DT_F32 || out_dtype == TPPX_DT_F16, TPPX_EINVAL, "%s: output must be fp32 or fp16 (dtype id %d)", who, out_dtype);
  TPPX_REQUIRE(post_op >= TPPX_POST_NONE && post_op <= TPPX_POST_RELU, TPPX_EINVAL, "%s: unknown post-op id %d", who, post_op);
  const bool need1 = post_op == TPPX_POST_MUL || post_op == TPPX_POST_ADD_SCALE || post_op == TPPX_POST_ADD2_SCALE;
  TPPX_REQUIRE(!need1 || post_in, TPPX_EINVAL, "%s: post-op %d needs post_in", who, post_op);
  TPPX_REQUIRE(post_op != TPPX_POST_ADD2_SCALE || post_in2, TPPX_EINVAL, "%s: post-op %d needs post_in2", who, post_op);
  TPPX_REQUIRE(count >= 0 && count < ((int64_t)1 << 40), TPPX_ESHAPE, "%s: count %ld out of range", who, (long)count);
  if (count == 0)
    return TPPX_OK;
  const unsigned blocks = (unsigned)((count + 255) / 256);
  if (out_dtype == TPPX_DT_F16)
    post_op_wide_kernel<true><<<blocks, 256, 0, (hipStream_t)stream>>>((const float*)acc_f32, post_in, post_in2, out, count, post_op, post_scale);
  else
    post_op_wide_kernel<false><<<blocks, 256, 0, (hipStream_t)stream>>>((const float*)acc_f32, post_in, post_in2, out, count, post_op, post_scale);
  return check_hip(hipGetLastError(), who);
}

extern "C" int tppx_linear_qint8_f32(const void* xq, const void* sa, const void* qw, const void* sw, const void* bias_f32,
                                     void* y_f32, int64_t M, int64_t N, int64_t K, int64_t qbs, tppx_stream_t stream) {
  const char* who = "tppx_linear_qint8_f32";
  if (int rc = check_linear_qint8(who, xq, sa, qw, sw, y_f32, M, N, K, qbs))
    return rc;
  if (M == 0)
    return TPPX_OK;
  const WideOut o = {bias_f32, nullptr, nullptr, y_f32, 1.0f, TPPX_DT_F32, 0, TPPX_POST_NONE, 0, 0, 0};
  return run_linear_qint8(who, xq, sa, qw, sw, o, M, N, K, qbs, (hipStream_t)stream);
}

extern "C" int tppx_linear_qint8_wide(const void* x, int dtype, void* xq, void* sa, const void* qw, const void* sw,
                                      const void* bias, int bias_dtype, const void* post_in, const void* post_in2, void* y,
                                      int64_t M, int64_t N, int64_t K, int64_t qbs, int post_op, float post_scale,
                                      tppx_stream_t stream) {
  const char* who = "tppx_linear_qint8_wide";
  TPPX_REQUIRE(dtype == TPPX_DT_F32 || dtype == TPPX_DT_F16, TPPX_EINVAL, "%s: compute type must be fp32 or fp16 (dtype id %d)", who, dtype);
  if (int rc = check_linear_qint8(who, xq, sa, qw, sw, y, M, N, K, qbs))
    return rc;
  const WideOut o = {bias, post_in, post_in2, y, post_scale, bias_dtype, dtype == TPPX_DT_F16, post_op, 0, 0, 0};
  if (int rc = check_out(who, o))
    return rc;
  if (M == 0)
    return TPPX_OK;
  if (x)
    if (int rc = check_hip(launch_quant_act_int8_wide(x, dtype, M, K, qbs, xq, sa, (hipStream_t)stream), who))
      return rc;
  return run_linear_qint8(who, xq, sa, qw, sw, o, M, N, K, qbs, (hipStream_t)stream);
}
