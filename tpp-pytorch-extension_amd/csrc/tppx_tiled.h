// What the kernels for many rows share: descriptors, the order of the tiles over the XCDs, epilogues.
#pragma once
#include <hip/hip_runtime.h>

#include "tppx_common.h"
#include "tppx_launch.h"

namespace tppx {

__device__ __forceinline__ bf16x8 tl_cvt_fp4x8(uint32_t codes, float scale) {
  bf16x2 c0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(codes, scale, 0);
  bf16x2 c1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(codes, scale, 1);
  bf16x2 c2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(codes, scale, 2);
  bf16x2 c3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(codes, scale, 3);
  bf16x8 w;
  w[0] = c0[0]; w[1] = c0[1]; w[2] = c1[0]; w[3] = c1[1];
  w[4] = c2[0]; w[5] = c2[1]; w[6] = c3[0]; w[7] = c3[1];
  return w;
}

// buffer descriptor of an operand below 4 GiB (addresses checked by the host, so without a bound of its own)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tl_rsrc(const void* q) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(q), 0, 0xffffffffu, 0x00020000);
}

// XCD-aware tile order: returns (bm, bn) of this workgroup.  Workgroup ids go round the 8 XCDs; XCD x gets a
// rectangle of the tile space and walks it row block fastest, so that the workgroups resident on an XCD at the same
// time share operand tiles in its L2.  xm = how many of the 8 rectangles lie along M (1: an XCD owns NB/8 channel
// blocks and all row blocks; 2, 4: 1/xm of the row blocks and xm/8 of the channel blocks).  Every XCD fetches
// 1/xm of the activations and xm/8 of the weights from memory.  The host passes an xm that divides evenly.
__device__ __forceinline__ void tile_of_block(int MB, int NB, int& bm, int& bn, int xm, int id) {
  const int T = MB * NB;
  if ((T & 7) == 0 && xm > 1) {
    const int x = id & 7, r = id >> 3;
    const int xn = 8 / xm;                // rectangles along N
    const int mb = MB / xm, nb = NB / xn; // the rectangle of XCD x: mb x nb tiles at (x % xm, x / xm)
    bm = (x % xm) * mb + r % mb;
    bn = (x / xm) * nb + r / mb;
    return;
  }
  // an eighth of the tiles in column-major order, whether or not NB divides by 8 (the first T mod 8 XCDs own one more);
  // dealt round the XCDs instead, each of them fetches most of the weights
  const int x = id & 7;
  id = x * (T >> 3) + min(x, T & 7) + (id >> 3);
  bm = id % MB;
  bn = id / MB;
}
__device__ __forceinline__ void tile_of_block(int MB, int NB, int& bm, int& bn, int xm = 1) {
  tile_of_block(MB, NB, bm, bn, xm, blockIdx.x);
}

// Several GEMMs over one activation (fused q/k/v) share a launch: the channel
// blocks of all segments form one grid.
struct BigParams {
  TiledParams seg[TPPX_MAX_SEGS];
  int nb0[TPPX_MAX_SEGS + 1]; // first channel block of each segment, then the total
  int n_seg;
  int xm;                     // XCD rectangles along M (see tile_of_block)
  int S;                      // K slices (grid y) whose sums go to `part`
  float* part;                // [S][workgroup][wave][tiles of the wave][64 lanes][4]
};

// Epilogue of a 128 x 64 wave tile through a wave-private LDS region: the
// fp32 sums of 64 rows at a time are written there (statically indexed, so the
// accumulators stay in registers), then read back row-contiguously; every
// lane finishes 8 adjacent channels and writes them with one 16-byte store.
// It is a chain at the end of every workgroup, so what bounds it is latency: the post-op is chosen once in front of it
// (chosen per output, every one of the 8 x 16 sat behind branches of its own) and its input is requested whole before
// the first sum is staged (requested in the loop, each of 16 rounds waited for memory).  QINT8 4096 x 4096 with residual
// at 1000 / 2048 rows 33.1 -> 28.7 / 51.6 -> 44.0 us, 11008 x 4096 at 1000 rows 87.8 -> 71.5; a four-layer prompt on bf16
// weights at 2048 tokens 3478 -> 3277, MXFP4 at 333 989 -> 919.
constexpr int EP_LD = 68; // floats per staged row of 64 channels: 64 + 4 keeps the 4-row lane groups on distinct banks
constexpr int ep_ld(int nt) { return nt * 16 + 4; }
template <int MT, int POST, int NT> // POST < 0: whatever p.post_op says; NT = 16-channel tiles of the wave tile (4, 3 or 2)
__device__ __forceinline__ void big_epilogue_post(const TiledParams& p, f32x4 (&acc)[MT][NT], float* stage, int m_base,
                                                  int tile_base) {
  constexpr bool INPUT = POST == TPPX_POST_MUL || POST == TPPX_POST_ADD_SCALE;
  const int lane = threadIdx.x & 63;
  // lanes per row, rows per wave instruction (three channel tiles: 10 rows, the last four lanes idle)
  constexpr int LPR = NT * 2, RPI = 64 / LPR, LD = ep_ld(NT);
  const int r0 = lane / LPR;
  const int cx = (lane % LPR) * 8; // first of this lane's 8 channels inside the wave tile
  const int tile = tile_base + (cx >> 4);
  const bool tile_ok = tile < p.tiles && r0 < RPI;
  const int n = min(tile, p.tiles - 1) * 16 + (cx & 15);
  // MH row tiles staged at a time: 64 rows, or the whole wave tile when it has fewer; the last time what is left
  constexpr int MH = MT < 4 ? MT : 4, NH = (MT + MH - 1) / MH;
  // every input of the post-op is requested before the first sum is staged (rows past the end read the last one)
  constexpr int NI = (MH * 16 + RPI - 1) / RPI;
  uint4 in[INPUT ? NH * NI : 1];
  if constexpr (INPUT) {
#pragma unroll
    for (int it = 0; it < NH * NI; it++)
      in[it] = *reinterpret_cast<const uint4*>(p.post_in + (int64_t)min(m_base + it / NI * (MH * 16) + it % NI * RPI + r0, p.M - 1) * p.N + n);
  }
  float bias[8];
#pragma unroll
  for (int e = 0; e < 8; e++)
    bias[e] = p.bias ? bf16_bits_to_f32(p.bias[n + e]) : 0.0f;
  static_for<0, NH>([&](auto H) {
    constexpr int h = decltype(H)::value, mh = MT - h * MH < MH ? MT - h * MH : MH, NR = (mh * 16 + RPI - 1) / RPI;
#pragma unroll
    for (int mt = 0; mt < mh; mt++)
#pragma unroll
      for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          stage[(mt * 16 + (lane >> 4) * 4 + r) * LD + nt * 16 + (lane & 15)] = acc[h * MH + mt][nt][r];
    // same wave wrote and reads: no barrier, the compiler orders the LDS accesses
    auto rows8 = [&](int it) {
      constexpr bool EVEN = mh * 16 % RPI == 0; // else the last rows are past the staged ones
      const int row = EVEN ? it * RPI + r0 : min(it * RPI + r0, mh * 16 - 1);
      const int m = m_base + h * (MH * 16) + row;
      const bool ok = tile_ok && m < p.M && (EVEN || it * RPI + r0 < mh * 16);
      const f32x4 v0 = *reinterpret_cast<const f32x4*>(stage + row * LD + cx);
      const f32x4 v1 = *reinterpret_cast<const f32x4*>(stage + row * LD + cx + 4);
      const int64_t o = (int64_t)m * p.N + n;
      uint32_t out[4];
      if constexpr (POST >= 0) {
        const uint4 i1 = INPUT ? in[INPUT ? h * NI + it : 0] : make_uint4(0, 0, 0, 0);
        const uint32_t w1[4] = {i1.x, i1.y, i1.z, i1.w};
#pragma unroll
        for (int e = 0; e < 4; e++)
          out[e] = apply_post_pair<POST>((e < 2 ? v0[2 * e] : v1[2 * e - 4]) + bias[2 * e],
                                         (e < 2 ? v0[2 * e + 1] : v1[2 * e - 3]) + bias[2 * e + 1], w1[e], p.post_scale);
        if (ok)
          *reinterpret_cast<uint4*>(p.y + o) = make_uint4(out[0], out[1], out[2], out[3]);
      } else if (ok) {
        uint4 i1 = make_uint4(0, 0, 0, 0), i2 = make_uint4(0, 0, 0, 0);
        if (p.post_in)
          i1 = *reinterpret_cast<const uint4*>(p.post_in + o);
        if (p.post_in2)
          i2 = *reinterpret_cast<const uint4*>(p.post_in2 + o);
        const uint32_t w1[4] = {i1.x, i1.y, i1.z, i1.w}, w2[4] = {i2.x, i2.y, i2.z, i2.w};
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float lo = (e < 2 ? v0[2 * e] : v1[2 * e - 4]) + bias[2 * e];
          const float hi = (e < 2 ? v0[2 * e + 1] : v1[2 * e - 3]) + bias[2 * e + 1];
          const uint32_t a = apply_post_bits(lo, p.post_op, w1[e] & 0xffffu, w2[e] & 0xffffu, p.post_scale);
          const uint32_t b = apply_post_bits(hi, p.post_op, w1[e] >> 16, w2[e] >> 16, p.post_scale);
          out[e] = (a & 0xffffu) | (b << 16);
        }
        *reinterpret_cast<uint4*>(p.y + o) = make_uint4(out[0], out[1], out[2], out[3]);
      }
    };
    if constexpr (POST >= 0) {
#pragma unroll
      for (int it = 0; it < NR; it++)
        rows8(it);
    } else {
      for (int it = 0; it < NR; it++)
        rows8(it);
    }
  });
}

template <int MT, int NT = 4>
__device__ __forceinline__ void big_epilogue(const TiledParams& p, f32x4 (&acc)[MT][NT], float* stage, int m_base,
                                             int tile_base) {
  switch (p.post_op) {
  case TPPX_POST_NONE: return big_epilogue_post<MT, TPPX_POST_NONE, NT>(p, acc, stage, m_base, tile_base);
  case TPPX_POST_SILU: return big_epilogue_post<MT, TPPX_POST_SILU, NT>(p, acc, stage, m_base, tile_base);
  case TPPX_POST_MUL: return big_epilogue_post<MT, TPPX_POST_MUL, NT>(p, acc, stage, m_base, tile_base);
  case TPPX_POST_ADD_SCALE: return big_epilogue_post<MT, TPPX_POST_ADD_SCALE, NT>(p, acc, stage, m_base, tile_base);
  default: return big_epilogue_post<MT, -1, NT>(p, acc, stage, m_base, tile_base);
  }
}

// The gate/up pair: the first half of the wave tile's channels are gate sums and the second the up sums of the SAME
// output channels, so silu(gate) * up is formed here, with the rounding points of SiluPostOp followed by MulPostOp, and
// only the product is written: a lane finishes 8 adjacent channels of one row (16-byte store, NT lanes per row).
template <int MT, int NT = 4>
__device__ __forceinline__ void big_epilogue_dual(const TiledParams& pg, const TiledParams& pu, f32x4 (&acc)[MT][NT],
                                                  float* stage, int m_base, int tile_base) {
  const int lane = threadIdx.x & 63;
  constexpr int LPR = NT, RPI = 64 / LPR, LD = ep_ld(NT);
  const int cx = (lane % LPR) * 8; // first of this lane's 8 channels among the wave's NT * 8
  const int tile = tile_base + (cx >> 4);
  const bool tile_ok = tile < pg.tiles;
  const int n = min(tile, pg.tiles - 1) * 16 + (cx & 15);
  float bg[8], bu[8];
#pragma unroll
  for (int e = 0; e < 8; e++) {
    bg[e] = pg.bias ? bf16_bits_to_f32(pg.bias[n + e]) : 0.0f;
    bu[e] = pu.bias ? bf16_bits_to_f32(pu.bias[n + e]) : 0.0f;
  }
  constexpr int MH = MT < 4 ? MT : 4; // row tiles staged at a time (the last time what is left)
  static_for<0, (MT + MH - 1) / MH>([&](auto H) {
    constexpr int h = decltype(H)::value, mh = MT - h * MH < MH ? MT - h * MH : MH;
#pragma unroll
    for (int mt = 0; mt < mh; mt++)
#pragma unroll
      for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          stage[(mt * 16 + (lane >> 4) * 4 + r) * LD + nt * 16 + (lane & 15)] = acc[h * MH + mt][nt][r];
    // same wave wrote and reads: no barrier, the compiler orders the LDS accesses
#pragma unroll
    for (int it = 0; it < (mh * 16 + RPI - 1) / RPI; it++) {
      constexpr bool EVEN = mh * 16 % RPI == 0; // else the last rows are past the staged ones
      const int row = EVEN ? it * RPI + lane / LPR : min(it * RPI + lane / LPR, mh * 16 - 1);
      const int m = m_base + h * (MH * 16) + row;
      const f32x4 g0 = *reinterpret_cast<const f32x4*>(stage + row * LD + cx);
      const f32x4 g1 = *reinterpret_cast<const f32x4*>(stage + row * LD + cx + 4);
      const f32x4 u0 = *reinterpret_cast<const f32x4*>(stage + row * LD + NT * 8 + cx);
      const f32x4 u1 = *reinterpret_cast<const f32x4*>(stage + row * LD + NT * 8 + cx + 4);
      if (tile_ok && m < pg.M && (EVEN || it * RPI + lane / LPR < mh * 16)) {
        uint32_t out[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float glo = (e < 2 ? g0[2 * e] : g1[2 * e - 4]) + bg[2 * e];
          const float ghi = (e < 2 ? g0[2 * e + 1] : g1[2 * e - 3]) + bg[2 * e + 1];
          const float ulo = (e < 2 ? u0[2 * e] : u1[2 * e - 4]) + bu[2 * e];
          const float uhi = (e < 2 ? u0[2 * e + 1] : u1[2 * e - 3]) + bu[2 * e + 1];
          const uint32_t gate = apply_post_pair<TPPX_POST_SILU>(glo, ghi, 0, 1.0f);
          out[e] = apply_post_pair<TPPX_POST_MUL>(ulo, uhi, gate, 1.0f);
        }
        *reinterpret_cast<uint4*>(pu.y + (int64_t)m * pu.N + n) = make_uint4(out[0], out[1], out[2], out[3]);
      }
    }
  });
}

// Wave tiles of the kernels in tppx_wide.h: MT x NT tiles of 16 rows x 16 channels per wave, w waves side by side; which weight
// formats are built, and whether with K in slices (MXFP4).  bf16 weights: 96 rows only --
// 4096 x 4096 and 4096 x 11008 at 576 .. 768 rows 46 -> 31 and 108 -> 75 us; the smaller wave tiles of two channel tiles lose to
// 64 x 128 or win by what their estimates err (fixed costs that depend on where the weights lie), three do not fit the registers.
struct WideForm {
  int mt, nt, w;
  bool mxfp4, bf16, split;
};
constexpr WideForm WIDE_FORMS[] = {
    {2, 1, 8, true, false, true},  {3, 2, 4, true, false, true},  {4, 2, 4, true, false, true},  {5, 2, 4, true, false, false},
    {6, 2, 4, false, true, false}, {4, 3, 4, true, false, false}, {5, 3, 4, true, false, false}, {5, 2, 8, true, false, false},
    {6, 2, 8, true, true, false},  {4, 3, 8, true, false, false}, {6, 3, 8, true, false, false},
};
constexpr int N_WIDE = sizeof(WIDE_FORMS) / sizeof(WIDE_FORMS[0]);
// K steps of 128 in the ring of a form
constexpr int wide_pd(int mt) { return mt <= 4 ? 4 : 3; }

// P.S > 1: K in slices, sums to P.part (launch_wide_sum adds them)
hipError_t launch_wide_mxfp4(const BigParams& P, int form, int wgs, bool dual, hipStream_t stream);
hipError_t launch_wide_bf16(const BigParams& P, int form, int wgs, bool dual, hipStream_t stream);
hipError_t launch_wide_sum(const BigParams& P, int form, int wgs, hipStream_t stream);

} // namespace tppx
