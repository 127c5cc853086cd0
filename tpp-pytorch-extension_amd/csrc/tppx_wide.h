// Many rows, bf16 activations: one wave tile of MT x NT MFMA tiles, W waves side by side (MXFP4 and bf16 weights).
#pragma once
#include "tppx_tiled.h"

namespace tppx {

// ---------------------------------------------------------------------------
// Launches of up to a few workgroups per CU: W waves side by side (one or two to a SIMD), each with a wave tile of MT*16 rows x
// NT*16 channels of its own weights; WIDE_FORMS has the tiles, the launcher takes the one whose workgroups fill a round of the CUs
// with the least padding (333 rows of a 2 x 11008 pair: 232 workgroups of 96 x 384 instead of 1032 of 64 x 128, whose second round
// ran at a third of the chip).  The weights go straight to registers, expanded once per workgroup; only the activations pass
// through LDS, a ring of PD stages of 128 K shared by the waves, and everything is requested PD - 1 steps ahead.  The operands of
// MFMA step j are read and expanded under the MFMAs of step j - 1, one of each behind every MFMA: a wave that is alone on its SIMD
// has nothing else to cover them.
// What bounds it: launches of few rows the intake of a CU (65 GB/s of activations and weights whatever the tile; with weights and
// rows at hand a step of 48 x 128 takes 0.25 us instead of 0.33, its MFMAs 0.16), so the small tiles run four stages (three:
// 4096 x 4096 at 333 rows 15.9 against 14.5 us); the large ones the matrix pipe at the clock the power limit leaves (96 x 384:
// 1.46 us a step with the chip full, 1.13 with 96 workgroups, the MFMAs 0.96 at 2.4 GHz), and about 5 us of launch, first loads
// and epilogue.  Tried: operands of two MFMA steps at a time, nothing; workgroups that start at different K, 5 .. 30 % slower (in
// step they share the lines in L2); five and six stages, nothing.
// Measured at 333 rows, MXFP4, against 64 x 128 workgroups of four waves, three per CU: 4096 x 4096 19.0 -> 14.5 us, 4096 x 11008
// 44 -> 34, 12288 x 4096 38.5 -> 31.5, 22016 x 4096 63 -> 52; 4096 x 4096 at 96 .. 256 rows 17 -> 12.  Over 888 random shapes of
// 65 .. 2048 rows 1.17 in the geometric mean.  All loads are buffer loads (scalar addresses; the compiler counts them beside the
// loads into LDS) and complete in issue order: a step waits until at most those of the PD - 2 younger steps are left.
// ---------------------------------------------------------------------------
template <int MT, int NT, int W, int PD, bool WBF16>
struct WideGeom {
  static constexpr int WGM = MT * 16, STAGE = WGM * 256;
  static constexpr int LB = WBF16 ? 4 * NT : 2 * NT; // weight (and scale) loads of a wave per step
  static constexpr int NA = (MT * 4 + W - 1) / W;    // and its 4-row pieces of A
  static constexpr int L = NA + LB;
  static constexpr int EP_ROWS = MT < 4 ? MT * 16 : 64;
  static constexpr size_t EP = (size_t)W * EP_ROWS * ep_ld(NT) * sizeof(float);
  static constexpr size_t EP_ODD = (NT & 1) ? (size_t)2 * (256 / W) * (W * 16 * NT + 4) * sizeof(float) : 0; // the pair with an odd NT
  static constexpr size_t EPB = EP > EP_ODD ? EP : EP_ODD;
  static constexpr size_t LDS = (size_t)PD * STAGE > EPB ? (size_t)PD * STAGE : EPB;
};

// The gate/up epilogue with the pairs of a workgroup dealt out over its four or eight waves (an odd NT): slot t = wave * NT + nt is the
// gate (t even) or the up tile of channel tile t / 2, so the sums of 256 / W rows at a time meet in LDS, two buffers in turn.
template <int MT, int NT, int W>
__device__ __forceinline__ void wide_epilogue_dual(const TiledParams& pg, const TiledParams& pu, f32x4 (&acc)[MT][NT],
                                                   float* lds, int m_base, int tile_base) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  constexpr int MH = 16 / W, LD = W * 16 * NT + 4, LPR = W * NT; // LPR groups of 8 output channels per row
  static_for<0, (MT + MH - 1) / MH>([&](auto H) {
    constexpr int h = decltype(H)::value, mh = MT - h * MH < MH ? MT - h * MH : MH;
    float* stage = lds + (h & 1) * (MH * 16 * LD);
#pragma unroll
    for (int mt = 0; mt < mh; mt++)
#pragma unroll
      for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          stage[(mt * 16 + (lane >> 4) * 4 + r) * LD + (wave * NT + nt) * 16 + (lane & 15)] = acc[h * MH + mt][nt][r];
    __syncthreads();
    constexpr int ITEMS = mh * 16 * LPR;
#pragma unroll
    for (int it = 0; it < (ITEMS + W * 64 - 1) / (W * 64); it++) {
      const int e = it * (W * 64) + tid;
      const int row = min(e / LPR, mh * 16 - 1), c = e % LPR;
      const int m = m_base + h * (MH * 16) + row, tile = tile_base + (c >> 1);
      const float* src = stage + row * LD + (c >> 1) * 32 + (c & 1) * 8;
      const f32x4 g0 = *reinterpret_cast<const f32x4*>(src), g1 = *reinterpret_cast<const f32x4*>(src + 4);
      const f32x4 u0 = *reinterpret_cast<const f32x4*>(src + 16), u1 = *reinterpret_cast<const f32x4*>(src + 20);
      if (e < ITEMS && tile < pg.tiles && m < pg.M) {
        const int n = tile * 16 + (c & 1) * 8;
        uint32_t out[4];
#pragma unroll
        for (int e2 = 0; e2 < 4; e2++) {
          const float bg0 = pg.bias ? bf16_bits_to_f32(pg.bias[n + 2 * e2]) : 0.0f, bg1 = pg.bias ? bf16_bits_to_f32(pg.bias[n + 2 * e2 + 1]) : 0.0f;
          const float bu0 = pu.bias ? bf16_bits_to_f32(pu.bias[n + 2 * e2]) : 0.0f, bu1 = pu.bias ? bf16_bits_to_f32(pu.bias[n + 2 * e2 + 1]) : 0.0f;
          const uint32_t gate = apply_post_pair<TPPX_POST_SILU>((e2 < 2 ? g0[2 * e2] : g1[2 * e2 - 4]) + bg0, (e2 < 2 ? g0[2 * e2 + 1] : g1[2 * e2 - 3]) + bg1, 0, 1.0f);
          out[e2] = apply_post_pair<TPPX_POST_MUL>((e2 < 2 ? u0[2 * e2] : u1[2 * e2 - 4]) + bu0, (e2 < 2 ? u0[2 * e2 + 1] : u1[2 * e2 - 3]) + bu1, gate, 1.0f);
        }
        *reinterpret_cast<uint4*>(pu.y + (int64_t)m * pu.N + n) = make_uint4(out[0], out[1], out[2], out[3]);
      }
    }
  });
}

template <int MT, int NT, int W, int PD, bool DUAL, bool WBF16, bool SPLIT>
__device__ __forceinline__ void wide_gemm_body(const BigParams& P) {
  using G = WideGeom<MT, NT, W, PD, WBF16>;
  constexpr int WGM = G::WGM, STAGE = G::STAGE, LB = G::LB, NA = G::NA, L = G::L;
  extern __shared__ __align__(16) uint8_t tl_lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int MB = (P.seg[0].M + WGM - 1) / WGM;
  int bm, bn;
  tile_of_block(MB, P.nb0[P.n_seg], bm, bn, P.xm);
  TiledParams p = P.seg[0];
  int nb_first = 0;
  if (!DUAL) {
#pragma unroll
    for (int i = 1; i < TPPX_MAX_SEGS; i++)
      if (i < P.n_seg && bn >= P.nb0[i]) {
        p = P.seg[i];
        nb_first = P.nb0[i];
      }
  }
  bn -= nb_first;
  const int KA = p.K >> 7, k0 = SPLIT ? KA * (int)blockIdx.y / P.S : 0, KT = SPLIT ? KA * ((int)blockIdx.y + 1) / P.S - k0 : KA, last = KT - 1;
  const int m_wg = bm * WGM;
  // DUAL: an even NT has the gate tiles, then the up tiles of the same channels; an odd one deals the workgroup's pairs out
  // gate, up, gate, .. over its waves
  constexpr bool ODD = DUAL && (NT & 1);
  const int tile_base = DUAL ? bn * (W / 2 * NT) + (ODD ? 0 : wave * (NT / 2)) : bn * (W * NT) + wave * NT;

  const auto xr = tl_rsrc(p.x);
  // piece i of this wave: rows (wave & 3)*4 .. + 3 of row tile i (W = 4), i*2 + wave/4 (W = 8; past the last one that again)
  uint32_t aoff[NA];
  auto piece_tile = [&](int i) { return W == 4 ? i : min(i * (W / 4) + (wave >> 2), MT - 1); };
  {
    const int r16 = (wave & 3) * 4 + (lane >> 4);
#pragma unroll
    for (int i = 0; i < NA; i++)
      aoff[i] = (uint32_t)min(m_wg + piece_tile(i) * 16 + r16, p.M - 1) * (uint32_t)p.K * 2u + (uint32_t)((lane & 15) ^ swz16(r16)) * 16u + (uint32_t)k0 * 256u;
  }
  __amdgpu_buffer_rsrc_t wr[NT], swr[NT];
  uint32_t woff[NT], swoff[NT];
#pragma unroll
  for (int nt = 0; nt < NT; nt++) {
    const int slot = wave * NT + nt;
    const bool up = ODD ? (slot & 1) != 0 : DUAL && nt >= NT / 2;
    const int tile = min(ODD ? tile_base + (slot >> 1) : DUAL ? tile_base + nt % (NT / 2 > 0 ? NT / 2 : 1) : tile_base + nt, p.tiles - 1);
    wr[nt] = tl_rsrc(up ? P.seg[1].qw : p.qw);
    swoff[nt] = ((uint32_t)tile * (uint32_t)KA + (uint32_t)k0) * 64u + (uint32_t)lane;
    if constexpr (WBF16) {
      woff[nt] = (((uint32_t)tile * (uint32_t)KA + (uint32_t)k0) * 256u + (uint32_t)lane) * 16u;
    } else {
      woff[nt] = swoff[nt] * 16u;
      swr[nt] = tl_rsrc(up ? P.seg[1].sw : p.sw);
    }
  }
  constexpr int BJ = WBF16 ? 4 : 1;
  i32x4 bw[PD][BJ][NT];
  uint32_t sc[PD][NT];
  auto load = [&](auto I, int s, auto SET) {
    constexpr int i = decltype(I)::value, set = decltype(SET)::value;
    s = min(s, last);
    if constexpr (i < LB) {
      if constexpr (WBF16)
        bw[set][i / NT][i % NT] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(wr[i % NT], woff[i % NT] + (i / NT) * 1024, s * 4096, 0));
      else if constexpr (i < NT)
        bw[set][0][i] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(wr[i], woff[i], s * 1024, 0));
      else
        sc[set][i - NT] = __builtin_amdgcn_raw_buffer_load_b8(swr[i - NT], swoff[i - NT], s * 64, 0);
    } else {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (__attribute__((address_space(3))) void*)(tl_lds + set * STAGE + (piece_tile(i - LB) * 4 + (wave & 3)) * 1024), 16,
                                               aoff[i - LB], s * 256, 0, 0);
    }
  };
  uint32_t rdb[4];
  {
    const int m = lane & 15, g = lane >> 4;
#pragma unroll
    for (int j = 0; j < 4; j++)
      rdb[j] = (uint32_t)((m >> 2) * 1024 + (m & 3) * 256 + ((g * 4 + j) ^ swz16(m)) * 16);
  }
  f32x4 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
      acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  static_for<0, PD - 1>([&](auto S) {
    static_for<0, L>([&](auto I) { load(I, decltype(S)::value, S); });
    __builtin_amdgcn_sched_barrier(0);
  });
  // the operands of MFMA step j are read (and expanded) under the MFMAs of the step before
  bf16x8 a[2][MT], b[2][NT];
#pragma unroll
  for (int i = 0; i < MT; i++)
    a[1][i] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < NT; i++)
    b[1][i] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
  auto mfmas = [&](auto SET) {
    constexpr int q = decltype(SET)::value;
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
      for (int nt = 0; nt < NT; nt++)
        acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[q][mt], b[q][nt], acc[mt][nt], 0, 0, 0);
  };
  // MORE: not one of the last steps, which request nothing any more and wait for all that is left.  (A load into registers
  // whose result is never used would not be there to be counted.)
  auto step = [&](auto MORE, auto SET, int s) {
    constexpr bool more = decltype(MORE)::value;
    constexpr int set = decltype(SET)::value, pset = (set + PD - 1) % PD;
    asm volatile("" : : : "memory");
    constexpr int vm = more ? L * (PD - 2) : 0;
    static_assert(vm < 64, "more loads than the counter holds");
    __builtin_amdgcn_s_waitcnt((vm & 15) | 7 << 4 | vm >> 4 << 14); // step s has landed, the reads of step s - 1 have returned
    asm volatile("s_barrier" : : : "memory");
    const uint8_t* ab = tl_lds + set * STAGE;
    float scale[NT];
    static_for<0, 4>([&](auto J) {
      constexpr int j = decltype(J)::value;
      if constexpr (j == 0 && !WBF16) {
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
          scale[nt] = e8m0_to_f32(sc[set][nt]);
      }
#pragma unroll
      for (int i = 0; i < MT; i++)
        a[j & 1][i] = *reinterpret_cast<const bf16x8*>(ab + i * 4096 + rdb[j]);
      mfmas(std::integral_constant<int, (j + 1) & 1>{});
#pragma unroll
      for (int nt = 0; nt < NT; nt++) {
        if constexpr (WBF16)
          b[j & 1][nt] = __builtin_bit_cast(bf16x8, bw[set][j][nt]);
        else
          b[j & 1][nt] = tl_cvt_fp4x8((uint32_t)bw[set][0][nt][j], scale[nt]);
      }
      if constexpr (more)
        static_for<L * j / 4, L * (j + 1) / 4>([&](auto I) { load(I, s + PD - 1, std::integral_constant<int, pset>{}); });
      // an MFMA, then one of each of the rest: operand reads first, the loads of a later step behind them
      static_for<0, MT * NT>([&](auto I) {
        constexpr int i = decltype(I)::value;
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if constexpr (i < MT)
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        if constexpr (!WBF16)
          __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);
        if constexpr (more && i >= MT && (i - MT) % 2 == 0)
          __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      });
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  int s = 0;
  for (; s + PD <= KT; s += PD)
    static_for<0, PD>([&](auto S) { step(std::true_type{}, S, s + decltype(S)::value); });
  static_for<0, PD - 1>([&](auto S) {
    if (s + decltype(S)::value < KT)
      step(std::false_type{}, S, s + decltype(S)::value);
  });
  mfmas(std::integral_constant<int, 1>{});
  if constexpr (SPLIT) { // (as they lie in the registers: a wave instruction is 1 KiB)
    f32x4* out = reinterpret_cast<f32x4*>(P.part) + (((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * W + wave) * (MT * NT * 64) + lane;
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
      for (int nt = 0; nt < NT; nt++)
        out[(mt * NT + nt) * 64] = acc[mt][nt];
    return;
  }
  __syncthreads(); // (waits for the loads still under way: the ring is free for the epilogue staging)
  if constexpr (ODD)
    wide_epilogue_dual<MT, NT, W>(p, P.seg[1], acc, reinterpret_cast<float*>(tl_lds), m_wg, tile_base);
  else {
    float* stage = reinterpret_cast<float*>(tl_lds) + wave * G::EP_ROWS * ep_ld(NT);
    if constexpr (DUAL)
      big_epilogue_dual<MT, NT>(p, P.seg[1], acc, stage, m_wg, tile_base);
    else
      big_epilogue<MT, NT>(p, acc, stage, m_wg, tile_base);
  }
}


template <int MT, int NT, int W, bool DUAL, bool WBF16, bool SPLIT>
__global__ void __launch_bounds__(W * 64, W / 4)
wide_kernel(const BigParams P) {
  wide_gemm_body<MT, NT, W, wide_pd(MT), DUAL, WBF16, SPLIT>(P);
}

// The other half of a launch split along K: a workgroup of one wave per wave tile adds the S slices' sums, in their order, and
// goes through the same epilogue.  Bound by those bytes and the launch.
template <int MT, int NT, int W, int S>
__global__ void __launch_bounds__(64)
wide_sum_kernel(const BigParams P) {
  __shared__ __align__(16) float stage[(MT < 4 ? MT : 4) * 16 * ep_ld(NT)];
  const int wg = (int)blockIdx.x / W, wave = (int)blockIdx.x % W, lane = threadIdx.x;
  const int MB = (P.seg[0].M + MT * 16 - 1) / (MT * 16), wgs = (int)gridDim.x / W;
  int bm, bn;
  tile_of_block(MB, P.nb0[P.n_seg], bm, bn, P.xm, wg);
  TiledParams p = P.seg[0];
  int nb_first = 0;
#pragma unroll
  for (int i = 1; i < TPPX_MAX_SEGS; i++)
    if (i < P.n_seg && bn >= P.nb0[i]) {
      p = P.seg[i];
      nb_first = P.nb0[i];
    }
  const f32x4* in = reinterpret_cast<const f32x4*>(P.part) + ((int64_t)wg * W + wave) * (MT * NT * 64) + lane;
  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT * NT; i++) {
    f32x4 v[S];
#pragma unroll
    for (int z = 0; z < S; z++)
      v[z] = in[(int64_t)z * wgs * W * (MT * NT * 64) + i * 64];
    acc[i / NT][i % NT] = v[0];
#pragma unroll
    for (int z = 1; z < S; z++)
      acc[i / NT][i % NT] += v[z];
  }
  big_epilogue<MT, NT>(p, acc, stage, bm * MT * 16, (bn - nb_first) * (W * NT) + wave * NT);
}

template <typename Kern>
static hipError_t wide_go(Kern kern, const BigParams& P, dim3 grid, int threads, size_t lds, hipStream_t stream) {
  TPPX_PLAN_ONLY(kern, grid, dim3(threads), lds);
  if (lds > 0)
    if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds); e != hipSuccess)
      return e;
  kern<<<grid, dim3(threads), lds, stream>>>(P);
  return hipGetLastError();
}

// form: index into WIDE_FORMS
template <bool WBF16, int F = 0>
static hipError_t wide_launch(const BigParams& P, int form, int wgs, bool dual, hipStream_t stream) {
  if constexpr (F < N_WIDE) {
    constexpr WideForm f = WIDE_FORMS[F];
    if constexpr (WBF16 ? f.bf16 : f.mxfp4)
      if (form == F) {
        constexpr size_t lds = WideGeom<f.mt, f.nt, f.w, wide_pd(f.mt), WBF16>::LDS;
        if constexpr (f.split && !WBF16)
          if (P.S > 1)
            return dual ? hipErrorInvalidValue
                        : wide_go(wide_kernel<f.mt, f.nt, f.w, false, WBF16, true>, P, dim3(wgs, P.S), f.w * 64, lds, stream);
        return dual ? wide_go(wide_kernel<f.mt, f.nt, f.w, true, WBF16, false>, P, dim3(wgs), f.w * 64, lds, stream)
                    : wide_go(wide_kernel<f.mt, f.nt, f.w, false, WBF16, false>, P, dim3(wgs), f.w * 64, lds, stream);
      }
    return wide_launch<WBF16, F + 1>(P, form, wgs, dual, stream);
  } else {
    return hipErrorInvalidValue;
  }
}

} // namespace tppx
