// Prefill-shape (large M) LDS-tiled MFMA kernels.
//
// Workgroup tile 128 (M) x 128 (N), 4 waves in a 2 x 2 grid, each wave 64 x 64
// = 4 x 4 MFMA tiles of 16 x 16.  Per K step of 128 input channels:
//   A (activations): global -> registers -> LDS, stored in MFMA operand order
//     so that a wave-wide ds_read_b128 is lane-contiguous (conflict free); two
//     LDS buffers, the global loads of step k+1 are in flight while step k is
//     multiplied.
//   B (weights): the native 1 KiB tiles ARE the MFMA operand layout, so every
//     wave loads its four channel tiles straight from global/L2 into registers
//     (one 128-bit load per lane and tile, next step prefetched) - no LDS, no
//     re-layout.  MXFP4 codes are expanded to bf16 in registers with the
//     hardware E8M0-scaled convert (exact) and multiplied with
//     v_mfma_f32_16x16x32_bf16; QINT8 uses v_mfma_i32_16x16x64_i8 with exact
//     int32 sums per K block and an fp32 scale-and-accumulate.
// Workgroup ids are remapped so that the workgroups of one XCD (ids equal
// mod 8) walk consecutive M blocks of the same N block: the weight tiles of
// that N block stay in the XCD's L2.
//
// MFMA operand convention (A = activations, B = weights):
//   lane l supplies row/col (l & 15) and K group (l >> 4);
//   result register r of lane l is D[m = (l >> 4) * 4 + r][n = l & 15].
#include <algorithm>
#include <string.h>
#include <type_traits>

#include "tppx_common.h"
#include "tppx_launch.h"
#include "tppx_tiled.h"

namespace tppx {

template <typename Acc>
__device__ __forceinline__ void tiled_epilogue(const TiledParams& p, Acc& acc, int m_base, int tile_base) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int nt = 0; nt < 4; nt++) {
    const int tile = tile_base + nt;
    if (tile >= p.tiles)
      continue;
    const int n = tile * 16 + (lane & 15);
    const float b = p.bias ? bf16_bits_to_f32(p.bias[n]) : 0.0f;
#pragma unroll
    for (int mt = 0; mt < 4; mt++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int m = m_base + mt * 16 + (lane >> 4) * 4 + r;
        if (m < p.M) {
          const int64_t o = (int64_t)m * p.N + n;
          uint32_t in1 = p.post_in ? p.post_in[o] : 0u;
          uint32_t in2 = p.post_in2 ? p.post_in2[o] : 0u;
          p.y[o] = (uint16_t)apply_post_bits(acc[mt][nt][r] + b, p.post_op, in1, in2, p.post_scale);
        }
      }
  }
}

// ---------------------------------------------------------------------------
// MXFP4, bf16 activations (exact reference numerics, fp32 accumulation over K)
// LDS A layout per buffer: [mt 8][j 4][lane 64] x 16 B  (32 KiB)
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
tiled_mxfp4_kernel(const TiledParams p) {
  extern __shared__ __align__(16) uint8_t tl_lds[];
  bf16x8* As = reinterpret_cast<bf16x8*>(tl_lds); // 2 buffers x 2048 slots
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  const int MB = (p.M + 127) >> 7, NB = (p.tiles + 7) >> 3;
  int bm, bn;
  tile_of_block(MB, NB, bm, bn);
  const int KT = p.K >> 7; // K steps of 128 = native tiles along K
  const int m_wg = bm * 128;
  const int tile_base = bn * 8 + wn * 4;

  const i32x4* wq[4];
  const uint8_t* wsc[4];
#pragma unroll
  for (int nt = 0; nt < 4; nt++) {
    const int64_t t = min(tile_base + nt, p.tiles - 1);
    wq[nt] = reinterpret_cast<const i32x4*>(p.qw) + t * KT * 64 + lane;
    wsc[nt] = reinterpret_cast<const uint8_t*>(p.sw) + t * KT * 64 + lane;
  }
  // A staging: thread handles LDS slots tid + 256*q  ->  (r16, g, j = wave, mt = q)
  const uint16_t* xb = reinterpret_cast<const uint16_t*>(p.x);
  const uint16_t* arow[8];
#pragma unroll
  for (int q = 0; q < 8; q++) {
    const int m = min(m_wg + q * 16 + (tid & 15), p.M - 1);
    arow[q] = xb + (int64_t)m * p.K + ((tid >> 4) & 3) * 32 + wave * 8;
  }

  bf16x8 areg[8];
  i32x4 breg[4];
  uint32_t bsc[4];
  auto load_a = [&](int ks) {
#pragma unroll
    for (int q = 0; q < 8; q++)
      areg[q] = *reinterpret_cast<const bf16x8*>(arow[q] + ks * 128);
  };
  auto load_b = [&](int ks) {
#pragma unroll
    for (int nt = 0; nt < 4; nt++) {
      breg[nt] = wq[nt][(int64_t)ks * 64];
      bsc[nt] = wsc[nt][(int64_t)ks * 64];
    }
  };
  auto store_a = [&](int buf) {
#pragma unroll
    for (int q = 0; q < 8; q++)
      As[buf * 2048 + q * 256 + tid] = areg[q];
  };

  f32x4 acc[4][4];
#pragma unroll
  for (int mt = 0; mt < 4; mt++)
#pragma unroll
    for (int nt = 0; nt < 4; nt++)
      acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};

  load_a(0);
  load_b(0);
  store_a(0);
  __syncthreads();
  for (int ks = 0; ks < KT; ks++) {
    const int buf = ks & 1;
    i32x4 bcur[4];
    float sc[4];
#pragma unroll
    for (int nt = 0; nt < 4; nt++) {
      bcur[nt] = breg[nt];
      sc[nt] = e8m0_to_f32(bsc[nt]);
    }
    if (ks + 1 < KT) {
      load_a(ks + 1);
      load_b(ks + 1);
    }
    const bf16x8* Ab = As + buf * 2048 + (wm * 4) * 256 + lane;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      bf16x8 a[4], b[4];
#pragma unroll
      for (int mt = 0; mt < 4; mt++)
        a[mt] = Ab[mt * 256 + j * 64];
#pragma unroll
      for (int nt = 0; nt < 4; nt++)
        b[nt] = tl_cvt_fp4x8((uint32_t)bcur[nt][j], sc[nt]);
#pragma unroll
      for (int mt = 0; mt < 4; mt++)
#pragma unroll
        for (int nt = 0; nt < 4; nt++)
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[mt], b[nt], acc[mt][nt], 0, 0, 0);
    }
    if (ks + 1 < KT)
      store_a(buf ^ 1);
    __syncthreads();
  }
  tiled_epilogue(p, acc, m_wg + wm * 64, tile_base);
}

// ---------------------------------------------------------------------------
// Unquantized bf16 weights at prefill shapes (the prompt pass of a model whose
// first-token weights stay bf16): the kernel above without the expansion.  The
// native bf16 tiles [N/16][K/128][4 j][64 lanes][16 B] hold the MFMA operands
// themselves, 4 KiB per (channel tile, K step) -- eight times the bytes of the
// packed codes -- so B runs as a ring of the four steps j of a K step: the
// operand of (ks, j) is requested right behind the MFMAs that consumed
// (ks - 1, j), a whole K step ahead, and no second register set is needed.
// All loads are ordinary register loads, so the compiler's partial waits hold.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
tiled_bf16_kernel(const TiledParams p) {
  extern __shared__ __align__(16) uint8_t tl_lds[];
  bf16x8* As = reinterpret_cast<bf16x8*>(tl_lds); // 2 buffers x 2048 slots
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  const int MB = (p.M + 127) >> 7, NB = (p.tiles + 7) >> 3;
  int bm, bn;
  tile_of_block(MB, NB, bm, bn);
  const int KT = p.K >> 7;
  const int m_wg = bm * 128;
  const int tile_base = bn * 8 + wn * 4;

  const i32x4* wq[4];
#pragma unroll
  for (int nt = 0; nt < 4; nt++) {
    const int64_t t = min(tile_base + nt, p.tiles - 1);
    wq[nt] = reinterpret_cast<const i32x4*>(p.qw) + t * KT * 256 + lane;
  }
  const uint16_t* xb = reinterpret_cast<const uint16_t*>(p.x);
  const uint16_t* arow[8];
#pragma unroll
  for (int q = 0; q < 8; q++) {
    const int m = min(m_wg + q * 16 + (tid & 15), p.M - 1);
    arow[q] = xb + (int64_t)m * p.K + ((tid >> 4) & 3) * 32 + wave * 8;
  }
  bf16x8 areg[8];
  i32x4 bring[4][4]; // [j][nt]
  auto load_a = [&](int ks) {
#pragma unroll
    for (int q = 0; q < 8; q++)
      areg[q] = *reinterpret_cast<const bf16x8*>(arow[q] + ks * 128);
  };
  auto load_b = [&](int ks, int j) {
#pragma unroll
    for (int nt = 0; nt < 4; nt++)
      bring[j][nt] = wq[nt][(int64_t)ks * 256 + j * 64];
  };
  auto store_a = [&](int buf) {
#pragma unroll
    for (int q = 0; q < 8; q++)
      As[buf * 2048 + q * 256 + tid] = areg[q];
  };

  f32x4 acc[4][4];
#pragma unroll
  for (int mt = 0; mt < 4; mt++)
#pragma unroll
    for (int nt = 0; nt < 4; nt++)
      acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};

  load_a(0);
#pragma unroll
  for (int j = 0; j < 4; j++)
    load_b(0, j);
  store_a(0);
  __syncthreads();
  for (int ks = 0; ks < KT; ks++) {
    const int buf = ks & 1;
    const bool more = ks + 1 < KT;
    if (more)
      load_a(ks + 1);
    const bf16x8* Ab = As + buf * 2048 + (wm * 4) * 256 + lane;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      bf16x8 a[4];
#pragma unroll
      for (int mt = 0; mt < 4; mt++)
        a[mt] = Ab[mt * 256 + j * 64];
#pragma unroll
      for (int mt = 0; mt < 4; mt++)
#pragma unroll
        for (int nt = 0; nt < 4; nt++)
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[mt], __builtin_bit_cast(bf16x8, bring[j][nt]), acc[mt][nt], 0, 0, 0);
      if (more)
        load_b(ks + 1, j);
    }
    if (more)
      store_a(buf ^ 1);
    __syncthreads();
  }
  tiled_epilogue(p, acc, m_wg + wm * 64, tile_base);
}

// ---------------------------------------------------------------------------
// QINT8 (W8A8): activations pre-quantised (int8 [M][K], f32 [M][K/qbs]).
// K step = 128 = two native tiles; LDS A layout per buffer:
// [mt 8][t 2][lane 64] x 16 B (16 KiB) + the activation scales of the step's
// K block for the 128 rows.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256, 2) // two workgroups per CU: without the bound the compiler spreads into 327 registers, one wave per SIMD
tiled_qint8_kernel(const TiledParams p) {
  extern __shared__ __align__(16) uint8_t tl_lds[];
  i32x4* As = reinterpret_cast<i32x4*>(tl_lds);                 // 2 x 1024 slots
  float* sa_s = reinterpret_cast<float*>(tl_lds + 2 * 1024 * 16); // 2 x 128
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  const int MB = (p.M + 127) >> 7, NB = (p.tiles + 7) >> 3;
  int bm, bn;
  tile_of_block(MB, NB, bm, bn);
  const int KS = p.K >> 7;        // K steps of 128
  const int KT = p.K >> 6;        // native tiles along K
  const int SPB = p.qbs >> 7;     // steps per K block (qbs is a multiple of 128 here)
  const int NBK = p.K / p.qbs;
  const int m_wg = bm * 128;
  const int tile_base = bn * 8 + wn * 4;

  const i32x4* wq[4];
  const float* wsc[4];
#pragma unroll
  for (int nt = 0; nt < 4; nt++) {
    const int64_t t = min(tile_base + nt, p.tiles - 1);
    wq[nt] = reinterpret_cast<const i32x4*>(p.qw) + t * KT * 64 + lane;
    wsc[nt] = reinterpret_cast<const float*>(p.sw) + t * NBK * 16 + (lane & 15);
  }
  // A staging: slots tid + 256*q -> (r16, g, t = wave & 1, mt = 2*q + (wave >> 1))
  const int8_t* xq = reinterpret_cast<const int8_t*>(p.xq);
  const int8_t* arow[4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int mt = q * 2 + (wave >> 1);
    const int m = min(m_wg + mt * 16 + (tid & 15), p.M - 1);
    arow[q] = xq + (int64_t)m * p.K + (wave & 1) * 64 + ((tid >> 4) & 3) * 16;
  }
  const int sa_row = min(m_wg + (tid & 127), p.M - 1);

  i32x4 areg[4], breg[2][4];
  float sareg = 0.f;
  auto load_a = [&](int ks) {
#pragma unroll
    for (int q = 0; q < 4; q++)
      areg[q] = *reinterpret_cast<const i32x4*>(arow[q] + ks * 128);
    if (ks % SPB == 0 && tid < 128)
      sareg = p.sa[(int64_t)sa_row * NBK + ks / SPB];
  };
  auto load_b = [&](int ks) {
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int nt = 0; nt < 4; nt++)
        breg[t][nt] = wq[nt][(int64_t)(ks * 2 + t) * 64];
  };
  auto store_a = [&](int ks, int buf) {
#pragma unroll
    for (int q = 0; q < 4; q++)
      As[buf * 1024 + q * 256 + tid] = areg[q];
    if (ks % SPB == 0 && tid < 128)
      sa_s[((ks / SPB) & 1) * 128 + tid] = sareg;
  };

  f32x4 facc[4][4];
  i32x4 iacc[4][4];
#pragma unroll
  for (int mt = 0; mt < 4; mt++)
#pragma unroll
    for (int nt = 0; nt < 4; nt++) {
      facc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
      iacc[mt][nt] = i32x4{0, 0, 0, 0};
    }

  load_a(0);
  load_b(0);
  store_a(0, 0);
  __syncthreads();
  for (int ks = 0; ks < KS; ks++) {
    const int buf = ks & 1;
    i32x4 bcur[2][4];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int nt = 0; nt < 4; nt++)
        bcur[t][nt] = breg[t][nt];
    if (ks + 1 < KS) {
      load_a(ks + 1);
      load_b(ks + 1);
    }
    // slot = (mt*2 + t)*64 + lane with mt = wm*4 + i
    const i32x4* Ab = As + buf * 1024 + (wm * 4) * 128 + lane;
#pragma unroll
    for (int t = 0; t < 2; t++) {
      i32x4 a[4];
#pragma unroll
      for (int mt = 0; mt < 4; mt++)
        a[mt] = Ab[mt * 128 + t * 64];
#pragma unroll
      for (int mt = 0; mt < 4; mt++)
#pragma unroll
        for (int nt = 0; nt < 4; nt++)
          iacc[mt][nt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[mt], bcur[t][nt], iacc[mt][nt], 0, 0, 0);
    }
    if ((ks + 1) % SPB == 0) { // K block complete: scale and fold into fp32
      const int b = ks / SPB;
      const float* sab = sa_s + (b & 1) * 128 + wm * 64 + (lane >> 4) * 4;
      float swv[4];
#pragma unroll
      for (int nt = 0; nt < 4; nt++)
        swv[nt] = wsc[nt][b * 16];
#pragma unroll
      for (int mt = 0; mt < 4; mt++) {
        const f32x4 sav = *reinterpret_cast<const f32x4*>(sab + mt * 16);
#pragma unroll
        for (int nt = 0; nt < 4; nt++)
#pragma unroll
          for (int r = 0; r < 4; r++) {
            facc[mt][nt][r] = fmaf((float)iacc[mt][nt][r], sav[r] * swv[nt], facc[mt][nt][r]);
            iacc[mt][nt][r] = 0;
          }
      }
    }
    if (ks + 1 < KS)
      store_a(ks + 1, buf ^ 1);
    __syncthreads();
  }
  tiled_epilogue(p, facc, m_wg + wm * 64, tile_base);
}

// ---------------------------------------------------------------------------
// Large-M MXFP4 kernel: workgroup tile 256 (M) x 256 (N), 8 waves in a 2 x 4
// grid (two per SIMD), each wave 128 x 64 = 8 x 4 MFMA tiles (128 accumulator
// registers).  Every expanded weight operand feeds 8 MFMAs, every activation
// operand read from LDS feeds 4 and is requested two MFMA groups ahead.
//   A: 4 rows x 256 B per wave instruction go from global memory straight
//      into LDS (global_load_lds, no staging registers), a whole K step ahead,
//      two buffers of 64 KiB.  The LDS image of such a load is lane-linear, so
//      the bank swizzle is applied on the source side: the lane at position c
//      of row m fetches chunk c ^ (m & 15), and the operand reads of a K group
//      fall on 16 different bank groups.
//   B: native tiles straight from global/L2, fetched half a K step ahead.
// LDS byte address of chunk ck of row m of row tile mt:
//   mt*4096 + (m>>2)*1024 + (m&3)*256 + ((ck ^ m) & 15)*16.
// ---------------------------------------------------------------------------
// LDS operand reads issued by hand, so that they can be kept several MFMA
// groups ahead of their use: the compiler does not track them, the waits are
// explicit (LDS operations complete in issue order, so "at most N younger
// operations outstanding" is enough) and are tied to the destination
// registers so that nothing using them can move above the wait.
template <int OFF>
__device__ __forceinline__ void lds_read_b128_async(i32x4& dst, uint32_t byte_addr) {
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(byte_addr), "n"(OFF));
}
template <int N>
__device__ __forceinline__ void lds_wait_keep(i32x4& r) {
  asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(r) : "n"(N));
}

// MT = 16-row tiles per wave along M (8).
// DUAL: the gate/up pair (seg[0] = gate, seg[1] = up, equal shapes).  A workgroup owns 128 output channels and
// computes their gate AND up sums (wave tile = 2 gate tiles + the 2 up tiles of the same channels); the epilogue
// writes silu(gate) * up once.  Channel blocks are 128 wide then.
// WM x WN waves, each with a wave tile of MT*16 rows x 64 channels:
//   2 x 4  workgroup tile 256 x 256, one workgroup per CU
//   1 x 4  128 x 256, 4 waves, TWO workgroups per CU: half-size workgroups for shapes whose last round of 256-row
//          workgroups would be mostly empty
//   1 x 8  128 x 512, one workgroup per CU: the same 65536 sums per CU as 2 x 4, but half the activation bytes per
//          K step (128 rows) and every weight tile fetched by ONE wave instead of by the two of a wave column -- half
//          the bytes moved from L2 into the CU per MFMA
// WBF16: unquantized bf16 weights in their native tiles ([N/16][K/128][4 j][64 lanes][16 B], the MFMA operands
// themselves) instead of packed codes + scales: 16 bytes per lane, tile and MFMA step, so they run as a ring of the
// four steps j of a K step -- (ks + 1, j) is requested right behind the last MFMA group of (ks, j), a whole K step
// ahead -- and no second register set is needed.  These loads are issued and waited for by hand (they complete in
// issue order, so "at most N younger loads outstanding" is the wait): with loads into LDS pending the compiler
// answers the first use of any loaded register, and the fence of __syncthreads(), with a wait for ALL loads.
template <int MT, bool DUAL, int WM, int WN, bool WBF16>
__device__ __forceinline__ void big_gemm_body(const BigParams& P) {
  constexpr int WGM = MT * 16 * WM; // rows per workgroup
  constexpr int NBLK = MT * 4 / WN; // blocks of 4 rows x 256 B of the A tile that a wave fetches per K step
  static_assert(NBLK % 4 == 0, "the swizzle below takes a wave's first block to be a multiple of 4");
  constexpr int ABUF = WGM * 256;  // bytes of one A buffer (rows x 128 K bf16)
  extern __shared__ __align__(16) uint8_t tl_lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6); // uniform: keeps LDS bases and block indices scalar
  const int wm = wave % WM, wn = wave / WM;
  const int MB = (P.seg[0].M + WGM - 1) / WGM;
  int bm, bn;
  tile_of_block(MB, P.nb0[P.n_seg], bm, bn, P.xm);
  // pick this block's GEMM with uniform selects (everything stays in scalar registers)
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
  const int KT = p.K >> 7;
  const int m_wg = bm * WGM;
  const int tile_base = DUAL ? bn * (WN * 2) + wn * 2 : bn * (WN * 4) + wn * 4;

  // Every global address below is a uniform base pointer plus a 32-bit byte
  // offset per lane (the launcher checks that the operands are smaller than
  // 4 GiB): one offset register instead of a 64-bit pointer pair per stream.
  const char* qwb = reinterpret_cast<const char*>(p.qw);
  const char* swb = reinterpret_cast<const char*>(p.sw);
  // DUAL: tiles 2 and 3 of the wave are the up projection's tiles of the channels of tiles 0 and 1
  const char* qwb2 = DUAL ? reinterpret_cast<const char*>(P.seg[1].qw) : qwb;
  const char* swb2 = DUAL ? reinterpret_cast<const char*>(P.seg[1].sw) : swb;
  uint32_t woff[4]; // slot index of this lane in tile nt at K step 0
#pragma unroll
  for (int nt = 0; nt < 4; nt++)
    woff[nt] = (uint32_t)(min(tile_base + (DUAL ? (nt & 1) : nt), p.tiles - 1) * KT * 64 + lane);

  // A tile (256 rows x 128 K, 64 KiB): 64 blocks of 4 rows x 256 B go from
  // global memory straight into LDS, one wave instruction per block (lane =
  // row r of the block, 16-byte chunk).  The LDS image of an instruction is
  // lane-linear, so the swizzle is applied on the global side: the lane at
  // position ch of row m fetches chunk ch ^ swz16(m & 15); operand reads
  // then fall on all the banks (see swz16).
  //   LDS byte address of chunk ck of row m of row tile mt:
  //     mt*4096 + (m>>2)*1024 + (m&3)*256 + (ck ^ swz16(m))*16
  const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>(tl_lds); // LDS byte address of the buffers
  uint32_t rdb[4]; // byte offset of this lane's operand for step j (+ mt*4096): chunk ck = g*4 + j
  {
    const int m = lane & 15, g = lane >> 4;
#pragma unroll
    for (int j = 0; j < 4; j++)
      rdb[j] = (uint32_t)((m >> 2) * 1024 + (m & 3) * 256 + ((g * 4 + j) ^ swz16(m)) * 16);
  }
  const char* xbase = reinterpret_cast<const char*>(p.x);
  // this wave's NBLK blocks: blk = wave*NBLK + i -> rows blk*4 + (lane>>4)
  const int rin = (lane >> 4);          // row inside the block
  const int ch = lane & 15;             // chunk position of this lane inside the row
  // source byte offset of block i at K step ks:
  //   row(i) * K * 2 + (ch ^ swz16(m16(i))) * 16 + ks * 256, row(i) = m_wg + (wave*8 + i)*4 + rin,
  //   m16(i) = (i & 3)*4 + rin (wave*8 is a multiple of 4)
  const bool full = m_wg + WGM <= p.M; // uniform
  const uint32_t xrow0 = (uint32_t)((m_wg + wave * (NBLK * 4) + rin) * p.K) * 2u;
  const uint32_t blk_stride = (uint32_t)(4 * p.K) * 2u; // uniform
  auto load_a_one = [&](auto I, int ks, int buf) {
    constexpr int i = decltype(I)::value;
    const uint32_t sw = (uint32_t)(ch ^ swz16((i & 3) * 4 + rin)) * 16u;
    uint32_t off;
    if (full) {
      off = xrow0 + (uint32_t)i * blk_stride + sw + (uint32_t)ks * 256u;
    } else { // past the end: re-read the last row (never stored)
      const int row = min(m_wg + (wave * NBLK + i) * 4 + rin, p.M - 1);
      off = (uint32_t)(row * p.K) * 2u + sw + (uint32_t)ks * 256u;
    }
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(xbase + (size_t)off),
                                     (__attribute__((address_space(3))) void*)(tl_lds + buf * ABUF + (wave * NBLK + i) * 1024),
                                     16, 0, 0);
  };
  auto load_a = [&](int ks, int buf) { static_for<0, NBLK>([&](auto I) { load_a_one(I, ks, buf); }); };
  // B of one K step: 4 tiles x 4 dwords (one per step j) and the scale factors
  uint32_t bc[4][4];
  float sc[4];
  i32x4 bnext[4];
  uint32_t snext[4];
  auto load_b = [&](int ks) {
#pragma unroll
    for (int nt = 0; nt < 4; nt++) {
      const uint32_t slot = woff[nt] + (uint32_t)ks * 64u;
      bnext[nt] = *reinterpret_cast<const i32x4*>((nt < 2 ? qwb : qwb2) + (size_t)(slot * 16u));
      snext[nt] = *reinterpret_cast<const uint8_t*>((nt < 2 ? swb : swb2) + (size_t)slot);
    }
  };
  auto take_b = [&]() {
#pragma unroll
    for (int nt = 0; nt < 4; nt++) {
#pragma unroll
      for (int j = 0; j < 4; j++)
        bc[nt][j] = (uint32_t)bnext[nt][j];
      sc[nt] = e8m0_to_f32(snext[nt]);
    }
  };
  i32x4 bw[4][4]; // WBF16: [j][nt]
  auto load_bw = [&](int ks, int j) {
#pragma unroll
    for (int nt = 0; nt < 4; nt++) {
      // native bf16 tiles: slot ((tile * KT + ks) * 4 + j) * 64 + lane, 16 bytes each
      const char* src = (nt < 2 ? qwb : qwb2) + (size_t)(((woff[nt] - (uint32_t)lane) * 4u + (uint32_t)(ks * 4 + j) * 64u + (uint32_t)lane) * 16u);
      asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(bw[j][nt]) : "v"(src));
    }
  };

  f32x4 acc[MT][4];
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int nt = 0; nt < 4; nt++)
      acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};

  load_a(0, 0);
  if constexpr (WBF16) {
#pragma unroll
    for (int j = 0; j < 4; j++)
      load_bw(0, j);
  } else {
    load_b(0);
  }
  __syncthreads();
  // One K step.  MORE: the next step's A tile is requested during this one, one block behind each of the first NBLK
  // MFMA groups (issued in one burst, a wave stands at its load instructions while the memory pipeline's queue
  // drains, and its MFMAs wait with it); it lands in the other buffer.
  auto step = [&](auto MORE, int ks) {
    constexpr bool more = decltype(MORE)::value;
    const int buf = ks & 1;
    if constexpr (!WBF16)
      take_b();
    // 4*MT operand reads per K step (q = j*MT + mt), kept RD ahead of the MFMAs
    // that consume them so the LDS latency is covered by 4*RD MFMAs
    const uint32_t abase = lds0 + (uint32_t)(buf * ABUF + wm * MT * 4096);
    constexpr int RD = 3; // operand reads in flight ahead of the MFMAs
    constexpr int NQ = 4 * MT;
    i32x4 ar[RD + 1];
    bf16x8 b[4];
    static_for<0, RD>([&](auto I) {
      constexpr int i = decltype(I)::value;
      lds_read_b128_async<(i % MT) * 4096>(ar[i], abase + rdb[i / MT]);
    });
    static_for<0, NQ>([&](auto Q) {
      constexpr int q = decltype(Q)::value;
      constexpr int j = q / MT, mt = q % MT;
      if constexpr (mt == 0 && WBF16) {
        // Step j's weights were requested a K step ago, behind group j * MT + MT - 1.  Behind them then: the later
        // steps' (4 each) and the blocks of A that K step still had to request (block d goes out behind group d);
        // in this K step, when it requests anything: the blocks of A behind the groups before this one and the
        // next K step's weights of the steps before j.
        constexpr int qj = j * MT + MT - 1;
        constexpr int younger = (3 - j) * 4 + (NBLK - 1 - qj > 0 ? NBLK - 1 - qj : 0) +
                                (more ? (j * MT < NBLK ? j * MT : NBLK) + j * 4 : 0);
        asm volatile("s_waitcnt vmcnt(%4)" : "+v"(bw[j][0]), "+v"(bw[j][1]), "+v"(bw[j][2]), "+v"(bw[j][3]) : "n"(younger));
#pragma unroll
        for (int nt = 0; nt < 4; nt++)
          b[nt] = __builtin_bit_cast(bf16x8, bw[j][nt]);
      }
      if constexpr (mt == 0 && !WBF16) {
#pragma unroll
        for (int nt = 0; nt < 4; nt++)
          b[nt] = tl_cvt_fp4x8(bc[nt][j], sc[nt]);
      }
      if constexpr (q + RD < NQ) {
        lds_read_b128_async<((q + RD) % MT) * 4096>(ar[(q + RD) % (RD + 1)], abase + rdb[(q + RD) / MT]);
        lds_wait_keep<RD>(ar[q % (RD + 1)]);
      } else {
        lds_wait_keep<NQ - 1 - q>(ar[q % (RD + 1)]);
      }
      const bf16x8 a = __builtin_bit_cast(bf16x8, ar[q % (RD + 1)]);
#pragma unroll
      for (int nt = 0; nt < 4; nt++)
        acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[nt], acc[mt][nt], 0, 0, 0);
      if constexpr (more && q < NBLK)
        load_a_one(std::integral_constant<int, q>{}, ks + 1, buf ^ 1);
      if constexpr (WBF16) {
        if constexpr (more && mt == MT - 1)
          load_bw(ks + 1, j); // the MFMAs that read step j's registers have been issued
      } else {
        if constexpr (more && q == NQ / 2 - 1)
          load_b(ks + 1); // dwords of steps 0 and 1 of the current B are dead by now
      }
    });
    if constexpr (WBF16 && more) {
      // this wave's loads into LDS have landed -- behind the last of them went out the next K step's weights of
      // every step j whose last group is not before that block's -- then everybody's; a bare barrier, see above
      constexpr int after = 4 * ((MT - 1 >= NBLK - 1) + (2 * MT - 1 >= NBLK - 1) + (3 * MT - 1 >= NBLK - 1) + (4 * MT - 1 >= NBLK - 1));
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"(after) : "memory");
    } else {
      __syncthreads(); // waits for this wave's direct-to-LDS loads, then for everybody's
    }
  };
  for (int ks = 0; ks + 1 < KT; ks++)
    step(std::true_type{}, ks);
  step(std::false_type{}, KT - 1);
  // every wave has left the main loop (barrier above): LDS is free for the epilogue staging
  if (DUAL)
    big_epilogue_dual<MT>(p, P.seg[1], acc, reinterpret_cast<float*>(tl_lds) + wave * 64 * EP_LD, m_wg + wm * (MT * 16),
                          tile_base);
  else
    big_epilogue<MT>(p, acc, reinterpret_cast<float*>(tl_lds) + wave * 64 * EP_LD, m_wg + wm * (MT * 16), tile_base);
}

// ---------------------------------------------------------------------------
// The same sums on bf16 weights, for launches of a few workgroups per CU and those of 128 x 256 that stand one to a CU:
// W waves side by side, each with a wave tile of MT*16 rows x 32 channels, K steps of 128, PD steps in flight.
// What bounds such a launch is what a step of one workgroup takes with nothing beside it: its intake and the latency of the
// step's loads.  So the weights of a wave are its own: they go straight to its registers, only the activations go through LDS,
// and everything is requested PD - 1 steps ahead.
// All loads are buffer loads: scalar addresses, and the compiler counts them exactly beside the loads into LDS (flat-
// addressed loads into LDS make it wait for everything).  Loads of the two kinds complete in issue order, so a step waits
// until at most those of the PD - 2 younger steps are left; one barrier per step.
// Measured at 333 rows: 4096 x 4096 with residual 25.4 -> 19.3 us, 4096 x 11008 76.9 -> 58.2; 64 x 256 at 1000 rows 4096 x 11008
// 152 -> 103; 128 x 256 at 2048 rows 167 -> 144.
// ---------------------------------------------------------------------------
template <int MT, int W, int PD>
struct SideGeom {
  static constexpr int WGM = MT * 16, STAGE = WGM * 256;
  static constexpr int NA = MT * 4 / W;             // 4-row pieces of A a wave fetches per step
  static constexpr int LB = 8;                      // weight loads of a wave per step
  static constexpr int L = NA + LB;
  static constexpr size_t EP = (size_t)W * (MT < 4 ? MT * 16 : 64) * ep_ld(2) * sizeof(float);
  static constexpr size_t LDS = (size_t)PD * STAGE > EP ? (size_t)PD * STAGE : EP;
};

template <int MT, int W, int PD, bool DUAL, bool SPLIT = false>
__device__ __forceinline__ void side_gemm_body(const BigParams& P) {
  using G = SideGeom<MT, W, PD>;
  constexpr int WGM = G::WGM, STAGE = G::STAGE, NA = G::NA, LB = G::LB, L = G::L;
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
  // K steps k0 .. k0 + KT - 1 of KA
  const int KA = p.K >> 7, k0 = SPLIT ? KA * (int)blockIdx.y / P.S : 0, KT = SPLIT ? KA * ((int)blockIdx.y + 1) / P.S - k0 : KA, last = KT - 1;
  const int m_wg = bm * WGM;
  const int tile_base = DUAL ? bn * W + wave : bn * (W * 2) + wave * 2; // DUAL: gate and up tile of the same 16 channels

  const auto xr = tl_rsrc(p.x);
  uint32_t aoff[NA];
#pragma unroll
  for (int i = 0; i < NA; i++) {
    const int blk = wave * NA + i, r16 = (blk & 3) * 4 + (lane >> 4);
    aoff[i] = (uint32_t)min(m_wg + blk * 4 + (lane >> 4), p.M - 1) * (uint32_t)p.K * 2u + (uint32_t)((lane & 15) ^ swz16(r16)) * 16u + (uint32_t)k0 * 256u;
  }
  __amdgpu_buffer_rsrc_t wr[2];
  uint32_t woff[2];
#pragma unroll
  for (int nt = 0; nt < 2; nt++) {
    const int tile = min(DUAL ? tile_base : tile_base + nt, p.tiles - 1);
    wr[nt] = tl_rsrc(DUAL && nt ? P.seg[1].qw : p.qw);
    woff[nt] = (((uint32_t)tile * (uint32_t)KA + (uint32_t)k0) * 256u + (uint32_t)lane) * 16u;
  }
  i32x4 bw[PD][4][2]; // weights of PD steps: the operands of the four MFMA steps
  // load i of step s (clamped to the last one: what is read past it is never used)
  auto load = [&](auto I, int s, auto SET) {
    constexpr int i = decltype(I)::value, set = decltype(SET)::value;
    s = min(s, last);
    if constexpr (i < LB) {
      bw[set][i >> 1][i & 1] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(wr[i & 1], woff[i & 1] + (i >> 1) * 1024, s * 4096, 0));
    } else {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (__attribute__((address_space(3))) void*)(tl_lds + set * STAGE + (wave * NA + i - LB) * 1024), 16,
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
  f32x4 acc[MT][2];
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
    acc[mt][0] = acc[mt][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  static_for<0, PD - 1>([&](auto S) {
    static_for<0, L>([&](auto I) { load(I, decltype(S)::value, S); });
    __builtin_amdgcn_sched_barrier(0); // (in this order: the waits count the loads behind those they wait for)
  });
  // Units of MU row tiles and one MFMA step j; the operands of unit q are read under the MFMAs
  // of unit q - 1, so the last unit of a step runs in the next one, under its first operand reads.
  constexpr int MU = 4, UJ = MT / MU, NQ = 4 * UJ;
  bf16x8 a[2][MU], b[2][2];
#pragma unroll
  for (int i = 0; i < MU; i++)
    a[1][i] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
  b[1][0] = b[1][1] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
  auto unit = [&](auto Q) {
    constexpr int q = decltype(Q)::value, j = q / UJ, mu = q % UJ;
#pragma unroll
    for (int i = 0; i < MU; i++)
#pragma unroll
      for (int nt = 0; nt < 2; nt++)
        acc[mu * MU + i][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[q & 1][i], b[j & 1][nt], acc[mu * MU + i][nt], 0, 0, 0);
  };
  // MORE: not one of the last steps, which request nothing any more and wait for all that is left.  (A load into registers
  // whose result is never used would not be there to be counted.)
  auto step = [&](auto MORE, auto SET, int s) {
    constexpr bool more = decltype(MORE)::value;
    constexpr int set = decltype(SET)::value, pset = (set + PD - 1) % PD;
    asm volatile("" : : : "memory");
    constexpr int vm = more ? L * (PD - 2) : 0;
    __builtin_amdgcn_s_waitcnt((vm & 15) | 7 << 4 | vm >> 4 << 14); // step s has landed, the reads of step s - 1 have returned
    asm volatile("s_barrier" : : : "memory");
    const uint8_t* ab = tl_lds + set * STAGE;
    static_for<0, NQ>([&](auto Q) {
      constexpr int q = decltype(Q)::value, j = q / UJ, mu = q % UJ;
#pragma unroll
      for (int i = 0; i < MU; i++)
        a[q & 1][i] = *reinterpret_cast<const bf16x8*>(ab + (mu * MU + i) * 4096 + rdb[j]);
      __builtin_amdgcn_sched_barrier(0);
      unit(std::integral_constant<int, (q + NQ - 1) % NQ>{});
      if constexpr (mu == 0) {
#pragma unroll
        for (int nt = 0; nt < 2; nt++)
          b[j & 1][nt] = __builtin_bit_cast(bf16x8, bw[set][j][nt]);
      }
      __builtin_amdgcn_sched_barrier(0);
      // the loads PD - 1 steps ahead, a few behind each unit (in one burst, a wave stands at its load instructions while
      // the memory pipeline's queue drains)
      if constexpr (more) {
        static_for<L * q / NQ, L * (q + 1) / NQ>([&](auto I) { load(I, s + PD - 1, std::integral_constant<int, pset>{}); });
        __builtin_amdgcn_sched_barrier(0);
      }
    });
  };
  int s = 0;
  for (; s + PD <= KT; s += PD)
    static_for<0, PD>([&](auto S) { step(std::true_type{}, S, s + decltype(S)::value); });
  static_for<0, PD - 1>([&](auto S) {
    if (s + decltype(S)::value < KT)
      step(std::false_type{}, S, s + decltype(S)::value);
  });
  unit(std::integral_constant<int, NQ - 1>{});
  if constexpr (SPLIT) { // (as they lie in the registers: a wave instruction is 1 KiB)
    f32x4* out = reinterpret_cast<f32x4*>(P.part) + (((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * W + wave) * (MT * 2 * 64) + lane;
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
      out[(mt * 2) * 64] = acc[mt][0];
      out[(mt * 2 + 1) * 64] = acc[mt][1];
    }
    return;
  }
  __syncthreads(); // (waits for the loads still under way: the ring is free for the epilogue staging)
  float* stage = reinterpret_cast<float*>(tl_lds) + wave * (MT < 4 ? MT * 16 : 64) * ep_ld(2);
  if (DUAL)
    big_epilogue_dual<MT, 2>(p, P.seg[1], acc, stage, m_wg, tile_base);
  else
    big_epilogue<MT, 2>(p, acc, stage, m_wg, tile_base);
}

// The other half of a launch split along K: a workgroup of one wave per wave tile adds the S slices' sums, in their order, and
// goes through the same epilogue.  Bound by those bytes, S * 32 KiB per 64 x 128 outputs, and the launch.
template <int MT, int W, int S>
__global__ void __launch_bounds__(64)
side_sum_kernel(const BigParams P) {
  __shared__ __align__(16) float stage[MT * 16 * ep_ld(2)];
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
  const f32x4* in = reinterpret_cast<const f32x4*>(P.part) + ((int64_t)wg * W + wave) * (MT * 2 * 64) + lane;
  f32x4 acc[MT][2];
#pragma unroll
  for (int i = 0; i < MT * 2; i++) {
    f32x4 v[S];
#pragma unroll
    for (int z = 0; z < S; z++)
      v[z] = in[(int64_t)z * wgs * W * (MT * 2 * 64) + i * 64];
    acc[i >> 1][i & 1] = v[0];
#pragma unroll
    for (int z = 1; z < S; z++)
      acc[i >> 1][i & 1] += v[z];
  }
  big_epilogue<MT, 2>(p, acc, stage, bm * MT * 16, (bn - nb_first) * (W * 2) + wave * 2);
}

constexpr int SIDE_PD = 3;
// MT <= 4: the forms for small launches, named by their workgroup tile (MT*16*WM rows x WN*64 channels) and threads
template <int MT, bool DUAL, int WM, int WN>
__global__ void __launch_bounds__(WM * WN * 64, 2)
big_bf16_kernel(const BigParams P) {
  if constexpr (MT <= 4)
    side_gemm_body<MT * WM, WM * WN, SIDE_PD, DUAL>(P);
  else
    big_gemm_body<MT, DUAL, WM, WN, true>(P);
}

// 64 x 128 with K in P.S slices (grid y), bf16 weights: launches of few workgroups and a long K.  A workgroup's time is its K
// steps whatever else the chip does, so 64 .. 192 of them with 86 steps leave most of it idle; several resident to a CU
// run S times as many with an S-th of the steps.  The sums go out as they lie in the registers, 32 KiB a workgroup, and a
// second launch adds them: with it 4096 x 11008 at 100 / 200 / 300 rows 56.9 -> 32.3, 61.2 -> 40.7, 66.4 -> 53.4 us, 2560 x 10240 at
// 200 rows 55.3 -> 28.5 (weights from memory).
__global__ void __launch_bounds__(256, 2)
side_split_kernel(const BigParams P) {
  side_gemm_body<4, 4, SIDE_PD, false, true>(P);
}

template <int MT, bool DUAL, int WM, int WN>
__global__ void __launch_bounds__(WM * WN * 64, WM * WN == 4 ? 2 : 1)
big_mxfp4_kernel(const BigParams P) {
  big_gemm_body<MT, DUAL, WM, WN, false>(P);
}

// ---------------------------------------------------------------------------
// Large-M QINT8 (W8A8, 256-wide blocks): W waves side by side, each with a wave tile of MT*16 rows x 32 channels, K step
// 256 = one scale block.  What bounds int8 at this size is the LDS and the fold, not the MFMA: a CU's LDS hands out
// 128 B/clk and takes in about half of that, the int8 MFMA runs at twice the bf16 rate, and every block's int32 sums
// have to be converted, scaled by sa[m] * sw[n] and added to the fp32 sums -- 3 vector instructions per output and block,
// 3 per MFMA, each of which stretches an MFMA's 16 cycles by about 4 (16.5 / 17.5 / 18 / 21.5 / 25.5 cycles with
// 0 / 1 / 2 / 3 / 4).  So:
//   * Weights never see the LDS: a wave owns its channels, so it loads their native tiles into registers, a whole step
//     ahead (two sets of 32 registers, the loop unrolled by two).  The form before brought both operands through LDS:
//     256 KB of operand reads and 96 KB of writes per step of a 128 x 256 workgroup, against 256 and 32 now, and a phase
//     of copying and a second barrier in every step.
//   * Activation rows and their scales go straight into LDS, two steps ahead in a ring of three stages; the bank swizzle
//     sits on the source side (the lane at position c of row m fetches chunk c ^ (m & 15)).  One barrier per step.
//   * All loads are buffer loads: the addresses are scalar, and the compiler counts them exactly beside the loads into
//     LDS (flat-addressed loads into LDS make it wait for everything).  Order per step: the next step's weights, then the
//     rows two steps ahead, one or two behind each MFMA step; loads return in order, so "at most LA + LB younger" is the
//     wait for a stage.
//   * The MFMAs run by groups of two row tiles (four sums of 16 x 16, all of K for them, then the next group), and the
//     fold of a group sits between the MFMAs of the next one, that of a step's last group under the next step's first
//     operand reads.
// Forms (the same sums in the same order, the same bits): 128 x 256 and 64 x 256 of eight waves, 64 x 128 of four.
// Measured, without the quantizer, against that earlier form, at 70 / 333 / 1000 / 2048 rows: 4096 x 4096 with residual
// 23.8 / 24.7 / 29.1 / 44.4 -> 13.7 / 15.0 / 24.5 / 43.0 us, 4096 x 11008 59.3 / 60.7 / 69.9 / 106 -> 30.6 / 31.9 / 56.2 /
// 97 us, pair 2 x 4096 x 11008 at 333 / 1000 rows 65 / 103 -> 49 / 94; 2.0 POP/s at 2048 rows.
// DUAL: the gate/up pair: a wave's two channel tiles are a gate tile and the up tile of the same channels, silu(gate) * up
// in the epilogue.  A launch per weight rounds its workgroups up to whole rounds of 256 twice, quantizes the rows twice
// and takes the gate matrix out to memory and back.
// ---------------------------------------------------------------------------
template <int MT, int W>
struct Qint8Geom {
  static constexpr int WGM = MT * 16, NB = 3;
  static constexpr int SA_OFF = WGM * 256;
  static constexpr int STAGE = SA_OFF + WGM * 4;
  static constexpr int NA = MT * 4 / W;              // 4-row pieces of A a wave fetches per step
  static constexpr int LA = NA + 1, LB = 10;     // loads per wave and step: rows + their scales; weights + their scales
  static constexpr size_t EP = (size_t)W * (MT < 4 ? MT * 16 : 64) * ep_ld(2) * sizeof(float);
  static constexpr size_t LDS = (size_t)NB * STAGE > EP ? (size_t)NB * STAGE : EP;
};

template <int MT, int W, bool DUAL, bool SPLIT = false>
__device__ __forceinline__ void big_qint8_body(const BigParams& P) {
  using G = Qint8Geom<MT, W>;
  constexpr int WGM = G::WGM, NB = G::NB, NA = G::NA, LA = G::LA, LB = G::LB, STAGE = G::STAGE;
  extern __shared__ __align__(16) uint8_t tl_lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int MB = (P.seg[0].M + WGM - 1) / WGM;
  int bm, bn;
  tile_of_block(MB, P.nb0[P.n_seg], bm, bn);
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
  // K steps k0 .. k0 + KS - 1 of KA
  const int KA = p.K >> 8, k0 = SPLIT ? KA * (int)blockIdx.y / P.S : 0, KS = SPLIT ? KA * ((int)blockIdx.y + 1) / P.S - k0 : KA;
  const int m_wg = bm * WGM;
  const int tile_base = DUAL ? bn * W + wave : bn * (W * 2) + wave * 2; // DUAL: gate and up tile of the same 16 channels

  const auto xr = tl_rsrc(p.xq), sar = tl_rsrc(p.sa);
  uint32_t aoff[NA];
#pragma unroll
  for (int i = 0; i < NA; i++) {
    const int blk = wave * NA + i, r16 = (blk & 3) * 4 + (lane >> 4);
    aoff[i] = (uint32_t)min(m_wg + blk * 4 + (lane >> 4), p.M - 1) * (uint32_t)p.K + (uint32_t)(((lane & 15) ^ r16) & 15) * 16u + (uint32_t)k0 * 256u;
  }
  const int sp = wave % (WGM / 64);
  const uint32_t saoff = (uint32_t)(min(m_wg + sp * 64 + lane, p.M - 1) * KA + k0) * 4u;
  auto load_a = [&](auto I, int s, int buf) {
    constexpr int i = decltype(I)::value;
    uint8_t* base = tl_lds + buf * STAGE;
    if constexpr (i < NA)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (__attribute__((address_space(3))) void*)(base + (wave * NA + i) * 1024), 16, aoff[i], s * 256, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(sar, (__attribute__((address_space(3))) void*)(base + G::SA_OFF + sp * 256), 4, saoff, s * 4, 0, 0);
  };
  __amdgpu_buffer_rsrc_t wr[2], swr[2];
  uint32_t woff[2], swoff[2];
#pragma unroll
  for (int nt = 0; nt < 2; nt++) {
    const int tile = min(DUAL ? tile_base : tile_base + nt, p.tiles - 1);
    wr[nt] = tl_rsrc(DUAL && nt ? P.seg[1].qw : p.qw);
    swr[nt] = tl_rsrc(DUAL && nt ? P.seg[1].sw : p.sw);
    woff[nt] = (((uint32_t)tile * (uint32_t)KA + (uint32_t)k0) * 256u + (uint32_t)lane) * 16u;
    swoff[nt] = (uint32_t)((tile * KA + k0) * 16 + (lane & 15)) * 4u;
  }
  i32x4 b[2][4][2]; // [set][j][nt]
  float swv[2][2];
  auto load_b = [&](auto I, int s, auto SET) {
    constexpr int i = decltype(I)::value, set = decltype(SET)::value;
    if constexpr (i < 8)
      b[set][i >> 1][i & 1] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(wr[i & 1], woff[i & 1] + (i >> 1) * 1024, s * 4096, 0));
    else
      swv[set][i & 1] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(swr[i & 1], swoff[i & 1], s * 64, 0));
  };
  uint32_t rdb[4];
  {
    const int m = lane & 15, g = lane >> 4;
#pragma unroll
    for (int j = 0; j < 4; j++)
      rdb[j] = (uint32_t)((m >> 2) * 1024 + (m & 3) * 256 + (((j * 4 + g) ^ m) & 15) * 16);
  }
  constexpr int NG = MT / 2, NQ = NG * 4; // groups of two row tiles; MFMA steps of a K step
  f32x4 facc[MT][2];
  i32x4 iacc[2][4];  // [group parity][row tile of the group * 2 + nt]
  f32x4 sav[2][2];   // [group parity][row tile]
  float swp[2] = {0.f, 0.f}; // channel scales of the step before
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int nt = 0; nt < 2; nt++)
      facc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 4; i++) {
    iacc[0][i] = iacc[1][i] = i32x4{0, 0, 0, 0};
    sav[i >> 1][i & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int last = KS - 1;
  // (in this order: the waits count the loads behind those they wait for)
  static_for<0, LA>([&](auto I) { load_a(I, 0, 0); });
  __builtin_amdgcn_sched_barrier(0);
  static_for<0, LB>([&](auto I) { load_b(I, 0, std::integral_constant<int, 0>{}); });
  __builtin_amdgcn_sched_barrier(0);
  static_for<0, LA>([&](auto I) { load_a(I, min(1, last), 1); });
  __builtin_amdgcn_sched_barrier(0);
  int buf = 0;
  // outputs e0 .. e1 (of 16) of group g's fold
  auto fold = [&](auto GI, auto E0, auto E1, const float (&sw)[2]) {
    constexpr int g = decltype(GI)::value;
    static_for<decltype(E0)::value, decltype(E1)::value>([&](auto E) {
      constexpr int e = decltype(E)::value, t = e >> 2, r = e & 3, rt = t >> 1, nt = t & 1;
      facc[g * 2 + rt][nt][r] = fmaf((float)iacc[g & 1][t][r], sav[g & 1][rt][r] * sw[nt], facc[g * 2 + rt][nt][r]);
    });
  };
  auto step = [&](auto SET, int s) {
    constexpr int set = decltype(SET)::value;
    asm volatile("" : : : "memory");
    constexpr int vm = LB + LA;
    __builtin_amdgcn_s_waitcnt((vm & 15) | 7 << 4 | vm >> 4 << 14); // A of step s has landed, reads of step s - 1 have returned
    asm volatile("s_barrier" : : : "memory");
    const int nbuf = buf == 0 ? NB - 1 : buf - 1;
    const uint8_t* ab = tl_lds + buf * STAGE;
    const float* sas = reinterpret_cast<const float*>(ab + G::SA_OFF) + (lane >> 4) * 4;
    constexpr int RD = 2;
    i32x4 ar[RD + 1][2];
    auto read = [&](auto Q) {
      constexpr int q = decltype(Q)::value, g = q >> 2, j = q & 3;
#pragma unroll
      for (int rt = 0; rt < 2; rt++)
        ar[q % (RD + 1)][rt] = *reinterpret_cast<const i32x4*>(ab + (g * 2 + rt) * 4096 + rdb[j]);
    };
    static_for<0, RD>([&](auto Q) { read(Q); });
    __builtin_amdgcn_sched_barrier(0);
    fold(std::integral_constant<int, NG - 1>{}, std::integral_constant<int, 0>{}, std::integral_constant<int, 16>{}, swp);
    __builtin_amdgcn_sched_barrier(0);
    static_for<0, NQ>([&](auto Q) {
      constexpr int q = decltype(Q)::value, g = q >> 2, j = q & 3;
      if constexpr (q + RD < NQ)
        read(std::integral_constant<int, q + RD>{});
      if constexpr (j == 0) {
#pragma unroll
        for (int rt = 0; rt < 2; rt++)
          sav[g & 1][rt] = *reinterpret_cast<const f32x4*>(sas + (g * 2 + rt) * 16);
      }
#pragma unroll
      for (int t = 0; t < 4; t++)
        iacc[g & 1][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ar[q % (RD + 1)][t >> 1], b[set][j][t & 1], j == 0 ? i32x4{0, 0, 0, 0} : iacc[g & 1][t], 0, 0, 0);
      if constexpr (g > 0)
        fold(std::integral_constant<int, g - 1>{}, std::integral_constant<int, j * 4>{}, std::integral_constant<int, j * 4 + 4>{}, swv[set]);
#pragma unroll
      for (int t = 0; t < 4; t++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if constexpr (g > 0)
          __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      // the next step's weights, then the rows two steps ahead, a few behind each MFMA step
      constexpr int NL = LB + LA, l0 = NL * q / NQ, l1 = NL * (q + 1) / NQ;
      static_for<l0, l1>([&](auto I) {
        constexpr int i = decltype(I)::value;
        if constexpr (i < LB)
          load_b(I, min(s + 1, last), std::integral_constant<int, set ^ 1>{});
        else
          load_a(std::integral_constant<int, i - LB>{}, min(s + 2, last), nbuf);
      });
      __builtin_amdgcn_sched_barrier(0);
    });
    swp[0] = swv[set][0];
    swp[1] = swv[set][1];
    buf = buf == NB - 1 ? 0 : buf + 1;
  };
  int s = 0;
  for (; s + 1 < KS; s += 2) {
    step(std::integral_constant<int, 0>{}, s);
    step(std::integral_constant<int, 1>{}, s + 1);
  }
  if (s < KS)
    step(std::integral_constant<int, 0>{}, s);
  fold(std::integral_constant<int, NG - 1>{}, std::integral_constant<int, 0>{}, std::integral_constant<int, 16>{}, swp);
  if constexpr (SPLIT) { // (as they lie in the registers: a wave instruction is 1 KiB)
    f32x4* out = reinterpret_cast<f32x4*>(P.part) + (((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * W + wave) * (MT * 2 * 64) + lane;
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
      out[(mt * 2) * 64] = facc[mt][0];
      out[(mt * 2 + 1) * 64] = facc[mt][1];
    }
    return;
  }
  __syncthreads(); // (waits for the loads still under way: the ring is free for the epilogue staging)
  float* stage = reinterpret_cast<float*>(tl_lds) + wave * (MT < 4 ? MT * 16 : 64) * ep_ld(2);
  if (DUAL)
    big_epilogue_dual<MT, 2>(p, P.seg[1], facc, stage, m_wg, tile_base);
  else
    big_epilogue<MT, 2>(p, facc, stage, m_wg, tile_base);
}

// 64 x 128 with K in P.S slices (grid y), as side_split_kernel
__global__ void __launch_bounds__(256, 2)
big_qint8_split_kernel(const BigParams P) {
  big_qint8_body<4, 4, false, true>(P);
}

__global__ void __launch_bounds__(512, 2)
big_qint8_kernel(const BigParams P) {
  big_qint8_body<8, 8, false>(P);
}

__global__ void __launch_bounds__(512, 2)
big_qint8_small_kernel(const BigParams P) {
  big_qint8_body<4, 8, false>(P);
}

__global__ void __launch_bounds__(256, 2)
big_qint8_narrow_kernel(const BigParams P) {
  big_qint8_body<4, 4, false>(P);
}

__global__ void __launch_bounds__(512, 2)
big_qint8_dual_kernel(const BigParams P) {
  big_qint8_body<8, 8, true>(P);
}

__global__ void __launch_bounds__(512, 2)
big_qint8_small_dual_kernel(const BigParams P) {
  big_qint8_body<4, 8, true>(P);
}

__global__ void __launch_bounds__(256, 2)
big_qint8_narrow_dual_kernel(const BigParams P) {
  big_qint8_body<4, 4, true>(P);
}

// ---------------------------------------------------------------------------
// Large-M MXFP4 weights x MXFP8 activations on the block-scaled MFMA
// (v_mfma_scale_f32_16x16x128_f8f6f4): the weights' E2M1 codes and E8M0 scales
// are the instruction's operands as they lie in the native tiles -- nothing is
// expanded -- and the activations arrive quantised in operand order
// (quant_act_mxfp8_kernel).  Not the reference's arithmetic (its activations
// stay bf16): an opt-in (TPPX_FLAG_ACT_FP8).
// Workgroup tile (MT*32) x 256, 8 waves (2 x 4), wave tile (MT*16) x 64 =
// 4*MT MFMAs of K = 128 per step; MT = 8 (256 rows) or 4 (128 rows).
// Everything a step needs -- both operands AND both sets of scale bytes -- goes
// from global memory straight into LDS (1 KiB per wave instruction for the
// operands: a native weight tile, half an activation tile, lane-linear on both
// sides, so operand reads are conflict-free 16-byte reads; 256 B per wave
// instruction for scales), NB - 1 steps ahead in a ring of NB stages.  All
// loads of the loop being of this one kind, they complete in issue order and
// the wait at the top of a step is a partial one (the younger stages stay in
// flight); one barrier per step.
// ---------------------------------------------------------------------------
typedef int i32x8 __attribute__((ext_vector_type(8)));

template <int N>
__device__ __forceinline__ void lds_wait_keep2(i32x4& a, i32x4& b) {
  asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(a), "+v"(b) : "n"(N));
}

template <int MT>
struct Fp8Geom {
  static constexpr int NB = MT == 8 ? 3 : 4;        // stages in the ring
  static constexpr int A_BYTES = MT * 4096;         // 2*MT row tiles of 2 KiB
  static constexpr int B_OFF = A_BYTES;             // 16 weight tiles of 1 KiB
  static constexpr int SA_OFF = B_OFF + 16384;      // MT/2 groups of 64 rows x 256 B
  static constexpr int SB_OFF = SA_OFF + MT * 128;  // 16 tiles x 64 B
  static constexpr int STAGE = SB_OFF + 1024;
  static constexpr int LPS = MT / 2 + 2 + 1;        // loads per wave and stage: A halves, weight tiles, one of scales
};

// DUAL: the gate/up pair as in big_mxfp4_kernel: 128 output channels per workgroup, the 16 weight tiles of a stage are
// 4 x (2 gate tiles, the 2 up tiles of the same channels), one group per wave column; silu(gate) * up in the epilogue.
template <int MT, bool DUAL>
__global__ void __launch_bounds__(512)
big_fp8_kernel(const BigParams P) {
  using G = Fp8Geom<MT>;
  constexpr int NB = G::NB, STAGE = G::STAGE, LPS = G::LPS;
  extern __shared__ __align__(16) uint8_t tl_lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int MB = (P.seg[0].M + MT * 32 - 1) / (MT * 32);
  int bm, bn;
  tile_of_block(MB, P.nb0[P.n_seg], bm, bn);
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
  const int KT = p.K >> 7;
  const int m_wg = bm * (MT * 32);
  const int tile_base = DUAL ? bn * 8 + wn * 2 : bn * 16 + wn * 4;
  // weight tile behind slot t (0..15) of a stage, and whether it is the up projection's (DUAL)
  auto slot_tile = [&](int t) { return DUAL ? bn * 8 + (t >> 2) * 2 + (t & 1) : bn * 16 + t; };
  auto slot_up = [&](int t) { return DUAL && (t & 2) != 0; };
  const int Q = (p.M + 63) >> 6; // 64-row groups of the quantised activations (rows padded to 64)

  // this wave's share of a stage: MT/2 activation half tiles, 2 weight tiles, one 256-byte piece of scales
  const char* xqb = reinterpret_cast<const char*>(p.xq);
  const char* qwb = reinterpret_cast<const char*>(p.qw);
  const char* a_src[MT / 2];
#pragma unroll
  for (int i = 0; i < MT / 2; i++) {
    const int j = wave * (MT / 2) + i; // half tile j of the 4*MT: row tile j >> 1, half j & 1
    a_src[i] = xqb + ((size_t)min(bm * (MT * 2) + (j >> 1), Q * 4 - 1) * KT * 2 + (j & 1)) * 1024 + (size_t)lane * 16;
  }
  const char* b_src[2];
#pragma unroll
  for (int i = 0; i < 2; i++)
    b_src[i] = (slot_up(wave * 2 + i) ? reinterpret_cast<const char*>(P.seg[1].qw) : qwb) +
               ((size_t)min(slot_tile(wave * 2 + i), p.tiles - 1) * KT) * 1024 + (size_t)lane * 16;
  const char* s_src;
  int s_dst, s_stride;
  if (wave < MT / 2) { // activation scales of 64-row group `wave`: [Q][KT][64 lanes][4 row tiles]
    s_src = reinterpret_cast<const char*>(p.sa) + (size_t)min(bm * (MT / 2) + wave, Q - 1) * KT * 256 + (size_t)lane * 4;
    s_dst = G::SA_OFF + wave * 256;
    s_stride = 256;
  } else { // weight scales of tiles 4i .. 4i+3: native [tile][KT][64]
    int i = wave - MT / 2;
    if (i >= 4)
      i -= 2; // 128-row form: waves 6, 7 repeat what 4, 5 fetch, so that every wave issues LPS loads per stage
    const int t = i * 4 + (lane >> 4);
    s_src = reinterpret_cast<const char*>(slot_up(t) ? P.seg[1].sw : p.sw) + (size_t)min(slot_tile(t), p.tiles - 1) * KT * 64 +
            (size_t)(lane & 15) * 4;
    s_dst = G::SB_OFF + i * 256;
    s_stride = 64;
  }
  // load number I (of LPS) of this wave's share of a stage
  auto dma_one = [&](auto I, int ks, int buf) {
    constexpr int i = decltype(I)::value;
    uint8_t* base = tl_lds + buf * STAGE;
    if constexpr (i < MT / 2)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(a_src[i] + (size_t)ks * 2048),
                                       (__attribute__((address_space(3))) void*)(base + (wave * (MT / 2) + i) * 1024), 16, 0, 0);
    else if constexpr (i < MT / 2 + 2)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(b_src[i - MT / 2] + (size_t)ks * 1024),
                                       (__attribute__((address_space(3))) void*)(base + G::B_OFF + (wave * 2 + i - MT / 2) * 1024), 16, 0, 0);
    else
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(s_src + (size_t)ks * s_stride),
                                       (__attribute__((address_space(3))) void*)(base + s_dst), 4, 0, 0);
  };
  auto dma = [&](int ks, int buf) { static_for<0, LPS>([&](auto I) { dma_one(I, ks, buf); }); };

  f32x4 acc[MT][4];
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int nt = 0; nt < 4; nt++)
      acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};

  const uint32_t lds0 = (uint32_t)(uintptr_t)tl_lds;
#pragma unroll
  for (int s = 0; s < NB - 1; s++)
    if (s < KT)
      dma(s, s);
  int buf = 0;
  // One K step.  DMA: the loads of stage ks + NB - 1 are issued one at a time behind the MFMA groups of the step
  // (issued in one burst at the top, a wave stands at its load instructions while the memory pipeline's queue
  // drains, and its MFMAs wait with it).
  auto step = [&](auto DMA, int ks) {
    constexpr bool with_dma = decltype(DMA)::value;
    // stage ks has landed for this wave (the NB - 2 younger ones may still be in flight) ...
    if (with_dma || ks + NB - 2 < KT)
      asm volatile("s_waitcnt vmcnt(%0)" : : "n"(LPS * (NB - 2)) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
    // ... and for every wave; nobody still reads the stage of step ks - 1, which the next loads overwrite
    asm volatile("s_barrier" : : : "memory");
    const int nbuf = buf == 0 ? NB - 1 : buf - 1;
    const uint8_t* base = tl_lds + buf * STAGE;
    i32x4 bw[4];
    int sbv[4];
    uint32_t sav[MT / 4];
#pragma unroll
    for (int nt = 0; nt < 4; nt++) {
      bw[nt] = *reinterpret_cast<const i32x4*>(base + G::B_OFF + (wn * 4 + nt) * 1024 + lane * 16);
      sbv[nt] = base[G::SB_OFF + (wn * 4 + nt) * 64 + lane];
    }
#pragma unroll
    for (int q = 0; q < MT / 4; q++)
      sav[q] = *reinterpret_cast<const uint32_t*>(base + G::SA_OFF + (wm * (MT / 4) + q) * 256 + lane * 4);
    // activation operands: the two halves of row tile mt, read two row tiles ahead of the MFMAs that use them
    const uint32_t abase = lds0 + (uint32_t)(buf * STAGE + wm * MT * 2048 + lane * 16);
    i32x4 alo[3], ahi[3];
    static_for<0, 2>([&](auto I) {
      constexpr int i = decltype(I)::value;
      lds_read_b128_async<i * 2048>(alo[i], abase);
      lds_read_b128_async<i * 2048 + 1024>(ahi[i], abase);
    });
    static_for<0, MT>([&](auto I) {
      constexpr int mt = decltype(I)::value;
      if constexpr (mt + 2 < MT) {
        lds_read_b128_async<(mt + 2) * 2048>(alo[(mt + 2) % 3], abase);
        lds_read_b128_async<(mt + 2) * 2048 + 1024>(ahi[(mt + 2) % 3], abase);
        lds_wait_keep2<4>(alo[mt % 3], ahi[mt % 3]);
      } else {
        lds_wait_keep2<(MT - 1 - mt) * 2>(alo[mt % 3], ahi[mt % 3]);
      }
      const i32x4 lo = alo[mt % 3], hi = ahi[mt % 3];
      const i32x8 a = i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      const int sa = (int)((sav[mt >> 2] >> ((mt & 3) * 8)) & 0xffu);
#pragma unroll
      for (int nt = 0; nt < 4; nt++) {
        const i32x8 b = i32x8{bw[nt][0], bw[nt][1], bw[nt][2], bw[nt][3], 0, 0, 0, 0};
        acc[mt][nt] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, acc[mt][nt], 0 /* A: E4M3 */,
                                                                       4 /* B: E2M1 */, 0, sa, 0, sbv[nt]);
      }
      if constexpr (with_dma) {
        // LPS loads over MT slots (LPS <= MT + 1: the last slot takes the remainder)
        if constexpr (mt < LPS)
          dma_one(std::integral_constant<int, mt>{}, ks + NB - 1, nbuf);
        if constexpr (mt == MT - 1)
          static_for<MT, (LPS > MT ? LPS : MT)>([&](auto J) { dma_one(J, ks + NB - 1, nbuf); });
      }
    });
    buf = buf == NB - 1 ? 0 : buf + 1;
  };
  int ks = 0;
  for (; ks + NB - 1 < KT; ks++)
    step(std::true_type{}, ks);
  for (; ks < KT; ks++)
    step(std::false_type{}, ks);
  __syncthreads(); // every wave has left the main loop: LDS is free for the epilogue staging
  if (DUAL)
    big_epilogue_dual<MT>(p, P.seg[1], acc, reinterpret_cast<float*>(tl_lds) + wave * 64 * EP_LD, m_wg + wm * (MT * 16),
                          tile_base);
  else
    big_epilogue<MT>(p, acc, reinterpret_cast<float*>(tl_lds) + wave * 64 * EP_LD, m_wg + wm * (MT * 16), tile_base);
}

// Workgroup tiles of the MXFP4 and bf16 launches:
//   256 x 256, 128 x 512  eight waves, one workgroup per CU; for launches that fill the chip several times over
//   128 x 256             four waves and two per CU; bf16 weights: up to 256 of them eight waves side by side, one per CU
//   64 x 128, 64 x 256    bf16 only: waves side by side
//   the rest              WIDE_FORMS: launches of up to a few workgroups per CU
enum { TILE_256_256 = 0, TILE_128_256, TILE_128_512, TILE_64_128, TILE_64_256, TILE_WIDE, N_TILES = TILE_WIDE + N_WIDE };
static constexpr int tile_rows(int tile) {
  constexpr int rows[TILE_WIDE] = {256, 128, 128, 64, 64};
  return tile < TILE_WIDE ? rows[tile] : WIDE_FORMS[tile - TILE_WIDE].mt * 16;
}
static constexpr int tile_cols16(int tile) { // 16-channel weight tiles (the pair: gate + up)
  constexpr int cols[TILE_WIDE] = {16, 16, 32, 8, 16};
  return tile < TILE_WIDE ? cols[tile] : WIDE_FORMS[tile - TILE_WIDE].nt * WIDE_FORMS[tile - TILE_WIDE].w;
}

// What a launch takes, in us, with r = its rounds of 256 workgroups, f = the filled part of the last one, s = K / 128 and w = the
// weights as MB of bf16:
//   one round     a + (b + c f) s + g w
//   more          p + q r + (u + v r + w f + z r s / 1000) s + h w     (z: the clock falls under the power limit as a launch grows)
//   K in slices   that for S times the workgroups and an S-th of the steps, and c0 + c1 us for each 32 KiB of the slices' sums
// and e us per round for the epilogue of a gate/up pair.  (Rounds also where several workgroups share a CU: three of one round's
// take about three times as long together.)
// MXFP4: fitted to 888 of 1184 shapes of 65 .. 2048 rows, 768 .. 37888 channels and K = 1024 .. 18944 with every tile forced, whole
// and in slices, weights in turn from 320 MB; on the others the tile and slices taken are 0.8 % off the fastest on average, 11 % in
// the worst hundredth.  Larger launches (28672 x 8192 pairs) are extrapolated and stay with the large tiles.
// MXFP4, K below 1024, more than a round: a workgroup is its first loads and its epilogue, which one alone on its CU has nothing
// beside.  Of 852 shapes of 65 .. 8192 rows and K = 128 .. 896 with every tile forced 256 x 256 is the fastest in 3 and by its estimate in
// 72, 128 x 512 in 34 and 81, so there they are not taken: 2 x 31616 x 512 at 3309 rows 285.9 us, on 128 x 256 246.2, 2 x 20544 x 256 at 1981
// 92 and 75; 1.4 % off the fastest on average, with them 2.4, and none more than 2.5 % slower for it.
// bf16: the large tiles, 64 x 128 and 64 x 256 fitted to 4100 launches, q/k/v groups among them, up to pairs of 28672 x 8192, most of
// all where the tile is within 20 % of the fastest, and with weights that come from memory: 96 of them, or as many as fill 2 GB, in
// turn.  (With four in turn most lie in the Infinity Cache, as they never do in a model, and the estimates came out 20 .. 30 %
// low.)  96 rows: fitted to 2956 more, times 0.96, which those take on the same shapes.
struct TileCost {
  double a, b, c, p, q, u, v, w, z, g, h, e, c0, c1;
};
static constexpr TileCost MXFP4_COST[N_TILES] = {
    {9.24, 1.85, 0.843, 2.85, 7.11, -1.18, 2.6, 1.32, 0.182, 0.0166, 0.0562, 0}, // 256 x 256
    {8.13, 1.15, 0.429, 2.31, 4.18, -0.632, 1.35, 0.85, 0, 0.0177, 0.00405, 0}, // 128 x 256
    {8.78, 1.83, 0.835, 1.79, 7.7, -1.27, 2.56, 1.42, 0, 0.0236, 0.0681, 0}, // 128 x 512
    {}, // 64 x 128
    {}, // 64 x 256
    {3.52, 0.203, 0.105, 3.27, 0.706, -0.0854, 0.243, 0.162, 0, 0.0109, 0.00497, 0, 2.91, 0.00848}, // 32 x 128
    {3.98, 0.254, 0.119, 3.01, 1.43, -0.0935, 0.289, 0.192, 0.037, 0.00615, 0.00283, 0, 3.05, 0.00707}, // 48 x 128
    {4.38, 0.277, 0.165, 2.79, 1.93, -0.191, 0.391, 0.21, 0.0643, 0.0034, 0, 0, 3.34, 0.00632}, // 64 x 128
    {4.33, 0.346, 0.196, 1.27, 2.63, -0.243, 0.472, 0.328, 0.0483, 0.0033, 0, 0}, // 80 x 128
    {}, // 96 x 128
    {5.36, 0.375, 0.235, 4.15, 2.87, -0.371, 0.647, 0.332, 0.00103, 0.00239, 0, 0}, // 64 x 192
    {5.54, 0.454, 0.247, 3.08, 3.4, -0.416, 0.758, 0.414, 0, 0.00417, 0, 0}, // 80 x 192
    {6.04, 0.498, 0.396, 2.68, 3.55, -0.583, 0.967, 0.565, 0, 0.00161, 0, 0}, // 80 x 256
    {6.4, 0.597, 0.463, 1.86, 4.66, -0.617, 1.08, 0.664, 0.0657, 0, 0, 0}, // 96 x 256
    {7.41, 0.585, 0.473, 2.65, 4.99, -0.639, 1.11, 0.671, 0, 0, 0, 0}, // 64 x 384
    {8.25, 0.935, 0.577, 1.79, 6.14, -0.789, 1.54, 0.962, 0, 0.00469, 0.00688, 0}, // 96 x 384
};
static constexpr TileCost BF16_COST[N_TILES] = {
    {9.19, 1.73, 0.784, 2.54, 6.07, -1.52, 2.92, 1.23, 0.155, 0.0249, 0.00722, 3.73}, // 256 x 256
    {7.3, 1.13, 0.298, 2.01, 3.53, -0.41, 1.25, 0.708, 0.288, 0.043, 0.0481, 1.07}, // 128 x 256
    {8.86, 1.81, 0.692, -1.47, 7.78, -1.4, 2.81, 1.4, 0.195, 0.0518, 0.0267, 3.63}, // 128 x 512
    {3.7, 0.613, 0.0187, 2.24, 0.731, 0.0345, 0.498, 0.186, 0.041, 0.0584, 0.069, 0.555, 2.2, 0.0115}, // 64 x 128
    {4.61, 1.02, 0.051, 1.68, 3.15, -0.354, 0.929, 0.634, 0.195, 0.0614, 0.0625, 1.05}, // 64 x 256
    {}, // 32 x 128
    {}, // 48 x 128
    {}, // 64 x 128
    {}, // 80 x 128
    {4.65, 0.631, 0.124, 3.46, 1.99, -0.287, 0.669, 0.398, 0.135, 0.0652, 0.0644, 0.6}, // 96 x 128
    {}, // 64 x 192
    {}, // 80 x 192
    {}, // 80 x 256
    {6.57, 1.09, 0.123, 0.575, 6.07, -0.269, 1.08, 0.729, 0.271, 0.0695, 0.0719, 0.6}, // 96 x 256
    {}, // 64 x 384
    {}, // 96 x 384
};
static double tile_us(const TileCost& k, int tile, int64_t wgs, double s, double weight_mb, bool dual) {
  const double r = (double)((wgs + 255) / 256), f = (double)wgs / 256.0 - (r - 1.0);
  if (r <= 1.0)
    return k.a + (k.b + k.c * f) * s + k.g * weight_mb + (dual ? k.e : 0.0);
  // (the z term at most as far as it was measured: 448 rounds x steps of 256 x 256, the same work in the other tiles)
  const double rs = std::min(r * s, 448.0 * 4096.0 / (tile_rows(tile) * tile_cols16(tile)));
  return k.p + k.q * r + (k.u + k.v * r + k.w * f + k.z * 1e-3 * rs * r) * s + k.h * weight_mb + (dual ? k.e * r : 0.0);
}

// How many of the 8 rectangles of tile_of_block lie along M: the split that moves the fewest bytes from memory into the L2s
// (every XCD fetches 1/xm of the activations and xm/8 of the weights)
static int xcd_split(int64_t mb, int64_t nb, double a_bytes, double w_bytes) {
  double best = 8.0 * (a_bytes + w_bytes / 8.0); // xm = 1: an eighth of the channel blocks each, whether or not 8 divides them
  int split = 1;
  for (int xm = 2; xm <= 4; xm *= 2)
    if (mb % xm == 0 && nb % (8 / xm) == 0) {
      const double fill = 8.0 * (a_bytes / xm + w_bytes * xm / 8.0);
      if (fill < best) {
        best = fill;
        split = xm;
      }
    }
  return split;
}

constexpr double MXFP4_WEIGHT_BYTES = 0.53;

// What the fits above do not have; a factor on tile_us.
// MXFP4, the wave tiles of up to 80 rows, more than a round of workgroups: without a split along M an XCD walks whole columns, and
// the columns of the workgroups that are resident together drift apart in K.  Against the estimate, with a split and up to 17 row
// blocks 0.92, 22 1.08, 25 1.12, from 28 on 1.15 .. 1.24; no such drift on the larger tiles.  1978 x 3136 x 10240 127.5 us, with it
// (96 x 384) 111.5; on 100 shapes of 390 .. 2048 rows with every tile forced the tile taken is 0.4 % off the fastest on average, 0.5
// without, 7.6 % in the worst case, 14 without.
// bf16, a single row block, all weights from memory once: 128 x 256 takes 1.13 of the estimate (1.3 in more than a round), 96 x 128
// in more than a round, where the last workgroups have the chip alone, 1.27, 96 x 256 1.2.  q/k/v of 3 x 10944 x 2304 at 93 rows
// 47.6 us, with it 40.0; 33024 x 5376 at 95 rows 103.6, 86.0; on 48 shapes 0.7 % off the fastest on average, 2.3 without.
template <bool WBF16>
static double tile_factor(int tile, int64_t mb, double s, int64_t wgs, int xm) {
  const bool more = wgs > 256;
  if (WBF16)
    return mb > 1 ? 1.0 : tile == TILE_128_256 ? (more ? 1.3 : 1.1) : tile < TILE_WIDE || !more ? 1.0 : tile_cols16(tile) == 8 ? 1.25 : 1.2;
  if (tile < TILE_WIDE || tile_cols16(tile) != 8 || !more || xm != 1)
    return 1.0;
  return 1.0 + std::max(0.0, std::min(0.33, 0.03 * (double)(mb - 17))) * std::min(1.0, std::max(0.0, (s - 8.0) / 12.0));
}

// the tiles a launch may take, one bit each
template <bool WBF16>
static unsigned big_tiles() {
  unsigned tiles = 1u << TILE_256_256 | 1u << TILE_128_256 | 1u << TILE_128_512;
  if (env_int("TPPX_TILED_SMALL", 1) == 0)
    return tiles;
  if (WBF16)
    tiles |= 1u << TILE_64_128 | 1u << TILE_64_256;
  for (int i = 0; i < N_WIDE; i++)
    if (WBF16 ? WIDE_FORMS[i].bf16 : WIDE_FORMS[i].mxfp4)
      tiles |= 1u << (TILE_WIDE + i);
  return tiles;
}

// bytes of the sums of one K slice of a workgroup
static int64_t slice_bytes(int tile) { return (int64_t)tile_rows(tile) * tile_cols16(tile) * 16 * 4; }

// The cheapest tile for n GEMMs of tiles[i] channel tiles over one activation (dual: the gate/up pair, tiles[0] each), *S its K
// slices (1: whole; only with room for their sums in part_bytes).  Slices have to look 3 % faster (bf16 weights 5 %, in more than
// a round 10 %): they are a second launch, behind and before other kernels (a GPT-J pass of three layers 699 .. 731 us in slices
// where whole K looked 4 % slower, whole 677 .. 688), and weights at hand in the Infinity Cache gain them less (bf16 8640 x 4608
// at 124 rows 32.9 and 32.1 us from memory, 22.4 and 25.8 at hand).
// Fewer than 2048 channels, MXFP4: up to K = 4096 not sliced (1024 channels at 160 .. 256 rows: decode kernels 9 us, slices 10), and
// the estimate that is weighed against the decode kernels is the one of whole K.  With a longer K and more rows than those run
// well a few dozen workgroups have all of it to walk: 1024 x 18176 at 320 rows 40.1 us whole, 22.5 in slices, 512 x 12288 at 677
// 24.6 and 17.8, 1920 x 8192 at 257 18.1 and 17.5.  Row blocks read the same weights: 1.5 % for each of 64 rows from the fifth to the
// sixteenth (768 x 12288 at 1400 rows 33.6 whole, 40.4 in slices; 64 x 12288 at 3421 24.4 and 19.3), and 8 % for six slices (1024 x
// 12288 at 320 rows 18.0, three 15.4).  On 228 shapes of 64 .. 1920 channels and 200 .. 6000 rows the one taken is 1 % off the fastest
// on average and at most 1.2 % slower than whole K.
template <bool WBF16>
static int cheapest_tile(int64_t M, int64_t K, const int* tiles, int n, bool dual, int64_t part_bytes, int* S, double* best_us = nullptr) {
  constexpr const TileCost* COST = WBF16 ? BF16_COST : MXFP4_COST;
  const unsigned allowed = big_tiles<WBF16>();
  const int forced = env_int("TPPX_TILED_SPLIT", 1);
  int64_t all = 0;
  for (int i = 0; i < n; i++)
    all += tiles[i];
  const double s = (double)(K / 128), mb = (double)(all * 32 * K) * 1e-6;
  int shape = 0;
  double best = 1e300, us = 1e300; // (us: without tile_factor, bf16 without what decides ties, as the decode kernels' estimates were weighed against it)
  *S = 1;
  for (int i = 0; i < N_TILES; i++) {
    if (!(allowed >> i & 1u) || (WBF16 && i >= TILE_WIDE && all < 48)) // (fewer than 768 channels: not measured)
      continue;
    const int tpw = tile_cols16(i) / (dual ? 2 : 1); // channel tiles of a workgroup (of each projection for the pair)
    int64_t nb = 0;
    for (int g = 0; g < (dual ? 1 : n); g++)
      nb += (tiles[g] + tpw - 1) / tpw;
    const int64_t rows = (M + tile_rows(i) - 1) / tile_rows(i), wgs = rows * nb;
    if (!WBF16 && K < 1024 && wgs > 256 && (i == TILE_256_256 || i == TILE_128_512)) // (two workgroups to a CU instead: see above)
      continue;
    // (a near tie goes to the large tiles, which read less)
    const double whole = tile_us(COST[i], i, wgs, s, mb, dual);
    double c = whole * (i >= TILE_64_128 && i != TILE_64_256 ? 1.01 : 1.0);
    us = std::min(us, WBF16 ? whole : c);
    c *= tile_factor<WBF16>(i, rows, s, wgs, xcd_split(rows, nb, (double)M, (double)nb * tile_cols16(i) * (WBF16 ? 16.0 : 8.0 * MXFP4_WEIGHT_BYTES)));
    if (c < best && !(forced > 1 && *S > 1)) {
      best = c;
      shape = i;
      *S = 1;
    }
    const bool narrow = !WBF16 && all < 128;
    if (dual || forced == 0 || !(COST[i].c0 > 0.0) || (forced == 1 && (WBF16 ? K <= 2560 || wgs > 320 : narrow && K <= 4096)))
      continue;
    for (int z : {2, 3, 4, 6}) {
      if (wgs * z * slice_bytes(i) > part_bytes || K / 128 < 4 * z || (forced == 1 && wgs * z > 1024)) // (as far as was measured)
        break;
      const double sliced = tile_us(COST[i], i, wgs * z, s / z, mb, false) + COST[i].c0 + COST[i].c1 * (double)(wgs * z * slice_bytes(i)) / 32768.0;
      c = sliced * (!WBF16 ? 1.03 : wgs <= 256 ? 1.05 : 1.10);
      if (narrow)
        c *= 1.0 + 0.015 * (double)std::min<int64_t>(12, std::max<int64_t>(0, (M + 63) / 64 - 4)) + (z == 6 ? 0.08 : 0.0);
      if (forced == z ? *S != z || c < best : forced == 1 && c < best) {
        if (!narrow || forced > 1)
          us = std::min(us, WBF16 ? sliced : c);
        best = c;
        shape = i;
        *S = z;
      }
    }
  }
  if (best_us)
    *best_us = us;
  return shape;
}

double tiled_mxfp4_us(int64_t M, int64_t K, int64_t n_tiles16, int64_t part_bytes) {
  const int tiles = (int)n_tiles16;
  double us;
  int S;
  cheapest_tile<false>(M, K, &tiles, 1, false, part_bytes, &S, &us);
  return us;
}

double tiled_bf16_us(int64_t M, int64_t K, int64_t n_tiles16, int64_t part_bytes) {
  const int tiles = (int)n_tiles16;
  double us;
  int S;
  cheapest_tile<true>(M, K, &tiles, 1, false, part_bytes, &S, &us);
  return us;
}

static bool big_fits(const TiledParams& p) {
  return (int64_t)p.M * p.K * 2 < ((int64_t)1 << 32) && (int64_t)p.tiles * 8 * p.K < ((int64_t)1 << 32);
}

bool tiled_mxfp4_takes_groups(const TiledParams& p) {
  return p.M >= big_min_rows() && big_fits(p);
}

template <typename Kern>
static hipError_t big_go(Kern kern, const BigParams& P, int wgs, int threads, size_t lds, hipStream_t stream) {
  TPPX_PLAN_ONLY(kern, dim3(wgs), dim3(threads), lds);
  if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds); e != hipSuccess)
    return e;
  kern<<<dim3(wgs), dim3(threads), lds, stream>>>(P);
  return hipGetLastError();
}

template <int MT, bool DUAL, int WM, int WN>
static hipError_t big_launch(const BigParams& P, int wgs, hipStream_t stream) {
  constexpr size_t lds = (size_t)WM * WN * 64 * EP_LD * sizeof(float); // epilogue staging per wave; >= the two A buffers
  static_assert(lds >= (size_t)2 * MT * 16 * WM * 256, "LDS plan");
  return big_go(big_mxfp4_kernel<MT, DUAL, WM, WN>, P, wgs, WM * WN * 64, lds, stream);
}

template <int MT, bool DUAL, int WM, int WN>
static hipError_t big_bf16_launch(const BigParams& P, int wgs, hipStream_t stream) {
  size_t lds = (size_t)WM * WN * 64 * EP_LD * sizeof(float);
  static_assert(MT <= 4 || (size_t)WM * WN * 64 * EP_LD * sizeof(float) >= (size_t)2 * MT * 16 * WM * 256, "LDS plan");
  if constexpr (MT <= 4)
    lds = SideGeom<MT * WM, WM * WN, SIDE_PD>::LDS;
  return big_go(big_bf16_kernel<MT, DUAL, WM, WN>, P, wgs, WM * WN * 64, lds, stream);
}

template <bool WBF16>
static int cheapest_tile(const TiledParams* t, int n, bool dual, int64_t part_bytes, int* S) {
  int tiles[TPPX_MAX_SEGS];
  for (int i = 0; i < n; i++)
    tiles[i] = t[i].tiles;
  return cheapest_tile<WBF16>(t[0].M, t[0].K, tiles, n, dual, part_bytes, S);
}

// fills P for n GEMMs over one activation with this workgroup tile; returns the workgroups of the launch
static int big_params(BigParams& P, const TiledParams* t, int n, bool dual, int tile, double bytes_per_weight) {
  const int tpw = tile_cols16(tile) / (dual ? 2 : 1), MB = (t[0].M + tile_rows(tile) - 1) / tile_rows(tile);
  memset(&P, 0, sizeof(P));
  int nb = 0;
  for (int i = 0; i < n; i++) {
    P.seg[i] = t[i];
    P.nb0[i] = nb;
    nb += (t[i].tiles + tpw - 1) / tpw;
  }
  if (dual) {
    nb = (t[0].tiles + tpw - 1) / tpw;
    P.nb0[1] = nb;
  }
  for (int i = n; i <= TPPX_MAX_SEGS; i++)
    P.nb0[i] = nb;
  P.n_seg = n;
  P.xm = xcd_split(MB, nb, (double)t[0].M * t[0].K * 2.0, (dual ? 2.0 : 1.0) * nb * tpw * 16.0 * t[0].K * bytes_per_weight);
  const int env_xm = env_int("TPPX_TILED_XCD_M", 0);
  if ((env_xm == 1 || env_xm == 2 || env_xm == 4) && MB % env_xm == 0 && nb % (8 / env_xm) == 0)
    P.xm = env_xm;
  return MB * nb;
}

// kern: 64 x 128 workgroups of four waves with K in S slices; part: S * wgs * 32 KiB
template <typename Kern>
static hipError_t split_launch(Kern kern, size_t lds, BigParams& P, int wgs, int S, float* part, hipStream_t stream) {
  P.S = S;
  P.part = part;
  auto gemm = [&]() -> hipError_t {
    TPPX_PLAN_ONLY(kern, dim3(wgs, S), dim3(256), lds);
    if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds); e != hipSuccess)
      return e;
    kern<<<dim3(wgs, S), dim3(256), lds, stream>>>(P);
    return hipGetLastError();
  };
  if (hipError_t e = gemm(); e != hipSuccess)
    return e;
  auto sum = [&](auto add) -> hipError_t {
    TPPX_PLAN_ONLY(add, dim3(wgs * 4), dim3(64), 0);
    add<<<dim3(wgs * 4), dim3(64), 0, stream>>>(P);
    return hipGetLastError();
  };
  return S == 2 ? sum(side_sum_kernel<4, 4, 2>) : S == 3 ? sum(side_sum_kernel<4, 4, 3>) : S == 4 ? sum(side_sum_kernel<4, 4, 4>)
                                                                                          : sum(side_sum_kernel<4, 4, 6>);
}

// TPPX_TILED_BIG_TILE: 1 = 256 x 256, 2 = 128 x 256, 3 = 128 x 512, 4 = 64 x 128, 6 = 64 x 256 (bf16 weights), from 7 on
// WIDE_FORMS; what is not built for the weights, 5 too, is left to the estimates
constexpr int wide_form(int mt, int nt, int w) {
  for (int i = 0; i < N_WIDE; i++)
    if (WIDE_FORMS[i].mt == mt && WIDE_FORMS[i].nt == nt && WIDE_FORMS[i].w == w)
      return i;
  return -1;
}
template <bool WBF16>
static int forced_tile() {
  constexpr int small = wide_form(4, 2, 4); // MXFP4's 64 x 128
  static_assert(small >= 0 && WIDE_FORMS[small].mxfp4);
  const int t = env_int("TPPX_TILED_BIG_TILE", 0);
  if (!WBF16 && t == 4)
    return TILE_WIDE + small;
  return t >= 1 && t <= 4 ? t - 1 : t == 6 ? TILE_64_256 : t >= 7 && t < 7 + N_WIDE ? TILE_WIDE + t - 7 : -1;
}

// K slices of a tile that TPPX_TILED_BIG_TILE forces: TPPX_TILED_SPLIT's, where the kernels are built and their sums have room
static int forced_slices(bool can, const TiledParams* t, int n, int tile, int64_t part_bytes) {
  const int S = env_int("TPPX_TILED_SPLIT", 1);
  int64_t nb = 0;
  for (int i = 0; i < n; i++)
    nb += (t[i].tiles + tile_cols16(tile) - 1) / tile_cols16(tile);
  const int64_t wgs = (t[0].M + tile_rows(tile) - 1) / tile_rows(tile) * nb;
  return can && (S == 2 || S == 3 || S == 4 || S == 6) && t[0].K / 128 >= 4 * S && wgs * S * slice_bytes(tile) <= part_bytes ? S : 1;
}

// dual: t[0] = gate, t[1] = up (equal shapes, n == 2); y[m][n] = silu(gate) * up goes to t[1].y
hipError_t launch_tiled_mxfp4_group(const TiledParams* t, int n, hipStream_t stream, bool dual, float* part, int64_t part_bytes) {
  if (dual && (n != 2 || t[0].tiles != t[1].tiles || t[0].K != t[1].K || t[0].M != t[1].M || t[0].x != t[1].x))
    return hipErrorInvalidValue;
  int shape = forced_tile<false>(), S = 1;
  if (shape < 0 || shape >= N_TILES || !(MXFP4_COST[shape].b > 0.0))
    shape = cheapest_tile<false>(t, n, dual, part ? part_bytes : 0, &S);
  else if (shape >= TILE_WIDE)
    S = forced_slices(WIDE_FORMS[shape - TILE_WIDE].split && !dual, t, n, shape, part ? part_bytes : 0);
  BigParams P;
  const int wgs = big_params(P, t, n, dual, shape, MXFP4_WEIGHT_BYTES);
  if (shape >= TILE_WIDE) {
    P.S = S;
    P.part = part;
    const hipError_t e = launch_wide_mxfp4(P, shape - TILE_WIDE, wgs, dual, stream);
    return S > 1 && e == hipSuccess ? launch_wide_sum(P, shape - TILE_WIDE, wgs, stream) : e;
  }
  switch (shape) {
  case TILE_128_512:
    return dual ? big_launch<8, true, 1, 8>(P, wgs, stream) : big_launch<8, false, 1, 8>(P, wgs, stream);
  case TILE_128_256:
    return dual ? big_launch<8, true, 1, 4>(P, wgs, stream) : big_launch<8, false, 1, 4>(P, wgs, stream);
  default:
    return dual ? big_launch<8, true, 2, 4>(P, wgs, stream) : big_launch<8, false, 2, 4>(P, wgs, stream);
  }
}

// MXFP4 weights x MXFP8 activations (t[i].xq = quantised activations in operand order, t[i].sa = their scale bytes)
template <int MT, bool DUAL>
static hipError_t fp8_launch(const BigParams& P, int wgs, hipStream_t stream) {
  const size_t ep = 8 * 64 * EP_LD * sizeof(float); // epilogue staging
  const size_t lds = std::max(ep, (size_t)Fp8Geom<MT>::NB * Fp8Geom<MT>::STAGE);
  TPPX_PLAN_ONLY((big_fp8_kernel<MT, DUAL>), dim3(wgs), dim3(512), lds);
  if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(big_fp8_kernel<MT, DUAL>), lds); e != hipSuccess)
    return e;
  big_fp8_kernel<MT, DUAL><<<dim3(wgs), dim3(512), lds, stream>>>(P);
  return hipGetLastError();
}

// dual: the gate/up pair (t[0] = gate, t[1] = up, equal shapes); silu(gate) * up goes to t[1].y
hipError_t launch_tiled_mxfp4_fp8_group(const TiledParams* t, int n, hipStream_t stream, bool dual) {
  if (dual && (n != 2 || t[0].tiles != t[1].tiles || t[0].K != t[1].K || t[0].M != t[1].M || t[0].xq != t[1].xq))
    return hipErrorInvalidValue;
  BigParams P;
  memset(&P, 0, sizeof(P));
  int nb = 0;
  for (int i = 0; i < n; i++) {
    P.seg[i] = t[i];
    P.nb0[i] = nb;
    nb += (t[i].tiles + 15) / 16;
  }
  if (dual) {
    nb = (t[0].tiles + 7) / 8; // 128 output channels (gate and up of each) per workgroup
    P.nb0[1] = nb;
  }
  for (int i = n; i <= TPPX_MAX_SEGS; i++)
    P.nb0[i] = nb;
  P.n_seg = n;
  // 256-row tiles unless 128-row ones fill the last round of workgroups (256 CUs, one workgroup each) better
  const int MB8 = (t[0].M + 255) / 256, MB4 = (t[0].M + 127) / 128;
  auto rounds = [](int wgs) { return (wgs + 255) / 256; };
  const double cost8 = rounds(MB8 * nb), cost4 = 0.5 * 1.15 * rounds(MB4 * nb);
  int mt = cost4 < cost8 ? 4 : 8;
  const int env_mt = env_int("TPPX_FP8_BIG_MT", 0);
  if (env_mt == 4 || env_mt == 8)
    mt = env_mt;
  if (mt == 4)
    return dual ? fp8_launch<4, true>(P, MB4 * nb, stream) : fp8_launch<4, false>(P, MB4 * nb, stream);
  return dual ? fp8_launch<8, true>(P, MB8 * nb, stream) : fp8_launch<8, false>(P, MB8 * nb, stream);
}

hipError_t launch_tiled_mxfp4(const TiledParams& p, hipStream_t stream, float* part, int64_t part_bytes) {
  if (tiled_mxfp4_takes_groups(p))
    return launch_tiled_mxfp4_group(&p, 1, stream, false, part, part_bytes);
  const int MB = (p.M + 127) / 128, NB = (p.tiles + 7) / 8;
  const size_t lds = 2 * 2048 * 16;
  TPPX_PLAN_ONLY(tiled_mxfp4_kernel, dim3(MB * NB), dim3(256), lds);
  if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(tiled_mxfp4_kernel), lds); e != hipSuccess)
    return e;
  tiled_mxfp4_kernel<<<dim3(MB * NB), dim3(256), lds, stream>>>(p);
  return hipGetLastError();
}

// silu(gate) * up over two bf16 tiles that already hold bias + dot (see the gate/up group launch)
__global__ void __launch_bounds__(256)
silu_mul_kernel(const uint16_t* __restrict__ gate, uint16_t* __restrict__ y, int64_t n8) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n8; i += (int64_t)gridDim.x * 256) {
    const uint4 g = reinterpret_cast<const uint4*>(gate)[i];
    const uint4 u = reinterpret_cast<const uint4*>(y)[i];
    const uint32_t gw[4] = {g.x, g.y, g.z, g.w}, uw[4] = {u.x, u.y, u.z, u.w};
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const uint32_t a0 = apply_post_bits(bf16_bits_to_f32(gw[e] & 0xffffu), TPPX_POST_SILU, 0, 0, 1.0f);
      const uint32_t a1 = apply_post_bits(bf16_bits_to_f32(gw[e] >> 16), TPPX_POST_SILU, 0, 0, 1.0f);
      const uint32_t b0 = apply_post_bits(bf16_bits_to_f32(uw[e] & 0xffffu), TPPX_POST_MUL, a0, 0, 1.0f);
      const uint32_t b1 = apply_post_bits(bf16_bits_to_f32(uw[e] >> 16), TPPX_POST_MUL, a1, 0, 1.0f);
      o[e] = (b0 & 0xffffu) | (b1 << 16);
    }
    reinterpret_cast<uint4*>(y)[i] = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

// prompt-sized passes; the kernel's 32-bit offsets want operands below 4 GiB
bool tiled_bf16_takes_groups(const TiledParams& p) {
  return p.M >= big_min_rows() && env_int("TPPX_BF16_BIG", 1) != 0 && (int64_t)p.M * p.K * 2 < ((int64_t)1 << 32) &&
         (int64_t)p.tiles * 32 * p.K < ((int64_t)1 << 32);
}

// n GEMMs over one activation in one launch (fuller last rounds: q/k/v of 4096 channels at 2048 rows 207 -> 167 us), or
// the gate/up pair (dual, as launch_tiled_mxfp4_group: 11008 x 4096 at 2048 rows 355 -> 310 us, 333 rows 148 -> 96)
hipError_t launch_tiled_bf16_group(const TiledParams* t, int n, hipStream_t stream, bool dual, float* part, int64_t part_bytes) {
  if (dual && (n != 2 || t[0].tiles != t[1].tiles || t[0].K != t[1].K || t[0].M != t[1].M || t[0].x != t[1].x))
    return hipErrorInvalidValue;
  int shape = forced_tile<true>(), S = 1;
  if (shape < 0 || shape >= N_TILES || !(BF16_COST[shape].b > 0.0))
    shape = cheapest_tile<true>(t, n, dual, part ? part_bytes : 0, &S);
  BigParams P;
  const int wgs = big_params(P, t, n, dual, shape, 2.0);
  if (shape >= TILE_WIDE)
    return launch_wide_bf16(P, shape - TILE_WIDE, wgs, dual, stream);
  if (S > 1)
    return split_launch(side_split_kernel, SideGeom<4, 4, SIDE_PD>::LDS, P, wgs, S, part, stream);
  switch (shape) {
  case TILE_128_512:
    return dual ? big_bf16_launch<8, true, 1, 8>(P, wgs, stream) : big_bf16_launch<8, false, 1, 8>(P, wgs, stream);
  case TILE_64_128:
    return dual ? big_bf16_launch<2, true, 2, 2>(P, wgs, stream) : big_bf16_launch<2, false, 2, 2>(P, wgs, stream);
  case TILE_64_256:
    return dual ? big_bf16_launch<2, true, 2, 4>(P, wgs, stream) : big_bf16_launch<2, false, 2, 4>(P, wgs, stream);
  case TILE_128_256:
    if (wgs <= 256 && env_int("TPPX_TILED_W8", 1) != 0) // at most one workgroup per CU: eight waves side by side
      return dual ? big_bf16_launch<4, true, 2, 4>(P, wgs, stream) : big_bf16_launch<4, false, 2, 4>(P, wgs, stream);
    return dual ? big_bf16_launch<8, true, 1, 4>(P, wgs, stream) : big_bf16_launch<8, false, 1, 4>(P, wgs, stream);
  default:
    return dual ? big_bf16_launch<8, true, 2, 4>(P, wgs, stream) : big_bf16_launch<8, false, 2, 4>(P, wgs, stream);
  }
}

hipError_t launch_tiled_bf16(const TiledParams& p, hipStream_t stream, float* part, int64_t part_bytes) {
  if (tiled_bf16_takes_groups(p))
    return launch_tiled_bf16_group(&p, 1, stream, false, part, part_bytes);
  const int MB = (p.M + 127) / 128, NB = (p.tiles + 7) / 8;
  const dim3 grid((unsigned)(MB * NB));
  const size_t lds = 2 * 2048 * 16;
  TPPX_PLAN_ONLY(tiled_bf16_kernel, grid, dim3(256), lds);
  hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(tiled_bf16_kernel), lds);
  if (e != hipSuccess)
    return e;
  tiled_bf16_kernel<<<grid, 256, lds, stream>>>(p);
  return hipGetLastError();
}

hipError_t launch_silu_mul(const uint16_t* gate, uint16_t* y, int64_t n, hipStream_t stream) {
  const int64_t n8 = n / 8;
  const unsigned blocks = (unsigned)((n8 + 255) / 256 < 256 * 16 ? (n8 + 255) / 256 : 256 * 16);
  TPPX_PLAN_ONLY(silu_mul_kernel, dim3(blocks), dim3(256), 0);
  silu_mul_kernel<<<dim3(blocks), dim3(256), 0, stream>>>(gate, y, n8);
  return hipGetLastError();
}

bool tiled_qint8_takes_groups(const TiledParams& p) {
  return p.qbs == 256 && p.M >= big_min_rows() && env_int("TPPX_TILED_BIG_QINT8", 1) != 0 &&
         (int64_t)p.M * p.K < ((int64_t)1 << 32) && (int64_t)p.tiles * 16 * p.K < ((int64_t)1 << 32);
}

// K slices (1: whole) of a QINT8 launch of nb blocks of 128 channels: as many as leave one round of 64 x 128 workgroups, for
// K from 6144 on (4096 x 4096: whole 17.0 us, in slices 16.7 .. 20) and slices of 1536 and more.  4096 x 11008, quantizer included:
// 100 rows (64 workgroups, 4 slices) 40.4 -> 25.1 us, 200 rows (128, 2) 42.3 -> 32.0, 333 rows (192) whole 43.3, in slices
// 45 .. 50; 2560 x 10240: 100 rows (40, 6) 33.4 -> 18.2, 333 rows (120, 2) 33.9 -> 27.5; 4096 x 16384 at 100 rows 53.4 -> 32.2.
int qint8_split(int64_t M, int64_t K, int64_t nb, int64_t part_bytes) {
  const int forced = env_int("TPPX_TILED_SPLIT", 1);
  const int64_t wgs = (M + 63) / 64 * nb;
  for (int S : {6, 4, 3, 2})
    if (wgs * S * 32768 <= part_bytes && (forced == S ? K / 256 >= S : forced == 1 && K >= 6144 && K >= 1536 * S && wgs * S <= 256))
      return S;
  return 1;
}

// n GEMMs over the same quantised activations (same M, K, xq, sa) in one launch of the large-M kernel
// dual: t[0] = gate, t[1] = up, as in launch_tiled_mxfp4_group
hipError_t launch_tiled_qint8_group(const TiledParams* t, int n, hipStream_t stream, bool dual, float* part, int64_t part_bytes) {
  if (dual && (n != 2 || t[0].tiles != t[1].tiles || t[0].K != t[1].K || t[0].M != t[1].M || t[0].xq != t[1].xq))
    return hipErrorInvalidValue;
  BigParams P;
  auto go = [&](auto kern, int rows, int waves, size_t lds) -> hipError_t {
    const dim3 grid((unsigned)((t[0].M + rows - 1) / rows * P.nb0[TPPX_MAX_SEGS])), block((unsigned)(waves * 64));
    TPPX_PLAN_ONLY(kern, grid, block, lds);
    if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds); e != hipSuccess)
      return e;
    kern<<<grid, block, lds, stream>>>(P);
    return hipGetLastError();
  };
  auto channel_blocks = [&](int waves) { // of 32 channels per wave; the pair: 16 of each projection
    memset(&P, 0, sizeof(P));
    int nb = 0;
    for (int i = 0; i < n; i++) {
      P.seg[i] = t[i];
      P.nb0[i] = nb;
      if (!dual)
        nb += (t[i].tiles + waves * 2 - 1) / (waves * 2);
      else if (i == 0)
        nb = (t[0].tiles + waves - 1) / waves;
    }
    for (int i = n; i <= TPPX_MAX_SEGS; i++)
      P.nb0[i] = nb;
    P.n_seg = n;
    return nb;
  };
  if (!dual && part) {
    const int nb = channel_blocks(4), S = qint8_split(t[0].M, t[0].K, nb, part_bytes);
    if (S > 1)
      return split_launch(big_qint8_split_kernel, Qint8Geom<4, 4>::LDS, P, (t[0].M + 63) / 64 * nb, S, part, stream);
  }
  const int64_t wgs64 = (int64_t)((t[0].M + 63) / 64) * channel_blocks(8); // workgroups of 64 x 256
  const bool small = env_int("TPPX_TILED_SMALL", 1) != 0;
  if (small && wgs64 <= 128) { // up to half the CUs: 64 x 128, twice as many, one round (4096 x 4096 at 333 rows 19.6 -> 15.0 us, at
                               // 512, exactly a round, 29.9 -> 21.9 with the quantizer; with 129 of 64 x 256 and more, where they
                               // take a second round, 64 x 128 loses: 24.5 against 25.7)
    channel_blocks(4);
    return dual ? go(big_qint8_narrow_dual_kernel, 64, 4, Qint8Geom<4, 4>::LDS) : go(big_qint8_narrow_kernel, 64, 4, Qint8Geom<4, 4>::LDS);
  }
  if (small && wgs64 <= 256) // one round of half-size workgroups (4096 x 4096 at 1000 rows 34.1 -> 24.5 us); two of them
                             // take longer than one of 128 x 256 (12288 x 4096 at 333 rows 39.9 against 32.3)
    return dual ? go(big_qint8_small_dual_kernel, 64, 8, Qint8Geom<4, 8>::LDS) : go(big_qint8_small_kernel, 64, 8, Qint8Geom<4, 8>::LDS);
  return dual ? go(big_qint8_dual_kernel, 128, 8, Qint8Geom<8, 8>::LDS) : go(big_qint8_kernel, 128, 8, Qint8Geom<8, 8>::LDS);
}

hipError_t launch_tiled_qint8(const TiledParams& p, hipStream_t stream, float* part, int64_t part_bytes) {
  if (tiled_qint8_takes_groups(p))
    return launch_tiled_qint8_group(&p, 1, stream, false, part, part_bytes);
  const int MB = (p.M + 127) / 128, NB = (p.tiles + 7) / 8;
  const size_t lds = 2 * 1024 * 16 + 2 * 128 * sizeof(float);
  TPPX_PLAN_ONLY(tiled_qint8_kernel, dim3(MB * NB), dim3(256), lds);
  tiled_qint8_kernel<<<dim3(MB * NB), dim3(256), lds, stream>>>(p);
  return hipGetLastError();
}

} // namespace tppx
