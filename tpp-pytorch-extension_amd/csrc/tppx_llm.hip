// Decode-side operators around the quantized linears of a Llama decoder layer:
// RMSNorm, rotary position embedding, KV-cache append and single-query
// (decode) attention.  All of them are bandwidth bound: one pass over their
// inputs with 128-bit coalesced accesses, reductions inside a wave with DPP,
// fp32 arithmetic, one bf16 rounding where the CPU path stores bf16.
#include <math.h>
#include <string.h>

#include <mutex>

#include "tppx_common.h"
#include "tppx_launch.h"
#include "tppx_norm.h"

namespace tppx {

__device__ __forceinline__ uint4 pack8(const float (&f)[8]) {
  uint32_t d[4];
#pragma unroll
  for (int i = 0; i < 4; i++)
    d[i] = f32x2_to_bf16_bits(f[2 * i], f[2 * i + 1]);
  return make_uint4(d[0], d[1], d[2], d[3]);
}

// ---------------------------------------------------------------------------
// RMSNorm: y = bf16( (x * rsqrt(mean(x^2) + eps)) * gamma ), fp32 inside.
// One workgroup of 256 threads per row; K a multiple of 8.
// ---------------------------------------------------------------------------
template <bool GAMMA_F32>
__global__ void __launch_bounds__(256)
rms_norm_kernel(const uint16_t* __restrict__ x, const void* __restrict__ gamma, uint16_t* __restrict__ y,
                int K, float eps) {
  __shared__ float red[4];
  const int row = blockIdx.x, tid = threadIdx.x;
  const uint4* xr = reinterpret_cast<const uint4*>(x + (int64_t)row * K);
  uint4* yr = reinterpret_cast<uint4*>(y + (int64_t)row * K);
  const int nchunk = K >> 3;
  float ss = 0.f;
  for (int i = tid; i < nchunk; i += 256) {
    float f[8];
    unpack8(xr[i], f);
#pragma unroll
    for (int e = 0; e < 8; e++)
      ss = fmaf(f[e], f[e], ss);
  }
  const float s = rms_scale(ss, red, K, eps);
  for (int i = tid; i < nchunk; i += 256) {
    float f[8], g[8];
    unpack8(xr[i], f); // second read hits L2/L1
    if (GAMMA_F32) {
      const float4* gp = reinterpret_cast<const float4*>(gamma) + 2 * i;
      const float4 g0 = gp[0], g1 = gp[1];
      g[0] = g0.x; g[1] = g0.y; g[2] = g0.z; g[3] = g0.w;
      g[4] = g1.x; g[5] = g1.y; g[6] = g1.z; g[7] = g1.w;
    } else {
      unpack8(reinterpret_cast<const uint4*>(gamma)[i], g);
    }
#pragma unroll
    for (int e = 0; e < 8; e++)
      f[e] = (f[e] * s) * g[e];
    yr[i] = pack8(f);
  }
}

// The same for K up to 8192 (NC = 16-byte chunks per thread, 1 .. 4): row and gamma are requested together and stay in
// registers, so that only one memory latency stands in the launch's way instead of two.  The same sums in the same order.
// Rows of 4096, us: 1 2.5 -> 2.1, 16 2.7 -> 2.3, 333 3.1 -> 2.9, 1000 5.2 -> 4.7, 2048 7.6 -> 6.8 (4.9 TB/s, what a copy moves); of
// 8192, 16 3.5 -> 2.6, 333 5.1 -> 4.2, 2048 15.7 -> 14.5.  Many rows of up to 1024 leave half of the threads or more to ask for the
// last chunk and its gamma again, and those run on the kernel above (f32 gamma, 8192 rows of 256 / 1024: 4.5 / 6.8 there, here
// 5.3 / 7.1; 1000 of 512 2.22, 2.30; 200 of 1024 2.11 either way, 16 2.04, here 1.90).  Waves past the end without requests, behind a
// branch: 2048 rows of 4096 5.6 -> 6.0, 1000 of 8192 5.8 -> 6.4.  2048 rows of 2304 and 2560 with f32 gamma lose 3 %, 1000 and 4096
// of them do not.
template <bool GAMMA_F32, int NC>
__global__ void __launch_bounds__(256)
rms_norm_regs_kernel(const uint16_t* __restrict__ x, const void* __restrict__ gamma, uint16_t* __restrict__ y, int K, float eps) {
  __shared__ float red[4];
  const int row = blockIdx.x, tid = threadIdx.x;
  const uint4* xr = reinterpret_cast<const uint4*>(x + (int64_t)row * K);
  uint4* yr = reinterpret_cast<uint4*>(y + (int64_t)row * K);
  const int nchunk = K >> 3;
  uint4 w[NC];
#pragma unroll
  for (int c = 0; c < NC; c++) // (threads past the end repeat the last chunk: no branch around a load)
    w[c] = xr[min(tid + c * 256, nchunk - 1)];
  float4 g4[NC][2];
  uint4 gb[NC];
#pragma unroll
  for (int c = 0; c < NC; c++) {
    const int i = min(tid + c * 256, nchunk - 1);
    if (GAMMA_F32) {
      g4[c][0] = reinterpret_cast<const float4*>(gamma)[2 * i];
      g4[c][1] = reinterpret_cast<const float4*>(gamma)[2 * i + 1];
    } else {
      gb[c] = reinterpret_cast<const uint4*>(gamma)[i];
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < NC; c++) {
    float f[8];
    unpack8(w[c], f);
    if (tid + c * 256 < nchunk) {
#pragma unroll
      for (int e = 0; e < 8; e++)
        ss = fmaf(f[e], f[e], ss);
    }
  }
  const float s = rms_scale(ss, red, K, eps);
#pragma unroll
  for (int c = 0; c < NC; c++) {
    if (tid + c * 256 >= nchunk)
      break;
    float f[8], g[8];
    unpack8(w[c], f);
    if (GAMMA_F32) {
      g[0] = g4[c][0].x; g[1] = g4[c][0].y; g[2] = g4[c][0].z; g[3] = g4[c][0].w;
      g[4] = g4[c][1].x; g[5] = g4[c][1].y; g[6] = g4[c][1].z; g[7] = g4[c][1].w;
    } else {
      unpack8(gb[c], g);
    }
#pragma unroll
    for (int e = 0; e < 8; e++)
      f[e] = (f[e] * s) * g[e];
    yr[tid + c * 256] = pack8(f);
  }
}

// ---------------------------------------------------------------------------
// LayerNorm (lyr_norm, fused_llm_infer.cpp:254-306; LayerNormFwdTPP,
// xsmm_functors.h:4749-4786): m = mean(x), v = max(mean(x^2) - m^2, 0),
// s = 1 / sqrt(v + eps), y = bf16( (x * s - s * m) * gamma + beta ), fp32 inside.
// One workgroup of 256 threads per row; K a multiple of 8.
// ---------------------------------------------------------------------------
template <bool PARAMS_F32>
__device__ __forceinline__ void load8_param(const void* p, int i, float (&g)[8]) {
  if (PARAMS_F32) {
    const float4* gp = reinterpret_cast<const float4*>(p) + 2 * i;
    const float4 g0 = gp[0], g1 = gp[1];
    g[0] = g0.x; g[1] = g0.y; g[2] = g0.z; g[3] = g0.w;
    g[4] = g1.x; g[5] = g1.y; g[6] = g1.z; g[7] = g1.w;
  } else {
    unpack8(reinterpret_cast<const uint4*>(p)[i], g);
  }
}

template <bool PARAMS_F32>
__global__ void __launch_bounds__(256)
layer_norm_kernel(const uint16_t* __restrict__ x, const void* __restrict__ gamma, const void* __restrict__ beta,
                  uint16_t* __restrict__ y, int K, float eps) {
  __shared__ float red[2][4];
  const int row = blockIdx.x, tid = threadIdx.x;
  const uint4* xr = reinterpret_cast<const uint4*>(x + (int64_t)row * K);
  uint4* yr = reinterpret_cast<uint4*>(y + (int64_t)row * K);
  const int nchunk = K >> 3;
  float sm = 0.f, ss = 0.f;
  for (int i = tid; i < nchunk; i += 256) {
    float f[8];
    unpack8(xr[i], f);
#pragma unroll
    for (int e = 0; e < 8; e++) {
      sm += f[e];
      ss = fmaf(f[e], f[e], ss);
    }
  }
  sm = wave_sum(sm);
  ss = wave_sum(ss);
  if ((tid & 63) == 0) {
    red[0][tid >> 6] = sm;
    red[1][tid >> 6] = ss;
  }
  __syncthreads();
  const float c = 1.0f / (float)K;
  const float m = ((red[0][0] + red[0][1]) + (red[0][2] + red[0][3])) * c;
  float v = ((red[1][0] + red[1][1]) + (red[1][2] + red[1][3])) * c;
  v = fmaxf(v - m * m, 0.0f);
  const float s = 1.0f / sqrtf(v + eps);
  const float b = -1.0f * s * m;
  for (int i = tid; i < nchunk; i += 256) {
    float f[8], g[8], bt[8];
    unpack8(xr[i], f); // second read hits L2/L1
    load8_param<PARAMS_F32>(gamma, i, g);
    load8_param<PARAMS_F32>(beta, i, bt);
#pragma unroll
    for (int e = 0; e < 8; e++)
      f[e] = (f[e] * s + b) * g[e] + bt[e];
    yr[i] = pack8(f);
  }
}

// The same for K up to 8192, row and parameters in registers, as rms_norm_regs_kernel.  Rows of 4096, us: 1 2.7 -> 2.1, 16 2.8 -> 2.4,
// 333 3.4 -> 3.0, 2048 8.5 -> 7.3; of 2560, 2048 6.7 -> 6.2.  (Rows of 1024 and less leave half of the threads idle: 1000 of them 3.0,
// here 3.1, so they stay with the kernel above.)
template <bool PARAMS_F32, int NC>
__global__ void __launch_bounds__(256)
layer_norm_regs_kernel(const uint16_t* __restrict__ x, const void* __restrict__ gamma, const void* __restrict__ beta,
                       uint16_t* __restrict__ y, int K, float eps) {
  __shared__ float red[2][4];
  const int row = blockIdx.x, tid = threadIdx.x;
  const uint4* xr = reinterpret_cast<const uint4*>(x + (int64_t)row * K);
  uint4* yr = reinterpret_cast<uint4*>(y + (int64_t)row * K);
  const int nchunk = K >> 3;
  constexpr int P = PARAMS_F32 ? 2 : 1; // 16-byte words of 8 parameters
  uint4 w[NC], g4[NC][P], b4[NC][P];
#pragma unroll
  for (int c = 0; c < NC; c++) // (threads past the end repeat the last chunk: no branch around a load)
    w[c] = xr[min(tid + c * 256, nchunk - 1)];
#pragma unroll
  for (int c = 0; c < NC; c++)
#pragma unroll
    for (int q = 0; q < P; q++) {
      const int i = min(tid + c * 256, nchunk - 1) * P + q;
      g4[c][q] = reinterpret_cast<const uint4*>(gamma)[i];
      b4[c][q] = reinterpret_cast<const uint4*>(beta)[i];
    }
  auto param = [](const uint4 (&p)[P], float (&f)[8]) {
    if constexpr (PARAMS_F32) {
#pragma unroll
      for (int q = 0; q < 2; q++) {
        f[4 * q] = __uint_as_float(p[q].x);
        f[4 * q + 1] = __uint_as_float(p[q].y);
        f[4 * q + 2] = __uint_as_float(p[q].z);
        f[4 * q + 3] = __uint_as_float(p[q].w);
      }
    } else {
      unpack8(p[0], f);
    }
  };
  float sm = 0.f, ss = 0.f;
#pragma unroll
  for (int c = 0; c < NC; c++) {
    float f[8];
    unpack8(w[c], f);
    if (tid + c * 256 < nchunk) {
#pragma unroll
      for (int e = 0; e < 8; e++) {
        sm += f[e];
        ss = fmaf(f[e], f[e], ss);
      }
    }
  }
  sm = wave_sum(sm);
  ss = wave_sum(ss);
  if ((tid & 63) == 0) {
    red[0][tid >> 6] = sm;
    red[1][tid >> 6] = ss;
  }
  __syncthreads();
  const float c1 = 1.0f / (float)K;
  const float m = ((red[0][0] + red[0][1]) + (red[0][2] + red[0][3])) * c1;
  float v = ((red[1][0] + red[1][1]) + (red[1][2] + red[1][3])) * c1;
  v = fmaxf(v - m * m, 0.0f);
  const float s = 1.0f / sqrtf(v + eps);
  const float b = -1.0f * s * m;
#pragma unroll
  for (int c = 0; c < NC; c++) {
    if (tid + c * 256 >= nchunk)
      break;
    float f[8], g[8], bt[8];
    unpack8(w[c], f);
    param(g4[c], g);
    param(b4[c], bt);
#pragma unroll
    for (int e = 0; e < 8; e++)
      f[e] = (f[e] * s + b) * g[e] + bt[e];
    yr[tid + c * 256] = pack8(f);
  }
}

// ---------------------------------------------------------------------------
// Llama rotary embedding, in place on t [B][S][N][H] (rotate-half pairs
// (h2, HR/2 + h2)), cos/sin table f32 [2][MP][HR], positions i64 [B_pos][S].
// Optionally the rotated key rows and the value rows are also written into
// the KV cache [B][N][Smax][H] at position offset + s (offset read from device
// memory), so that one launch covers rotary(q), rotary(k) and the cache append.
// A workgroup works on one token: its position, the table rows and the cache slot are the same for all of its threads.  A
// thread takes one unit of work: a rotation pair of 8-wide chunks (both halves read and written once; GPT-J: one chunk, its
// pairs lie inside), or one chunk that is only copied into the cache.  What bounds a prompt's launch is the way to memory
// and back (112 MB for 2048 tokens x 3 x 32 heads of 128); numbering the chunks of all tokens in one row of threads took two
// 64-bit divisions per thread (190 vector instructions) and read every chunk twice: 2048 tokens 26.5 -> 19.3 us, 1000 tokens
// 14.6 -> 10.2, 2048 x (64 + 2 x 8) heads 22.8 -> 14.8.
// ---------------------------------------------------------------------------
struct RotaryParams {
  uint16_t* q;         // [B][S][Nq][H] or null
  uint16_t* k;         // [B][S][Nkv][H] or null
  const uint16_t* v;   // [B][S][Nkv][H] or null (append only)
  uint16_t* kc;        // [B][Nkv][Smax][H] or null
  uint16_t* vc;
  const float* emb;    // [2][MP][HR] or null (append without rotation)
  const int64_t* pos;  // [B_pos][S]
  const int32_t* offset; // device scalar: cache length before this append
  int B, S, Nq, Nkv, H, MP, HR, B_pos, Smax;
  int gptj;            // 1: GPT-J pairs (h, h + 1) and a sin | cos table f32 [MP][HR] (fused_llm_infer.cpp:150-205)
  int rot, uq, uk, uv; // units of a head: rotations, then all of a query's, a key's and a value's
  uint32_t mq, mk, mv; // ceil(2^32 / units), for the division by them
};

__global__ void __launch_bounds__(256)
rotary_append_kernel(const RotaryParams p) {
  const int tok = blockIdx.x, b = tok / p.S, s = tok - b * p.S; // (uniform, as everything up to the unit)
  const int nq = p.q ? p.Nq * p.uq : 0, nk = p.k ? p.Nkv * p.uk : 0, nv = p.v && p.vc ? p.Nkv * p.uv : 0;
  const int64_t pp = p.pos[(int64_t)(p.B_pos == 1 ? 0 : b) * p.S + s];
  const bool rotate = p.emb && pp >= 0 && pp < p.MP; // positions outside the table are left unrotated
  const int at = p.kc || p.vc ? *p.offset + s : 0;
  const bool room = at < p.Smax;
  int i = blockIdx.y * 256 + threadIdx.x;
  if (i >= nq + nk + nv)
    return;
  if (i >= nq + nk) { // value rows: plain copy into the cache
    i -= nq + nk;
    const int n = p.uv == 1 ? i : (int)__umulhi((uint32_t)i, p.mv), c = i - n * p.uv;
    if (room)
      reinterpret_cast<uint4*>(p.vc + (((int64_t)b * p.Nkv + n) * p.Smax + at) * p.H)[c] =
          reinterpret_cast<const uint4*>(p.v + ((int64_t)tok * p.Nkv + n) * p.H)[c];
    return;
  }
  const bool is_k = i >= nq;
  if (is_k)
    i -= nq;
  const int units = is_k ? p.uk : p.uq;
  const int n = units == 1 ? i : (int)__umulhi((uint32_t)i, is_k ? p.mk : p.mq), u = i - n * units;
  uint4* row = reinterpret_cast<uint4*>(is_k ? p.k + ((int64_t)tok * p.Nkv + n) * p.H : p.q + ((int64_t)tok * p.Nq + n) * p.H);
  uint4* crow = is_k && p.kc && room ? reinterpret_cast<uint4*>(p.kc + (((int64_t)b * p.Nkv + n) * p.Smax + at) * p.H) : nullptr;
  if (u >= p.rot) { // behind the rotated dims: copied only
    const int c = (p.HR >> 3) + u - p.rot;
    if (crow)
      crow[c] = row[c];
    return;
  }
  if (p.gptj) { // a chunk of 8 holds four whole pairs (h, h + 1); sin at [p][h / 2], cos at [p][HR / 2 + h / 2]
    uint4 w = row[u];
    if (rotate) {
      float a[8], r[8];
      unpack8(w, a);
      const float* sn = p.emb + pp * p.HR + u * 4;
      const float* cs = sn + (p.HR >> 1);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        r[2 * e] = rotate_first(a[2 * e], a[2 * e + 1], cs[e], sn[e]);
        r[2 * e + 1] = rotate_second(a[2 * e], a[2 * e + 1], cs[e], sn[e]);
      }
      w = pack8(r);
      row[u] = w;
    }
    if (crow)
      crow[u] = w;
    return;
  }
  uint4 w0 = row[u], w1 = row[u + p.rot]; // chunk u of the first half and its partner
  if (rotate) {
    float a[8], o[8], r0[8], r1[8];
    unpack8(w0, a);
    unpack8(w1, o);
    const float* cs = p.emb + pp * p.HR + u * 8;
    const float* sn = p.emb + ((int64_t)p.MP + pp) * p.HR + u * 8;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      r0[e] = rotate_first(a[e], o[e], cs[e], sn[e]);
      r1[e] = rotate_second(a[e], o[e], cs[e], sn[e]);
    }
    w0 = pack8(r0);
    w1 = pack8(r1);
    row[u] = w0;
    row[u + p.rot] = w1;
  }
  if (crow) {
    crow[u] = w0;
    crow[u + p.rot] = w1;
  }
}

// ---------------------------------------------------------------------------
// Decode attention (one query token per sequence), head size 128, cache
// [B][Nkv][Smax][128] bf16.  Grid (B*Nq, splits); split y takes the trips
// y, y + splits, ... of the key range, whose length is a device scalar.  Two
// kernels with a workgroup per query head share the split merge (attn_finish):
//   attn_decode_kernel       4 waves, a wave instruction reads 4 keys (lane =
//     key l>>4, 16-byte chunk l&15), 64 keys per trip with the next trip
//     requested ahead; every 16-lane row keeps its own running (max, sum, 8
//     output dims per lane), merged at the end through LDS: the long loops of
//     larger batches;
//   attn_decode_wide_kernel  128 keys per trip on the packed bf16 dot
//     instruction: the one- or two-trip workgroups of small batches, where
//     the arithmetic above costs more than the cache stream.
// Scores: fp32 dot * 1/sqrt(H) + mask; probabilities are rounded to bf16
// before they multiply V (as the CPU path stores them), sums and the output
// accumulate in fp32.
// A third, attn_decode_group_kernel below, takes several query heads per K/V head.
// ---------------------------------------------------------------------------
struct AttnParams {
  const uint16_t* q;    // [B][Nq][128]
  const uint16_t* kc;   // [B][Nkv][Smax][128]
  const uint16_t* vc;
  const uint16_t* mask; // bf16 [B][mask_ld] additive, or null
  const int32_t* kv_len; // device scalar; valid keys = *kv_len + kv_len_add
  int kv_len_add;
  uint16_t* out;        // [B][Nq][128]
  float* part;          // [B*Nq][splits][130]
  int B, Nq, Nkv, Smax, mask_ld, splits;
  unsigned int* counters; // the caller's arrival counters, or null:
  int ticket0;          // >= 0: first of the library's (the last split to arrive merges); < 0: second kernel
  float scale;
  // ROT: the query and the step's new key / value arrive unrotated and not yet in the cache
  const uint16_t* k_new; // [B][Nkv][128]
  const uint16_t* v_new; // [B][Nkv][128]
  const float* emb;      // f32 [2][MP][128] cos / sin
  const int64_t* pos;    // i64 [B_pos] position of the new token
  int MP, B_pos;
};

// Arrival counters of the split launches, one per (sequence, head): zero between launches (the counting
// instruction wraps on the last arrival).  A caller that gives counters with its workspace orders its launches on both
// alike.  Without them a launch of 128-wide heads takes a window of the library's, handed out in rotation by the host:
// windows come round again after 4096 counters, so launches queued on other streams, and graphs replayed beside eager
// work, can hold the same one.
// The counters of a launch are all hit within a microsecond or two; side by side they would queue up at the atomic
// unit of one memory channel, so each one has 256 bytes to itself.
constexpr int ATTN_TICKETS = 4096;
constexpr int ATTN_TICKET_STRIDE = 64; // in counters
__device__ unsigned int attn_tickets[ATTN_TICKETS * ATTN_TICKET_STRIDE];

__global__ void attn_clear_tickets_kernel(int first, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n)
    attn_tickets[(first + i) * ATTN_TICKET_STRIDE] = 0;
}

// Counts an arrival of group `i` of a launch; true for the last of `splits`.
__device__ __forceinline__ bool attn_arrive(unsigned int* counters, int ticket0, int i, int splits) {
  unsigned int* c = counters ? counters : attn_tickets + (int64_t)ticket0 * ATTN_TICKET_STRIDE;
  const unsigned int last = (unsigned int)splits - 1;
  return atomicInc(c + (int64_t)i * ATTN_TICKET_STRIDE, last) == last;
}

__device__ __forceinline__ uint4 as_uint4(const i32x4& v) {
  return make_uint4((uint32_t)v[0], (uint32_t)v[1], (uint32_t)v[2], (uint32_t)v[3]);
}

// Shared end of the single-query kernels.  Threads tid < 128 hold output dimension tid of this workgroup's state: the
// running max M, the sum Ls and the unnormalised output o.  One split: normalise and store.  Several: store the state;
// with arrival counters the split that arrives last merges all of them inside the launch.  hold(): right before the arrival.
template <typename Hold>
__device__ __forceinline__ void attn_finish(const AttnParams& p, int bh, int tid, float M, float Ls, float o, Hold&& hold) {
  if (tid < 128) {
    if (p.splits == 1) {
      p.out[(int64_t)bh * 128 + tid] = (uint16_t)f32_to_bf16_bits(Ls > 0.f ? o / Ls : 0.f);
    } else if (p.ticket0 < 0 && !p.counters) {
      float* dst = p.part + ((int64_t)bh * p.splits + blockIdx.y) * 130;
      dst[2 + tid] = o;
      if (tid == 0) {
        dst[0] = M;
        dst[1] = Ls;
      }
    } else {
      // device-scope atomic stores: written through to the level all XCDs share, no cache write-back needed
      float* dst = p.part + ((int64_t)bh * p.splits + blockIdx.y) * 130;
      __hip_atomic_store(dst + 2 + tid, o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (tid == 0) {
        __hip_atomic_store(dst, M, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(dst + 1, Ls, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  if (p.splits == 1 || (p.ticket0 < 0 && !p.counters))
    return;
  // The split that arrives last merges all of them, in split order (the same sums whichever split that is).
  // Order: every thread waits until its own stores above have been acknowledged (vmcnt counts stores on this
  // target; a workgroup barrier by itself does not wait for the global stores of the other waves), then the
  // barrier, then the ticket, then the device-scope loads of the other splits' results.  Nobody waits for anybody.
  __shared__ int arrived_last;
  hold();
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0)
    arrived_last = attn_arrive(p.counters, p.ticket0, bh, p.splits);
  __syncthreads();
  if (!arrived_last || tid >= 128)
    return;
  const float* src = p.part + (int64_t)bh * p.splits * 130;
  float pm[32], pl[32], po[32]; // every load in flight at once (at most 32 splits)
#pragma unroll
  for (int i = 0; i < 32; i++) {
    pm[i] = -3.0e38f;
    pl[i] = po[i] = 0.f;
    if (i < p.splits) {
      pm[i] = __hip_atomic_load(src + i * 130, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      pl[i] = __hip_atomic_load(src + i * 130 + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      po[i] = __hip_atomic_load(src + i * 130 + 2 + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  M = -3.0e38f;
#pragma unroll
  for (int i = 0; i < 32; i++)
    if (i < p.splits)
      M = fmaxf(M, pm[i]);
  Ls = 0.f;
  o = 0.f;
#pragma unroll
  for (int i = 0; i < 32; i++)
    if (i < p.splits) {
      const float w = __expf(pm[i] - M);
      Ls = fmaf(w, pl[i], Ls);
      o = fmaf(w, po[i], o);
    }
  p.out[(int64_t)bh * 128 + tid] = (uint16_t)f32_to_bf16_bits(Ls > 0.f ? o / Ls : 0.f);
}


// ROT: the launch also does what the rotary + append launch did before it (fused_llm_infer.cpp:1252-1253 and
// LayerCache::update, attn.h:198-222): q and the new key arrive unrotated, every workgroup rotates its query, the
// key / value of the new token (cache position *kv_len) are taken from registers wherever that position is read,
// and one workgroup per KV head writes them into the cache.  Rotated values are rounded to bf16 first, as stored.
template <bool ROT>
__global__ void __launch_bounds__(256)
attn_decode_kernel(const AttnParams p) {
  __shared__ float sm[16], sl[16];
  __shared__ float sacc[16][128];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, c = lane & 15;
  const int bh = blockIdx.x, b = bh / p.Nq, hq = bh - b * p.Nq;
  const int hk = hq / (p.Nq / p.Nkv);
  const uint4* kb = reinterpret_cast<const uint4*>(p.kc + ((int64_t)b * p.Nkv + hk) * p.Smax * 128) + c;
  const uint4* vb = reinterpret_cast<const uint4*>(p.vc + ((int64_t)b * p.Nkv + hk) * p.Smax * 128) + c;
  constexpr int NU = 4; // keys per DPP row and trip (8 measured no better)
  // One trip = 64 keys per workgroup, 4 * NU per wave (NU per DPP row).  Split y takes trips y, y + splits, ...: the
  // splits differ by at most one trip whatever the length is, and the first trip's rows do not depend on the length
  // (a device scalar), so they are requested here, before anything else is read: the cache stream starts with the
  // launch.  Rows are clamped to the cache's last row; a trip past the end is read and never used (at most one per
  // workgroup).  Inside the loop the next trip is requested before this trip's arithmetic.
  i32x4 kw[NU], vw[NU], kn[NU], vn[NU];
  auto load_kv = [&](int base, i32x4 (&kd)[NU], i32x4 (&vd)[NU]) {
#pragma unroll
    for (int u = 0; u < NU; u++) {
      const int kk = min(base + u * 4 + g, p.Smax - 1);
      kd[u] = __builtin_nontemporal_load(reinterpret_cast<const i32x4*>(kb + (int64_t)kk * 16));
      vd[u] = __builtin_nontemporal_load(reinterpret_cast<const i32x4*>(vb + (int64_t)kk * 16));
    }
  };
  load_kv(blockIdx.y * 64 + wave * (4 * NU), kw, vw);
  const int len0 = *p.kv_len;
  const int L = max(0, min(len0 + p.kv_len_add, p.Smax));
  const int nk = (ROT && len0 >= 0 && len0 < p.Smax) ? len0 : -1; // cache position of the new token
  const int trips = (L + 63) >> 6;
  // the split whose trips contain the new token's position (wave-uniform)
  const bool has_new = ROT && nk >= 0 && nk < L && ((nk >> 6) % p.splits) == (int)blockIdx.y;

  float qf[8];
  i32x4 knew = {0, 0, 0, 0}, vnew = {0, 0, 0, 0};
  if (!ROT) {
    unpack8(reinterpret_cast<const uint4*>(p.q + (int64_t)bh * 128)[c], qf);
  } else {
    // chunk c holds first halves (c < 8) or second halves of the rotation pairs (h2, 64 + h2); partner chunk c ^ 8
    const bool first = c < 8;
    const int64_t pp = p.pos[p.B_pos == 1 ? 0 : b];
    const bool rot = p.emb != nullptr && pp >= 0 && pp < p.MP;
    float cs[8], sn[8];
#pragma unroll
    for (int e = 0; e < 8; e++)
      cs[e] = sn[e] = 0.f;
    if (rot) { // rows of 128 floats, 8 per chunk: 32-byte aligned
      const f32x4* cp = reinterpret_cast<const f32x4*>(p.emb + pp * 128 + (c & 7) * 8);
      const f32x4* sp = reinterpret_cast<const f32x4*>(p.emb + ((int64_t)p.MP + pp) * 128 + (c & 7) * 8);
      const f32x4 c0 = cp[0], c1 = cp[1], s0 = sp[0], s1 = sp[1];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        cs[e] = c0[e];
        cs[4 + e] = c1[e];
        sn[e] = s0[e];
        sn[4 + e] = s1[e];
      }
    }
    auto rotate = [&](const uint16_t* row, float (&r)[8]) -> uint4 {
      const uint4 w = reinterpret_cast<const uint4*>(row)[c];
      if (!rot) {
        unpack8(w, r);
        return w;
      }
      const uint4 wo = reinterpret_cast<const uint4*>(row)[c ^ 8];
      float a[8], o[8];
      unpack8(w, a);
      unpack8(wo, o);
#pragma unroll
      for (int e = 0; e < 8; e++)
        r[e] = first ? rotate_first(a[e], o[e], cs[e], sn[e]) : rotate_second(o[e], a[e], cs[e], sn[e]);
      const uint4 out = pack8(r);
      unpack8(out, r); // the rotated row is a bf16 tensor
      return out;
    };
    rotate(p.q + (int64_t)bh * 128, qf);
    if (has_new) { // only the split that reads the new token's position needs its key and value
      float kr[8];
      const uint4 kw4 = rotate(p.k_new + ((int64_t)b * p.Nkv + hk) * 128, kr);
      knew = i32x4{(int)kw4.x, (int)kw4.y, (int)kw4.z, (int)kw4.w};
      vnew = *reinterpret_cast<const i32x4*>(p.v_new + ((int64_t)b * p.Nkv + hk) * 128 + c * 8);
      // one workgroup per KV head appends: the first query head of the group
      if (hq == hk * (p.Nq / p.Nkv) && tid < 16) {
        const int64_t o = (((int64_t)b * p.Nkv + hk) * p.Smax + nk) * 128 + c * 8;
        *reinterpret_cast<i32x4*>(const_cast<uint16_t*>(p.kc) + o) = knew;
        *reinterpret_cast<i32x4*>(const_cast<uint16_t*>(p.vc) + o) = vnew;
      }
    }
  }
#pragma unroll
  for (int e = 0; e < 8; e++)
    qf[e] *= p.scale;
  const uint16_t* mrow = p.mask ? p.mask + (int64_t)b * p.mask_ld : nullptr;

  float m = -3.0e38f, l = 0.f, acc[8];
#pragma unroll
  for (int e = 0; e < 8; e++)
    acc[e] = 0.f;
  // the new token is not in the cache yet (or is being written by another workgroup right now): wherever its
  // position was read, the registers replace what the load returned
  auto patch_new = [&](int base, i32x4 (&kd)[NU], i32x4 (&vd)[NU]) {
    if (has_new) {
#pragma unroll
      for (int u = 0; u < NU; u++)
        if (base + u * 4 + g == nk) {
          kd[u] = knew;
          vd[u] = vnew;
        }
    }
  };
  patch_new(blockIdx.y * 64 + wave * (4 * NU), kw, vw);
  for (int t = blockIdx.y; t < trips; t += p.splits) {
    const int base = t * 64 + wave * (4 * NU);
    load_kv(base + p.splits * 64, kn, vn); // unconditional (rows are clamped): a branch here would drain the queue
    patch_new(base + p.splits * 64, kn, vn);
    int key[NU];
#pragma unroll
    for (int u = 0; u < NU; u++)
      key[u] = base + u * 4 + g;
    float sc[NU];
#pragma unroll
    for (int u = 0; u < NU; u++) {
      float kf[8];
      unpack8(as_uint4(kw[u]), kf);
      float d = 0.f;
#pragma unroll
      for (int e = 0; e < 8; e++)
        d = fmaf(qf[e], kf[e], d);
      d = row16_sum(d);
      if (mrow && key[u] < p.mask_ld && key[u] < L)
        d += bf16_bits_to_f32(mrow[key[u]]);
      sc[u] = key[u] < L ? d : -3.0e38f;
    }
    if (t * 64 + 64 > L) { // the last trip only (wave-uniform): rows past the end may hold anything, NaN included
#pragma unroll
      for (int u = 0; u < NU; u++)
        if (key[u] >= L)
          vw[u] = i32x4{0, 0, 0, 0};
    }
    float mn = m;
#pragma unroll
    for (int u = 0; u < NU; u++)
      mn = fmaxf(mn, sc[u]);
    const float alpha = __expf(m - mn);
    l *= alpha;
#pragma unroll
    for (int e = 0; e < 8; e++)
      acc[e] *= alpha;
#pragma unroll
    for (int u = 0; u < NU; u++) {
      const float pr = key[u] < L ? __expf(sc[u] - mn) : 0.f;
      l += pr;
      const float pb = round_bf16(pr);
      float vf[8];
      unpack8(as_uint4(vw[u]), vf);
#pragma unroll
      for (int e = 0; e < 8; e++)
        acc[e] = fmaf(pb, vf[e], acc[e]);
    }
    m = mn;
#pragma unroll
    for (int u = 0; u < NU; u++) {
      kw[u] = kn[u];
      vw[u] = vn[u];
    }
  }
  // merge the 16 (wave, row) states
  const int st = wave * 4 + g;
  if (c == 0) {
    sm[st] = m;
    sl[st] = l;
  }
#pragma unroll
  for (int e = 0; e < 8; e++)
    sacc[st][c * 8 + e] = acc[e];
  __syncthreads();
  float M = -3.0e38f, Ls = 0.f, o = 0.f;
  if (tid < 128) {
    M = sm[0];
#pragma unroll
    for (int i = 1; i < 16; i++)
      M = fmaxf(M, sm[i]);
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const float w = __expf(sm[i] - M);
      Ls = fmaf(w, sl[i], Ls);
      o = fmaf(w, sacc[i][tid], o);
    }
  }
  attn_finish(p, bh, tid, M, Ls, o, [] {});
}

// ---------------------------------------------------------------------------
// The same single-query attention for few trips per workgroup: at batch 1 the
// cache of one head is a few hundred KB, every workgroup makes one or two
// trips, and the vector arithmetic of the kernel above (bf16 unpacking, one
// multiply-add per element, a 16-lane reduction per 4 keys) costs more than
// the cache stream.  Here a lane owns an eighth (16 dims, chunks j*8 + q8) of
// FOUR keys per trip -- a wave instruction reads 8 whole rows, a wave covers
// 32 keys, the workgroup 128 -- and:
//   * q . k runs on v_dot2c_f32_bf16 (two bf16 products per instruction, no
//     unpacking), followed by an 8-lane reduction;
//   * the wave shares one running max (one exp per key and lane);
//   * p . v pairs the lane's keys: (v_a[e], v_b[e]) . (p_a, p_b), again on
//     the dot instruction, the pair assembled by one byte permute;
//   * the query is rotated once per workgroup (wave 0, one rotation pair per
//     lane) and handed to the lanes through LDS; the new key only in the
//     split that reads its position.
// The per-lane outputs (16 dims, partial over the lane's keys) are added up
// through LDS at the end.  The first trip's K and V rows (16 KB per wave) are
// requested before anything else, a later trip's K rows once this trip's scores
// have freed their registers and its V rows behind this trip's sums, so that a
// workgroup of many trips never stands without requests; in those lanes past the
// length share its last row (a last trip of one key fetched 128), while the first
// is requested before the length is known, up to the cache's end.  Against requests at
// the start of a trip, rows up to the cache's end, 32 heads: 16 sequences of 2048
// keys 90 -> 85 us (6.3 TB/s, ends of the launch included), a step of four layers
// of 32 of 1300 741 -> 707, 2 of 2048 229 -> 222, 1 of 2000 201 -> 199.
// ---------------------------------------------------------------------------
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
__device__ __forceinline__ float dot2_bf16(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, a), __builtin_bit_cast(bf16x2_t, b), c, false);
}
__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, dpp_mov<0xB1>(v));
  v = fmaxf(v, dpp_mov<0x4E>(v));
  v = fmaxf(v, dpp_mov<0x141>(v));
  v = fmaxf(v, dpp_mov<0x140>(v));
  const float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0));
  const float b = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16));
  const float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
  const float d = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 48));
  return fmaxf(fmaxf(a, b), fmaxf(c, d));
}

constexpr int ATTN_WIDE_KEYS = 128; // keys per workgroup and trip

template <bool ROT>
__global__ void __launch_bounds__(256, 4) // four workgroups per CU: at most 128 registers
attn_decode_wide_kernel(const AttnParams p) {
  __shared__ __align__(16) uint16_t q_s[128], k_s[128];
  __shared__ float sm[4], sl[4];
  __shared__ __align__(16) float sacc[4][8][132];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kq = lane >> 3, q8 = lane & 7;
  const int bh = blockIdx.x, b = bh / p.Nq, hq = bh - b * p.Nq;
  const int hk = hq / (p.Nq / p.Nkv);
  const int S = p.splits;
  const char* kb = reinterpret_cast<const char*>(p.kc + ((int64_t)b * p.Nkv + hk) * p.Smax * 128) + q8 * 16;
  const char* vb = reinterpret_cast<const char*>(p.vc + ((int64_t)b * p.Nkv + hk) * p.Smax * 128) + q8 * 16;
  // key set s of a trip: keys base + s*8 + kq; register [s][j] holds dims (j*8 + q8)*8 .. +7 as four bf16 pairs
  i32x4 kr[4][2], vr[4][2];
  auto load_rows = [&](const char* src, int base, int end, i32x4 (&dst)[4][2]) {
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const int key = min(base + s * 8 + kq, end - 1); // past the end: read, never used
#pragma unroll
      for (int j = 0; j < 2; j++)
        dst[s][j] = __builtin_nontemporal_load(reinterpret_cast<const i32x4*>(src + (int64_t)key * 256 + j * 128));
    }
  };
  // A wave's loads return in the order of their issue.  Wave 0 prepares the query (and the new key): it asks for
  // those few values first, so that they do not queue behind its 16 KB of rows, and rotates them while the rows of
  // all four waves are on their way.  Lane i owns the rotation pair (i, 64 + i).
  i32x4 qp[2];
  float qx1 = 0.f, qx2 = 0.f, kx1 = 0.f, kx2 = 0.f, cs = 1.f, sn = 0.f;
  bool rot = false;
  if (!ROT) {
#pragma unroll
    for (int j = 0; j < 2; j++)
      qp[j] = reinterpret_cast<const i32x4*>(p.q + (int64_t)bh * 128)[j * 8 + q8];
  } else if (wave == 0) {
    const uint16_t* qrow = p.q + (int64_t)bh * 128;
    const uint16_t* krow = p.k_new + ((int64_t)b * p.Nkv + hk) * 128;
    qx1 = bf16_bits_to_f32(qrow[lane]);
    qx2 = bf16_bits_to_f32(qrow[64 + lane]);
    kx1 = bf16_bits_to_f32(krow[lane]);
    kx2 = bf16_bits_to_f32(krow[64 + lane]);
    const int64_t pp = p.pos[p.B_pos == 1 ? 0 : b];
    rot = p.emb != nullptr && pp >= 0 && pp < p.MP; // positions outside the table are left unrotated
    if (rot) {
      cs = p.emb[pp * 128 + lane];
      sn = p.emb[((int64_t)p.MP + pp) * 128 + lane];
    }
  }
  load_rows(kb, blockIdx.y * ATTN_WIDE_KEYS + wave * 32, p.Smax, kr);
  load_rows(vb, blockIdx.y * ATTN_WIDE_KEYS + wave * 32, p.Smax, vr);
  const int len0 = *p.kv_len;
  const int L = max(0, min(len0 + p.kv_len_add, p.Smax));
  const int nk = (ROT && len0 >= 0 && len0 < p.Smax) ? len0 : -1; // cache position of the new token
  const int trips = (L + ATTN_WIDE_KEYS - 1) / ATTN_WIDE_KEYS;
  // the split whose trips contain the new token's position (uniform over the workgroup)
  const bool has_new = ROT && nk >= 0 && nk < L && ((nk / ATTN_WIDE_KEYS) % S) == (int)blockIdx.y;

  if (ROT) {
    if (wave == 0) {
      q_s[lane] = (uint16_t)f32_to_bf16_bits(rot ? rotate_first(qx1, qx2, cs, sn) : qx1);
      q_s[64 + lane] = (uint16_t)f32_to_bf16_bits(rot ? rotate_second(qx1, qx2, cs, sn) : qx2);
      if (has_new) {
        k_s[lane] = (uint16_t)f32_to_bf16_bits(rot ? rotate_first(kx1, kx2, cs, sn) : kx1);
        k_s[64 + lane] = (uint16_t)f32_to_bf16_bits(rot ? rotate_second(kx1, kx2, cs, sn) : kx2);
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 2; j++)
      qp[j] = reinterpret_cast<const i32x4*>(q_s)[j * 8 + q8];
    // one workgroup per KV head appends: the first query head of the group, in the split that reads the position
    if (has_new && hq == hk * (p.Nq / p.Nkv) && tid < 16) {
      const int64_t o = (((int64_t)b * p.Nkv + hk) * p.Smax + nk) * 128 + tid * 8;
      *reinterpret_cast<i32x4*>(const_cast<uint16_t*>(p.kc) + o) = reinterpret_cast<const i32x4*>(k_s)[tid];
      *reinterpret_cast<i32x4*>(const_cast<uint16_t*>(p.vc) + o) =
          *reinterpret_cast<const i32x4*>(p.v_new + ((int64_t)b * p.Nkv + hk) * 128 + tid * 8);
    }
  }
  const uint16_t* mrow = p.mask ? p.mask + (int64_t)b * p.mask_ld : nullptr;

  float m = -3.0e38f, l = 0.f; // m is the same in every lane of the wave
  float acc[16];
#pragma unroll
  for (int e = 0; e < 16; e++)
    acc[e] = 0.f;
  // a trip in two halves: the scores of its keys, which frees the K registers, then the sums, which free the V registers
  float sc[4];
  auto scores = [&](int base) {
    if (has_new && nk >= base && nk < base + 32) {
      // the new token is not in the cache yet (or is being written right now): its lanes take the rotated key from
      // LDS and the value from the step's input
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const i32x4 kv = reinterpret_cast<const i32x4*>(k_s)[j * 8 + q8];
        const i32x4 vv = *reinterpret_cast<const i32x4*>(p.v_new + ((int64_t)b * p.Nkv + hk) * 128 + (j * 8 + q8) * 8);
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
          for (int r = 0; r < 4; r++) { // (selects: stores under a condition end up indexed, and the rows in scratch memory)
            kr[s][j][r] = nk == base + s * 8 + kq ? kv[r] : kr[s][j][r];
            vr[s][j][r] = nk == base + s * 8 + kq ? vv[r] : vr[s][j][r];
          }
      }
    }
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const int key = base + s * 8 + kq;
      float d = 0.f;
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          d = dot2_bf16((uint32_t)kr[s][j][r], (uint32_t)qp[j][r], d);
      d += dpp_mov<0xB1>(d);  // the eight parts of the key: quad_perm [1,0,3,2], [2,3,0,1], row_half_mirror
      d += dpp_mov<0x4E>(d);
      d += dpp_mov<0x141>(d);
      d *= p.scale;
      if (mrow && key < p.mask_ld && key < L)
        d += bf16_bits_to_f32(mrow[key]);
      sc[s] = key < L ? d : -3.0e38f;
    }
  };
  auto sums = [&](int base) {
    const float mn = fmaxf(m, wave_max(fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3]))));
    if (mn > m) { // wave-uniform; rare once the first trips have passed
      const float alpha = __expf(m - mn);
      l *= alpha;
#pragma unroll
      for (int e = 0; e < 16; e++)
        acc[e] *= alpha;
      m = mn;
    }
    uint32_t pk[2] = {0, 0}; // probabilities of the key pairs (0, 1) and (2, 3) as packed bf16
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const int key = base + s * 8 + kq;
      const float pr = key < L ? __expf(sc[s] - m) : 0.f;
      l += pr;
      pk[s >> 1] |= f32_to_bf16_bits(pr) << (16 * (s & 1));
      if (base + 32 > L && key >= L) { // rows past the end may hold anything, NaN included
#pragma unroll
        for (int j = 0; j < 2; j++)
          vr[s][j] = i32x4{0, 0, 0, 0};
      }
    }
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const uint32_t va = (uint32_t)vr[2 * h][j][r], vb2 = (uint32_t)vr[2 * h + 1][j][r];
          // v_perm_b32: selector bytes 0..3 pick from the second operand, 4..7 from the first
          const uint32_t lo = __builtin_amdgcn_perm(vb2, va, 0x05040100u); // (a.dim 2r, b.dim 2r)
          const uint32_t hi = __builtin_amdgcn_perm(vb2, va, 0x07060302u); // (a.dim 2r+1, b.dim 2r+1)
          acc[j * 8 + 2 * r] = dot2_bf16(lo, pk[h], acc[j * 8 + 2 * r]);
          acc[j * 8 + 2 * r + 1] = dot2_bf16(hi, pk[h], acc[j * 8 + 2 * r + 1]);
        }
  };
  int t = blockIdx.y;
  for (; t + S < trips; t += S) { // (the last trip on its own: a load under a condition would make every wait one for all)
    const int base = t * ATTN_WIDE_KEYS + wave * 32, next = (t + S) * ATTN_WIDE_KEYS + wave * 32;
    scores(base);
    __builtin_amdgcn_sched_barrier(0);
    load_rows(kb, next, L, kr); // lanes past the end share the last row: a trip of one key fetches one
    __builtin_amdgcn_sched_barrier(0);
    sums(base);
    __builtin_amdgcn_sched_barrier(0);
    load_rows(vb, next, L, vr);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (t < trips) {
    scores(t * ATTN_WIDE_KEYS + wave * 32);
    sums(t * ATTN_WIDE_KEYS + wave * 32);
  }
  // add up the lanes' partial outputs: [wave][kq][dim], rows padded against bank conflicts
#pragma unroll
  for (int j = 0; j < 2; j++) {
    float* dst = &sacc[wave][kq][(j * 8 + q8) * 8];
    *reinterpret_cast<f32x4*>(dst) = f32x4{acc[j * 8], acc[j * 8 + 1], acc[j * 8 + 2], acc[j * 8 + 3]};
    *reinterpret_cast<f32x4*>(dst + 4) = f32x4{acc[j * 8 + 4], acc[j * 8 + 5], acc[j * 8 + 6], acc[j * 8 + 7]};
  }
  // every key's l sits in the eight lanes of the key: the wave sum counts it eight times (exactly, a power of two)
  const float lw = wave_sum(l) * 0.125f;
  if (lane == 0) {
    sm[wave] = m;
    sl[wave] = lw;
  }
  __syncthreads();
  float M = -3.0e38f, Ls = 0.f, o = 0.f;
  if (tid < 128) {
    M = fmaxf(fmaxf(sm[0], sm[1]), fmaxf(sm[2], sm[3]));
#pragma unroll
    for (int w = 0; w < 4; w++) {
      float so = 0.f;
#pragma unroll
      for (int i = 0; i < 8; i++)
        so += sacc[w][i][tid];
      const float wt = __expf(sm[w] - M);
      Ls = fmaf(wt, sl[w], Ls);
      o = fmaf(wt, so, o);
    }
  }
  // A workgroup without keys gets here with its rows still on their way.  Their registers stay taken until its state is
  // stored: the first reuse of one would wait for all of them in front of the sums over the waves, and the last of the nine
  // or so workgroups of a head would arrive that much later (32 heads, 130 keys of 2048: 7.36 us, so 6.99; 12 of 64, 4 x 300 of 1024: 5.91, so 5.60).
  auto hold = [&] {
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int j = 0; j < 2; j++)
        asm volatile("" : : "v"(kr[s][j]), "v"(vr[s][j]), "v"(qp[j]));
  };
  attn_finish(p, bh, tid, M, Ls, o, hold);
}

__global__ void __launch_bounds__(128)
attn_combine_kernel(const AttnParams p) {
  const int bh = blockIdx.x, tid = threadIdx.x;
  const float* src = p.part + (int64_t)bh * p.splits * 130;
  float M = -3.0e38f;
  for (int i = 0; i < p.splits; i++)
    M = fmaxf(M, src[i * 130]);
  float Ls = 0.f, o = 0.f;
  for (int i = 0; i < p.splits; i++) {
    const float w = __expf(src[i * 130] - M);
    Ls = fmaf(w, src[i * 130 + 1], Ls);
    o = fmaf(w, src[i * 130 + 2 + tid], o);
  }
  p.out[(int64_t)bh * 128 + tid] = (uint16_t)f32_to_bf16_bits(Ls > 0.f ? o / Ls : 0.f);
}

// ---------------------------------------------------------------------------
// Prompt attention: S query tokens per sequence at positions past .. past+S-1
// over the cache [B][Nkv][Smax][128], causal (query i sees keys 0 .. past+i).
// Grid (ceil(S/64), B*Nq); 4 waves of 16 queries each share the K and V tiles
// of 64 keys through LDS.  Both products run on the 16x16x32 bf16 MFMA in
// transposed form, so that no probability ever changes lanes:
//   scores^T[key][query] = K tile (rows = keys) x Q^T      (4 MFMAs per 16 keys)
//   out^T[dim][query]   += V^T tile (rows = dims) x P^T    (2 MFMAs per 16 dims)
// The score tile's result layout -- lane (g, c) holds keys g*4+r of query c --
// is, after rounding to bf16, already the second operand of the V product
// (its 32 K slots filled with the lane's keys of two score tiles; the V^T
// operand picks the same keys).  V is transposed on its way into LDS.
// Online softmax per query: fp32 scores * 1/sqrt(H) + mask, running max and
// sum, probabilities rounded to bf16 before they multiply V, sum and output
// in fp32 (the same arithmetic as the single-query kernel above).
// ---------------------------------------------------------------------------
struct AttnPrefillParams {
  const uint16_t* q;    // [B][S][Nq][128]
  const uint16_t* kc;   // [B][Nkv][Smax][128]
  const uint16_t* vc;
  const uint16_t* mask; // bf16 [B][mask_ld] additive, or null
  uint16_t* out;        // [B][S][Nq][128]
  int B, S, Nq, Nkv, Smax, mask_ld, past;
  float scale;
  int H;                // head size (attn_prefill_hd_kernel; the kernel for 128 does not read it)
};

constexpr int AP_VP = 68; // LDS row pitch of the hd kernel's V^T tile (64 keys + 4: rows 8-byte aligned)

// Prompt attention, head size 128: W waves of 16 queries share the K and V tiles of 64 keys (8: 128 queries, four waves per
// SIMD with two workgroups on a CU; 4: 64 queries, for launches of few workgroups).
// K and V tiles go straight into LDS, a tile ahead, two stages of 2 x 16 KiB, one barrier per tile; the swizzle sits on the
// source side (K: position ch of row r holds chunk ch ^ (r & 15); V: ch ^ 2 (r & 7)), so that the rows of an operand read
// fall on different bank groups.  V's operand is read by the transposing LDS read: of a 16-lane group lane i fetches 8 bytes
// of key (i >> 2) and gets the four keys of dim i.
// What bounds it is the chain scores -> softmax -> output of a wave, not one unit (MFMA a third busy, vector issue a half), so
// waves per SIMD count more than operand reads per MFMA (32 queries per wave, half the reads: 57 us where 16 took 50).  The
// tile's maximum is taken across lanes and the sums are rescaled only where some query's running maximum moves, everything
// else being a factor of exactly 1: the bits of doing it in every tile.  Two links of that chain stand still: the 16 operand
// reads of 32 keys' V are waited for as they are issued, twice per tile (124 of 128 registers are taken, none are left to read
// ahead), and with a mask its values, requested behind the next tile, arrive behind it.
// Measured against registers in between, V transposed by byte permutes and a rescaling per tile: 2048 tokens x 32 heads
// 74 -> 57.5 us, 64 heads on 8 of K/V 152 -> 88, 1000 x 32 28 -> 22.3, 333 x 32 12.6 -> 9.9, 3 x 600 behind 500 with a mask 107
// -> 48.5 (the mask was read under a branch per key).
// Tried beside it: a running maximum that is a power of two and moves by 8 at a time, exact as well but with other roundings
// of the probabilities (49.5); the next tile's scores under this one's softmax in a wave (256 registers and scratch); two
// halves of the keys on eight waves (54.8), the same half a turn apart (60).
typedef int i32x2 __attribute__((ext_vector_type(2)));
// The transposing reads of 32 keys' V operands (8 dim tiles x 2 runs of 16 keys), issued and waited for in one block: around
// the builtin the compiler waits for every load into LDS under way, that is for the next tile.
template <int OFF>
__device__ __forceinline__ void read_v_operands(i32x2 (&v)[8][2], const uint32_t (&a)[8]) {
  asm volatile("ds_read_b64_tr_b16 %0, %16 offset:%24\n\tds_read_b64_tr_b16 %1, %16 offset:%25\n\t"
               "ds_read_b64_tr_b16 %2, %17 offset:%24\n\tds_read_b64_tr_b16 %3, %17 offset:%25\n\t"
               "ds_read_b64_tr_b16 %4, %18 offset:%24\n\tds_read_b64_tr_b16 %5, %18 offset:%25\n\t"
               "ds_read_b64_tr_b16 %6, %19 offset:%24\n\tds_read_b64_tr_b16 %7, %19 offset:%25\n\t"
               "ds_read_b64_tr_b16 %8, %20 offset:%24\n\tds_read_b64_tr_b16 %9, %20 offset:%25\n\t"
               "ds_read_b64_tr_b16 %10, %21 offset:%24\n\tds_read_b64_tr_b16 %11, %21 offset:%25\n\t"
               "ds_read_b64_tr_b16 %12, %22 offset:%24\n\tds_read_b64_tr_b16 %13, %22 offset:%25\n\t"
               "ds_read_b64_tr_b16 %14, %23 offset:%24\n\tds_read_b64_tr_b16 %15, %23 offset:%25\n\t"
               "s_waitcnt lgkmcnt(0)"
               : "=&v"(v[0][0]), "=&v"(v[0][1]), "=&v"(v[1][0]), "=&v"(v[1][1]), "=&v"(v[2][0]), "=&v"(v[2][1]), "=&v"(v[3][0]),
                 "=&v"(v[3][1]), "=&v"(v[4][0]), "=&v"(v[4][1]), "=&v"(v[5][0]), "=&v"(v[5][1]), "=&v"(v[6][0]), "=&v"(v[6][1]),
                 "=&v"(v[7][0]), "=&v"(v[7][1])
               : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(a[5]), "v"(a[6]), "v"(a[7]), "n"(OFF), "n"(OFF + 4096)
               : "memory");
}

// maximum over the four 16-lane groups: swapped with itself a register gives both halves, no trip through the LDS
__device__ __forceinline__ float max_of_groups(float v) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
// a product that is not fused into what follows it
__device__ __forceinline__ float scaled(float v, float by) {
#pragma clang fp contract(off)
  return v * by;
}

template <int W>
__global__ void __launch_bounds__(W * 64, W == 8 ? 4 : 2)
attn_prefill_kernel(const AttnPrefillParams p) {
  constexpr int STAGE = 32768;
  __shared__ __align__(16) uint8_t lds[2 * STAGE]; // per stage: K [64 keys][256 B] | V [64 keys][256 B]
  constexpr int QB = 16 * W; // queries per workgroup
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c = lane & 15;
  // The last query blocks see the most keys: start them first.  Two workgroups share a CU, and the dispatcher puts
  // workgroup i + 256 beside workgroup i: every other run of whole query blocks within 256 workgroups is walked the other way
  // round, so that a long block meets a short one.  Heads go round the XCDs, those of one K/V head to the same one.
  const int heads = p.B * p.Nq, nblk = (p.S + QB - 1) / QB;
  const int per = heads < 256 ? 256 / heads : 1;
  int k = (int)blockIdx.x / heads;
  if (const int chunk = k / per; (chunk & 1) && (chunk + 1) * per <= nblk)
    k = chunk * per + per - 1 - k % per;
  const int qblk = nblk - 1 - k, bh = (int)blockIdx.x % heads, b = bh / p.Nq;
  const int hr = bh - b * p.Nq, hk = hr % p.Nkv, hq = hk * (p.Nq / p.Nkv) + hr / p.Nkv;
  const int q0 = qblk * QB + wave * 16;
  const int last_key = p.past + p.S - 1;

  const float scale2 = p.scale * 1.44269504f; // scores in the base-2 domain; positive
  const int qi = min(q0 + c, p.S - 1), qpos = p.past + qi; // this lane's query and the last key it sees (past the end: the last one, not stored)
  const uint16_t* qrow = p.q + (((int64_t)b * p.S + qi) * p.Nq + hq) * 128;
  bf16x8 qreg[4];
#pragma unroll
  for (int j = 0; j < 4; j++)
    qreg[j] = *reinterpret_cast<const bf16x8*>(qrow + j * 32 + g * 8);
  const int64_t head = ((int64_t)b * p.Nkv + hk) * p.Smax * 128;
  const uint16_t* mrow = p.mask ? p.mask + (int64_t)b * p.mask_ld : nullptr;

  constexpr int NP = 16 / W; // pieces of 4 rows x 256 B of K and of V that a wave brings (rows past the last key repeat it)
  auto request = [&](int kb, int stage) {
    const int64_t at = head + (int64_t)kb * (64 * 128); // (a descriptor per tile: no limit on the keys of a head)
    const auto kr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.kc + at), 0, 0xffffffffu, 0x00020000);
    const auto vr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.vc + at), 0, 0xffffffffu, 0x00020000);
    const int rows = last_key - kb * 64;
#pragma unroll
    for (int i = 0; i < NP; i++) {
      const int pc = wave * NP + i;
      const uint32_t row = (uint32_t)min(pc * 4 + g, rows) * 256u;
      uint8_t* const dst = lds + stage * STAGE + pc * 1024;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(kr, (__attribute__((address_space(3))) void*)dst, 16, row + (uint32_t)(c ^ ((pc & 3) * 4 + g)) * 16u, 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(vr, (__attribute__((address_space(3))) void*)(dst + 16384), 16, row + (uint32_t)(c ^ (((pc & 1) * 4 + g) * 2)) * 16u, 0, 0, 0);
    }
  };
  uint32_t kaddr[4], vaddr[8]; // this lane's operands inside a stage: K chunk j * 4 + g of row c; V dims dt * 16 .. + 15
#pragma unroll
  for (int j = 0; j < 4; j++)
    kaddr[j] = (uint32_t)(c * 256 + (((j * 4 + g) ^ c) & 15) * 16);
  {
    const int r = g * 4 + (c >> 2); // key of this lane's 8 bytes inside a run of 16
#pragma unroll
    for (int dt = 0; dt < 8; dt++)
      vaddr[dt] = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds + (uint32_t)(r * 256 + ((dt * 2 + ((c >> 1) & 1)) ^ ((r & 7) * 2)) * 16 + (c & 1) * 8);
  }

  float m = -3.0e38f, l = 0.f;
  f32x4 acc[8];
#pragma unroll
  for (int dt = 0; dt < 8; dt++)
    acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  // key tiles up to the one holding the last key of the workgroup's last query (the same for all four waves)
  const int nkb = (p.past + min(qblk * QB + QB - 1, p.S - 1)) / 64 + 1;
  auto tile = [&](auto STAGE_, int kb) {
    constexpr int stage = decltype(STAGE_)::value, V_AT = stage * STAGE + 16384;
    // this tile has landed and the other stage has been read, for this wave and then for every wave
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" : : : "memory");
    if (kb + 1 < nkb)
      request(kb + 1, stage ^ 1); // in flight during the arithmetic below
    if (kb * 64 > p.past + q0 + 15)
      return; // past the causal edge of all of this wave's queries
    const uint8_t* st = lds + stage * STAGE;

    f32x4 sc[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
      sc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 4; j++)
        sc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(st + kaddr[j] + t * 4096), qreg[j], sc[t], 0, 0, 0);
    }
    // Scores in the base-2 domain (scale * log2 e folded into one multiplier, the product rounded): a probability is one exp2.
    // The additive mask is read only when there is one (wave-uniform branch: no addresses, no predicated loads).
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        sc[t][r] = scaled(sc[t][r], scale2);
    if (mrow) {
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int key = kb * 64 + (i >> 2) * 16 + g * 4 + (i & 3);
        const float mv = bf16_bits_to_f32(mrow[min(key, p.mask_ld - 1)]) * 1.44269504f; // (no branch per key)
        sc[i >> 2][i & 3] += key < p.mask_ld ? mv : 0.f;
      }
    }
    // only the tiles that reach past the position of this wave's first query hide anything (wave-uniform)
    if (kb * 64 + 63 > p.past + q0) {
#pragma unroll
      for (int t = 0; t < 4; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int key = kb * 64 + t * 16 + g * 4 + r;
          // keys past the causal edge get -inf, whose exp2 is exactly 0 against the finite running maximum
          sc[t][r] = key <= qpos ? sc[t][r] : -INFINITY;
        }
    }
    float mx = -3.0e38f;
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        mx = fmaxf(mx, sc[t][r]);
    float alpha = 1.0f;
    if (__builtin_amdgcn_ballot_w64(mx > m) != 0) { // some query's maximum moves (otherwise every factor below is 1)
      mx = max_of_groups(mx);
      const float mn = fmaxf(m, mx); // finite from the first tile on: key 0 is visible to every query
      alpha = __builtin_amdgcn_exp2f(m - mn);
#pragma unroll
      for (int dt = 0; dt < 8; dt++)
        acc[dt] *= alpha;
      m = mn;
    }
    bf16x8 pb[2];
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const float pr = __builtin_amdgcn_exp2f(sc[2 * u + (j >> 2)][j & 3] - m);
        l = u == 0 && j == 0 ? fmaf(l, alpha, pr) : l + pr;
        pb[u][j] = (__bf16)pr;
      }
    // K slots g*8 .. g*8+7 of the operand = keys u*32 + g*4 .. +3 and u*32 + 16 + g*4 .. +3 of the tile, the keys pb[.][u]
    // holds in the same slots
    static_for<0, 2>([&](auto U) {
      constexpr int u = decltype(U)::value;
      i32x2 vv[8][2];
      read_v_operands<V_AT + u * 8192>(vv, vaddr);
#pragma unroll
      for (int dt = 0; dt < 8; dt++) {
        const i32x4 av = {vv[dt][0][0], vv[dt][0][1], vv[dt][1][0], vv[dt][1][1]};
        acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av), pb[u], acc[dt], 0, 0, 0);
      }
    });
  };
  request(0, 0);
  for (int kb = 0; kb < nkb; kb += 2) {
    tile(std::integral_constant<int, 0>{}, kb);
    if (kb + 1 < nkb)
      tile(std::integral_constant<int, 1>{}, kb + 1);
  }
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
  if (q0 + c < p.S) {
    uint16_t* orow = p.out + (((int64_t)b * p.S + q0 + c) * p.Nq + hq) * 128;
#pragma unroll
    for (int dt = 0; dt < 8; dt++) {
      uint32_t w[2];
#pragma unroll
      for (int e = 0; e < 2; e++)
        w[e] = f32x2_to_bf16_bits(l > 0.f ? acc[dt][2 * e] / l : 0.f, l > 0.f ? acc[dt][2 * e + 1] / l : 0.f);
      *reinterpret_cast<uint2*>(orow + dt * 16 + g * 4) = make_uint2(w[0], w[1]);
    }
  }
}

// ---------------------------------------------------------------------------
// Single-query attention where several query heads share a K/V head (grouped-query attention), head size 128: a workgroup
// per (sequence, K/V head, up to 16 of its query heads, split of the keys).  The query heads are the columns of the MFMA
// operand that the prompt kernel above fills with queries, so a key row is read once for all of them.
// What bounds it is the cache stream.  A wave works by itself on tiles of 32 keys (8 KiB of K and of V, in two stages of its
// own LDS, brought by loads straight into LDS; no barrier in the loop), the first one requested before the length is known;
// 2 waves = 64 KiB, so that two workgroups of a CU have 64 to 128 KiB under way.  Scores, maximum, probabilities and sums as in
// attn_decode_wide_kernel; the waves and then the splits are merged in order, the latter by the last to arrive.
// The relative error against float64 is that kernel's (28 heads on 4, 64 on 8: 0.98 .. 1.00 of it over 33 .. 2500 keys), up to
// 1.02 times it where fewer splits leave more keys to a running maximum (32 on 16, 16 x 700: 2.15e-3 and 2.11e-3).  With the
// probabilities as two bf16 terms it would be 1.66e-3, for 1 to 2 % of the time.
// Against a workgroup per query head (attn_decode_wide_kernel), which reads every row Nq / Nkv times through the L2s and does
// its arithmetic on the vector units each time, us per launch: 28 heads on 4 of K/V, 16 sequences of 2500 keys 101 -> 20.6,
// 48 of 1500 169 -> 32.7, 4 of 2000 27.6 -> 10.4, 1 of 4000 15.7 -> 11.8, 1 of 100 6.9 -> 6.3; 64 heads on 8, 16 of 2048
// 164 -> 28.7; 32 on 16, 16 of 1000 44 -> 26.4 (5 TB/s of cache).  With a head per K/V head the other kernel is the faster one
// from some 30 MB of cache on (32 heads, 16 of 2048 87 against 96 us: more waves with requests of their own).
// ---------------------------------------------------------------------------
constexpr int AG_WAVES = 2, AG_KEYS = 32 * AG_WAVES; // keys per workgroup and trip

// the K operands of 32 keys (2 runs of 16 keys x 4 steps of 32 dims), issued and waited for in one block
template <int OFF>
__device__ __forceinline__ void read_k_operands(i32x4 (&k)[2][4], const uint32_t (&a)[4]) {
  asm volatile("ds_read_b128 %0, %8 offset:%12\n\tds_read_b128 %1, %9 offset:%12\n\t"
               "ds_read_b128 %2, %10 offset:%12\n\tds_read_b128 %3, %11 offset:%12\n\t"
               "ds_read_b128 %4, %8 offset:%13\n\tds_read_b128 %5, %9 offset:%13\n\t"
               "ds_read_b128 %6, %10 offset:%13\n\tds_read_b128 %7, %11 offset:%13\n\t"
               "s_waitcnt lgkmcnt(0)"
               : "=&v"(k[0][0]), "=&v"(k[0][1]), "=&v"(k[0][2]), "=&v"(k[0][3]), "=&v"(k[1][0]), "=&v"(k[1][1]), "=&v"(k[1][2]), "=&v"(k[1][3])
               : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "n"(OFF), "n"(OFF + 4096)
               : "memory");
}

template <bool ROT>
__global__ void __launch_bounds__(AG_WAVES * 64, 1)
attn_decode_group_kernel(const AttnParams p) {
  constexpr int STAGE = 16384, WAVE_LDS = 2 * STAGE; // per stage: K [32 keys][256 B] | V [32 keys][256 B]
  constexpr int OP = 132;                            // pitch of a merged output row in floats
  __shared__ __align__(16) uint8_t lds[AG_WAVES * WAVE_LDS];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c = lane & 15;
  const int G = p.Nq / p.Nkv, blocks = (G + 15) >> 4; // query heads of a K/V head, workgroups they take
  const int gb = (int)blockIdx.x % blocks, bkv = (int)blockIdx.x / blocks, b = bkv / p.Nkv, hk = bkv - b * p.Nkv;
  const int heads = min(16, G - gb * 16);             // of this workgroup
  const int head0 = b * p.Nq + hk * G + gb * 16;      // the first of them
  const int S = p.splits;

  // rows past the cache's end repeat its last one; rows past the length are masked below
  auto request = [&](int base, int stage) {
    const int first = min(base, p.Smax - 1), rows = p.Smax - 1 - first;
    const int64_t at = ((int64_t)bkv * p.Smax + first) * 128;
    const auto kr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.kc + at), 0, 0xffffffffu, 0x00020000);
    const auto vr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.vc + at), 0, 0xffffffffu, 0x00020000);
    uint8_t* const dst = lds + wave * WAVE_LDS + stage * STAGE;
#pragma unroll
    for (int pc = 0; pc < 8; pc++) // pieces of 4 rows x 256 B
      __builtin_amdgcn_raw_ptr_buffer_load_lds(kr, (__attribute__((address_space(3))) void*)(dst + pc * 1024), 16,
                                               (uint32_t)min(pc * 4 + g, rows) * 256u + (uint32_t)(c ^ ((pc & 3) * 4 + g)) * 16u, 0, 0, 0);
#pragma unroll
    for (int pc = 0; pc < 8; pc++)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(vr, (__attribute__((address_space(3))) void*)(dst + 8192 + pc * 1024), 16,
                                               (uint32_t)min(pc * 4 + g, rows) * 256u + (uint32_t)(c ^ (((pc & 1) * 4 + g) * 2)) * 16u, 0, 0, 0);
  };
  // the query: head c, dims j * 32 + g * 8 .. + 7 (columns past the heads repeat the last one, never stored)
  i32x4 qw[4];
  {
    const uint16_t* qrow = p.q + (int64_t)(head0 + min(c, heads - 1)) * 128 + g * 8;
#pragma unroll
    for (int j = 0; j < 4; j++)
      qw[j] = *reinterpret_cast<const i32x4*>(qrow + j * 32);
  }
  const int64_t pp = ROT ? p.pos[p.B_pos == 1 ? 0 : b] : 0;
  const bool rot = ROT && p.emb != nullptr && pp >= 0 && pp < p.MP; // positions outside the table are left unrotated
  if (rot) { // rotation pairs (i, 64 + i): operands j and j + 2 of the same lane
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const f32x4* cp = reinterpret_cast<const f32x4*>(p.emb + pp * 128 + j * 32 + g * 8);
      const f32x4* sp = reinterpret_cast<const f32x4*>(p.emb + ((int64_t)p.MP + pp) * 128 + j * 32 + g * 8);
      const f32x4 cs[2] = {cp[0], cp[1]}, sn[2] = {sp[0], sp[1]};
#pragma unroll
      for (int d = 0; d < 4; d++) {
        uint32_t lo[2], hi[2];
#pragma unroll
        for (int e = 0; e < 2; e++) {
          const float x1 = bf16_bits_to_f32(((uint32_t)qw[j][d] >> (16 * e)) & 0xffffu);
          const float x2 = bf16_bits_to_f32(((uint32_t)qw[j + 2][d] >> (16 * e)) & 0xffffu);
          const float cv = cs[d >> 1][(d & 1) * 2 + e], sv = sn[d >> 1][(d & 1) * 2 + e];
          lo[e] = f32_to_bf16_bits(rotate_first(x1, x2, cv, sv));
          hi[e] = f32_to_bf16_bits(rotate_second(x1, x2, cv, sv));
        }
        qw[j][d] = (int)(lo[0] | lo[1] << 16);
        qw[j + 2][d] = (int)(hi[0] | hi[1] << 16);
      }
    }
  }
  request(blockIdx.y * AG_KEYS + wave * 32, 0);
  const int len0 = *p.kv_len;
  const int L = max(0, min(len0 + p.kv_len_add, p.Smax));
  const int nk = (ROT && len0 >= 0 && len0 < p.Smax) ? len0 : -1; // cache position of the new token
  const int trips = (L + AG_KEYS - 1) / AG_KEYS;
  const uint16_t* mrow = p.mask ? p.mask + (int64_t)b * p.mask_ld : nullptr;

  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds + wave * WAVE_LDS;
  uint32_t kaddr[4], vaddr[8]; // this lane's operands inside a stage: K chunk j * 4 + g of row c; V dims dt * 16 .. + 15
#pragma unroll
  for (int j = 0; j < 4; j++)
    kaddr[j] = lds0 + (uint32_t)(c * 256 + (((j * 4 + g) ^ c) & 15) * 16);
  {
    const int r = g * 4 + (c >> 2); // key of this lane's 8 bytes inside a run of 16
#pragma unroll
    for (int dt = 0; dt < 8; dt++)
      vaddr[dt] = lds0 + (uint32_t)(r * 256 + ((dt * 2 + ((c >> 1) & 1)) ^ ((r & 7) * 2)) * 16 + (c & 1) * 8);
  }
  float m = -3.0e38f, l = 0.f;
  f32x4 acc[8];
#pragma unroll
  for (int dt = 0; dt < 8; dt++)
    acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto tile = [&](auto STAGE_, int base, bool more) {
    constexpr int stage = decltype(STAGE_)::value;
    if (more) // the next tile's 16 loads stay under way
      asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (ROT && nk >= base && nk < base + 32) {
      // the new token is not in the cache yet: its row of the tile becomes the rotated key (lane i: pair (i, 64 + i)) and the
      // step's value; one workgroup per K/V head writes both into the cache
      uint8_t* const st = lds + wave * WAVE_LDS + stage * STAGE;
      const int r = nk - base;
      const uint16_t* krow = p.k_new + (int64_t)bkv * 128;
      const uint16_t* vrow = p.v_new + (int64_t)bkv * 128;
      const float x1 = bf16_bits_to_f32(krow[lane]), x2 = bf16_bits_to_f32(krow[64 + lane]);
      const float cv = rot ? p.emb[pp * 128 + lane] : 1.f, sv = rot ? p.emb[((int64_t)p.MP + pp) * 128 + lane] : 0.f;
      const uint16_t k1 = (uint16_t)f32_to_bf16_bits(rot ? rotate_first(x1, x2, cv, sv) : x1), k2 = (uint16_t)f32_to_bf16_bits(rot ? rotate_second(x1, x2, cv, sv) : x2);
      const i32x4 vn = *reinterpret_cast<const i32x4*>(vrow + c * 8);
      uint16_t* const kt = reinterpret_cast<uint16_t*>(st + r * 256);
      kt[((lane >> 3) ^ (r & 15)) * 8 + (lane & 7)] = k1;
      kt[((8 + (lane >> 3)) ^ (r & 15)) * 8 + (lane & 7)] = k2;
      if (g == 0)
        *reinterpret_cast<i32x4*>(st + 8192 + r * 256 + (c ^ ((r & 7) * 2)) * 16) = vn;
      if (gb == 0) {
        const int64_t o = ((int64_t)bkv * p.Smax + nk) * 128;
        uint16_t* const kd = const_cast<uint16_t*>(p.kc) + o;
        kd[lane] = k1;
        kd[64 + lane] = k2;
        if (g == 0)
          *reinterpret_cast<i32x4*>(const_cast<uint16_t*>(p.vc) + o + c * 8) = vn;
      }
      // (the builtin, so that the compiler knows these loads done: it would wait for the next tile at the join otherwise)
      __builtin_amdgcn_s_waitcnt(0x0070); // vmcnt(0) lgkmcnt(0)
      asm volatile("" ::: "memory");
    }
    f32x4 sc[2];
    {
      i32x4 kw[2][4];
      read_k_operands<stage * STAGE>(kw, kaddr);
#pragma unroll
      for (int t = 0; t < 2; t++) {
        sc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; j++)
          sc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kw[t][j]), __builtin_bit_cast(bf16x8, qw[j]), sc[t], 0, 0, 0);
      }
    }
    const bool tail = base + 32 > L; // wave-uniform
#pragma unroll
    for (int i = 0; i < 8; i++)
      sc[i >> 2][i & 3] = scaled(sc[i >> 2][i & 3], p.scale);
    if (mrow) {
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int key = base + (i >> 2) * 16 + g * 4 + (i & 3);
        const float mv = bf16_bits_to_f32(mrow[min(key, p.mask_ld - 1)]); // (no branch per key)
        sc[i >> 2][i & 3] += key < p.mask_ld ? mv : 0.f;
      }
    }
    if (tail) {
#pragma unroll
      for (int i = 0; i < 8; i++) // past the end: -inf, whose exponential is exactly 0 against the finite maximum
        sc[i >> 2][i & 3] = base + (i >> 2) * 16 + g * 4 + (i & 3) < L ? sc[i >> 2][i & 3] : -INFINITY;
    }
    float mx = m;
#pragma unroll
    for (int i = 0; i < 8; i++)
      mx = fmaxf(mx, sc[i >> 2][i & 3]);
    if (__builtin_amdgcn_ballot_w64(mx > m) != 0) { // some head's maximum moves
      mx = max_of_groups(mx);
      const float alpha = __expf(m - mx);
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < 8; dt++)
        acc[dt] *= alpha;
      m = mx;
    }
    bf16x8 pb;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const float pr = __expf(sc[i >> 2][i & 3] - m);
      l += pr;
      pb[i] = (__bf16)pr;
    }
    // K slots g*8 .. +7 of the operand = keys g*4 .. +3 and 16 + g*4 .. +3, the keys pb holds in the same slots
    i32x2 vv[8][2];
    read_v_operands<stage * STAGE + 8192>(vv, vaddr);
    if (tail) { // rows past the end may hold anything, NaN included
      const int left = L - base - g * 4; // keys of this lane's first run that count
      auto keep = [](int n) { return n <= 0 ? 0 : n == 1 ? 0xffff : -1; };
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int k0 = keep(left - h * 16), k1 = keep(left - h * 16 - 2);
#pragma unroll
        for (int dt = 0; dt < 8; dt++) {
          vv[dt][h][0] &= k0;
          vv[dt][h][1] &= k1;
        }
      }
    }
#pragma unroll
    for (int dt = 0; dt < 8; dt++) {
      const i32x4 av = {vv[dt][0][0], vv[dt][0][1], vv[dt][1][0], vv[dt][1][1]};
      acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av), pb, acc[dt], 0, 0, 0);
    }
  };
  // Tiles of this wave: base + i * S * AG_KEYS while they begin before the end of the keys.  While tile i is worked on tile
  // i + 1 is under way in the other stage; a stage is asked for again once its tile has been read.
  const int step = S * AG_KEYS;
  int base = blockIdx.y * AG_KEYS + wave * 32;
  if (base + step < L)
    request(base + step, 1);
  for (; base < L; base += 2 * step) {
    tile(std::integral_constant<int, 0>{}, base, base + step < L);
    if (base + 2 * step < L)
      request(base + 2 * step, 0);
    if (base + step < L) {
      tile(std::integral_constant<int, 1>{}, base + step, base + 2 * step < L);
      if (base + 3 * step < L)
        request(base + 3 * step, 1);
    }
  }
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);

  // the waves' states through LDS (every load into it has landed, also a first tile that lies past the keys)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  float* const mo = reinterpret_cast<float*>(lds);           // [wave][head][OP]
  float* const sm = mo + AG_WAVES * 16 * OP;                 // [wave][head] maximum
  float* const sl = sm + AG_WAVES * 16;                      // [wave][head] sum
  float* const sw = sl + AG_WAVES * 16;                      // [head][32] weight of a split
  float* const sws = sw + 16 * 32;                           // [head][32] its sum
  int* const arrived_last = reinterpret_cast<int*>(sws + 16 * 32);
#pragma unroll
  for (int dt = 0; dt < 8; dt++)
    *reinterpret_cast<f32x4*>(mo + (wave * 16 + c) * OP + dt * 16 + g * 4) = acc[dt];
  if (g == 0) {
    sm[wave * 16 + c] = m;
    sl[wave * 16 + c] = l;
  }
  __syncthreads();
  float* const part_o = p.part;                                            // [head][split][128]
  float* const part_ml = p.part + (int64_t)p.B * p.Nq * S * 128;           // [head][split][2]
  auto store4 = [&](int h, int d4, f32x4 o, float Ls) {
    uint32_t w[2];
#pragma unroll
    for (int e = 0; e < 2; e++)
      w[e] = f32x2_to_bf16_bits(Ls > 0.f ? o[2 * e] / Ls : 0.f, Ls > 0.f ? o[2 * e + 1] / Ls : 0.f);
    *reinterpret_cast<uint2*>(p.out + (int64_t)(head0 + h) * 128 + d4 * 4) = make_uint2(w[0], w[1]);
  };
  for (int i = tid; i < heads * 32; i += AG_WAVES * 64) {
    const int h = i >> 5, d4 = i & 31;
    float M = sm[h];
#pragma unroll
    for (int w = 1; w < AG_WAVES; w++)
      M = fmaxf(M, sm[w * 16 + h]);
    float Ls = 0.f;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < AG_WAVES; w++) {
      const float wt = __expf(sm[w * 16 + h] - M);
      Ls = fmaf(wt, sl[w * 16 + h], Ls);
      const f32x4 ow = *reinterpret_cast<const f32x4*>(mo + (w * 16 + h) * OP + d4 * 4);
#pragma unroll
      for (int e = 0; e < 4; e++)
        o[e] = fmaf(wt, ow[e], o[e]);
    }
    if (S == 1) {
      store4(h, d4, o, Ls);
      continue;
    }
    if (p.ticket0 < 0 && !p.counters) { // attn_combine_kernel follows
      float* const dst = p.part + ((int64_t)(head0 + h) * S + blockIdx.y) * 130;
#pragma unroll
      for (int e = 0; e < 4; e++)
        dst[2 + d4 * 4 + e] = o[e];
      if (d4 == 0) {
        dst[0] = M;
        dst[1] = Ls;
      }
      continue;
    }
    // device-scope stores: written through to the level all XCDs share
    const int64_t at = (int64_t)(head0 + h) * S + blockIdx.y;
    uint64_t* const dst = reinterpret_cast<uint64_t*>(part_o + at * 128 + d4 * 4);
    __hip_atomic_store(dst, __builtin_bit_cast(uint64_t, make_float2(o[0], o[1])), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(dst + 1, __builtin_bit_cast(uint64_t, make_float2(o[2], o[3])), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (d4 == 0)
      __hip_atomic_store(reinterpret_cast<uint64_t*>(part_ml + at * 2), __builtin_bit_cast(uint64_t, make_float2(M, Ls)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (S == 1 || (p.ticket0 < 0 && !p.counters))
    return;
  // The split that arrives last merges all of them, in split order; the ordering argument is attn_finish's: own stores
  // acknowledged, barrier, ticket, device-scope loads.  Nobody waits for anybody.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0)
    *arrived_last = attn_arrive(p.counters, p.ticket0, (int)blockIdx.x, S);
  __syncthreads();
  if (!*arrived_last)
    return;
  auto load2 = [](const float* src) {
    return __builtin_bit_cast(float2, __hip_atomic_load(reinterpret_cast<const uint64_t*>(src), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  };
  // 16 lanes per head: every lane two splits at most
  for (int i = tid; i < heads * 16; i += AG_WAVES * 64) {
    const int h = i >> 4, s0 = i & 15;
    float2 ml[2] = {{-3.0e38f, 0.f}, {-3.0e38f, 0.f}};
#pragma unroll
    for (int u = 0; u < 2; u++)
      if (s0 + 16 * u < S)
        ml[u] = load2(part_ml + ((int64_t)(head0 + h) * S + s0 + 16 * u) * 2);
    float M = fmaxf(ml[0].x, ml[1].x);
    M = fmaxf(M, dpp_mov<0xB1>(M));
    M = fmaxf(M, dpp_mov<0x4E>(M));
    M = fmaxf(M, dpp_mov<0x141>(M));
    M = fmaxf(M, dpp_mov<0x140>(M));
#pragma unroll
    for (int u = 0; u < 2; u++) {
      sw[h * 32 + s0 + 16 * u] = __expf(ml[u].x - M);
      sws[h * 32 + s0 + 16 * u] = ml[u].y;
    }
  }
  __syncthreads();
  for (int i = tid; i < heads * 32; i += AG_WAVES * 64) {
    const int h = i >> 5, d4 = i & 31;
    const float* src = part_o + (int64_t)(head0 + h) * S * 128 + d4 * 4;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    float Ls = 0.f;
    for (int s0 = 0; s0 < S; s0 += 8) { // eight splits' loads in flight
      float2 a[8][2];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const float* at = src + (int64_t)min(s0 + u, S - 1) * 128;
        a[u][0] = load2(at);
        a[u][1] = load2(at + 2);
      }
#pragma unroll
      for (int u = 0; u < 8; u++) {
        if (s0 + u < S) {
          const float wt = sw[h * 32 + s0 + u];
          Ls = fmaf(wt, sws[h * 32 + s0 + u], Ls);
          o[0] = fmaf(wt, a[u][0].x, o[0]);
          o[1] = fmaf(wt, a[u][0].y, o[1]);
          o[2] = fmaf(wt, a[u][1].x, o[2]);
          o[3] = fmaf(wt, a[u][1].y, o[3]);
        }
      }
    }
    store4(h, d4, o, Ls);
  }
}

// ---------------------------------------------------------------------------
// Prompt attention at head sizes other than 128: attn_prefill_kernel with the head size padded to HD = 64, 128 or
// 256 (H a multiple of 8, H <= HD; dims past H are staged as zeros and not stored), the K tile 64 x (HD + 8) and the
// V^T tile HD x 68 in dynamic LDS, HD / 32 MFMAs per 16 keys for the scores and HD / 16 output tiles per query group.
// Same arithmetic and rounding points as the kernel for 128.
// TEAMS = 2: launches of few workgroups, where four waves walk one key tile after another and wait for each: two teams of four
// waves take every other tile, with K and V tiles of their own, and the second one's sums (fp32, with the row maxima) meet the
// first one's in LDS at the end.  96 workgroups of 80 wide behind 13 tiles 20.9 -> 17.4 us, 192 of 64 wide over 16 tiles
// 17.9 -> 14.0.
// ---------------------------------------------------------------------------
template <int QG, int HD, int TEAMS>
__global__ void __launch_bounds__(256 * TEAMS)
attn_prefill_hd_kernel(const AttnPrefillParams p) {
  extern __shared__ __align__(16) uint16_t ap_lds[];
  constexpr int KP = HD + 8, VP = AP_VP, NJ = HD / 32, NDT = HD / 16, CH = HD / 8;
  constexpr int VI = (CH + 15) / 16; // value chunks per thread: 16 threads (key quads) x 16 chunks per pass
  static_assert(TEAMS == 1 || QG == 1, "teams hand over one query group");
  constexpr int TILE = 64 * KP + HD * VP; // elements of a team's tiles
  const int team = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8);
  uint16_t* ks = ap_lds + team * TILE; // [64 keys][KP]
  uint16_t* vt = ks + 64 * KP;         // [HD dims][VP]
  constexpr int QB = 64 * QG;
  const int H = p.H, HC = H >> 3;  // real 8-dim chunks per row
  const int tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, c = lane & 15;
  const int bh = blockIdx.y, b = bh / p.Nq, hq = bh - b * p.Nq;
  const int hk = hq / (p.Nq / p.Nkv);
  // the last query blocks see the most keys: start them first; the heads of every other run of 256 workgroups the
  // other way round, so that the workgroups that share a CU (i, i + 256, ...) are a long one and a short one (one
  // order per head, taken from the head's first workgroup)
  const int wg0 = (int)(blockIdx.y * gridDim.x);
  const int qblk = ((wg0 >> 8) & 1) ? (int)blockIdx.x : (int)gridDim.x - 1 - (int)blockIdx.x;
  const int q0 = qblk * QB + wave * (16 * QG);
  const int last_key = p.past + p.S - 1;
  const i32x4 zero4 = {0, 0, 0, 0};

  int qpos[QG];
  bf16x8 qreg[QG][NJ];
#pragma unroll
  for (int qg = 0; qg < QG; qg++) {
    const int qi = min(q0 + qg * 16 + c, p.S - 1);
    qpos[qg] = p.past + qi;
    const uint16_t* qrow = p.q + (((int64_t)b * p.S + qi) * p.Nq + hq) * H;
#pragma unroll
    for (int j = 0; j < NJ; j++) {
      const int ch = j * 4 + g;
      qreg[qg][j] = __builtin_bit_cast(bf16x8, ch < HC ? *reinterpret_cast<const i32x4*>(qrow + ch * 8) : zero4);
    }
  }
  const uint16_t* kbase = p.kc + ((int64_t)b * p.Nkv + hk) * (int64_t)p.Smax * H;
  const uint16_t* vbase = p.vc + ((int64_t)b * p.Nkv + hk) * (int64_t)p.Smax * H;
  const uint16_t* mrow = p.mask ? p.mask + (int64_t)b * p.mask_ld : nullptr;

  // staging registers: K rows chunk-fastest; V: a thread takes one chunk of FOUR consecutive keys per pass
  i32x4 kst[NJ], vst[VI][4];
  const int vq = tid & 15;
  auto load_tile = [&](int kb) {
#pragma unroll
    for (int i = 0; i < NJ; i++) {
      const int idx = tid + i * 256;
      const int key = idx / CH, ch = idx % CH;
      const int kk = min(kb * 64 + key, last_key);
      kst[i] = ch < HC ? *reinterpret_cast<const i32x4*>(kbase + (int64_t)kk * H + ch * 8) : zero4;
    }
#pragma unroll
    for (int it = 0; it < VI; it++) {
      const int vch = (tid >> 4) + it * 16;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int kv = min(kb * 64 + vq * 4 + i, last_key);
        vst[it][i] = vch < HC ? *reinterpret_cast<const i32x4*>(vbase + (int64_t)kv * H + vch * 8) : zero4;
      }
    }
  };
  auto store_tile = [&]() {
#pragma unroll
    for (int i = 0; i < NJ; i++) {
      const int idx = tid + i * 256;
      *reinterpret_cast<i32x4*>(ks + (idx / CH) * KP + (idx % CH) * 8) = kst[i];
    }
#pragma unroll
    for (int it = 0; it < VI; it++) {
      const int vch = (tid >> 4) + it * 16;
      if (vch < CH) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const uint32_t sel = (e & 1) ? 0x07060302u : 0x05040100u;
          const uint32_t lo = __builtin_amdgcn_perm((uint32_t)vst[it][1][e >> 1], (uint32_t)vst[it][0][e >> 1], sel);
          const uint32_t hi = __builtin_amdgcn_perm((uint32_t)vst[it][3][e >> 1], (uint32_t)vst[it][2][e >> 1], sel);
          *reinterpret_cast<uint2*>(vt + (vch * 8 + e) * VP + vq * 4) = make_uint2(lo, hi);
        }
      }
    }
  };

  const float scale2 = p.scale * 1.44269504f;
  float m[QG], l[QG];
  f32x4 acc[QG][NDT];
#pragma unroll
  for (int qg = 0; qg < QG; qg++) {
    m[qg] = -3.0e38f;
    l[qg] = 0.f;
#pragma unroll
    for (int dt = 0; dt < NDT; dt++)
      acc[qg][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int nkb = (p.past + min(qblk * QB + QB - 1, p.S - 1)) / 64 + 1;
  load_tile(team); // (past the last tile: the last key again, never used)
  for (int kb0 = 0; kb0 < nkb; kb0 += TEAMS) {
    const int kb = kb0 + team;
    __syncthreads(); // the previous tile has been read by every wave
    store_tile();
    __syncthreads();
    if (kb + TEAMS < nkb)
      load_tile(kb + TEAMS); // in flight during the arithmetic below
    if (TEAMS > 1 && kb >= nkb)
      continue; // the last round of a team without a tile (its barriers are behind it)

    f32x4 sc[QG][4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
#pragma unroll
      for (int qg = 0; qg < QG; qg++)
        sc[qg][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < NJ; j++) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(ks + (t * 16 + c) * KP + j * 32 + g * 8);
#pragma unroll
        for (int qg = 0; qg < QG; qg++)
          sc[qg][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, qreg[qg][j], sc[qg][t], 0, 0, 0);
      }
    }
#pragma unroll
    for (int qg = 0; qg < QG; qg++)
#pragma unroll
      for (int t = 0; t < 4; t++)
        sc[qg][t] *= scale2;
    if (mrow) {
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int key = kb * 64 + (i >> 2) * 16 + g * 4 + (i & 3);
        const float mk = key < p.mask_ld ? bf16_bits_to_f32(mrow[key]) * 1.44269504f : 0.f;
#pragma unroll
        for (int qg = 0; qg < QG; qg++)
          sc[qg][i >> 2][i & 3] += mk;
      }
    }
    bf16x8 pb[QG][2];
    const bool edge = kb * 64 + 63 > p.past + q0;
#pragma unroll
    for (int qg = 0; qg < QG; qg++) {
      if (edge) {
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const int key = kb * 64 + t * 16 + g * 4 + r;
            sc[qg][t][r] = key <= qpos[qg] ? sc[qg][t][r] : -INFINITY;
          }
      }
      float mx = -3.0e38f;
#pragma unroll
      for (int t = 0; t < 4; t++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          mx = fmaxf(mx, sc[qg][t][r]);
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      const float mn = fmaxf(m[qg], mx);
      const float alpha = __builtin_amdgcn_exp2f(m[qg] - mn);
      l[qg] *= alpha;
#pragma unroll
      for (int dt = 0; dt < NDT; dt++)
        acc[qg][dt] *= alpha;
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int j = 0; j < 8; j++) {
          const float pr = __builtin_amdgcn_exp2f(sc[qg][2 * u + (j >> 2)][j & 3] - mn);
          l[qg] += pr;
          pb[qg][u][j] = (__bf16)pr;
        }
      m[qg] = mn;
    }
#pragma unroll
    for (int dt = 0; dt < NDT; dt++)
#pragma unroll
      for (int u = 0; u < 2; u++) {
        const uint16_t* vrow = vt + (dt * 16 + c) * VP + u * 32 + g * 4;
        const uint2 lo = *reinterpret_cast<const uint2*>(vrow), hi = *reinterpret_cast<const uint2*>(vrow + 16);
        const i32x4 av = {(int)lo.x, (int)lo.y, (int)hi.x, (int)hi.y};
#pragma unroll
        for (int qg = 0; qg < QG; qg++)
          acc[qg][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av), pb[qg][u], acc[qg][dt], 0, 0, 0);
      }
  }
#pragma unroll
  for (int qg = 0; qg < QG; qg++) {
    l[qg] += __shfl_xor(l[qg], 16);
    l[qg] += __shfl_xor(l[qg], 32);
  }
  if constexpr (TEAMS > 1) {
    // the other teams leave their sums where their tiles were ([wave][dim tile][lane] x 16 bytes, then maximum and sum per
    // query); the first one adds them in team order
    float* sums = reinterpret_cast<float*>(ks);
    float* ml = sums + HD * 64;
    static_assert(HD * 256 + 512 <= TILE * 2, "a team's sums fit its tiles");
    __syncthreads();
    if (team > 0) {
#pragma unroll
      for (int dt = 0; dt < NDT; dt++)
        *reinterpret_cast<f32x4*>(sums + ((wave * NDT + dt) * 64 + lane) * 4) = acc[0][dt];
      if (g == 0) {
        ml[(wave * 16 + c) * 2] = m[0];
        ml[(wave * 16 + c) * 2 + 1] = l[0];
      }
    }
    __syncthreads();
    if (team > 0)
      return;
#pragma unroll
    for (int t = 1; t < TEAMS; t++) {
      const float* ot = reinterpret_cast<const float*>(ap_lds + t * TILE);
      const float om = ot[HD * 64 + (wave * 16 + c) * 2], ol = ot[HD * 64 + (wave * 16 + c) * 2 + 1];
      const float mn = fmaxf(m[0], om);
      const float wa = __builtin_amdgcn_exp2f(m[0] - mn), wb = __builtin_amdgcn_exp2f(om - mn);
#pragma unroll
      for (int dt = 0; dt < NDT; dt++) {
        const f32x4 o = *reinterpret_cast<const f32x4*>(ot + ((wave * NDT + dt) * 64 + lane) * 4);
#pragma unroll
        for (int r = 0; r < 4; r++)
          acc[0][dt][r] = acc[0][dt][r] * wa + o[r] * wb;
      }
      l[0] = l[0] * wa + ol * wb;
      m[0] = mn;
    }
  }
#pragma unroll
  for (int qg = 0; qg < QG; qg++) {
    const float ls = l[qg];
    const int qi = q0 + qg * 16 + c;
    if (qi < p.S) {
      uint16_t* orow = p.out + (((int64_t)b * p.S + qi) * p.Nq + hq) * H;
#pragma unroll
      for (int dt = 0; dt < NDT; dt++) {
        if (dt * 16 + g * 4 < H) { // H is a multiple of 8: the four dims of this lane exist together
          uint32_t w[2];
#pragma unroll
          for (int h = 0; h < 2; h++)
            w[h] = f32x2_to_bf16_bits(ls > 0.f ? acc[qg][dt][2 * h] / ls : 0.f, ls > 0.f ? acc[qg][dt][2 * h + 1] / ls : 0.f);
          *reinterpret_cast<uint2*>(orow + dt * 16 + g * 4) = make_uint2(w[0], w[1]);
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Greedy step of a generation loop: next token = argmax of the row's logits (the first maximal index; a NaN counts
// as maximal, as torch.argmax has it), stored as int64; the position of the row moves on by one; the token's
// embedding row becomes the row of the next step's hidden states; workgroup 0 moves the cache length on by one.
// One workgroup of 1024 threads per row: 16-byte loads, (value, index) maxima through DPP-free LDS steps.
// ---------------------------------------------------------------------------
struct GreedyKey {
  float v;
  int i;
};
__device__ __forceinline__ bool greedy_before(float v, int i, float bv, int bi) {
  // total order: NaN above everything, then larger value, then smaller index
  const bool vn = v != v, bn = bv != bv;
  if (vn != bn)
    return vn;
  if (!vn && v != bv)
    return v > bv;
  return i < bi;
}

__global__ void __launch_bounds__(1024)
greedy_next_kernel(const uint16_t* __restrict__ logits, int V, const uint16_t* __restrict__ embed, int hidden,
                   int64_t* __restrict__ tokens, int64_t* __restrict__ pos, int32_t* __restrict__ seq_len,
                   uint16_t* __restrict__ h_next) {
  __shared__ float sv[1024];
  __shared__ int si[1024];
  const int b = blockIdx.x, tid = threadIdx.x;
  const uint16_t* row = logits + (size_t)b * V;
  float bv = -INFINITY;
  int bi = 0x7fffffff;
  for (int c = tid * 8; c < V; c += 1024 * 8) { // V % 8 == 0
    const uint4 raw = *reinterpret_cast<const uint4*>(row + c);
    const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const float v = bf16_bits_to_f32((w[e >> 1] >> ((e & 1) * 16)) & 0xffffu);
      if (greedy_before(v, c + e, bv, bi)) {
        bv = v;
        bi = c + e;
      }
    }
  }
  sv[tid] = bv;
  si[tid] = bi;
  __syncthreads();
  for (int step = 512; step > 0; step >>= 1) {
    if (tid < step && greedy_before(sv[tid + step], si[tid + step], sv[tid], si[tid])) {
      sv[tid] = sv[tid + step];
      si[tid] = si[tid + step];
    }
    __syncthreads();
  }
  const int tok = si[0];
  if (tid == 0) {
    tokens[b] = tok;
    if (pos)
      pos[b] += 1;
    if (seq_len && b == 0)
      seq_len[0] += 1;
  }
  if (h_next)
    for (int c = tid * 8; c < hidden; c += 1024 * 8) // hidden % 8 == 0
      *reinterpret_cast<uint4*>(h_next + (size_t)b * hidden + c) = *reinterpret_cast<const uint4*>(embed + (size_t)tok * hidden + c);
}

} // namespace tppx

using namespace tppx;

extern "C" int tppx_greedy_next(const void* logits, int64_t B, int64_t V, const void* embed, int64_t hidden, void* tokens,
                                void* pos, void* seq_len, void* h_next, tppx_stream_t stream) {
  const char* who = "tppx_greedy_next";
  TPPX_REQUIRE(logits && tokens, TPPX_EINVAL, "%s: null pointer", who);
  TPPX_REQUIRE(aligned16(logits), TPPX_EINVAL, "%s: logits not 16-byte aligned", who);
  TPPX_REQUIRE(B > 0 && B < (1 << 16) && V > 0 && V % 8 == 0 && V < ((int64_t)1 << 31), TPPX_ESHAPE,
               "%s: bad shape B=%ld V=%ld (V must be a multiple of 8)", who, (long)B, (long)V);
  TPPX_REQUIRE(!h_next || (embed && aligned16(embed) && aligned16(h_next) && hidden > 0 && hidden % 8 == 0), TPPX_EINVAL,
               "%s: the next hidden states need a 16-byte aligned embedding table and output with hidden %% 8 == 0", who);
  greedy_next_kernel<<<dim3((unsigned)B), dim3(1024), 0, (hipStream_t)stream>>>(
      (const uint16_t*)logits, (int)V, (const uint16_t*)embed, (int)hidden, (int64_t*)tokens, (int64_t*)pos, (int32_t*)seq_len,
      (uint16_t*)h_next);
  return check_hip(hipGetLastError(), who);
}

extern "C" int tppx_rms_norm(const void* x, const void* gamma, int gamma_dtype, void* y, int64_t rows, int64_t K,
                             float eps, tppx_stream_t stream) {
  TPPX_REQUIRE(x && gamma && y, TPPX_EINVAL, "tppx_rms_norm: null pointer");
  TPPX_REQUIRE(aligned16(x) && aligned16(gamma) && aligned16(y), TPPX_EINVAL, "tppx_rms_norm: pointer not 16-byte aligned");
  TPPX_REQUIRE(gamma_dtype == TPPX_DT_F32 || gamma_dtype == TPPX_DT_BF16, TPPX_EINVAL, "tppx_rms_norm: unknown gamma dtype %d", gamma_dtype);
  TPPX_REQUIRE(rows > 0 && rows < ((int64_t)1 << 31) && K > 0 && K % 8 == 0 && K < (1 << 24), TPPX_ESHAPE,
               "tppx_rms_norm: bad shape rows=%ld K=%ld (K must be a multiple of 8)", (long)rows, (long)K);
  const auto go = [&](auto F32) {
    constexpr bool f32 = decltype(F32)::value;
    const dim3 grid((unsigned)rows), block(256);
    const uint16_t* xp = (const uint16_t*)x;
    const hipStream_t st = (hipStream_t)stream;
    switch (K > 1024 || rows <= 512 ? (K + 2047) / 2048 : 0) {
      case 1: rms_norm_regs_kernel<f32, 1><<<grid, block, 0, st>>>(xp, gamma, (uint16_t*)y, (int)K, eps); break;
      case 2: rms_norm_regs_kernel<f32, 2><<<grid, block, 0, st>>>(xp, gamma, (uint16_t*)y, (int)K, eps); break;
      case 3: rms_norm_regs_kernel<f32, 3><<<grid, block, 0, st>>>(xp, gamma, (uint16_t*)y, (int)K, eps); break;
      case 4: rms_norm_regs_kernel<f32, 4><<<grid, block, 0, st>>>(xp, gamma, (uint16_t*)y, (int)K, eps); break;
      default: rms_norm_kernel<f32><<<grid, block, 0, st>>>(xp, gamma, (uint16_t*)y, (int)K, eps);
    }
  };
  if (gamma_dtype == TPPX_DT_F32)
    go(std::true_type{});
  else
    go(std::false_type{});
  return check_hip(hipGetLastError(), "tppx_rms_norm");
}

extern "C" int tppx_layer_norm(const void* x, const void* gamma, const void* beta, int param_dtype, void* y,
                               int64_t rows, int64_t K, float eps, tppx_stream_t stream) {
  TPPX_REQUIRE(x && gamma && beta && y, TPPX_EINVAL, "tppx_layer_norm: null pointer");
  TPPX_REQUIRE(aligned16(x) && aligned16(gamma) && aligned16(beta) && aligned16(y), TPPX_EINVAL,
               "tppx_layer_norm: pointer not 16-byte aligned");
  TPPX_REQUIRE(param_dtype == TPPX_DT_F32 || param_dtype == TPPX_DT_BF16, TPPX_EINVAL,
               "tppx_layer_norm: unknown gamma / beta dtype %d", param_dtype);
  TPPX_REQUIRE(rows > 0 && rows < ((int64_t)1 << 31) && K > 0 && K % 8 == 0 && K < (1 << 24), TPPX_ESHAPE,
               "tppx_layer_norm: bad shape rows=%ld K=%ld (K must be a multiple of 8)", (long)rows, (long)K);
  const auto go = [&](auto F32) {
    constexpr bool f32 = decltype(F32)::value;
    const dim3 grid((unsigned)rows), block(256);
    const uint16_t* xp = (const uint16_t*)x;
    const hipStream_t st = (hipStream_t)stream;
    switch (K > 1024 ? (K + 2047) / 2048 : 0) {
      case 1: layer_norm_regs_kernel<f32, 1><<<grid, block, 0, st>>>(xp, gamma, beta, (uint16_t*)y, (int)K, eps); break;
      case 2: layer_norm_regs_kernel<f32, 2><<<grid, block, 0, st>>>(xp, gamma, beta, (uint16_t*)y, (int)K, eps); break;
      case 3: layer_norm_regs_kernel<f32, 3><<<grid, block, 0, st>>>(xp, gamma, beta, (uint16_t*)y, (int)K, eps); break;
      case 4: layer_norm_regs_kernel<f32, 4><<<grid, block, 0, st>>>(xp, gamma, beta, (uint16_t*)y, (int)K, eps); break;
      default: layer_norm_kernel<f32><<<grid, block, 0, st>>>(xp, gamma, beta, (uint16_t*)y, (int)K, eps);
    }
  };
  if (param_dtype == TPPX_DT_F32)
    go(std::true_type{});
  else
    go(std::false_type{});
  return check_hip(hipGetLastError(), "tppx_layer_norm");
}

static int rotary_common(const char* who, RotaryParams& p, hipStream_t stream) {
  TPPX_REQUIRE(p.B > 0 && p.S > 0 && p.H >= 8 && p.H <= 512 && p.H % 8 == 0, TPPX_ESHAPE,
               "%s: bad shape B=%d S=%d H=%d (head size must be a multiple of 8 up to 512)", who, p.B, p.S, p.H);
  if (p.emb)
    TPPX_REQUIRE(p.HR > 0 && p.HR <= p.H && p.HR % 16 == 0 && p.MP > 0, TPPX_ESHAPE,
                 "%s: rotary_dim=%d must be a multiple of 16 and <= H=%d", who, p.HR, p.H);
  TPPX_REQUIRE(p.B_pos == 1 || p.B_pos == p.B, TPPX_ESHAPE, "%s: position_ids shape not compatible", who);
  const int heads = (p.q ? p.Nq : 0) + (p.k ? p.Nkv : 0) + ((p.v && p.vc) ? p.Nkv : 0);
  const int64_t total = (int64_t)p.B * p.S * heads * (p.H / 8);
  TPPX_REQUIRE(total > 0 && total < ((int64_t)1 << 40), TPPX_ESHAPE, "%s: nothing to do", who);
  if (!p.emb)
    p.HR = 0; // append without rotation: a key row is copied whole
  p.rot = p.gptj ? p.HR / 8 : p.HR / 16;
  p.uq = p.rot;
  p.uk = p.rot + (p.H - p.HR) / 8;
  p.uv = p.H / 8;
  auto magic = [](int units) { return units > 1 ? (uint32_t)((((uint64_t)1 << 32) + units - 1) / units) : 0u; };
  p.mq = magic(p.uq);
  p.mk = magic(p.uk);
  p.mv = magic(p.uv);
  const int64_t units = (int64_t)(p.q ? p.Nq : 0) * p.uq + (int64_t)(p.k ? p.Nkv : 0) * p.uk + (p.v && p.vc ? (int64_t)p.Nkv * p.uv : 0);
  if (units == 0)
    return TPPX_OK;
  TPPX_REQUIRE(units <= (int64_t)65535 * 256 && (int64_t)p.B * p.S < ((int64_t)1 << 31), TPPX_ESHAPE, "%s: too many heads or tokens", who);
  rotary_append_kernel<<<dim3((unsigned)(p.B * p.S), (unsigned)((units + 255) / 256)), dim3(256), 0, stream>>>(p);
  return check_hip(hipGetLastError(), who);
}

extern "C" int tppx_rotary_llama(void* t, const void* emb_pos, const void* pos, int64_t B, int64_t S, int64_t N,
                                 int64_t H, int64_t MP, int64_t HR, int64_t B_pos, tppx_stream_t stream) {
  TPPX_REQUIRE(t && emb_pos && pos, TPPX_EINVAL, "tppx_rotary_llama: null pointer");
  TPPX_REQUIRE(aligned16(t), TPPX_EINVAL, "tppx_rotary_llama: pointer not 16-byte aligned");
  TPPX_REQUIRE(N > 0, TPPX_ESHAPE, "tppx_rotary_llama: N=%ld", (long)N);
  RotaryParams p;
  memset(&p, 0, sizeof(p));
  p.q = (uint16_t*)t;
  p.emb = (const float*)emb_pos;
  p.pos = (const int64_t*)pos;
  p.B = (int)B; p.S = (int)S; p.Nq = (int)N; p.H = (int)H; p.MP = (int)MP; p.HR = (int)HR; p.B_pos = (int)B_pos;
  return rotary_common("tppx_rotary_llama", p, (hipStream_t)stream);
}

extern "C" int tppx_rotary_kv_append_llama(void* q, void* k, const void* v, const void* emb_pos, const void* pos,
                                           void* kcache, void* vcache, const void* offset_dev, int64_t B,
                                           int64_t S, int64_t Nq, int64_t Nkv, int64_t H, int64_t MP, int64_t HR,
                                           int64_t B_pos, int64_t Smax, tppx_stream_t stream) {
  const char* who = "tppx_rotary_kv_append_llama";
  TPPX_REQUIRE(k && v && kcache && vcache && offset_dev && pos, TPPX_EINVAL, "%s: null pointer", who);
  TPPX_REQUIRE(aligned16(k) && aligned16(v) && aligned16(kcache) && aligned16(vcache) && (!q || aligned16(q)),
               TPPX_EINVAL, "%s: pointer not 16-byte aligned", who);
  TPPX_REQUIRE(Nkv > 0 && Smax > 0 && (!q || Nq > 0), TPPX_ESHAPE, "%s: bad head counts / capacity", who);
  RotaryParams p;
  memset(&p, 0, sizeof(p));
  p.q = (uint16_t*)q; p.k = (uint16_t*)k; p.v = (const uint16_t*)v;
  p.kc = (uint16_t*)kcache; p.vc = (uint16_t*)vcache;
  p.emb = (const float*)emb_pos; p.pos = (const int64_t*)pos; p.offset = (const int32_t*)offset_dev;
  p.B = (int)B; p.S = (int)S; p.Nq = (int)Nq; p.Nkv = (int)Nkv; p.H = (int)H; p.MP = (int)MP; p.HR = (int)HR;
  p.B_pos = (int)B_pos; p.Smax = (int)Smax;
  return rotary_common(who, p, (hipStream_t)stream);
}

extern "C" int tppx_rotary_gptj(void* t, const void* emb_pos, const void* pos, int64_t B, int64_t S, int64_t N,
                                int64_t H, int64_t MP, int64_t HR, int64_t B_pos, tppx_stream_t stream) {
  TPPX_REQUIRE(t && emb_pos && pos, TPPX_EINVAL, "tppx_rotary_gptj: null pointer");
  TPPX_REQUIRE(aligned16(t), TPPX_EINVAL, "tppx_rotary_gptj: pointer not 16-byte aligned");
  TPPX_REQUIRE(N > 0, TPPX_ESHAPE, "tppx_rotary_gptj: N=%ld", (long)N);
  RotaryParams p;
  memset(&p, 0, sizeof(p));
  p.q = (uint16_t*)t;
  p.emb = (const float*)emb_pos;
  p.pos = (const int64_t*)pos;
  p.B = (int)B; p.S = (int)S; p.Nq = (int)N; p.H = (int)H; p.MP = (int)MP; p.HR = (int)HR; p.B_pos = (int)B_pos;
  p.gptj = 1;
  return rotary_common("tppx_rotary_gptj", p, (hipStream_t)stream);
}

extern "C" int tppx_rotary_kv_append_gptj(void* q, void* k, const void* v, const void* emb_pos, const void* pos,
                                          void* kcache, void* vcache, const void* offset_dev, int64_t B, int64_t S,
                                          int64_t Nq, int64_t Nkv, int64_t H, int64_t MP, int64_t HR, int64_t B_pos,
                                          int64_t Smax, tppx_stream_t stream) {
  const char* who = "tppx_rotary_kv_append_gptj";
  TPPX_REQUIRE(k && v && kcache && vcache && offset_dev && pos && emb_pos, TPPX_EINVAL, "%s: null pointer", who);
  TPPX_REQUIRE(aligned16(k) && aligned16(v) && aligned16(kcache) && aligned16(vcache) && (!q || aligned16(q)),
               TPPX_EINVAL, "%s: pointer not 16-byte aligned", who);
  TPPX_REQUIRE(Nkv > 0 && Smax > 0 && (!q || Nq > 0), TPPX_ESHAPE, "%s: bad head counts / capacity", who);
  RotaryParams p;
  memset(&p, 0, sizeof(p));
  p.q = (uint16_t*)q; p.k = (uint16_t*)k; p.v = (const uint16_t*)v;
  p.kc = (uint16_t*)kcache; p.vc = (uint16_t*)vcache;
  p.emb = (const float*)emb_pos; p.pos = (const int64_t*)pos; p.offset = (const int32_t*)offset_dev;
  p.B = (int)B; p.S = (int)S; p.Nq = (int)Nq; p.Nkv = (int)Nkv; p.H = (int)H; p.MP = (int)MP; p.HR = (int)HR;
  p.B_pos = (int)B_pos; p.Smax = (int)Smax;
  p.gptj = 1;
  return rotary_common(who, p, (hipStream_t)stream);
}

// a caller's arrival counters: zero before their first launch, zero again behind every launch
struct AttnCounters {
  void* p = nullptr;
  int64_t bytes = 0;
  unsigned int* of(int64_t groups) const { // null: too few
    return groups * ATTN_TICKET_STRIDE * (int64_t)sizeof(unsigned int) <= bytes ? (unsigned int*)p : nullptr;
  }
};

static int check_counters(const char* who, const AttnCounters& c) {
  TPPX_REQUIRE(c.bytes >= 0 && (c.bytes == 0 || c.p), TPPX_EINVAL, "%s: size of the counters given with a null pointer", who);
  TPPX_REQUIRE(((uintptr_t)c.p & 3u) == 0, TPPX_EINVAL, "%s: counters not 4-byte aligned", who);
  return TPPX_OK;
}

// window of the library's arrival counters (at most ATTN_TICKETS), handed out in rotation
static int attn_take_tickets(int64_t tickets) {
  static std::mutex mu;
  static int cursor = 0;
  std::lock_guard<std::mutex> lock(mu);
  if (cursor + tickets > ATTN_TICKETS)
    cursor = 0;
  const int first = cursor;
  cursor += (int)tickets;
  return first;
}

// shared tail of the single-query entry points for 128-wide heads: split planning, counters, launch
static int attn_decode_launch(const char* who, AttnParams& p, bool rot, int64_t B, int64_t Nq, int64_t Smax, void* ws,
                              int64_t ws_bytes, AttnCounters counters, hipStream_t stream) {
  // The wide kernel (128 keys per workgroup and trip) is the default: measured against the row kernel (64 keys per
  // trip) over 32 heads, it is faster at every batch size from 1 to 64 and context from 100 to 8000 keys once its
  // workgroups make about two trips each (batch 16, 2048 keys: 3660 -> 3739 tokens/s for the whole decode step;
  // batch 1, 8000 keys: 29.1 us with the row kernel, 32.1 with 9 wide splits per head, 27.0 with 16).  Splits per
  // head: two trips per workgroup, but no fewer workgroups than 288 (about one per CU: fewer leave CUs idle) and no
  // more than 512 (more splits mean more states to merge); the row kernel (TPPX_ATTN_WIDE=0) wants about two
  // workgroups per CU.  At most one split per trip and at most 32 (the merge holds every split's state in registers).
  const int wide_env = (int)env_int("TPPX_ATTN_WIDE", -1);
  const int64_t target_env = env_int("TPPX_ATTN_TARGET_WGS", 0);
  const bool wide = wide_env != 0;
  const int64_t heads = B * Nq;
  int64_t splits;
  if (target_env > 0 || !wide) {
    splits = ((target_env > 0 ? target_env : 512) + heads - 1) / heads;
  } else {
    const int64_t lo = (288 + heads - 1) / heads, hi = (512 + heads - 1) / heads;
    splits = ((Smax + ATTN_WIDE_KEYS - 1) / ATTN_WIDE_KEYS + 1) / 2;
    splits = splits < lo ? lo : splits > hi ? hi : splits;
  }
  const int64_t trip_keys = wide ? ATTN_WIDE_KEYS : 64;
  const int64_t max_by_len = (Smax + trip_keys - 1) / trip_keys;
  if (splits > max_by_len)
    splits = max_by_len;
  if (splits > 32)
    splits = 32;
  const bool one_launch = env_int("TPPX_ATTN_ONE_LAUNCH", 1) != 0;
  // Several query heads per K/V head: one workgroup for up to 16 of them.  Splits for about one workgroup per CU (16 groups of
  // 2000 keys: 16 splits 10.4 us, 32 13.2: more states to merge); from 129 groups on as many as two workgroups per CU take
  // in one round (160 groups of 900 keys: 3 splits 20.4, 2 21.8).  At least a trip each.
  const int64_t groups = B * p.Nkv * ((Nq / p.Nkv + 15) / 16);
  int64_t gsplits = target_env > 0 ? (target_env + groups - 1) / groups : groups <= 128 ? (256 + groups - 1) / groups : 500 / groups;
  gsplits = std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>(gsplits, 32), (Smax + AG_KEYS - 1) / AG_KEYS));
  if (gsplits > 1 && (B * Nq * gsplits * 130 * (int64_t)sizeof(float) > ws_bytes || !aligned16(ws)))
    gsplits = 1;
  const bool group = wide && Nq > p.Nkv && env_int("TPPX_ATTN_GROUP", 1) != 0;
  if (p.mask_ld <= 0)
    p.mask = nullptr; // a mask of no keys: the grouped kernel clamps its reads to the mask's last key
  if (group)
    splits = gsplits;
  const int64_t need = B * Nq * splits * 130 * (int64_t)sizeof(float);
  if (splits > 1 && need > ws_bytes)
    splits = 1; // no room for partial results: one workgroup per head
  p.splits = (int)splits;
  p.part = (float*)ws;
  p.ticket0 = -1;
  const int64_t tickets = group ? groups : B * Nq;
  if (splits > 1 && one_launch) {
    p.counters = counters.of(tickets);
    if (!p.counters && tickets <= ATTN_TICKETS)
      p.ticket0 = attn_take_tickets(tickets);
  }
  const dim3 grid((unsigned)(group ? groups : B * Nq), (unsigned)splits);
  if (group && rot)
    attn_decode_group_kernel<true><<<grid, dim3(AG_WAVES * 64), 0, stream>>>(p);
  else if (group)
    attn_decode_group_kernel<false><<<grid, dim3(AG_WAVES * 64), 0, stream>>>(p);
  else if (wide && rot)
    attn_decode_wide_kernel<true><<<grid, dim3(256), 0, stream>>>(p);
  else if (wide)
    attn_decode_wide_kernel<false><<<grid, dim3(256), 0, stream>>>(p);
  else if (rot)
    attn_decode_kernel<true><<<grid, dim3(256), 0, stream>>>(p);
  else
    attn_decode_kernel<false><<<grid, dim3(256), 0, stream>>>(p);
  int rc = check_hip(hipGetLastError(), who);
  if (rc && p.ticket0 >= 0) {
    // the refused launch leaves its counter window as it found it, but whoever gets the window next relies on zeros
    const int n = (int)tickets;
    attn_clear_tickets_kernel<<<dim3((n + 255) / 256), dim3(256), 0, stream>>>(p.ticket0, n);
    (void)hipGetLastError();
  }
  if (rc || splits == 1 || p.ticket0 >= 0 || p.counters)
    return rc;
  attn_combine_kernel<<<dim3((unsigned)(B * Nq)), dim3(128), 0, stream>>>(p);
  return check_hip(hipGetLastError(), who);
}

// ---------------------------------------------------------------------------
// Attention for head sizes other than 128 (attn<T>, src/csrc/llm/attn.cpp:781-955, is generic in the head size; the
// kernels above are built for 128), H a multiple of 8 up to 256.  The single-query step runs on
// attn_hd_step_kernel below, prompt passes on attn_prefill_hd_kernel above; this first, plain kernel serves
// both when those are switched off (TPPX_ATTN_GENERIC_ROWS=0, TPPX_ATTN_PREFILL_MFMA=0).  One wave per (sequence,
// query token, query head), four per workgroup, no barrier: 64 keys per trip,
// a lane takes the whole dot product of its key (16-byte loads along its row, the query as fp32 in wave-private
// LDS, read as broadcasts), online softmax over the trip with the probabilities rounded to bf16 before they multiply
// V and the normaliser summing the unrounded ones, then lanes turn to output dimensions (lane, lane + 64, ...) and
// walk the trip's value rows.  A plain kernel for the shapes the tuned ones do not take, not a tuned one.
// ---------------------------------------------------------------------------
struct AttnGenParams {
  const uint16_t* q;   // [B][S][Nq][H]
  const uint16_t* kc;  // [B][Nkv][Smax][H]
  const uint16_t* vc;
  const uint16_t* mask; // bf16 [B][mask_ld] additive, or null
  const int32_t* kv_len; // single-query step: device scalar, valid keys = *kv_len + kv_len_add; null: prompt pass
  int kv_len_add;
  uint16_t* out;       // [B][S][Nq][H]
  int B, S, Nq, Nkv, H, Smax, mask_ld, past; // prompt pass: query i sees keys 0 .. past + i
  float scale;
  // single-query step (attn_hd_step_kernel):
  int splits;          // workgroups per query
  unsigned int* counters; // splits > 1: the caller's arrival counters, or null: attn_hd_merge_kernel follows
  float* part;         // splits > 1: [query][split][2 + H] floats (running maximum, sum, unnormalised output)
  // APP: the query and the step's new key / value arrive unrotated and not yet in the cache
  const uint16_t* k_new; // [B][Nkv][H]
  const uint16_t* v_new;
  const float* emb;      // cos / sin [2][MP][HR] (Llama pairs) or sin | cos [MP][HR] (gptj), or null: no rotation
  const int64_t* pos;    // i64 [B_pos]
  int MP, HR, B_pos, gptj;
};

__global__ void __launch_bounds__(256)
attn_generic_kernel(const AttnGenParams p) {
  __shared__ __align__(16) float q_s[4][256];
  __shared__ float p_s[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t qi = (int64_t)blockIdx.x * 4 + wave;
  if (qi >= (int64_t)p.B * p.S * p.Nq) // whole waves; nothing below synchronises across waves
    return;
  const int h = (int)(qi % p.Nq), sq = (int)((qi / p.Nq) % p.S), b = (int)(qi / ((int64_t)p.Nq * p.S));
  const int hk = h / (p.Nq / p.Nkv), H = p.H;
  int L = p.kv_len ? p.kv_len[0] + p.kv_len_add : p.past + sq + 1;
  L = max(min(L, p.Smax), 0);
  const uint16_t* qrow = p.q + qi * H;
  for (int d = lane; d < H; d += 64)
    q_s[wave][d] = bf16_bits_to_f32(qrow[d]);
  // the lanes of a wave hand values to one another through LDS: the LDS serves a wave's accesses in order; the
  // fence and the wave barrier keep the compiler from moving the reads above the writes
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  const uint16_t* kb = p.kc + ((int64_t)b * p.Nkv + hk) * (int64_t)p.Smax * H;
  const uint16_t* vb = p.vc + ((int64_t)b * p.Nkv + hk) * (int64_t)p.Smax * H;
  const uint16_t* mrow = p.mask ? p.mask + (int64_t)b * p.mask_ld : nullptr;
  float m = -3.0e38f, l = 0.f, acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int c0 = 0; c0 < L; c0 += 64) {
    const int key = c0 + lane;
    const uint16_t* krow = kb + (int64_t)min(key, L - 1) * H;
    float d = 0.f;
    for (int e = 0; e < H; e += 8) {
      const i32x4 kv = *reinterpret_cast<const i32x4*>(krow + e);
      const f32x4 qa = *reinterpret_cast<const f32x4*>(&q_s[wave][e]), qb = *reinterpret_cast<const f32x4*>(&q_s[wave][e + 4]);
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const uint32_t w = (uint32_t)kv[j];
        const float q0 = j < 2 ? qa[2 * j] : qb[2 * j - 4], q1 = j < 2 ? qa[2 * j + 1] : qb[2 * j - 3];
        d = fmaf(bf16_bits_to_f32(w & 0xffffu), q0, d);
        d = fmaf(bf16_bits_to_f32(w >> 16), q1, d);
      }
    }
    d *= p.scale;
    if (mrow && key < p.mask_ld && key < L)
      d += bf16_bits_to_f32(mrow[key]);
    const float sc = key < L ? d : -3.0e38f;
    const float mn = fmaxf(m, wave_max(sc));
    const float alpha = __expf(m - mn); // 1 when the maximum stays
    m = mn;
    const float pr = key < L ? __expf(sc - m) : 0.f;
    l = l * alpha + wave_sum(pr);
#pragma unroll
    for (int i = 0; i < 4; i++)
      acc[i] *= alpha;
    __builtin_amdgcn_wave_barrier(); // (the previous trip's reads of p_s are done)
    p_s[wave][lane] = round_bf16(pr);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int nk = min(64, L - c0);
    for (int j = 0; j < nk; j++) {
      const float pj = p_s[wave][j];
      const uint16_t* vrow = vb + (int64_t)(c0 + j) * H;
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (lane + 64 * i < H)
          acc[i] = fmaf(pj, bf16_bits_to_f32(vrow[lane + 64 * i]), acc[i]);
    }
  }
  uint16_t* orow = p.out + qi * H;
#pragma unroll
  for (int i = 0; i < 4; i++)
    if (lane + 64 * i < H)
      orow[lane + 64 * i] = (uint16_t)f32_to_bf16_bits(l > 0.f ? acc[i] / l : 0.f);
}

// The single-query step at those head sizes, laid out like attn_decode_wide_kernel: G lanes share a key, a lane owns its
// chunks j*G + c (8 dims of 16 bytes each; chunks past H / 8 idle) of NU keys, so a wave instruction reads 64 / G whole
// (part) rows and a trip's K and V rows -- up to 16 KB a wave -- are requested at once, the first trip's before the length is
// known.  q . k and p . v run on the bf16 dot instruction, the wave shares one running maximum, the lanes' outputs are added
// up through LDS.  A probability enters p . v as two bf16 terms: rounded to one, against a maximum that a whole wave shares, it
// made the relative error against float64 1.98 / 2.02 / 1.98e-3 for heads of 256 / 80 / 64, where rounding it against the maximum
// of a lane group (the larger ones are then the 1 that bf16 holds exactly) gives 1.87 / 1.82 / 1.80e-3; in two terms it is 1.65 /
// 1.63 / 1.63e-3, the rounding of the output, for at most 1 % of the time (64 heads of 80, 2500 keys 67.1 -> 68.0 us).
// Grid (B * Nq, splits): split y takes the trips y, y + splits, ...; where the caller gives arrival counters the split that
// arrives last merges all of them in the launch.
// APP: the launch also does what the rotary + append launch did before it (LayerCache::update, attn.h:198-222): wave 0
// rotates the query and, in the split that reads its position, the new key -- rounded to bf16, as stored -- and that
// position's lanes take key and value from there; one workgroup per KV head writes them into the cache.
// What bounds a step of a few sequences is this chain of launches and of dependent loads, many the bytes.  In a graph of
// steps, against rotary + append, attention and the merge as launches of their own: 16 heads of 256, 1 x 2000 keys
// 24.2 -> 12.5 us, 4 x 700 18.1 -> 12.2, 16 x 2500 106.5 (6.2 TB/s) either way; 32 heads of 80, 1 x 2000 14.3 -> 9.7,
// 4 x 140 7.8 -> 7.0, 48 x 1400 113.7 -> 108.3.  (80 as 8 lanes x 2 chunks, the second a quarter live, 117.4.)
// Later trips' rows are requested as in attn_decode_wide_kernel: a graph of four layers with 16 heads of 256, 1 x 2000 keys
// 205.8 -> 199.4 us, 16 x 2500 619.8 -> 607.2, with 32 heads of 80, 1 x 2000 181.9 -> 176.1, 48 x 1400 677.7 -> 671.3.
template <int G, int J, int NU, bool APP>
__global__ void __launch_bounds__(256, 4)
attn_hd_step_kernel(const AttnGenParams p) {
  constexpr int KPI = 64 / G;            // keys per wave instruction
  constexpr int WK = NU * KPI;           // keys per wave and trip
  constexpr int TRIP = 4 * WK;           // keys per workgroup and trip
  constexpr int OP = G * J * 8 + 4;      // pitch of a lane group's output in floats
  __shared__ __align__(16) uint16_t q_s[G * J * 8], k_s[G * J * 8];
  __shared__ float sm[4], sl[4];
  __shared__ __align__(16) float sacc[4][KPI][OP];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = lane / G, c = lane % G;
  const int H = p.H, C = H >> 3, S = p.splits;
  const int bh = blockIdx.x, b = bh / p.Nq, hq = bh - b * p.Nq;
  const int hk = hq / (p.Nq / p.Nkv);
  const int64_t kv_head = (int64_t)b * p.Nkv + hk;
  const uint16_t* kb = p.kc + kv_head * p.Smax * H;
  const uint16_t* vb = p.vc + kv_head * p.Smax * H;
  bool live[J];                          // this lane's chunks that exist; the others re-read the last one
  int at[J];
#pragma unroll
  for (int j = 0; j < J; j++) {
    live[j] = j * G + c < C;
    at[j] = min(j * G + c, C - 1) * 8;
  }
  i32x4 kr[NU][J], vr[NU][J];
  auto load_rows = [&](const uint16_t* src, int base, int end, i32x4 (&dst)[NU][J]) {
#pragma unroll
    for (int u = 0; u < NU; u++) {
      const int64_t row = (int64_t)min(base + u * KPI + grp, end - 1) * H; // past the end: read, never used
#pragma unroll
      for (int j = 0; j < J; j++)
        dst[u][j] = __builtin_nontemporal_load(reinterpret_cast<const i32x4*>(src + row + at[j]));
    }
  };
  // A wave's loads return in the order of their issue: wave 0 asks for the query and the new key first (dims lane + 64 i)
  constexpr int D = G * J / 8;           // head dims per lane of wave 0
  i32x4 qp[J];
  float qx[D], qo[D], kx[D], ko[D], cs[D], sn[D]; // value, its pair's other half, cos, signed sin
  bool turned[D];
  if (!APP) {
#pragma unroll
    for (int j = 0; j < J; j++)
      qp[j] = *reinterpret_cast<const i32x4*>(p.q + (int64_t)bh * H + at[j]);
  } else if (wave == 0) {
    const uint16_t* qrow = p.q + (int64_t)bh * H;
    const uint16_t* krow = p.k_new + kv_head * H;
    const int64_t pp = p.emb ? p.pos[p.B_pos == 1 ? 0 : b] : -1;
    const bool rot = pp >= 0 && pp < p.MP; // positions outside the table are left unrotated
    const int half = p.HR >> 1;
#pragma unroll
    for (int i = 0; i < D; i++) {
      const int d = min(lane + 64 * i, H - 1);
      const bool turn = rot && d < p.HR;
      const bool second = p.gptj ? (d & 1) : d >= half;
      const int o = !turn ? d : p.gptj ? d ^ 1 : second ? d - half : d + half;
      const int e = p.gptj ? d >> 1 : second ? d - half : d;
      qx[i] = bf16_bits_to_f32(qrow[d]);
      qo[i] = bf16_bits_to_f32(qrow[o]);
      kx[i] = bf16_bits_to_f32(krow[d]);
      ko[i] = bf16_bits_to_f32(krow[o]);
      cs[i] = sn[i] = 0.f;
      turned[i] = turn;
      if (turn) {
        cs[i] = p.gptj ? p.emb[pp * p.HR + half + e] : p.emb[pp * p.HR + e];
        sn[i] = p.gptj ? p.emb[pp * p.HR + e] : p.emb[((int64_t)p.MP + pp) * p.HR + e];
        if (!second)
          sn[i] = -sn[i];
      }
    }
  }
  load_rows(kb, blockIdx.y * TRIP + wave * WK, p.Smax, kr);
  load_rows(vb, blockIdx.y * TRIP + wave * WK, p.Smax, vr);
  const int len0 = *p.kv_len;
  const int L = max(0, min(len0 + p.kv_len_add, p.Smax));
  const int nk = (APP && len0 >= 0 && len0 < p.Smax) ? len0 : -1; // cache position of the new token
  const int trips = (L + TRIP - 1) / TRIP;
  // the split whose trips contain the new token's position (uniform over the workgroup)
  const bool has_new = APP && nk >= 0 && nk < L && (nk / TRIP) % S == (int)blockIdx.y;
  if (APP) {
    if (wave == 0) {
#pragma unroll
      for (int i = 0; i < D; i++) {
        const int d = lane + 64 * i;
        if (d < H) {
          // rotate_first and rotate_second, the sign in sn
          q_s[d] = (uint16_t)f32_to_bf16_bits(turned[i] ? fmaf(qx[i], cs[i], __fmul_rn(qo[i], sn[i])) : qx[i]);
          k_s[d] = (uint16_t)f32_to_bf16_bits(turned[i] ? fmaf(kx[i], cs[i], __fmul_rn(ko[i], sn[i])) : kx[i]);
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < J; j++)
      qp[j] = *reinterpret_cast<const i32x4*>(q_s + at[j]);
    // one workgroup per KV head appends: the first query head of the group, in the split that reads the position
    if (has_new && hq == hk * (p.Nq / p.Nkv) && tid < C) {
      const int64_t o = (kv_head * p.Smax + nk) * H + tid * 8;
      *reinterpret_cast<i32x4*>(const_cast<uint16_t*>(p.kc) + o) = reinterpret_cast<const i32x4*>(k_s)[tid];
      *reinterpret_cast<i32x4*>(const_cast<uint16_t*>(p.vc) + o) = reinterpret_cast<const i32x4*>(p.v_new + kv_head * H)[tid];
    }
  }
  const uint16_t* mrow = p.mask ? p.mask + (int64_t)b * p.mask_ld : nullptr;
  float m = -3.0e38f, l = 0.f; // m is the same in every lane of the wave
  float acc[J * 8];
#pragma unroll
  for (int e = 0; e < J * 8; e++)
    acc[e] = 0.f;
  // a trip in two halves, as in attn_decode_wide_kernel
  float sc[NU], mx;
  auto scores = [&](int base) {
    if (has_new && nk >= base && nk < base + WK) {
#pragma unroll
      for (int j = 0; j < J; j++) {
        const i32x4 kv = *reinterpret_cast<const i32x4*>(k_s + at[j]);
        const i32x4 vv = *reinterpret_cast<const i32x4*>(p.v_new + kv_head * H + at[j]);
#pragma unroll
        for (int u = 0; u < NU; u++)
#pragma unroll
          for (int r = 0; r < 4; r++) { // (selects, not stores under a condition)
            kr[u][j][r] = nk == base + u * KPI + grp ? kv[r] : kr[u][j][r];
            vr[u][j][r] = nk == base + u * KPI + grp ? vv[r] : vr[u][j][r];
          }
      }
    }
    mx = -3.0e38f;
#pragma unroll
    for (int u = 0; u < NU; u++) {
      const int key = base + u * KPI + grp;
      float d = 0.f;
#pragma unroll
      for (int j = 0; j < J; j++) {
        float dj = 0.f;
#pragma unroll
        for (int r = 0; r < 4; r++)
          dj = dot2_bf16((uint32_t)kr[u][j][r], (uint32_t)qp[j][r], dj);
        d += live[j] ? dj : 0.f;
      }
      d += dpp_mov<0xB1>(d);  // the parts of the key: quad_perm [1,0,3,2], [2,3,0,1], row_half_mirror, row_mirror
      d += dpp_mov<0x4E>(d);
      d += dpp_mov<0x141>(d);
      if (G == 16)
        d += dpp_mov<0x140>(d);
      d *= p.scale;
      if (mrow && key < p.mask_ld && key < L)
        d += bf16_bits_to_f32(mrow[key]);
      sc[u] = key < L ? d : -3.0e38f;
      mx = fmaxf(mx, sc[u]);
    }
  };
  auto sums = [&](int base) {
    const float mn = fmaxf(m, wave_max(mx));
    if (mn > m) { // wave-uniform; rare once the first trips have passed
      const float alpha = __expf(m - mn);
      l *= alpha;
#pragma unroll
      for (int e = 0; e < J * 8; e++)
        acc[e] *= alpha;
      m = mn;
    }
    uint32_t pk[NU / 2], pk2[NU / 2]; // probabilities of the key pairs as packed bf16: the leading bits, the rest
#pragma unroll
    for (int u = 0; u < NU; u++) {
      const int key = base + u * KPI + grp;
      const float pr = key < L ? __expf(sc[u] - m) : 0.f;
      l += pr;
      const uint32_t pb = __float_as_uint(pr) >> 16, p2 = f32_to_bf16_bits(pr - __uint_as_float(pb << 16));
      if (u & 1) {
        pk[u >> 1] |= pb << 16;
        pk2[u >> 1] |= p2 << 16;
      } else {
        pk[u >> 1] = pb;
        pk2[u >> 1] = p2;
      }
      if (base + WK > L && key >= L) { // rows past the end may hold anything, NaN included
#pragma unroll
        for (int j = 0; j < J; j++)
          vr[u][j] = i32x4{0, 0, 0, 0};
      }
    }
#pragma unroll
    for (int h = 0; h < NU / 2; h++)
#pragma unroll
      for (int j = 0; j < J; j++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const uint32_t va = (uint32_t)vr[2 * h][j][r], vb2 = (uint32_t)vr[2 * h + 1][j][r];
          const uint32_t lo = __builtin_amdgcn_perm(vb2, va, 0x05040100u); // (a.dim 2r, b.dim 2r)
          const uint32_t hi = __builtin_amdgcn_perm(vb2, va, 0x07060302u); // (a.dim 2r+1, b.dim 2r+1)
          acc[j * 8 + 2 * r] = dot2_bf16(lo, pk[h], dot2_bf16(lo, pk2[h], acc[j * 8 + 2 * r]));
          acc[j * 8 + 2 * r + 1] = dot2_bf16(hi, pk[h], dot2_bf16(hi, pk2[h], acc[j * 8 + 2 * r + 1]));
        }
  };
  int t = blockIdx.y;
  for (; t + S < trips; t += S) {
    const int base = t * TRIP + wave * WK, next = (t + S) * TRIP + wave * WK;
    scores(base);
    __builtin_amdgcn_sched_barrier(0);
    load_rows(kb, next, L, kr);
    __builtin_amdgcn_sched_barrier(0);
    sums(base);
    __builtin_amdgcn_sched_barrier(0);
    load_rows(vb, next, L, vr);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (t < trips) {
    scores(t * TRIP + wave * WK);
    sums(t * TRIP + wave * WK);
  }
#pragma unroll
  for (int j = 0; j < J; j++) {
    float* dst = &sacc[wave][grp][(j * G + c) * 8];
    *reinterpret_cast<f32x4*>(dst) = f32x4{acc[j * 8], acc[j * 8 + 1], acc[j * 8 + 2], acc[j * 8 + 3]};
    *reinterpret_cast<f32x4*>(dst + 4) = f32x4{acc[j * 8 + 4], acc[j * 8 + 5], acc[j * 8 + 6], acc[j * 8 + 7]};
  }
  const float lw = wave_sum(l) * (1.0f / G); // every key's l sits in its G lanes: counted G times, a power of two
  if (lane == 0) {
    sm[wave] = m;
    sl[wave] = lw;
  }
  __syncthreads();
  float M = fmaxf(fmaxf(sm[0], sm[1]), fmaxf(sm[2], sm[3])), Ls = 0.f, o = 0.f;
  float* st = p.part + ((int64_t)bh * S + blockIdx.y) * (H + 2);
  if (tid < H) {
#pragma unroll
    for (int w = 0; w < 4; w++) {
      float so = 0.f;
#pragma unroll
      for (int i = 0; i < KPI; i++)
        so += sacc[w][i][tid];
      const float wt = __expf(sm[w] - M);
      Ls = fmaf(wt, sl[w], Ls);
      o = fmaf(wt, so, o);
    }
    if (S == 1) {
      p.out[(int64_t)bh * H + tid] = (uint16_t)f32_to_bf16_bits(Ls > 0.f ? o / Ls : 0.f);
    } else { // device scope: written through to the level all XCDs share
      __hip_atomic_store(st + 2 + tid, o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (tid == 0) {
        __hip_atomic_store(st, M, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(st + 1, Ls, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  if (S == 1 || !p.counters) // (without counters attn_hd_merge_kernel follows)
    return;
  // as in attn_finish: own stores acknowledged, barrier, ticket, then the device-scope loads; nobody waits for anybody
  __shared__ int arrived_last;
#pragma unroll
  for (int u = 0; u < NU; u++)
#pragma unroll
    for (int j = 0; j < J; j++)
      asm volatile("" : : "v"(kr[u][j]), "v"(vr[u][j]), "v"(qp[j])); // (see attn_decode_wide_kernel)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0)
    arrived_last = attn_arrive(p.counters, 0, bh, S);
  __syncthreads();
  if (!arrived_last || tid >= H)
    return;
  const float* src = p.part + (int64_t)bh * S * (H + 2);
  float pm[32], pl[32], po[32]; // every load in flight at once (at most 32 splits)
  M = -3.0e38f;
#pragma unroll
  for (int i = 0; i < 32; i++) {
    pm[i] = -3.0e38f;
    pl[i] = po[i] = 0.f;
    if (i < S) {
      pm[i] = __hip_atomic_load(src + i * (H + 2), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      pl[i] = __hip_atomic_load(src + i * (H + 2) + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      po[i] = __hip_atomic_load(src + i * (H + 2) + 2 + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
#pragma unroll
  for (int i = 0; i < 32; i++)
    if (i < S)
      M = fmaxf(M, pm[i]);
  Ls = 0.f;
  o = 0.f;
#pragma unroll
  for (int i = 0; i < 32; i++)
    if (i < S) {
      const float w = __expf(pm[i] - M); // a split without keys carries sum 0 and output 0
      Ls = fmaf(w, pl[i], Ls);
      o = fmaf(w, po[i], o);
    }
  p.out[(int64_t)bh * H + tid] = (uint16_t)f32_to_bf16_bits(Ls > 0.f ? o / Ls : 0.f);
}

// Without arrival counters: one wave per query, the splits' (maximum, sum, output) states, in split order, become the
// normalised output -- the sums of the merge above.
__global__ void __launch_bounds__(64)
attn_hd_merge_kernel(const AttnGenParams p) {
  const int lane = threadIdx.x;
  const int64_t qi = blockIdx.x;
  const int H = p.H;
  const float* st = p.part + qi * p.splits * (int64_t)(H + 2);
  float M = -3.0e38f;
  for (int i = 0; i < p.splits; i++)
    M = fmaxf(M, st[i * (H + 2)]);
  float Ls = 0.f, o[4] = {0.f, 0.f, 0.f, 0.f};
  for (int i = 0; i < p.splits; i++) {
    const float* si = st + i * (int64_t)(H + 2);
    const float w = __expf(si[0] - M); // a split without keys carries sum 0 and output 0
    Ls = fmaf(w, si[1], Ls);
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (lane + 64 * j < H)
        o[j] = fmaf(w, si[2 + lane + 64 * j], o[j]);
  }
  uint16_t* orow = p.out + qi * H;
#pragma unroll
  for (int j = 0; j < 4; j++)
    if (lane + 64 * j < H)
      orow[lane + 64 * j] = (uint16_t)f32_to_bf16_bits(Ls > 0.f ? o[j] / Ls : 0.f);
}

static int attn_generic_launch(const char* who, AttnGenParams& p, hipStream_t stream, void* ws = nullptr,
                               int64_t ws_bytes = 0, AttnCounters counters = {}) {
  TPPX_REQUIRE(p.H >= 8 && p.H <= 256 && p.H % 8 == 0, TPPX_EUNSUPPORTED,
               "%s: head size %d (multiples of 8 up to 256)", who, p.H);
  const int64_t queries = (int64_t)p.B * p.S * p.Nq;
  p.splits = 1;
  if (p.kv_len && p.S == 1 && env_int("TPPX_ATTN_GENERIC_ROWS", 1) != 0) {
    TPPX_REQUIRE(queries < ((int64_t)1 << 31), TPPX_ESHAPE, "%s: problem too large", who);
    // Workgroups per (sequence, head), as for 128-wide heads: two trips each at the cache's capacity (the length itself is
    // a device scalar: splits whose trips lie past the keys leave empty states), but no fewer than 288 workgroups and no
    // more than 512 in all; at most one per trip and 32; of that count, one less and one more the one that fills the rounds
    // of 256 best (192 heads of 80, 3000 keys: three 39.0 us, four 34.2; 160: four 31.4, three 29.1; 224 heads of 64: three
    // 33.0, two 31.6).  One for caches of three trips (50 keys in 178 of one sequence: 4.6 us against 6.5 with two), from
    // 256 heads on (16 x 16 x 700 keys: 30.5 against 31.6 with two), more than 128 wide, where a workgroup moves twice the
    // bytes, from 160 on (208 heads of 256, 3000 keys: 98 against 108 with three, 160 heads 80 against 83 with four; 96
    // heads 76 against 49 with five), and where the workspace cannot hold the states.
    const int64_t trip = p.H <= 128 ? 128 : 64, most = ((int64_t)p.Smax + trip - 1) / trip;
    int64_t want = env_int("TPPX_ATTN_GENERIC_SPLITS", 0);
    if (want <= 0 && (most <= 3 || queries >= (p.H > 128 ? 160 : 256))) {
      want = 1;
    } else if (want <= 0) {
      const int64_t least = (288 + queries - 1) / queries, w = std::max(least, std::min((most + 1) / 2, (512 + queries - 1) / queries));
      const auto fill = [&](int64_t n) { return (double)(n * queries) / (double)((n * queries + 255) / 256); };
      want = w;
      for (int64_t n = std::max(least, w - 1); n <= std::min(w + 1, std::max(w, (most + 1) / 2)); n++)
        if (n < want ? fill(n) >= fill(want) : fill(n) > fill(want))
          want = n;
    }
    want = std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>(want, 32), most));
    if (want > 1 && ws && queries * want * (p.H + 2) * (int64_t)sizeof(float) <= ws_bytes) {
      p.splits = (int)want;
      p.part = (float*)ws;
      p.counters = env_int("TPPX_ATTN_ONE_LAUNCH", 1) != 0 ? counters.of(queries) : nullptr;
    }
    const dim3 grid((unsigned)queries, (unsigned)p.splits);
    auto go = [&](auto app) {
      constexpr bool APP = decltype(app)::value;
      if (p.H <= 64)
        attn_hd_step_kernel<8, 1, 4, APP><<<grid, dim3(256), 0, stream>>>(p);
      else if (p.H <= 128)
        attn_hd_step_kernel<16, 1, 8, APP><<<grid, dim3(256), 0, stream>>>(p);
      else
        attn_hd_step_kernel<16, 2, 4, APP><<<grid, dim3(256), 0, stream>>>(p);
    };
    if (p.k_new)
      go(std::true_type{});
    else
      go(std::false_type{});
    int rc = check_hip(hipGetLastError(), who);
    if (rc || p.splits == 1 || p.counters)
      return rc;
    attn_hd_merge_kernel<<<dim3((unsigned)queries), dim3(64), 0, stream>>>(p);
    return check_hip(hipGetLastError(), who);
  }
  TPPX_REQUIRE(!p.k_new, TPPX_EUNSUPPORTED, "%s: the single-query kernel is switched off", who);
  const int64_t waves = queries;
  TPPX_REQUIRE(waves > 0 && (waves + 3) / 4 < ((int64_t)1 << 31), TPPX_ESHAPE, "%s: problem too large", who);
  attn_generic_kernel<<<dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, stream>>>(p);
  return check_hip(hipGetLastError(), who);
}

static int run_attn_decode(const char* who, const void* q, const void* kcache, const void* vcache, const void* mask,
                           int64_t mask_ld, const void* kv_len_dev, int64_t kv_len_add, void* out, int64_t B, int64_t Nq,
                           int64_t Nkv, int64_t H, int64_t Smax, void* ws, int64_t ws_bytes, const AttnCounters& counters,
                           tppx_stream_t stream) {
  if (int rc = check_counters(who, counters))
    return rc;
  TPPX_REQUIRE(q && kcache && vcache && kv_len_dev && out, TPPX_EINVAL, "%s: null pointer", who);
  TPPX_REQUIRE(aligned16(q) && aligned16(kcache) && aligned16(vcache) && aligned16(out), TPPX_EINVAL,
               "%s: pointer not 16-byte aligned", who);
  TPPX_REQUIRE(B > 0 && Nq > 0 && Nkv > 0 && Nq % Nkv == 0 && Smax > 0 && B * Nq < (1 << 30), TPPX_ESHAPE,
               "%s: bad shape B=%ld Nq=%ld Nkv=%ld Smax=%ld", who, (long)B, (long)Nq, (long)Nkv, (long)Smax);
  TPPX_REQUIRE(ws_bytes >= 0 && (ws_bytes == 0 || ws), TPPX_EINVAL, "%s: workspace size given with a null workspace", who);
  if (H != 128) { // other head sizes: the plain kernel
    AttnGenParams g;
    memset(&g, 0, sizeof(g));
    g.q = (const uint16_t*)q; g.kc = (const uint16_t*)kcache; g.vc = (const uint16_t*)vcache; g.mask = (const uint16_t*)mask;
    g.kv_len = (const int32_t*)kv_len_dev; g.kv_len_add = (int)kv_len_add; g.out = (uint16_t*)out;
    g.B = (int)B; g.S = 1; g.Nq = (int)Nq; g.Nkv = (int)Nkv; g.H = (int)H; g.Smax = (int)Smax; g.mask_ld = (int)mask_ld;
    g.scale = 1.0f / sqrtf((float)H);
    return attn_generic_launch(who, g, (hipStream_t)stream, ws, ws_bytes, counters);
  }
  AttnParams p;
  memset(&p, 0, sizeof(p));
  p.q = (const uint16_t*)q; p.kc = (const uint16_t*)kcache; p.vc = (const uint16_t*)vcache;
  p.mask = (const uint16_t*)mask; p.kv_len = (const int32_t*)kv_len_dev; p.kv_len_add = (int)kv_len_add; p.out = (uint16_t*)out;
  p.B = (int)B; p.Nq = (int)Nq; p.Nkv = (int)Nkv; p.Smax = (int)Smax; p.mask_ld = (int)mask_ld;
  p.scale = 1.0f / sqrtf((float)H);
  return attn_decode_launch(who, p, false, B, Nq, Smax, ws, ws_bytes, counters, (hipStream_t)stream);
}

static int run_attn_decode_rotary(const char* who, const void* q, const void* k, const void* v, const void* emb_pos,
                                  const void* pos, int64_t B_pos, int64_t MP, int64_t HR, void* kcache, void* vcache,
                                  const void* mask, int64_t mask_ld, const void* kv_len_dev, void* out, int64_t B,
                                  int64_t Nq, int64_t Nkv, int64_t H, int64_t Smax, void* ws, int64_t ws_bytes,
                                  const AttnCounters& counters, tppx_stream_t stream) {
  if (int rc = check_counters(who, counters))
    return rc;
  TPPX_REQUIRE(q && k && v && pos && kcache && vcache && kv_len_dev && out, TPPX_EINVAL, "%s: null pointer", who);
  TPPX_REQUIRE(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(kcache) && aligned16(vcache) && aligned16(out) &&
                   (!emb_pos || aligned16(emb_pos)),
               TPPX_EINVAL, "%s: pointer not 16-byte aligned", who);
  TPPX_REQUIRE(H == 128 && (!emb_pos || HR == 128), TPPX_EUNSUPPORTED,
               "%s: head size %ld / rotary size %ld (only 128 with a full-width rotation is built)", who, (long)H, (long)HR);
  TPPX_REQUIRE(B > 0 && Nq > 0 && Nkv > 0 && Nq % Nkv == 0 && Smax > 0 && B * Nq < (1 << 30) && (B_pos == 1 || B_pos == B) &&
                   (!emb_pos || MP > 0),
               TPPX_ESHAPE, "%s: bad shape B=%ld Nq=%ld Nkv=%ld Smax=%ld B_pos=%ld MP=%ld", who, (long)B, (long)Nq,
               (long)Nkv, (long)Smax, (long)B_pos, (long)MP);
  TPPX_REQUIRE(ws_bytes >= 0 && (ws_bytes == 0 || ws), TPPX_EINVAL, "%s: workspace size given with a null workspace", who);
  AttnParams p;
  memset(&p, 0, sizeof(p));
  p.q = (const uint16_t*)q; p.kc = (const uint16_t*)kcache; p.vc = (const uint16_t*)vcache;
  p.mask = (const uint16_t*)mask; p.kv_len = (const int32_t*)kv_len_dev; p.kv_len_add = 1; p.out = (uint16_t*)out;
  p.B = (int)B; p.Nq = (int)Nq; p.Nkv = (int)Nkv; p.Smax = (int)Smax; p.mask_ld = (int)mask_ld;
  p.scale = 1.0f / sqrtf((float)H);
  p.k_new = (const uint16_t*)k; p.v_new = (const uint16_t*)v; p.emb = (const float*)emb_pos; p.pos = (const int64_t*)pos;
  p.MP = (int)MP; p.B_pos = (int)B_pos;
  return attn_decode_launch(who, p, true, B, Nq, Smax, ws, ws_bytes, counters, (hipStream_t)stream);
}

static int run_attn_decode_append(const char* who, const void* q, const void* k, const void* v, const void* emb_pos,
                                  int gptj, const void* pos, int64_t B_pos, int64_t MP, int64_t HR, void* kcache,
                                  void* vcache, const void* mask, int64_t mask_ld, const void* kv_len_dev, void* out,
                                  int64_t B, int64_t Nq, int64_t Nkv, int64_t H, int64_t Smax, void* ws, int64_t ws_bytes,
                                  const AttnCounters& counters, tppx_stream_t stream) {
  if (int rc = check_counters(who, counters))
    return rc;
  TPPX_REQUIRE(q && k && v && pos && kcache && vcache && kv_len_dev && out, TPPX_EINVAL, "%s: null pointer", who);
  TPPX_REQUIRE(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(kcache) && aligned16(vcache) && aligned16(out),
               TPPX_EINVAL, "%s: pointer not 16-byte aligned", who);
  TPPX_REQUIRE(H != 128, TPPX_EUNSUPPORTED, "%s: 128-wide heads have kernels of their own", who);
  TPPX_REQUIRE(B > 0 && Nq > 0 && Nkv > 0 && Nq % Nkv == 0 && Smax > 0 && B * Nq < (1 << 30) && (B_pos == 1 || B_pos == B),
               TPPX_ESHAPE, "%s: bad shape B=%ld Nq=%ld Nkv=%ld Smax=%ld B_pos=%ld", who, (long)B, (long)Nq, (long)Nkv,
               (long)Smax, (long)B_pos);
  TPPX_REQUIRE(!emb_pos || (HR > 0 && HR <= H && HR % 16 == 0 && MP > 0), TPPX_ESHAPE,
               "%s: rotary_dim=%ld must be a multiple of 16 and <= H=%ld", who, (long)HR, (long)H);
  TPPX_REQUIRE(ws_bytes >= 0 && (ws_bytes == 0 || ws), TPPX_EINVAL, "%s: workspace size given with a null workspace", who);
  AttnGenParams g;
  memset(&g, 0, sizeof(g));
  g.q = (const uint16_t*)q; g.kc = (const uint16_t*)kcache; g.vc = (const uint16_t*)vcache; g.mask = (const uint16_t*)mask;
  g.kv_len = (const int32_t*)kv_len_dev; g.kv_len_add = 1; g.out = (uint16_t*)out;
  g.B = (int)B; g.S = 1; g.Nq = (int)Nq; g.Nkv = (int)Nkv; g.H = (int)H; g.Smax = (int)Smax; g.mask_ld = (int)mask_ld;
  g.scale = 1.0f / sqrtf((float)H);
  g.k_new = (const uint16_t*)k; g.v_new = (const uint16_t*)v; g.emb = (const float*)emb_pos; g.pos = (const int64_t*)pos;
  g.MP = (int)MP; g.HR = emb_pos ? (int)HR : 0; g.B_pos = (int)B_pos; g.gptj = gptj != 0;
  return attn_generic_launch(who, g, (hipStream_t)stream, ws, ws_bytes, counters);
}

extern "C" int tppx_attn_decode(const void* q, const void* kcache, const void* vcache, const void* mask, int64_t mask_ld,
                                const void* kv_len_dev, int64_t kv_len_add, void* out, int64_t B, int64_t Nq, int64_t Nkv,
                                int64_t H, int64_t Smax, void* ws, int64_t ws_bytes, tppx_stream_t stream) {
  return run_attn_decode("tppx_attn_decode", q, kcache, vcache, mask, mask_ld, kv_len_dev, kv_len_add, out, B, Nq, Nkv, H,
                         Smax, ws, ws_bytes, {}, stream);
}

extern "C" int tppx_attn_decode_counted(const void* q, const void* kcache, const void* vcache, const void* mask,
                                        int64_t mask_ld, const void* kv_len_dev, int64_t kv_len_add, void* out, int64_t B,
                                        int64_t Nq, int64_t Nkv, int64_t H, int64_t Smax, void* ws, int64_t ws_bytes,
                                        void* counters, int64_t counter_bytes, tppx_stream_t stream) {
  return run_attn_decode("tppx_attn_decode_counted", q, kcache, vcache, mask, mask_ld, kv_len_dev, kv_len_add, out, B, Nq,
                         Nkv, H, Smax, ws, ws_bytes, {counters, counter_bytes}, stream);
}

extern "C" int tppx_attn_decode_rotary(const void* q, const void* k, const void* v, const void* emb_pos, const void* pos,
                                       int64_t B_pos, int64_t MP, int64_t HR, void* kcache, void* vcache,
                                       const void* mask, int64_t mask_ld, const void* kv_len_dev, void* out, int64_t B,
                                       int64_t Nq, int64_t Nkv, int64_t H, int64_t Smax, void* ws, int64_t ws_bytes,
                                       tppx_stream_t stream) {
  return run_attn_decode_rotary("tppx_attn_decode_rotary", q, k, v, emb_pos, pos, B_pos, MP, HR, kcache, vcache, mask,
                                mask_ld, kv_len_dev, out, B, Nq, Nkv, H, Smax, ws, ws_bytes, {}, stream);
}

extern "C" int tppx_attn_decode_rotary_counted(const void* q, const void* k, const void* v, const void* emb_pos,
                                               const void* pos, int64_t B_pos, int64_t MP, int64_t HR, void* kcache,
                                               void* vcache, const void* mask, int64_t mask_ld, const void* kv_len_dev,
                                               void* out, int64_t B, int64_t Nq, int64_t Nkv, int64_t H, int64_t Smax,
                                               void* ws, int64_t ws_bytes, void* counters, int64_t counter_bytes,
                                               tppx_stream_t stream) {
  return run_attn_decode_rotary("tppx_attn_decode_rotary_counted", q, k, v, emb_pos, pos, B_pos, MP, HR, kcache, vcache,
                                mask, mask_ld, kv_len_dev, out, B, Nq, Nkv, H, Smax, ws, ws_bytes,
                                {counters, counter_bytes}, stream);
}

extern "C" int tppx_attn_decode_append(const void* q, const void* k, const void* v, const void* emb_pos, int gptj,
                                       const void* pos, int64_t B_pos, int64_t MP, int64_t HR, void* kcache, void* vcache,
                                       const void* mask, int64_t mask_ld, const void* kv_len_dev, void* out, int64_t B,
                                       int64_t Nq, int64_t Nkv, int64_t H, int64_t Smax, void* ws, int64_t ws_bytes,
                                       tppx_stream_t stream) {
  return run_attn_decode_append("tppx_attn_decode_append", q, k, v, emb_pos, gptj, pos, B_pos, MP, HR, kcache, vcache,
                                mask, mask_ld, kv_len_dev, out, B, Nq, Nkv, H, Smax, ws, ws_bytes, {}, stream);
}

extern "C" int tppx_attn_decode_append_counted(const void* q, const void* k, const void* v, const void* emb_pos, int gptj,
                                               const void* pos, int64_t B_pos, int64_t MP, int64_t HR, void* kcache,
                                               void* vcache, const void* mask, int64_t mask_ld, const void* kv_len_dev,
                                               void* out, int64_t B, int64_t Nq, int64_t Nkv, int64_t H, int64_t Smax,
                                               void* ws, int64_t ws_bytes, void* counters, int64_t counter_bytes,
                                               tppx_stream_t stream) {
  return run_attn_decode_append("tppx_attn_decode_append_counted", q, k, v, emb_pos, gptj, pos, B_pos, MP, HR, kcache,
                                vcache, mask, mask_ld, kv_len_dev, out, B, Nq, Nkv, H, Smax, ws, ws_bytes,
                                {counters, counter_bytes}, stream);
}

extern "C" int tppx_attn_prefill(const void* q, const void* kcache, const void* vcache, const void* mask,
                                 int64_t mask_ld, int64_t past_len, void* out, int64_t B, int64_t S, int64_t Nq,
                                 int64_t Nkv, int64_t H, int64_t Smax, tppx_stream_t stream) {
  const char* who = "tppx_attn_prefill";
  TPPX_REQUIRE(q && kcache && vcache && out, TPPX_EINVAL, "%s: null pointer", who);
  TPPX_REQUIRE(aligned16(q) && aligned16(kcache) && aligned16(vcache) && aligned16(out), TPPX_EINVAL,
               "%s: pointer not 16-byte aligned", who);
  TPPX_REQUIRE(B > 0 && S > 0 && Nq > 0 && Nkv > 0 && Nq % Nkv == 0 && Smax > 0 && B * Nq < 65536 &&
                   S < ((int64_t)1 << 24) && Smax < ((int64_t)1 << 30),
               TPPX_ESHAPE, "%s: bad shape B=%ld S=%ld Nq=%ld Nkv=%ld Smax=%ld", who, (long)B, (long)S, (long)Nq,
               (long)Nkv, (long)Smax);
  TPPX_REQUIRE(past_len >= 0 && past_len + S <= Smax, TPPX_ESHAPE,
               "%s: %ld cached + %ld new keys exceed the cache capacity %ld", who, (long)past_len, (long)S, (long)Smax);
  TPPX_REQUIRE(!mask || mask_ld > 0, TPPX_EINVAL, "%s: mask given with mask_ld=%ld", who, (long)mask_ld);
  if (H != 128 && env_int("TPPX_ATTN_PREFILL_MFMA", 1) == 0) { // other head sizes on the plain kernel
    AttnGenParams g;
    memset(&g, 0, sizeof(g));
    g.q = (const uint16_t*)q; g.kc = (const uint16_t*)kcache; g.vc = (const uint16_t*)vcache; g.mask = (const uint16_t*)mask;
    g.out = (uint16_t*)out;
    g.B = (int)B; g.S = (int)S; g.Nq = (int)Nq; g.Nkv = (int)Nkv; g.H = (int)H; g.Smax = (int)Smax; g.mask_ld = (int)mask_ld;
    g.past = (int)past_len;
    g.scale = 1.0f / sqrtf((float)H);
    return attn_generic_launch(who, g, (hipStream_t)stream);
  }
  AttnPrefillParams p;
  memset(&p, 0, sizeof(p));
  p.q = (const uint16_t*)q; p.kc = (const uint16_t*)kcache; p.vc = (const uint16_t*)vcache;
  p.mask = (const uint16_t*)mask; p.out = (uint16_t*)out;
  p.B = (int)B; p.S = (int)S; p.Nq = (int)Nq; p.Nkv = (int)Nkv; p.Smax = (int)Smax; p.mask_ld = (int)mask_ld;
  p.past = (int)past_len;
  p.scale = 1.0f / sqrtf((float)H);
  p.H = (int)H;
  if (H != 128) { // other head sizes: the same kernel over a padded head size
    TPPX_REQUIRE(H >= 8 && H <= 256 && H % 8 == 0, TPPX_EUNSUPPORTED,
                 "%s: head size %ld (multiples of 8 up to 256)", who, (long)H);
    const int hd = H <= 64 ? 64 : H <= 128 ? 128 : 256;
    const long wgs2h = ((S + 127) / 128) * B * Nq;
    const bool two = hd != 256 && S > 64 && env_int("TPPX_ATTN_QG", wgs2h >= 512 ? 2 : 1) == 2;
    const dim3 grid((unsigned)((S + (two ? 127 : 63)) / (two ? 128 : 64)), (unsigned)(B * Nq));
    const int64_t tiles = (past_len + S + 63) / 64;
    // One workgroup per CU or less: two teams over the key tiles from five of them on (3: 6.0 us either way at 64 wide, 7.4
    // against 7.5 at 80; 5: 8.0 -> 7.4 and 10.2 -> 9.7).  Beyond 256 workgroups they share CUs as it is (512 of 80 wide 26.6
    // us, in teams 31.6), and at 256 wide the LDS reads of one team fill a CU (13 tiles 35.0 against 33.8, 5 tiles 17.6
    // against 18.4).
    const bool teams = hd != 256 && !two && tiles > 1 &&
                       env_int("TPPX_ATTN_TEAMS", (int64_t)grid.x * grid.y <= 256 && tiles >= 5 ? 2 : 1) == 2;
    hipError_t e = hipSuccess;
#define TPPX_AP_HD(QG_, HD_, T_)                                                                                      \
  do {                                                                                                               \
    const size_t lds = (size_t)T_ * (64 * (HD_ + 8) + HD_ * AP_VP) * sizeof(uint16_t);                               \
    e = allow_dynamic_lds(reinterpret_cast<const void*>(attn_prefill_hd_kernel<QG_, HD_, T_>), lds);                 \
    if (e == hipSuccess)                                                                                             \
      attn_prefill_hd_kernel<QG_, HD_, T_><<<grid, dim3(256 * T_), lds, (hipStream_t)stream>>>(p);                   \
  } while (0)
    if (hd == 64 && two)
      TPPX_AP_HD(2, 64, 1);
    else if (hd == 64 && teams)
      TPPX_AP_HD(1, 64, 2);
    else if (hd == 64)
      TPPX_AP_HD(1, 64, 1);
    else if (hd == 128 && two)
      TPPX_AP_HD(2, 128, 1);
    else if (hd == 128 && teams)
      TPPX_AP_HD(1, 128, 2);
    else if (hd == 128)
      TPPX_AP_HD(1, 128, 1);
    else
      TPPX_AP_HD(1, 256, 1);
#undef TPPX_AP_HD
    if (e != hipSuccess)
      return check_hip(e, who);
    return check_hip(hipGetLastError(), who);
  }
  // 128 queries per workgroup from 400 of them on (3 x 600 tokens behind 500 x 28 heads, 420 of them: 15 % faster); below that
  // twice as many of 64 (1000 tokens x 32 heads, 256: 12 % faster, 2 x 700, 384: 7 %)
  const int64_t wgs = (S + 127) / 128 * B * Nq;
  const bool wide = env_int("TPPX_ATTN_QG", wgs >= 400 ? 2 : 1) == 2;
  auto go = [&](auto kern, int64_t rows, int threads) -> hipError_t {
    kern<<<dim3((unsigned)((S + rows - 1) / rows * B * Nq)), dim3(threads), 0, (hipStream_t)stream>>>(p);
    return hipGetLastError();
  };
  return check_hip(wide && S > 64 ? go(attn_prefill_kernel<8>, 128, 512) : go(attn_prefill_kernel<4>, 64, 256), who);
}
