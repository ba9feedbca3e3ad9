// llm_ops.hip — hand-written CDNA4 (gfx950 / MI355X) kernels for the
// Llama-3.2 / Gemma-2 decode + prefill forward pass.
//
// Design notes (MI355X-first):
//  - wave64 everywhere; block sizes are multiples of 64
//  - bf16 I/O, fp32 accumulation; all bf16 traffic vectorized 16 B/lane
//  - products of one row, of few and of many are in gemv.hip, row_gemm.hip
//    and gemm_prompt.hip, attention in attn_decode.hip and attn_prefill.hip
//  - attention never materializes QK^T: online softmax in registers
//  - KV cache is a preallocated pool, written in place (decode: inside
//    the fused attention kernel; prefill: k_rope_cache) — replaces the
//    reference's O(T^2) concat cache (llama3.2_model.py:325)
//  - every kernel is hipGraph-capture-safe (no mallocs/syncs; sequence
//    position and sampled token ids live in device memory)
//
// What stands here for the reference's GPU pieces:
//  K1 softmax RawKernel      -> online softmax in k_attn_dec /
//                               k_attn_rows / k_attn
//  K2 cuBLAS GEMM/GEMV       -> k_gemv (decode), k_row_gemm (few rows),
//                               k_gemm_prompt (prefill)
//  K3 elementwise ufuncs     -> fused GEMV staging (NORM/GLU/NORM2), epilogues
//                               of products, k_rmsnorm, k_softcap, k_addinto,
//                               k_glu
//  K4 KV concat              -> in-place pool writes
//  K5 repeat_kv              -> attention indexes kv_head = q_head/groups
//  K7 torch.multinomial      -> k_logit_max + k_sample_pick (last-block commit)

#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstdio>
#include <cstdlib>

#include "common.h"
#include "gemv.h"

DEVINL float stage_red_sum(float* red) {
  const int nw = blockDim.x >> 6;
  float t = 0.f;
  for (int w = 0; w < nw; w++) t += red[w];
  return t;
}

typedef uint32_t u4v __attribute__((ext_vector_type(4)));  // = u4v_ alias

// ====================================================================
// Multi-x fp8 GEMV (batched decode, B = 2..8 lockstep sequences):
// ONE non-temporal weight stream feeds B accumulators — weight reuse
// turns B-way decode into ~single-sequence step time (the 128-row MFMA
// GEMM path wastes >90% of each tile at B<=8).  All staging modes of
// the single-x GEMV, applied per row; XF32 stages fp32 pairs for
// fp32 FMAs (LDS B*K*4), falling back to bf16 staging (B*K*2) for
// deep-K shapes.  BT = compile-time row capacity (2/4/8); the actual
// B <= BT, with clamped source rows.
// ====================================================================

// per-row staging into xs + b*K (f32 or bf16 element type)
template <bool XF32>
DEVINL void gemv_stage_mx_row(char* smem, int b, const u16* xb,
                              const u16* x2b, const float* g,
                              const float* g2, u16* houtb, int K, int BT,
                              int stage, int act, float eps, float escale,
                              float* red, bool persist) {
  const int STRIDE = blockDim.x * 8;
  float* xf = (float*)smem + (size_t)b * K;
  u16* xh = (u16*)smem + (size_t)b * K;
#define MXSTORE(i, v) do { if (XF32) xf[i] = (v); else xh[i] = f2b(v); } while (0)
  if (stage == STAGE_RAW || stage == STAGE_NORM ||
      stage == STAGE_NORM_EMBED) {
    float ss = 0.f;
    for (int i = threadIdx.x * 8; i < K; i += STRIDE) {
      s8v v = *(const s8v*)(xb + i);
#pragma unroll
      for (int j = 0; j < 8; j++) {
        float f = b2f(((u16*)&v)[j]);
        if (stage == STAGE_NORM_EMBED) {
          f = b2f(f2b(f * escale));
          if (persist) houtb[i + j] = f2b(f);
        }
        MXSTORE(i + j, f);
        ss += f * f;
      }
    }
    if (stage == STAGE_RAW) return;
    ss = wave_reduce_sum(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    float rnorm = rsqrtf(stage_red_sum(red) / (float)K + eps);
    __syncthreads();  // red reused by the next row's reduction
    for (int i = threadIdx.x * 8; i < K; i += STRIDE) {
#pragma unroll
      for (int j = 0; j < 8; j++) {
        float f = (XF32 ? xf[i + j] : b2f(xh[i + j])) * rnorm * g[i + j];
        MXSTORE(i + j, f);
      }
    }
  } else if (stage == STAGE_GLU) {
    for (int i = threadIdx.x * 8; i < K; i += STRIDE) {
      s8v gv = *(const s8v*)(xb + i);
      s8v uv = *(const s8v*)(x2b + i);
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const float a = gate_act(b2f(((u16*)&gv)[j]), act);
        MXSTORE(i + j, a * b2f(((u16*)&uv)[j]));
      }
    }
  } else if (stage == STAGE_NORM2) {
    const u16* h = x2b;
    float ss = 0.f;
    for (int i = threadIdx.x * 8; i < K; i += STRIDE) {
      s8v v = *(const s8v*)(xb + i);
#pragma unroll
      for (int j = 0; j < 8; j++) {
        float f = b2f(((u16*)&v)[j]);
        ss += f * f;
      }
    }
    ss = wave_reduce_sum(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    float rnorm_a = rsqrtf(stage_red_sum(red) / (float)K + eps);
    __syncthreads();
    float ss2 = 0.f;
    for (int i = threadIdx.x * 8; i < K; i += STRIDE) {
      s8v v = *(const s8v*)(xb + i);
      s8v hv = *(const s8v*)(h + i);
      f4v ga = *(const f4v*)(g + i);
      f4v gb = *(const f4v*)(g + i + 4);
      u16 o[8];
#pragma unroll
      for (int j = 0; j < 8; j++) {
        float f = b2f(((u16*)&v)[j]) * rnorm_a * (j < 4 ? ga[j] : gb[j - 4])
                  + b2f(((u16*)&hv)[j]);
        o[j] = f2b(f);
        float fr = b2f(o[j]);
        MXSTORE(i + j, fr);
        ss2 += fr * fr;
      }
      if (persist) *(s8v*)(houtb + i) = *(s8v*)o;
    }
    ss2 = wave_reduce_sum(ss2);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss2;
    __syncthreads();
    float rnorm_b = rsqrtf(stage_red_sum(red) / (float)K + eps);
    __syncthreads();
    for (int i = threadIdx.x * 8; i < K; i += STRIDE) {
#pragma unroll
      for (int j = 0; j < 8; j++) {
        float f = (XF32 ? xf[i + j] : b2f(xh[i + j])) * rnorm_b * g2[i + j];
        MXSTORE(i + j, f);
      }
    }
  }
#undef MXSTORE
}

template <int BT, bool XF32>
__global__ void __launch_bounds__(256)
k_gemv_fp8_mx(const uint8_t* __restrict__ W,
              const float* __restrict__ scales, const u16* __restrict__ x,
              long xstride, const u16* __restrict__ x2, long x2stride,
              const float* __restrict__ g, const float* __restrict__ g2,
              void* __restrict__ y, long ystride,
              const u16* __restrict__ res, long rstride,
              u16* __restrict__ hout, long hstride, int N, int K, int B,
              int stage, int act, float eps, int out_f32, float softcap,
              float escale) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* red = (float*)(smem + (size_t)BT * K * (XF32 ? 4 : 2));
  for (int b = 0; b < BT; b++) {
    int bs = b < B ? b : B - 1;  // clamp padded rows to a valid source
    const u16* xb = x + (size_t)bs * xstride;
    if (stage == STAGE_NORM_EMBED)  // x = table, x2 = per-row token ids
      xb = x + (size_t)((const int*)x2)[bs] * (size_t)K;
    const u16* x2b = (stage == STAGE_NORM_EMBED || x2 == nullptr)
                         ? nullptr : x2 + (size_t)bs * x2stride;
    u16* houtb = hout ? hout + (size_t)bs * hstride : nullptr;
    __syncthreads();
    gemv_stage_mx_row<XF32>(smem, b, xb, x2b, g, g2, houtb, K, BT, stage,
                            act, eps, escale, red, blockIdx.x == 0);
  }
  __syncthreads();

  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int wpb = blockDim.x >> 6;
  const float* xsf = (const float*)smem;
  const u16* xsh = (const u16*)smem;
  for (int row = blockIdx.x * wpb + wave; row < N; row += gridDim.x * wpb) {
    const uint8_t* Wr = W + (size_t)row * K;
    f2v a0[BT], a1[BT];
#pragma unroll
    for (int b = 0; b < BT; b++) {
      a0[b] = (f2v){0.f, 0.f};
      a1[b] = (f2v){0.f, 0.f};
    }
    for (int k = lane * 16; k < K; k += 1024) {
      u4v w0 = __builtin_nontemporal_load((const u4v*)(Wr + k));
#pragma unroll
      for (int q = 0; q < 4; q++) {
        f2v ca = __builtin_amdgcn_cvt_pk_f32_fp8(w0[q], false);
        f2v cb = __builtin_amdgcn_cvt_pk_f32_fp8(w0[q], true);
#pragma unroll
        for (int b = 0; b < BT; b++) {
          f2v xa, xb2;
          if (XF32) {
            xa = *(const f2v*)(xsf + (size_t)b * K + k + q * 4);
            xb2 = *(const f2v*)(xsf + (size_t)b * K + k + q * 4 + 2);
          } else {
            const u16* p = xsh + (size_t)b * K + k + q * 4;
            xa = (f2v){b2f(p[0]), b2f(p[1])};
            xb2 = (f2v){b2f(p[2]), b2f(p[3])};
          }
          a0[b] += ca * xa;
          a1[b] += cb * xb2;
        }
      }
    }
    const float sc = scales[row];
#pragma unroll
    for (int b = 0; b < BT; b++) {
      f2v s = a0[b] + a1[b];
      float acc = wave_reduce_sum(s[0] + s[1]) * sc;
      if (lane == 0 && b < B) {
        if (softcap > 0.f) acc = softcap * tanhf(acc / softcap);
        if (res && stage != STAGE_NORM2 && stage != STAGE_NORM_EMBED)
          acc += b2f(res[(size_t)b * rstride + row]);
        if (out_f32) ((float*)y)[(size_t)b * ystride + row] = acc;
        else ((u16*)y)[(size_t)b * ystride + row] = f2b(acc);
      }
    }
  }
}

extern "C" hipError_t launch_gemv_fp8_mx(
    const void* W, const void* scales, const void* x, long xstride,
    const void* x2, long x2stride, const void* g, const void* g2, void* y,
    long ystride, const void* res, long rstride, void* hout, long hstride,
    int N, int K, int B, int stage, int act, float eps, int out_f32,
    float softcap, float escale, hipStream_t stream) {
  if (B < 1 || B > 8 || K % 16 != 0) return hipErrorInvalidValue;
  int BT = B <= 2 ? 2 : (B <= 4 ? 4 : 8);
  bool xf32 = ((size_t)BT * K * 4 + 64) <= 128 * 1024;
  size_t lds = (size_t)BT * K * (xf32 ? 4 : 2) + 64;
  if (lds > 160 * 1024) return hipErrorInvalidValue;
  static bool raised = false;
  if (lds > 65536 && !raised) {
#define MXRAISE(BTV, XFV)                                                   \
    hipFuncSetAttribute((const void*)&k_gemv_fp8_mx<BTV, XFV>,              \
                        hipFuncAttributeMaxDynamicSharedMemorySize,         \
                        160 * 1024)
    MXRAISE(2, true); MXRAISE(2, false);
    MXRAISE(4, true); MXRAISE(4, false);
    MXRAISE(8, true); MXRAISE(8, false);
#undef MXRAISE
    raised = true;
  }
  int threads = 256;
  int wpb = threads / 64;
  int blocks = (N + wpb - 1) / wpb;
  if (blocks > 1024) blocks = 1024;
#define MX_CASE(BTV, XFV)                                                   \
  hipLaunchKernelGGL((k_gemv_fp8_mx<BTV, XFV>), dim3(blocks),               \
                     dim3(threads), lds, stream, (const uint8_t*)W,         \
                     (const float*)scales, (const u16*)x, xstride,          \
                     (const u16*)x2, x2stride, (const float*)g,             \
                     (const float*)g2, y, ystride, (const u16*)res,         \
                     rstride, (u16*)hout, hstride, N, K, B, stage, act,     \
                     eps, out_f32, softcap, escale)
  if (BT == 2) { if (xf32) MX_CASE(2, true); else MX_CASE(2, false); }
  else if (BT == 4) { if (xf32) MX_CASE(4, true); else MX_CASE(4, false); }
  else { if (xf32) MX_CASE(8, true); else MX_CASE(8, false); }
#undef MX_CASE
  return hipGetLastError();
}

// ====================================================================
// RMSNorm of bf16 rows: y = [res +] norm(x) * g (g fp32, Gemma's +1 folded
// in); with g2 also y2 = norm(y) * g2, the norm that follows a sandwich's
// residual, or the same as e4m3 rows (16 rows ahead of a product: each of its
// 256 blocks took 5 us for the norm and the rounding).  Without g2 norm(x) * g
// itself may go to e4m3, from fp32: of rows that are too long for the product
// to norm.
//
// A block of four waves a row, which stays in their registers; g and the
// residual are on the way before anything is summed.  Bound by the launch and
// a trip to memory where rows are few, by the trip and the two barriers' share
// of a CU where they are many.  us, by 1024 threads that asked for g after the
// sum -> here: 37x2048 3.95 -> 2.2, 1999x2048 15.2 -> 5.2, 2048x2304 with a
// residual 20.3 -> 7.4 (and the norm behind it: 40.6 -> 10.0).  A wave a row,
// without barriers: 37x2048 2.9, 1999x2048 5.5.
// ====================================================================

template <int NC>
__global__ void __launch_bounds__(256)
k_rmsnorm(const u16* __restrict__ x, const float* __restrict__ g,
          const u16* res, u16* y, const float* __restrict__ g2,
          u16* __restrict__ y2, uint8_t* __restrict__ q2,
          float* __restrict__ s2, int H, float eps) {
  __shared__ float red[3][4];
  const size_t at = (size_t)blockIdx.x * H;
  s8v v[NC], r[NC];
  f4v gg[NC][2], hh[NC][2];
  int k[NC];
#pragma unroll
  for (int c = 0; c < NC; c++) {
    k[c] = (c * 256 + threadIdx.x) * 8;
    const int q = min(k[c], H - 8);
    v[c] = *(const s8v*)(x + at + q);
    if (res) r[c] = *(const s8v*)(res + at + q);
    gg[c][0] = *(const f4v*)(g + q);
    gg[c][1] = *(const f4v*)(g + q + 4);
    if (g2) {
      hh[c][0] = *(const f4v*)(g2 + q);
      hh[c][1] = *(const f4v*)(g2 + q + 4);
    }
  }
  auto norm = [&](float* sums) {
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < NC; c++)
      if (k[c] < H)
#pragma unroll
        for (int j = 0; j < 8; j++) {
          const float f = b2f(((u16*)&v[c])[j]);
          ss += f * f;
        }
    ss = wave_reduce_sum(ss);
    if ((threadIdx.x & 63) == 0) sums[threadIdx.x >> 6] = ss;
    __syncthreads();
    ss = (sums[0] + sums[1]) + (sums[2] + sums[3]);
    return rsqrtf(ss / (float)H + eps);
  };
  float rm = norm(red[0]);
  if (y) {
#pragma unroll
    for (int c = 0; c < NC; c++) {
      u16 o[8];
#pragma unroll
      for (int j = 0; j < 8; j++) {
        float f = b2f(((u16*)&v[c])[j]) * rm * gg[c][j / 4][j % 4];
        if (res) f += b2f(((u16*)&r[c])[j]);
        o[j] = f2b(f);
      }
      v[c] = *(s8v*)o;
      if (k[c] < H) *(s8v*)(y + at + k[c]) = v[c];
    }
    if (!g2) return;
    rm = norm(red[1]);
  } else {
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
      for (int i = 0; i < 2; i++) hh[c][i] = gg[c][i];
  }
  if (!q2) {
#pragma unroll
    for (int c = 0; c < NC; c++) {
      u16 o[8];
#pragma unroll
      for (int j = 0; j < 8; j++)
        o[j] = f2b(b2f(((u16*)&v[c])[j]) * rm * hh[c][j / 4][j % 4]);
      if (k[c] < H) *(s8v*)(y2 + at + k[c]) = *(s8v*)o;
    }
    return;
  }
  // rows for an e4m3 product: what it would do to them in each of its blocks
  float am = 0.f;
#pragma unroll
  for (int c = 0; c < NC; c++)
#pragma unroll
    for (int j = 0; j < 8; j++) {
      hh[c][j / 4][j % 4] *= b2f(((u16*)&v[c])[j]) * rm;
      am = fmaxf(am, k[c] < H ? fabsf(hh[c][j / 4][j % 4]) : 0.f);
    }
#pragma unroll
  for (int w = 1; w < 64; w <<= 1) am = fmaxf(am, __shfl_xor(am, w));
  if ((threadIdx.x & 63) == 0) red[2][threadIdx.x >> 6] = am;
  __syncthreads();
  am = fmaxf(fmaxf(red[2][0], red[2][1]), fmaxf(red[2][2], red[2][3]));
  am = fmaxf(am, 1e-8f) / 448.0f;
  if (threadIdx.x == 0) s2[blockIdx.x] = am;
#pragma unroll
  for (int c = 0; c < NC; c++) {
    float f[8];
#pragma unroll
    for (int j = 0; j < 8; j++) f[j] = hh[c][j / 4][j % 4];
    if (k[c] < H)
      *(unsigned long long*)(q2 + at + k[c]) = f32x8_to_fp8(f, 1.0f / am);
  }
}

extern "C" hipError_t launch_rmsnorm(const void* x, const void* g,
                                     const void* res, void* y, const void* g2,
                                     void* y2, void* q2, void* s2, int M,
                                     int H, float eps, hipStream_t stream) {
  // a row stays in the registers of four waves
  if (M < 0 || H < 8 || H > 16384 || H % 8 != 0 || !q2 != !s2 ||
      (y ? !g2 != (!y2 && !q2) || (y2 && q2) : !q2 || g2 || y2 || res))
    return hipErrorInvalidValue;
  if (M == 0) return hipSuccess;
#define RMS_GO(NC)                                                           \
  hipLaunchKernelGGL(k_rmsnorm<NC>, dim3(M), dim3(256), 0, stream,           \
                     (const u16*)x, (const float*)g, (const u16*)res,        \
                     (u16*)y, (const float*)g2, (u16*)y2, (uint8_t*)q2,      \
                     (float*)s2, H, eps)
  if (H <= 2048) RMS_GO(1);
  else if (H <= 4096) RMS_GO(2);
  else if (H <= 8192) RMS_GO(4);
  else RMS_GO(8);
#undef RMS_GO
  return hipGetLastError();
}

// ====================================================================
// RoPE + KV-pool write.
// q inout [M, nh*hd]; k_in/v_in [M, kvh*hd]; caches [kvh, S, hd] bf16, or
// e4m3 with one fp32 scale per (kv_head, position): absmax/448 over the
// head_dim values, the same scheme as the fp8 weights.
// Position of row m is *pos_ptr + m (device scalar: graph-replay-safe), or
// rows[m] in cache rows[M + m] of several.
// cos/sin tables fp32 [max_seq, hd/2].
//
// Bound by memory where rows are many and by the trips of one thread where
// they are few, so a thread has 16 values of one head, eight of either half,
// and the hd/16 threads of a head meet for its e4m3 scale in registers.
// us, by a block a row that took its heads in turn, two bytes at a time
// (e4m3: a meeting of the block for every one) -> here:
//   bf16  5 rows of 24/8 heads of 128 4.3 -> 2.9, 1999 of 32/8 of 64 8.4 ->
//         6.2, 2048 of 32/8 of 128 13 -> 9.3 (37 of 32/8 of 64: 3.9 both)
//   e4m3  120 rows of 8/4 heads of 256 8.8 -> 3.3, 2048 of 32/8 of 128
//         27.4 -> 10.0
// ====================================================================

template <bool KV8>
__global__ void __launch_bounds__(256)
k_rope_rows(u16* __restrict__ q, const u16* __restrict__ kin,
            const u16* __restrict__ vin, void* __restrict__ kc,
            void* __restrict__ vc, float* __restrict__ kS,
            float* __restrict__ vS, const float* __restrict__ cost,
            const float* __restrict__ sint, const int* __restrict__ pos_ptr,
            const int* __restrict__ rows, int M, int nh, int kvh, int hd,
            int S, int ldq, int ldkv) {
  const int G = hd / 16, per = (nh + 2 * kvh) * G, hd2 = hd / 2;
  const int at = blockIdx.x * 256 + threadIdx.x;
  const bool there = at < M * per;
  const int id = there ? at : M * per - 1;
  const int m = id / per, u = id - m * per, h = u / G, t = u - h * G;
  const int pos = rows ? rows[m] : *pos_ptr + m;
  const size_t pool = rows ? (size_t)rows[M + m] * kvh * S : 0;
  const u16* src = h < nh ? q + (size_t)m * ldq + h * hd
                   : h < nh + kvh ? kin + (size_t)m * ldkv + (h - nh) * hd
                   : vin + (size_t)m * ldkv + (h - nh - kvh) * hd;
  const s8v lo = *(const s8v*)(src + t * 8);
  const s8v hi = *(const s8v*)(src + hd2 + t * 8);
  float a[8], b[8];
#pragma unroll
  for (int j = 0; j < 8; j++) {
    a[j] = b2f(((const u16*)&lo)[j]);
    b[j] = b2f(((const u16*)&hi)[j]);
  }
  if (h < nh + kvh) {
    const float* cp = cost + (size_t)pos * hd2 + t * 8;
    const float* sp = sint + (size_t)pos * hd2 + t * 8;
    const f4v c[2] = {*(const f4v*)cp, *(const f4v*)(cp + 4)};
    const f4v s[2] = {*(const f4v*)sp, *(const f4v*)(sp + 4)};
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const float x1 = a[j], x2 = b[j], cj = c[j / 4][j % 4];
      const float sj = s[j / 4][j % 4];
      a[j] = x1 * cj - x2 * sj;
      b[j] = x2 * cj + x1 * sj;
    }
  }
  const int kh = h < nh + kvh ? h - nh : h - nh - kvh;   // of a key or value
  const size_t row = pool + (size_t)(h < nh ? 0 : kh) * S + pos;
  if constexpr (KV8) {
    // all lanes of the wave, also those that rotate queries
    float am = 0.f;
#pragma unroll
    for (int j = 0; j < 8; j++)
      am = fmaxf(am, fmaxf(fabsf(a[j]), fabsf(b[j])));
    for (int w = 1; w < G; w <<= 1) am = fmaxf(am, __shfl_xor(am, w));
    if (!there) return;
    if (h >= nh) {
      const float sc = fmaxf(am, 1e-8f) / 448.0f;
      uint8_t* dst = (uint8_t*)(h < nh + kvh ? kc : vc) + row * hd + t * 8;
      if (t == 0) (h < nh + kvh ? kS : vS)[row] = sc;
      *(unsigned long long*)dst = f32x8_to_fp8(a, 1.0f / sc);
      *(unsigned long long*)(dst + hd2) = f32x8_to_fp8(b, 1.0f / sc);
      return;
    }
  }
  if (!there) return;
  u16* dst = h < nh ? q + (size_t)m * ldq + h * hd
                    : (u16*)(h < nh + kvh ? kc : vc) + row * hd;
  u16 o[8], p[8];
#pragma unroll
  for (int j = 0; j < 8; j++) {
    o[j] = f2b(a[j]);
    p[j] = f2b(b[j]);
  }
  *(s8v*)(dst + t * 8) = *(s8v*)o;
  *(s8v*)(dst + hd2 + t * 8) = *(s8v*)p;
}

// Any head size and alignment.
extern "C" __global__ void __launch_bounds__(256)
k_rope_cache(u16* __restrict__ q, const u16* __restrict__ kin,
             const u16* __restrict__ vin, u16* __restrict__ kc,
             u16* __restrict__ vc, const float* __restrict__ cost,
             const float* __restrict__ sint, const int* __restrict__ pos_ptr,
             int nh, int kvh, int hd, int S, int ldq, int ldkv) {
  const int m = blockIdx.x;
  const int pos = *pos_ptr + m;
  const int hd2 = hd / 2;
  const float* cp = cost + (size_t)pos * hd2;
  const float* sp = sint + (size_t)pos * hd2;

  // q rotation in place
  u16* qr = q + (size_t)m * ldq;
  for (int idx = threadIdx.x; idx < nh * hd2; idx += 256) {
    int h = idx / hd2, i = idx % hd2;
    float x1 = b2f(qr[h * hd + i]);
    float x2 = b2f(qr[h * hd + i + hd2]);
    float c = cp[i], s = sp[i];
    qr[h * hd + i] = f2b(x1 * c - x2 * s);
    qr[h * hd + i + hd2] = f2b(x2 * c + x1 * s);
  }
  // k rotation -> cache; v copy -> cache
  const u16* kr = kin + (size_t)m * ldkv;
  const u16* vr = vin + (size_t)m * ldkv;
  for (int idx = threadIdx.x; idx < kvh * hd2; idx += 256) {
    int h = idx / hd2, i = idx % hd2;
    float x1 = b2f(kr[h * hd + i]);
    float x2 = b2f(kr[h * hd + i + hd2]);
    float c = cp[i], s = sp[i];
    u16* dst = kc + ((size_t)h * S + pos) * hd;
    dst[i] = f2b(x1 * c - x2 * s);
    dst[i + hd2] = f2b(x2 * c + x1 * s);
  }
  for (int idx = threadIdx.x; idx < kvh * hd; idx += 256) {
    int h = idx / hd, i = idx % hd;
    vc[((size_t)h * S + pos) * hd + i] = vr[h * hd + i];
  }
}

extern "C" __global__ void __launch_bounds__(256)
k_rope_cache_fp8(u16* __restrict__ q, const u16* __restrict__ kin,
                 const u16* __restrict__ vin, uint8_t* __restrict__ kc,
                 uint8_t* __restrict__ vc, float* __restrict__ kS,
                 float* __restrict__ vS, const float* __restrict__ cost,
                 const float* __restrict__ sint,
                 const int* __restrict__ pos_ptr,
                 int nh, int kvh, int hd, int S, int ldq, int ldkv) {
  __shared__ float row[256];
  __shared__ float red[4];
  const int m = blockIdx.x;
  const int pos = *pos_ptr + m;
  const int hd2 = hd / 2;
  const float* cp = cost + (size_t)pos * hd2;
  const float* sp = sint + (size_t)pos * hd2;
  const int tid = threadIdx.x;

  // q rotation in place (q stays bf16)
  u16* qr = q + (size_t)m * ldq;
  for (int idx = tid; idx < nh * hd2; idx += 256) {
    int h = idx / hd2, i = idx % hd2;
    float x1 = b2f(qr[h * hd + i]);
    float x2 = b2f(qr[h * hd + i + hd2]);
    float c = cp[i], s = sp[i];
    qr[h * hd + i] = f2b(x1 * c - x2 * s);
    qr[h * hd + i + hd2] = f2b(x2 * c + x1 * s);
  }

  const u16* kr = kin + (size_t)m * ldkv;
  const u16* vr = vin + (size_t)m * ldkv;
  for (int h = 0; h < kvh; h++) {
    // rotated k row -> LDS floats
    __syncthreads();
    if (tid < hd2) {
      float x1 = b2f(kr[h * hd + tid]);
      float x2 = b2f(kr[h * hd + tid + hd2]);
      float c = cp[tid], s = sp[tid];
      row[tid] = x1 * c - x2 * s;
      row[tid + hd2] = x2 * c + x1 * s;
    }
    __syncthreads();
    float am = 0.f;
    for (int i = tid; i < hd; i += 256) am = fmaxf(am, fabsf(row[i]));
#pragma unroll
    for (int w = 1; w < 64; w <<= 1) am = fmaxf(am, __shfl_xor(am, w));
    if ((tid & 63) == 0) red[tid >> 6] = am;
    __syncthreads();
    am = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    float sc = fmaxf(am, 1e-8f) / 448.0f;
    if (tid == 0) kS[(size_t)h * S + pos] = sc;
    if (tid * 8 < hd)
      *(unsigned long long*)(kc + ((size_t)h * S + pos) * hd + tid * 8) =
          f32x8_to_fp8(&row[tid * 8], 1.0f / sc);
    // v row (no rotation)
    __syncthreads();
    for (int i = tid; i < hd; i += 256) row[i] = b2f(vr[h * hd + i]);
    __syncthreads();
    am = 0.f;
    for (int i = tid; i < hd; i += 256) am = fmaxf(am, fabsf(row[i]));
#pragma unroll
    for (int w = 1; w < 64; w <<= 1) am = fmaxf(am, __shfl_xor(am, w));
    if ((tid & 63) == 0) red[tid >> 6] = am;
    __syncthreads();
    am = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    sc = fmaxf(am, 1e-8f) / 448.0f;
    if (tid == 0) vS[(size_t)h * S + pos] = sc;
    if (tid * 8 < hd)
      *(unsigned long long*)(vc + ((size_t)h * S + pos) * hd + tid * 8) =
          f32x8_to_fp8(&row[tid * 8], 1.0f / sc);
  }
}

extern "C" hipError_t launch_rope_cache(void* q, const void* kin,
                                        const void* vin, void* kc, void* vc,
                                        void* kS, void* vS, int kv8,
                                        const void* cost, const void* sint,
                                        const void* pos_ptr, const void* rows,
                                        int M, int nh,
                                        int kvh, int hd, int S, int ldq,
                                        int ldkv, hipStream_t stream) {
  // 16 bytes at a time; e4m3: a head's threads are a power of two
  const size_t low = (size_t)q | (size_t)kin | (size_t)vin | (size_t)kc |
                     (size_t)vc | (size_t)cost | (size_t)sint;
  const int G = hd / 16;
  if (hd >= 16 && hd % 16 == 0 && ldq % 8 == 0 && ldkv % 8 == 0 &&
      low % 16 == 0 && (!kv8 || (G <= 64 && (G & (G - 1)) == 0)) &&
      (long)M * (nh + 2 * kvh) * G < 1L << 30) {
    const dim3 grid((M * (nh + 2 * kvh) * G + 255) / 256);
#define ROPE_GO(KV8)                                                         \
  hipLaunchKernelGGL(k_rope_rows<KV8>, grid, dim3(256), 0, stream, (u16*)q,  \
                     (const u16*)kin, (const u16*)vin, kc, vc, (float*)kS,   \
                     (float*)vS, (const float*)cost, (const float*)sint,     \
                     (const int*)pos_ptr, (const int*)rows, M, nh, kvh, hd,  \
                     S, ldq, ldkv)
    if (kv8) ROPE_GO(true);
    else ROPE_GO(false);
#undef ROPE_GO
    return hipGetLastError();
  }
  if (rows) return hipErrorInvalidValue;
  if (kv8) {
    hipLaunchKernelGGL(k_rope_cache_fp8, dim3(M), dim3(256), 0, stream,
                       (u16*)q, (const u16*)kin, (const u16*)vin,
                       (uint8_t*)kc, (uint8_t*)vc, (float*)kS, (float*)vS,
                       (const float*)cost, (const float*)sint,
                       (const int*)pos_ptr, nh, kvh, hd, S, ldq, ldkv);
  } else {
    hipLaunchKernelGGL(k_rope_cache, dim3(M), dim3(256), 0, stream, (u16*)q,
                       (const u16*)kin, (const u16*)vin, (u16*)kc, (u16*)vc,
                       (const float*)cost, (const float*)sint,
                       (const int*)pos_ptr, nh, kvh, hd, S, ldq, ldkv);
  }
  return hipGetLastError();
}

// ====================================================================
// GQA attention with online softmax (decode + per-query prefill).
// NOTE: with every shipped preset at head_dim in {64,128,256} the MFMA
// prefill kernel below is taken instead; this per-query VALU kernel is
// kept as the reachable fallback for odd head_dims and as the simple
// DEBUGGING reference the fused kernels are compared against in tests.
// grid (nh, M): block = head h, query row m (absolute pos = *len_ptr + m,
// attends keys [start, pos+1)).  4 waves split the KV range; each lane
// owns (sub-position, 8-dim chunk); merge within wave then across waves.
// Sliding window + attention-logit softcap = real Gemma-2 semantics
// (the reference omitted both).
// ====================================================================

template <bool KV8>
__global__ void __launch_bounds__(256)
k_attn_t(const u16* __restrict__ q, const void* __restrict__ kc,
         const void* __restrict__ vc, u16* __restrict__ out,
         const int* __restrict__ len_ptr, const float* __restrict__ kS,
         const float* __restrict__ vS, int nh, int kvh, int hd, int ldq, int S,
         float scale, float softcap, int window) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* red = (float*)smem;  // [4][hd] acc + [4][2] m,l

  const int h = blockIdx.x, m = blockIdx.y;
  const int kvhead = h / (nh / kvh);
  const int pos = *len_ptr + m;
  const int T = pos + 1;
  int start = 0;
  if (window > 0 && T - window > 0) start = T - window;

  const int LP = hd / 8;        // lanes per position
  const int PP = 64 / LP;       // positions per wave-iteration
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int p = lane / LP, d0 = (lane % LP) * 8;

  // q fragment for this head (8 dims), fp32
  float qf[8];
  {
    s8v v = *(const s8v*)(q + (size_t)m * ldq + h * hd + d0);
#pragma unroll
    for (int j = 0; j < 8; j++) qf[j] = b2f(((u16*)&v)[j]);
  }

  const u16* K0 = (const u16*)kc + (size_t)kvhead * S * hd;
  const u16* V0 = (const u16*)vc + (size_t)kvhead * S * hd;
  const uint8_t* K08 = (const uint8_t*)kc + (size_t)kvhead * S * hd;
  const uint8_t* V08 = (const uint8_t*)vc + (size_t)kvhead * S * hd;
  const float* kS0 = KV8 ? kS + (size_t)kvhead * S : nullptr;
  const float* vS0 = KV8 ? vS + (size_t)kvhead * S : nullptr;

  float mrun = -INFINITY, lrun = 0.f, acc[8];
#pragma unroll
  for (int j = 0; j < 8; j++) acc[j] = 0.f;

  {
    int t0 = start + wave * PP;
    if (t0 < T) {
      int t = t0 + p;
      bool valid = t < T;
      int tl = valid ? t : start;
      s8v kv, vv;
      unsigned long long kraw = 0, vraw = 0;
      float ksc = 1.f, vsc = 1.f;
      if (KV8) {
        kraw = *(const unsigned long long*)(K08 + (size_t)tl * hd + d0);
        vraw = *(const unsigned long long*)(V08 + (size_t)tl * hd + d0);
        ksc = kS0[tl]; vsc = vS0[tl];
      } else {
        kv = *(const s8v*)(K0 + (size_t)tl * hd + d0);
        vv = *(const s8v*)(V0 + (size_t)tl * hd + d0);
      }
      for (; t0 < T; t0 += 4 * PP) {
        int t0n = t0 + 4 * PP;
        s8v kvn, vvn;
        unsigned long long krawn = 0, vrawn = 0;
        float kscn = 1.f, vscn = 1.f;
        bool validn = false;
        if (t0n < T) {
          int tn = t0n + p;
          validn = tn < T;
          int tln = validn ? tn : start;
          if (KV8) {
            krawn = *(const unsigned long long*)(K08 + (size_t)tln * hd + d0);
            vrawn = *(const unsigned long long*)(V08 + (size_t)tln * hd + d0);
            kscn = kS0[tln]; vscn = vS0[tln];
          } else {
            kvn = *(const s8v*)(K0 + (size_t)tln * hd + d0);
            vvn = *(const s8v*)(V0 + (size_t)tln * hd + d0);
          }
        }
        float partial = 0.f;
        if (KV8) {
          // dequant straight to f32 in the dot (4 cvt + 8 fma per 8
          // elems — cheaper than the bf16 path's 8 shifts + 8 fma)
          f2v c0_ = __builtin_amdgcn_cvt_pk_f32_fp8((uint32_t)kraw, false);
          f2v c1_ = __builtin_amdgcn_cvt_pk_f32_fp8((uint32_t)kraw, true);
          f2v c2_ = __builtin_amdgcn_cvt_pk_f32_fp8((uint32_t)(kraw >> 32),
                                                    false);
          f2v c3_ = __builtin_amdgcn_cvt_pk_f32_fp8((uint32_t)(kraw >> 32),
                                                    true);
          partial = qf[0] * c0_[0] + qf[1] * c0_[1] + qf[2] * c1_[0] +
                    qf[3] * c1_[1] + qf[4] * c2_[0] + qf[5] * c2_[1] +
                    qf[6] * c3_[0] + qf[7] * c3_[1];
        } else {
#pragma unroll
          for (int j = 0; j < 8; j++) partial += qf[j] * b2f(((u16*)&kv)[j]);
        }
        for (int w = 1; w < LP; w <<= 1) partial += __shfl_xor(partial, w);
        float score = partial * (KV8 ? ksc : 1.f) * scale;
        if (softcap > 0.f) score = softcap * tanhf(score / softcap);
        if (!valid) score = -INFINITY;
        float mnew = fmaxf(mrun, score);
        float alpha = (mnew == -INFINITY) ? 0.f : __expf(mrun - mnew);
        float pv = (mnew == -INFINITY) ? 0.f : __expf(score - mnew);
        lrun = lrun * alpha + pv;
        if (KV8) {
          float pvv = pv * vsc;
          f2v d0_ = __builtin_amdgcn_cvt_pk_f32_fp8((uint32_t)vraw, false);
          f2v d1_ = __builtin_amdgcn_cvt_pk_f32_fp8((uint32_t)vraw, true);
          f2v d2_ = __builtin_amdgcn_cvt_pk_f32_fp8((uint32_t)(vraw >> 32),
                                                    false);
          f2v d3_ = __builtin_amdgcn_cvt_pk_f32_fp8((uint32_t)(vraw >> 32),
                                                    true);
          float vf[8] = {d0_[0], d0_[1], d1_[0], d1_[1],
                         d2_[0], d2_[1], d3_[0], d3_[1]};
#pragma unroll
          for (int j = 0; j < 8; j++)
            acc[j] = acc[j] * alpha + pvv * vf[j];
        } else {
#pragma unroll
          for (int j = 0; j < 8; j++)
            acc[j] = acc[j] * alpha + pv * b2f(((u16*)&vv)[j]);
        }
        if (mnew != -INFINITY) mrun = mnew;
        kv = kvn; vv = vvn; kraw = krawn; vraw = vrawn;
        valid = validn; ksc = kscn; vsc = vscn;
      }
    }
  }

  // merge across position-groups within the wave (lanes l, l^LP, l^2LP, ...)
  for (int w = LP; w < 64; w <<= 1) {
    float mo = __shfl_xor(mrun, w);
    float lo = __shfl_xor(lrun, w);
    float mn = fmaxf(mrun, mo);
    float sa = (mrun == -INFINITY && mo == -INFINITY) ? 0.f : __expf(mrun - mn);
    float sb = (mrun == -INFINITY && mo == -INFINITY) ? 0.f : __expf(mo - mn);
#pragma unroll
    for (int j = 0; j < 8; j++) {
      float ao = __shfl_xor(acc[j], w);
      acc[j] = acc[j] * sa + ao * sb;
    }
    lrun = lrun * sa + lo * sb;
    mrun = mn;
  }

  // merge across the 4 waves via LDS
  float* accs = red;             // [4][hd]
  float* mls = red + 4 * hd;     // [4][2]
  if (lane < LP) {
#pragma unroll
    for (int j = 0; j < 8; j++) accs[wave * hd + d0 + j] = acc[j];
  }
  if (lane == 0) {
    mls[wave * 2] = mrun;
    mls[wave * 2 + 1] = lrun;
  }
  __syncthreads();
  if (wave == 0) {
    float mt = fmaxf(fmaxf(mls[0], mls[2]), fmaxf(mls[4], mls[6]));
    float lt = 0.f, sc[4];
#pragma unroll
    for (int w = 0; w < 4; w++) {
      sc[w] = (mls[w * 2] == -INFINITY) ? 0.f : __expf(mls[w * 2] - mt);
      lt += mls[w * 2 + 1] * sc[w];
    }
    float inv = 1.f / lt;
    for (int d = lane; d < hd; d += 64) {
      float v = 0.f;
#pragma unroll
      for (int w = 0; w < 4; w++) v += accs[w * hd + d] * sc[w];
      out[((size_t)m * nh + h) * hd + d] = f2b(v * inv);
    }
  }
}

extern "C" hipError_t launch_attn(const void* q, const void* kc,
                                  const void* vc, void* out,
                                  const void* len_ptr, const void* kS,
                                  const void* vS, int kv8, int M, int nh,
                                  int kvh, int hd, int ldq, int S, float scale,
                                  float softcap, int window,
                                  hipStream_t stream) {
  size_t lds = (4 * hd + 8) * sizeof(float);
#define ATTN_CASE(KV8V)                                                     \
  hipLaunchKernelGGL((k_attn_t<KV8V>), dim3(nh, M), dim3(256), lds, stream, \
                     (const u16*)q, kc, vc, (u16*)out,                      \
                     (const int*)len_ptr, (const float*)kS,                 \
                     (const float*)vS, nh, kvh, hd, ldq, S, scale, softcap, \
                     window)
  if (kv8) ATTN_CASE(true);
  else ATTN_CASE(false);
#undef ATTN_CASE
  return hipGetLastError();
}

// ====================================================================
// GLU activations: out = act(gate) * up ; act 0 = SiLU, 1 = tanh-GELU, for
// halves that are there already (products take theirs as they store)
// ====================================================================

extern "C" __global__ void __launch_bounds__(256)
k_glu(const u16* __restrict__ gate, const u16* __restrict__ up,
      u16* __restrict__ out, long total, int act) {
  long i = ((long)blockIdx.x * 256 + threadIdx.x) * 8;
  if (i >= total) return;
  s8v g = *(const s8v*)(gate + i);
  s8v u = *(const s8v*)(up + i);
  u16 o[8];
#pragma unroll
  for (int j = 0; j < 8; j++) {
    o[j] = f2b(gate_act(b2f(((u16*)&g)[j]), act) * b2f(((u16*)&u)[j]));
  }
  *(s8v*)(out + i) = *(s8v*)o;
}

extern "C" hipError_t launch_glu(const void* gate, const void* up, void* out,
                                 long total, int act, hipStream_t stream) {
  long blocks = (total / 8 + 255) / 256;
  hipLaunchKernelGGL(k_glu, dim3((uint32_t)blocks), dim3(256), 0, stream,
                     (const u16*)gate, (const u16*)up, (u16*)out, total, act);
  return hipGetLastError();
}

// ====================================================================
// Embedding gather: h[m] = embed[ids[m]] * scale  (ids live on device so
// the decode graph can feed back the sampled token without host sync)
// ====================================================================

extern "C" __global__ void __launch_bounds__(256)
k_embed(const u16* __restrict__ embed, const int* __restrict__ ids,
        u16* __restrict__ out, int H, float scale) {
  const int m = blockIdx.x;
  const int id = ids[m];
  const u16* src = embed + (size_t)id * H;
  u16* dst = out + (size_t)m * H;
  for (int i = threadIdx.x * 8; i < H; i += 2048) {
    s8v v = *(const s8v*)(src + i);
    u16 o[8];
#pragma unroll
    for (int j = 0; j < 8; j++) o[j] = f2b(b2f(((u16*)&v)[j]) * scale);
    *(s8v*)(dst + i) = *(s8v*)o;
  }
}

extern "C" hipError_t launch_embed(const void* embed, const void* ids,
                                   void* out, int M, int H, float scale,
                                   hipStream_t stream) {
  hipLaunchKernelGGL(k_embed, dim3(M), dim3(256), 0, stream,
                     (const u16*)embed, (const int*)ids, (u16*)out, H, scale);
  return hipGetLastError();
}

// ====================================================================
// Sampling: greedy argmax or min-p + Gumbel-argmax multinomial.
//   keep tokens with p >= min_p * p_max  <=>  logit >= max + ln(min_p);
//   winner = argmax over kept of (logit + Gumbel noise).
// Writes the token to *next_token (feeds the next decode graph step),
// appends to out_ring, bumps *len_ptr and *nout — all device-side, so the
// whole decode step is graph-replayable.
// ====================================================================

DEVINL uint32_t hash32(uint32_t x) {
  x ^= x >> 16; x *= 0x7feb352du;
  x ^= x >> 15; x *= 0x846ca68bu;
  x ^= x >> 16;
  return x;
}

// order-preserving float->u32 key (monotone for max); invertible
DEVINL uint32_t fkey(float f) {
  union { float f; uint32_t u; } c; c.f = f;
  return (c.u & 0x80000000u) ? ~c.u : (c.u ^ 0x80000000u);
}
DEVINL float fkey_inv(uint32_t k) {
  union { float f; uint32_t u; } c;
  c.u = (k & 0x80000000u) ? (k ^ 0x80000000u) : ~k;
  return c.f;
}

// pack (key, idx): ties prefer the SMALLEST index (matches np.argmax)
DEVINL uint64_t pack_ki(uint32_t key, int idx) {
  return ((uint64_t)key << 32) | (uint32_t)(0x7fffffff - idx);
}
DEVINL int unpack_idx(uint64_t p) { return 0x7fffffff - (int)(uint32_t)p; }

// pass 1 (min-p only): global max logit -> gmax[b] (packed).
// Batched: grid.y = sequence row b (lbf16: logits stored bf16 — the
// batched lm_head GEMM path emits bf16 rows).
#define SMP_U 4         // logits of a thread at a time

template <int NT>       // threads of a block
__global__ void __launch_bounds__(NT)
k_logit_max(const void* __restrict__ logits, int V, int lbf16,
            unsigned long long* __restrict__ gmax,
            uint64_t* __restrict__ ctr) {
  const int b = blockIdx.y;
  gmax += b;
  // advance the shared RNG counter HERE: stream order guarantees every
  // k_sample_pick block then reads the same post-bump value (bumping
  // from pick's commit raced with straggler blocks still reading it)
  if (ctr && blockIdx.x == 0 && b == 0 && threadIdx.x == 0) *ctr += 1;
  const float* lf = (const float*)logits + (size_t)b * V;
  const u16* lh = (const u16*)logits + (size_t)b * V;
  float mv = -INFINITY;
  int mi = 0;
  for (int i0 = blockIdx.x * NT * SMP_U + threadIdx.x; i0 < V;
       i0 += gridDim.x * NT * SMP_U) {
    float v[SMP_U];
#pragma unroll
    for (int u = 0; u < SMP_U; u++) {
      const int i = min(i0 + u * NT, V - 1);
      v[u] = lbf16 ? b2f(lh[i]) : lf[i];
    }
#pragma unroll
    for (int u = 0; u < SMP_U; u++) {
      const int i = min(i0 + u * NT, V - 1);
      if (v[u] > mv || (v[u] == mv && i < mi)) { mv = v[u]; mi = i; }
    }
  }
  uint64_t pk = pack_ki(fkey(mv), mi);
#pragma unroll
  for (int w = 1; w < 64; w <<= 1) {
    uint64_t o = __shfl_xor((unsigned long long)pk, w);
    if (o > pk) pk = o;
  }
  __shared__ unsigned long long ws[NT / 64];
  if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = pk;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t b = ws[0];
    for (int w = 1; w < NT / 64; w++) if (ws[w] > b) b = ws[w];
    atomicMax(gmax, (unsigned long long)b);
  }
}

// pass 2: winner = argmax over kept tokens of (logit/T [+ Gumbel]) -> *pick,
// and the LAST-arriving block (G16 ticket) commits it: write *next_token,
// append to out_ring, bump len/ctr, re-zero the scratch — the former
// k_sample_fin's 1-thread launch (~4 us) folded away.
// Temperature folds into both the min-p keep-set and the Gumbel score:
//   p_i(T) >= min_p * p_max(T)  <=>  l_i >= l_max + T*ln(min_p)
//   Gumbel-argmax over p(T)     <=>  argmax of l_i/T + G_i
//
// TOPS: one row, whose logits' producer left the largest of several shares of
// them (`tops`), so that no launch goes through all of them ahead: each block
// goes through the shares, its first logits already on the way.  The last to
// arrive advances the RNG counter, which all have read by then.
// us a step by min-p, both launches -> here: 32000 logits 7.6 -> 5.1, 128256
// 8.2 -> 5.2, 256000 8.6 -> 5.5.
template <int NT, bool TOPS>
__global__ void __launch_bounds__(NT)
k_sample_pick(const void* __restrict__ logits, int V, int lbf16,
              long ring_stride, float min_p,
              int greedy, uint64_t seed, float inv_temp,
              unsigned long long* __restrict__ gmax,
              uint64_t* __restrict__ ctr,
              unsigned long long* __restrict__ pick,
              int* __restrict__ cnt, int* __restrict__ next_token,
              int* __restrict__ out_ring, int* __restrict__ nout,
              int* __restrict__ len_ptr, int bump_len,
              const float* __restrict__ tops, int ntops) {
  const int b = blockIdx.y;
  gmax += b; pick += b; cnt += b; nout += b;
  out_ring += (size_t)b * ring_stride;
  const float* lf = (const float*)logits + (size_t)b * V;
  const u16* lh = (const u16*)logits + (size_t)b * V;
  float vs[SMP_U];
  auto load = [&](int i0) {
#pragma unroll
    for (int u = 0; u < SMP_U; u++) {
      const int i = min(i0 + u * NT, V - 1);
      vs[u] = lbf16 ? b2f(lh[i]) : lf[i];
    }
  };
  const int step = gridDim.x * NT * SMP_U;
  int i0 = blockIdx.x * NT * SMP_U + threadIdx.x;
  load(i0);
  float thresh = -INFINITY;
  if constexpr (TOPS) {
    __shared__ float top[NT / 64];
    float m = -INFINITY;
    for (int i = threadIdx.x; i < ntops; i += NT) m = fmaxf(m, tops[i]);
    m = wave_reduce_max(m);
    if ((threadIdx.x & 63) == 0) top[threadIdx.x >> 6] = m;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NT / 64; w++) m = fmaxf(m, top[w]);
    thresh = m + __logf(min_p) / inv_temp;
  } else if (!greedy) {
    thresh = fkey_inv((uint32_t)(*gmax >> 32)) + __logf(min_p) / inv_temp;
  }
  const uint32_t c = ((uint32_t)(*ctr) + (TOPS ? 1u : 0u)) ^
                     ((uint32_t)b * 0x85ebca6bu);
  float bv = -INFINITY;
  int bi = 0x7fffffff;
  for (; i0 < V; i0 += step) {
    if (i0 >= step) load(i0);
#pragma unroll
    for (int u = 0; u < SMP_U; u++) {
      const int i = min(i0 + u * NT, V - 1);
      const float v = vs[u];
      if (v < thresh) continue;
      float sc = v;
      if (!greedy) {
        uint32_t r = hash32(hash32((uint32_t)i ^ (c * 0x9e3779b9u)) ^
                            (uint32_t)seed);
        float u1 = (r + 1.0f) * 2.3283064e-10f;  // (0,1]
        sc = v * inv_temp - __logf(-__logf(u1));
      }
      if (sc > bv || (sc == bv && i < bi)) { bv = sc; bi = i; }
    }
  }
  uint64_t pk = pack_ki(fkey(bv), bi);
#pragma unroll
  for (int w = 1; w < 64; w <<= 1) {
    uint64_t o = __shfl_xor((unsigned long long)pk, w);
    if (o > pk) pk = o;
  }
  __shared__ unsigned long long ws[NT / 64];
  __shared__ int lastflag;
  if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = pk;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t b = ws[0];
    for (int w = 1; w < NT / 64; w++) if (ws[w] > b) b = ws[w];
    // atomics of the device both, one after the other: nothing to write back
    atomicMax(pick, (unsigned long long)b);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    int t = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
    lastflag = (t == (int)gridDim.x - 1);
  }
  __syncthreads();
  if (!lastflag || threadIdx.x != 0) return;
  // last arriver: commit the winner, reset scratch, advance state
  *cnt = 0;
  int winner = unpack_idx(
      __hip_atomic_load(pick, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  if (winner < 0 || winner >= V) winner = 0;  // NaN-logit insurance
  next_token[b] = winner;
  int n = *nout;
  out_ring[n] = winner;
  *nout = n + 1;
  // per-row position advances (ragged batch); the shared RNG counter
  // was already advanced by k_logit_max ahead of this kernel
  if (TOPS) *ctr += 1;
  if (bump_len) len_ptr[b] += 1;
  *pick = 0ull;
  *gmax = 0ull;
}

extern "C" hipError_t launch_sample(const void* logits, int V, int lbf16,
                                    int batch, long ring_stride, float min_p,
                                    int greedy, uint64_t seed, float inv_temp,
                                    void* ctr, void* gmax, void* pick,
                                    void* cnt, void* next_token,
                                    void* out_ring, void* nout,
                                    void* len_ptr, int bump_len,
                                    const void* tops, int ntops,
                                    hipStream_t stream) {
  if (tops && (batch != 1 || ntops < 1)) return hipErrorInvalidValue;
  // Every block queues up at a word of its row, twice in the pick, and the
  // words of a group's rows share lines: some 25 ns a block, of whatever row.
  // A trip of a block through its logits takes some 0.65 us.  One row: 63
  // blocks of 2048 logits, 128256 of them greedy in 5.3 us (501 blocks of 256:
  // 14.0).  A group takes larger blocks, and fewer of a row where there are
  // many; us, greedy and min-p, in blocks of 256 threads, 16 of a row or more
  // (as before) -> in 16 of 512 -> here:
  //   16 rows of 32768   10.3, 16.5 ->  9.5, 14.4 ->  7.1, 11.8
  //   16 rows of 256000  20.9, 33.4 -> 15.6, 25.3 -> 12.5, 20.6
  //   64 rows of 128256  35.0, 48.6 -> 33.0, 48.8 -> 19.8, 34.2
  //   64 rows of 256000  43.8, 65.8 -> 49.6, 71.6 -> 34.1, 52.6
  const int nt = batch > 4 ? 1024 : 512;
  int blocks = (V + nt * SMP_U - 1) / (nt * SMP_U);
  const int most = batch > 32  ? 8
                   : batch > 4 ? 16
                               : 64 / (batch > 0 ? batch : 1);
  if (blocks > most) blocks = most;
#define SMP_PICK(NT, TOPS)                                                   \
  hipLaunchKernelGGL((k_sample_pick<NT, TOPS>), dim3(blocks, batch),         \
                     dim3(NT), 0, stream, logits, V, lbf16, ring_stride,     \
                     min_p, greedy, seed, inv_temp,                          \
                     (unsigned long long*)gmax, (uint64_t*)ctr,              \
                     (unsigned long long*)pick, (int*)cnt,                   \
                     (int*)next_token, (int*)out_ring, (int*)nout,           \
                     (int*)len_ptr, bump_len, (const float*)tops, ntops)
  if (tops && !greedy) {
    SMP_PICK(512, true);
    return hipGetLastError();
  }
#define SMP_GO(NT)                                                           \
  if (!greedy)                                                               \
    hipLaunchKernelGGL(k_logit_max<NT>, dim3(blocks, batch), dim3(NT), 0,    \
                       stream, logits, V, lbf16, (unsigned long long*)gmax,  \
                       (uint64_t*)ctr);                                      \
  SMP_PICK(NT, false)
  if (nt == 1024) {
    SMP_GO(1024);
  } else {
    SMP_GO(512);
  }
#undef SMP_GO
#undef SMP_PICK
  return hipGetLastError();
}

// ====================================================================
// MXFP4 weight quantization: 4-bit e2m1 values packed 2/byte with one
// e8m0 (power-of-two) scale per 32-element block — the OCP MX format.
// Decode is weights-only quantization: the GEMV dequantizes via
// v_cvt_scalef32_pk_f32_fp4, which applies the block scale INSIDE the
// hardware convert (same VALU per element as the fp8 path, HALF the
// weight bytes -> ~1.5x on stream-bound shapes).
// ====================================================================

extern "C" __global__ void __launch_bounds__(256)
k_quant_fp4_rows(const u16* __restrict__ X, uint8_t* __restrict__ Q,
                 uint8_t* __restrict__ E, int K) {
  const int row = blockIdx.x;
  const u16* xr = X + (size_t)row * K;
  uint8_t* qr = Q + (size_t)row * (K / 2);
  uint8_t* er = E + (size_t)row * (K / 32);
  // each thread owns whole 32-element blocks
  for (int blk = threadIdx.x; blk < K / 32; blk += 256) {
    float v[32];
    float am = 0.f;
#pragma unroll
    for (int j = 0; j < 32; j++) {
      v[j] = b2f(xr[blk * 32 + j]);
      am = fmaxf(am, fabsf(v[j]));
    }
    // e2m1 max magnitude = 6.0: scale = 2^e with absmax/2^e <= 6
    int e = 0;
    if (am > 0.f) {
      int ee;
      frexpf(am / 6.0f, &ee);  // am/6 = m * 2^ee, m in [0.5, 1)
      e = ee;                  // 2^ee >= am/6
      if (ldexpf(6.0f, e - 1) >= am) e -= 1;  // exact-power tightening
    }
    if (e < -126) e = -126;
    if (e > 127) e = 127;
    union { float f; uint32_t u; } sc;
    sc.u = (uint32_t)(e + 127) << 23;       // 2^e
    er[blk] = (uint8_t)(e + 127);
#pragma unroll
    for (int d = 0; d < 4; d++) {           // 4 dwords of 8 nibbles
      // HW semantics (device-verified): encode fp4 = RNE(v / scale),
      // decode = v * scale -> pass the SAME 2^e both ways; the pair
      // selector must be a literal
      uint32_t w = 0;
      w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(
          w, v[d * 8 + 0], v[d * 8 + 1], sc.f, 0);
      w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(
          w, v[d * 8 + 2], v[d * 8 + 3], sc.f, 1);
      w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(
          w, v[d * 8 + 4], v[d * 8 + 5], sc.f, 2);
      w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(
          w, v[d * 8 + 6], v[d * 8 + 7], sc.f, 3);
      *(uint32_t*)(qr + blk * 16 + d * 4) = w;
    }
  }
}

extern "C" hipError_t launch_quant_fp4(const void* X, void* Q, void* E,
                                       int M, int K, hipStream_t stream) {
  if (K % 32 != 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_quant_fp4_rows, dim3(M), dim3(256), 0, stream,
                     (const u16*)X, (uint8_t*)Q, (uint8_t*)E, K);
  return hipGetLastError();
}

// ====================================================================
// fp8 row quantization: Q[N,K] = e4m3(X / s_n), s_n = absmax_n / 448.
// One block per row.  Used (a) at load time to quantize weights ON
// DEVICE (on the host a 9B model took ~90 s, and a duplicate bf16 copy
// stayed), (b) per prefill GEMM to quantize the
// activation rows so BOTH MFMA operands are fp8.
// HW convert: v_cvt_pk_fp8_f32 (OCP e4m3fn on gfx950, saturating).
// ====================================================================

// Few rows take 1024 threads each (a row is then read once, into registers;
// 16 rows of 14336: 2.7 us, by 256 threads 4.4), many rows 256.
DEVINL void load8(const u16* p, float* f) {
  const s8v v = *(const s8v*)p;
#pragma unroll
  for (int j = 0; j < 8; j++) f[j] = b2f(((u16*)&v)[j]);
}
DEVINL void load8(const float* p, float* f) {
  *(f4v*)f = *(const f4v*)p;
  *(f4v*)(f + 4) = *(const f4v*)(p + 4);
}

template <typename T, int NT>
__global__ void __launch_bounds__(NT)
k_quant_fp8_rows(const T* __restrict__ X, uint8_t* __restrict__ Q,
                 float* __restrict__ S, int K) {
  constexpr int KEEP = 3;                    // chunks that stay in registers
  __shared__ float wmax[NT / 64];
  const int row = blockIdx.x;
  const T* xr = X + (size_t)row * K;
  uint8_t* qr = Q + (size_t)row * K;

  float amax = 0.f, kept[KEEP][8];
#pragma unroll
  for (int c = 0; c < KEEP; c++) {
    const int i = (c * NT + threadIdx.x) * 8;
    if (i < K) {
      load8(xr + i, kept[c]);
#pragma unroll
      for (int j = 0; j < 8; j++) amax = fmaxf(amax, fabsf(kept[c][j]));
    }
  }
  for (int i = (KEEP * NT + threadIdx.x) * 8; i < K; i += NT * 8) {
    float f[8];
    load8(xr + i, f);
#pragma unroll
    for (int j = 0; j < 8; j++) amax = fmaxf(amax, fabsf(f[j]));
  }
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) amax = fmaxf(amax, __shfl_xor(amax, m));
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = amax;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NT / 64; w++) amax = fmaxf(amax, wmax[w]);
  const float s = fmaxf(amax, 1e-8f) / 448.0f;
  const float rs = 1.0f / s;
  if (threadIdx.x == 0) S[row] = s;

#pragma unroll
  for (int c = 0; c < KEEP; c++) {
    const int i = (c * NT + threadIdx.x) * 8;
    if (i < K)
      *(unsigned long long*)(qr + i) = f32x8_to_fp8(kept[c], rs);
  }
  for (int i = (KEEP * NT + threadIdx.x) * 8; i < K; i += NT * 8) {
    float f[8];
    load8(xr + i, f);
    *(unsigned long long*)(qr + i) = f32x8_to_fp8(f, rs);
  }
}

extern "C" hipError_t launch_quant_fp8(const void* X, void* Q, void* S,
                                       int f32, int M, int K,
                                       hipStream_t stream) {
  if (K % 8 != 0) return hipErrorInvalidValue;
#define QUANT_CASE(T, NT)                                                    \
  hipLaunchKernelGGL((k_quant_fp8_rows<T, NT>), dim3(M), dim3(NT), 0, stream, \
                     (const T*)X, (uint8_t*)Q, (float*)S, K)
  const bool few = M <= 64 && K > 2048;
  if (f32) { if (few) QUANT_CASE(float, 1024); else QUANT_CASE(float, 256); }
  else { if (few) QUANT_CASE(u16, 1024); else QUANT_CASE(u16, 256); }
#undef QUANT_CASE
  return hipGetLastError();
}

// ====================================================================
// Weight prefetcher (side-stream): stream a tensor through L2/MALL with
// plain (retaining) loads so the 256 MB Infinity Cache holds the NEXT
// layer's weights before its compute kernel issues.  The sink write
// keeps the loads alive; modest grid so compute keeps its CUs.
// ====================================================================

extern "C" __global__ void __launch_bounds__(256)
k_prefetch(const u16* __restrict__ p, long n, float* __restrict__ sink) {
  float acc = 0.f;
  for (long i = ((long)blockIdx.x * 256 + threadIdx.x) * 8; i < n;
       i += (long)gridDim.x * 256 * 8) {
    s8v v = *(const s8v*)(p + i);
    acc += b2f(((u16*)&v)[0]);  // one live use per 16 B line segment
  }
  if (acc == 1e30f) sink[blockIdx.x] = acc;  // never true; keeps loads
}

extern "C" hipError_t launch_prefetch(const void* p, long n_elems,
                                      void* sink, hipStream_t stream) {
  hipLaunchKernelGGL(k_prefetch, dim3(128), dim3(256), 0, stream,
                     (const u16*)p, n_elems, (float*)sink);
  return hipGetLastError();
}

// ====================================================================
// elementwise tanh soft-cap: y = cap * tanh(x / cap)  (bf16)
// (Gemma-2 final-logit capping on the all-positions GEMM path; the
// decode GEMV fuses this into its epilogue instead)
// ====================================================================

extern "C" __global__ void __launch_bounds__(256)
k_softcap(u16* __restrict__ y, long total, float cap) {
  long i = ((long)blockIdx.x * 256 + threadIdx.x) * 8;
  if (i >= total) return;
  s8v v = *(const s8v*)(y + i);
  u16 o[8];
#pragma unroll
  for (int j = 0; j < 8; j++)
    o[j] = f2b(cap * tanhf(b2f(((u16*)&v)[j]) / cap));
  *(s8v*)(y + i) = *(s8v*)o;
}

extern "C" hipError_t launch_softcap(void* y, long total, float cap,
                                     hipStream_t stream) {
  long blocks = (total / 8 + 255) / 256;
  hipLaunchKernelGGL(k_softcap, dim3((uint32_t)blocks), dim3(256), 0, stream,
                     (u16*)y, total, cap);
  return hipGetLastError();
}

// ====================================================================
// y += a (bf16, fp32 math).  Used on the TP path where the RCCL
// all-reduce sits between the row-parallel GEMV and the residual add.
// ====================================================================

extern "C" __global__ void __launch_bounds__(256)
k_addinto(u16* __restrict__ y, const u16* __restrict__ a, long total) {
  long i = ((long)blockIdx.x * 256 + threadIdx.x) * 8;
  if (i >= total) return;
  s8v yv = *(const s8v*)(y + i);
  s8v av = *(const s8v*)(a + i);
  u16 o[8];
#pragma unroll
  for (int j = 0; j < 8; j++)
    o[j] = f2b(b2f(((u16*)&yv)[j]) + b2f(((u16*)&av)[j]));
  *(s8v*)(y + i) = *(s8v*)o;
}

extern "C" hipError_t launch_addinto(void* y, const void* a, long total,
                                     hipStream_t stream) {
  long blocks = (total / 8 + 255) / 256;
  hipLaunchKernelGGL(k_addinto, dim3((uint32_t)blocks), dim3(256), 0, stream,
                     (u16*)y, (const u16*)a, total);
  return hipGetLastError();
}

// ====================================================================
// Grid-wide barrier (device-side, graph-replay-safe).  Used by the
// fused-layer decode path: phases of one layer run inside ONE kernel
// with barriers instead of kernel boundaries (~4 us launch/ramp floor
// each).
//
// Protocol: `cnt` is a MONOTONIC u64 arrive counter (never reset — the
// launch invariant is cnt % nblocks == 0, preserved because every
// launch/replay runs the same barrier count with the same grid);
// `seq` is the completed-barrier counter.  Each block reads base_seq
// once at kernel start (stable: seq cannot change until every block
// has arrived at barrier 0, which implies every block already read it)
// and spins for seq > base_seq + bar_idx.  Bounded spin -> err flag,
// not a hung GPU.
// ====================================================================

DEVINL int grid_barrier(unsigned long long* cnt, unsigned long long* seq,
                        unsigned long long base_seq, int bar_idx,
                        int nblocks, long spin_limit,
                        uint32_t* err) {
  __shared__ int ok;
  __syncthreads();
  if (threadIdx.x == 0) {
    ok = 1;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    unsigned long long t = __hip_atomic_fetch_add(
        cnt, 1ull, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
    if (t % (unsigned long long)nblocks ==
        (unsigned long long)nblocks - 1ull) {
      __hip_atomic_store(seq, base_seq + bar_idx + 1, __ATOMIC_RELEASE,
                         __HIP_MEMORY_SCOPE_AGENT);
    } else {
      long spins = 0;
      while (__hip_atomic_load(seq, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT) <=
             base_seq + bar_idx) {
        if (++spins > spin_limit) {
          __hip_atomic_store(err, 1u, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
          ok = 0;
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  __syncthreads();
  return ok;
}

// microbenchmark: nbar back-to-back barriers (measures the phase-
// boundary cost that replaces a kernel launch in the fused path)
extern "C" __global__ void __launch_bounds__(256)
k_gbar_bench(unsigned long long* cnt, unsigned long long* seq,
             uint32_t* err, int nbar, long spin_limit) {
  const unsigned long long base =
      __hip_atomic_load(seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (int b = 0; b < nbar; b++)
    if (!grid_barrier(cnt, seq, base, b, gridDim.x, spin_limit, err))
      return;
}

extern "C" hipError_t launch_gbar_bench(void* cnt, void* seq, void* err,
                                        int nblocks, int nbar,
                                        long spin_limit,
                                        hipStream_t stream) {
  hipLaunchKernelGGL(k_gbar_bench, dim3(nblocks), dim3(256), 0, stream,
                     (unsigned long long*)cnt, (unsigned long long*)seq,
                     (uint32_t*)err, nbar, spin_limit);
  return hipGetLastError();
}

// ====================================================================
// Utility: device-side int32 set/add (for seq-length bookkeeping inside
// graphs where needed)
// ====================================================================

extern "C" __global__ void k_i32_set(int* p, int v) { *p = v; }

extern "C" hipError_t launch_i32_set(void* p, int v, hipStream_t stream) {
  hipLaunchKernelGGL(k_i32_set, dim3(1), dim3(1), 0, stream, (int*)p, v);
  return hipGetLastError();
}
// ====================================================================
// Mixtral sparse-MoE helpers (the reference has no MoE).
// k_moe_route fuses the per-row RMSNorm, the router dots
// against Wg[E,H] (f32 accum — bf16 router logits would risk top-k
// flips), the softmax over E, and the HF top-k renormalization
// (modeling_mixtral MixtralTopKRouter), emitting compact (idx, w)
// pairs for the expert-indexed products and optionally a dense M x E
// weight grid.
// One block per row; E <= 64, topk <= 8.  Bound by its chain of trips: the
// row and gamma together, then all experts' weights at once (eight waves, an
// expert each at a time), then one wave with an expert a lane.  Experts one
// after the other, two barriers each, and the choice by one thread took 17.3
// us for a row of 2048 and eight experts; here 3.8 (60 experts 8.1).
// ====================================================================

extern "C" __global__ void __launch_bounds__(512)
k_moe_route(const u16* __restrict__ h, const float* __restrict__ g,
            const u16* __restrict__ wg, int M, int H, int E, int topk,
            float eps, int* __restrict__ idx, float* __restrict__ wout,
            float* __restrict__ dense) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* xf = (float*)smem;           // H floats: normed row
  float* red = xf + H;                // 8 wave partials
  float* el = red + 8;                // E router logits
  const int m = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const u16* hr = h + (size_t)m * H;
  float ss = 0.f;
  for (int i = tid; i < H; i += 512) {
    const float v = b2f(hr[i]), gv = g[i];
    xf[i] = v * gv;
    ss += v * v;
  }
  ss = wave_reduce_sum(ss);
  if (lane == 0) red[wave] = ss;
  __syncthreads();
  ss = 0.f;
#pragma unroll
  for (int w = 0; w < 8; w++) ss += red[w];
  const float rn = __frsqrt_rn(ss / H + eps);
  for (int e = wave; e < E; e += 8) {
    const u16* wr = wg + (size_t)e * H;
    float d = 0.f;
    int i = lane * 2;
    if (H % 2 == 0) {                 // pairs: rows are 4-byte aligned
#pragma unroll 8
      for (; i < H; i += 128) {
        const uint32_t w = *(const uint32_t*)(wr + i);
        d += xf[i] * __uint_as_float(w << 16) +
             xf[i + 1] * __uint_as_float(w & 0xffff0000u);
      }
    } else {
      for (i = lane; i < H; i += 64) d += xf[i] * b2f(wr[i]);
    }
    d = wave_reduce_sum(d);
    if (lane == 0) el[e] = d * rn;
  }
  __syncthreads();
  if (wave != 0) return;
  const float NONE = -INFINITY;
  float v = lane < E ? el[lane] : NONE;
  auto most = [&](float x) {
#pragma unroll
    for (int w = 1; w < 64; w <<= 1) x = fmaxf(x, __shfl_xor(x, w));
    return x;
  };
  const float top = most(v);          // by all lanes, also those without one
  float p = lane < E ? __expf(v - top) : 0.f;
  if (!(p == p)) p = 0.f;             // an index is one of an expert, whatever
  if (dense && lane < E) dense[(size_t)m * E + lane] = 0.f;
  // top-k by repeated argmax (ties -> smallest index, matching the
  // oracle's stable argsort); renormalize the kept probs by their sum
  float left = lane < E ? p : -2.f, wsum = 0.f, mine = 0.f;
  int slot = -1;
  for (int j = 0; j < topk; j++) {
    const float bv = most(left);
    const int be = __ffsll((unsigned long long)__ballot(left == bv)) - 1;
    wsum += bv;
    if (lane == be) {
      slot = j;
      mine = bv;
      left = -1.f;
    }
  }
  if (slot >= 0) {
    const float wv = mine / wsum;
    idx[(size_t)m * topk + slot] = lane;
    wout[(size_t)m * topk + slot] = wv;
    if (dense) dense[(size_t)m * E + lane] = wv;
  }
}

extern "C" hipError_t launch_moe_route(const void* h, const void* g,
                                       const void* wg, int M, int H, int E,
                                       int topk, float eps, void* idx,
                                       void* wout, void* dense,
                                       hipStream_t stream) {
  if (E < 1 || E > 64 || topk < 1 || topk > 8 || topk > E)
    return hipErrorInvalidValue;
  size_t lds = (size_t)H * 4 + 32 + (size_t)E * 4;
  if (lds > 64 * 1024 + 16) return hipErrorInvalidValue;
  static const hipError_t raised = hipFuncSetAttribute(
      (const void*)&k_moe_route, hipFuncAttributeMaxDynamicSharedMemorySize,
      64 * 1024 + 16);
  (void)raised;
  hipLaunchKernelGGL(k_moe_route, dim3(M), dim3(512), lds, stream,
                     (const u16*)h, (const float*)g, (const u16*)wg, M, H,
                     E, topk, eps, (int*)idx, (float*)wout, (float*)dense);
  return hipGetLastError();
}

// y[m, :H] += w[m * wstride] * x[m, :H]  (bf16 I/O, f32 math): one expert's
// results for all rows, weighted by a column of the dense grid (0 if
// unrouted).
extern "C" __global__ void __launch_bounds__(256)
k_moe_scale_add(u16* __restrict__ y, const u16* __restrict__ xin,
                const float* __restrict__ w, long wstride, int M, int H) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long)M * H) return;
  const float wv = w[(size_t)(i / H) * wstride];
  if (wv != 0.f) y[i] = f2b(b2f(y[i]) + wv * b2f(xin[i]));
}

extern "C" hipError_t launch_moe_scale_add(void* y, const void* x,
                                           const void* w, long wstride,
                                           int M, int H,
                                           hipStream_t stream) {
  long total = (long)M * H;
  hipLaunchKernelGGL(k_moe_scale_add,
                     dim3((uint32_t)((total + 255) / 256)), dim3(256), 0,
                     stream, (u16*)y, (const u16*)x, (const float*)w,
                     wstride, M, H);
  return hipGetLastError();
}
