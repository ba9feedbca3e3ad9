// head_rows.hip — the head of several rows beside e4m3 weights, rows that are
// not rounded to e4m3: Y[M, N] = norm(x) W[N, K]^T, M up to 16, fp32 out.
//
// The prompts of a group end in a row each.  A product a row streamed W as
// often (16 rows of 32768x3584: 16 times 21 us); here it is read once.  A normed
// value stands as the sum of three bf16 numbers (8 bits of its mantissa each),
// W is bf16 without a rounding, so that products are exact on the matrix cores
// and sums fp32, as they are on the vector units for one row.
//
// Bound by W: a wave takes 64 rows of it over a quarter of K, x in parts comes
// out of the L2, one and a half times the bytes of W.  us, a launch a row -> here,
// W from memory, 2 and 16 rows: 32768x3584 43 -> 40 and 313 -> 53, 128256x4096
// 160 -> 148 and 1273 -> 214, 32768x2304 33 -> 30 and 239 -> 37.
#include "common.h"

typedef __bf16 hr_b8 __attribute__((ext_vector_type(8)));
typedef __bf16 hr_b2 __attribute__((ext_vector_type(2)));

#define HR_M 16
#define HR_NW 4
#define HR_TN 4                            // tiles of 16 rows of W a wave

// parts [3][16][K] of the rows' normed values; row i is rows[i] of x
__global__ void __launch_bounds__(256)
k_head_parts(const u16* __restrict__ x, const int* __restrict__ rows,
             const float* __restrict__ g, u16* __restrict__ parts, int K,
             float eps) {
  __shared__ float red[4];
  const int m = blockIdx.x, tid = threadIdx.x;
  const u16* xr = x + (size_t)rows[m] * K;
  float ss = 0.f;
  for (int i = tid * 8; i < K; i += 2048) {
    const s8v v = *(const s8v*)(xr + i);
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const float f = b2f(((const u16*)&v)[j]);
      ss += f * f;
    }
  }
  ss = wave_reduce_sum(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  const float rn = rsqrtf((red[0] + red[1] + red[2] + red[3]) / (float)K + eps);
  for (int i = tid * 8; i < K; i += 2048) {
    const s8v v = *(const s8v*)(xr + i);
    union { __bf16 e[8]; s8v s; } o[3];
#pragma unroll
    for (int j = 0; j < 8; j++) {
      float f = b2f(((const u16*)&v)[j]) * rn * g[i + j];
#pragma unroll
      for (int q = 0; q < 3; q++) {
        o[q].e[j] = (__bf16)f;
        f -= (float)o[q].e[j];
      }
    }
#pragma unroll
    for (int q = 0; q < 3; q++)
      *(s8v*)(parts + ((size_t)q * HR_M + m) * K + i) = o[q].s;
  }
}

__global__ void __launch_bounds__(64 * HR_NW)
k_head_rows(const uint8_t* __restrict__ W, const float* __restrict__ ws,
            const u16* __restrict__ parts, float* __restrict__ y, int M, int N,
            int K, float softcap) {
  __shared__ f4v sums[HR_NW][HR_TN][64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, gq = lane >> 4;
  const int n0 = blockIdx.x * (HR_TN * 16);
  // slabs of 64 k; a lane's 16 bytes are two operands, k 16 gq + 0..7 and 8..15
  const int slabs = K / 64;
  const uint8_t* wr[HR_TN];
#pragma unroll
  for (int t = 0; t < HR_TN; t++)
    wr[t] = W + (size_t)min(n0 + t * 16 + lr, N - 1) * K + gq * 16;
  const u16* xr = parts + (size_t)min(lr, M - 1) * K + gq * 16;
  f4v acc[HR_TN];
#pragma unroll
  for (int t = 0; t < HR_TN; t++) acc[t] = {0.f, 0.f, 0.f, 0.f};
  union Op { u4v_ u; hr_b8 v; hr_b2 p[4]; };
  struct Slab { u4v_ w[HR_TN]; Op x[3][2]; };
  auto load = [&](Slab& d, int s) {
    const size_t k = (size_t)min(s, slabs - 1) * 64;
#pragma unroll
    for (int t = 0; t < HR_TN; t++)
      d.w[t] = __builtin_nontemporal_load((const u4v_*)(wr[t] + k));
#pragma unroll
    for (int q = 0; q < 3; q++)
#pragma unroll
      for (int h = 0; h < 2; h++)
        d.x[q][h].u = *(const u4v_*)(xr + (size_t)q * HR_M * K + k + h * 8);
  };
  auto mul = [&](const Slab& d) {
#pragma unroll
    for (int t = 0; t < HR_TN; t++)
#pragma unroll
      for (int h = 0; h < 2; h++) {
        Op w;
#pragma unroll
        for (int e = 0; e < 2; e++) {
          const uint32_t u = d.w[t][h * 2 + e];
          w.p[e * 2] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(u, 1.0f, false);
          w.p[e * 2 + 1] =
              __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(u, 1.0f, true);
        }
#pragma unroll
        for (int q = 2; q >= 0; q--)       // the smallest first
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.v, d.x[q][h].v,
                                                           acc[t], 0, 0, 0);
      }
  };
  Slab a, b;
  int s = wave;
  if (s < slabs) {
    load(a, s);
    for (; s + HR_NW < slabs; s += 2 * HR_NW) {
      load(b, s + HR_NW);
      mul(a);
      load(a, s + 2 * HR_NW);              // at the end: of the last again
      mul(b);
    }
    if (s < slabs) mul(a);
  }
#pragma unroll
  for (int t = 0; t < HR_TN; t++) sums[wave][t][lane] = acc[t];
  __syncthreads();
  // tile `wave`: row lr of x, outputs 4 gq + 0..3 of the tile
  f4v v = sums[0][wave][lane];
#pragma unroll
  for (int k = 1; k < HR_NW; k++) v += sums[k][wave][lane];
  if (lr >= M) return;
  const int n = n0 + wave * 16 + gq * 4;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    if (n + r >= N) continue;
    float f = v[r] * ws[n + r];
    if (softcap > 0.f) f = softcap * tanhf(f / softcap);
    y[(size_t)lr * N + n + r] = f;
  }
}
static_assert(HR_TN == HR_NW, "a wave finishes a tile");

// x: bf16 rows of K, of which rows[0 .. M) are taken (device); parts: scratch
// of 3 * 16 * K bf16; y [M, N]
extern "C" hipError_t launch_head_rows(const void* x, const void* rows,
                                       const void* g, const void* w,
                                       const void* ws, void* parts, void* y,
                                       int M, int N, int K, float eps,
                                       float softcap, hipStream_t stream) {
  if (!x || !rows || !g || !w || !ws || !parts || !y || M < 1 || M > HR_M ||
      N < 1 || K < 64 || K % 64 ||
      ((size_t)x | (size_t)w | (size_t)parts) % 16)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_head_parts, dim3(M), dim3(256), 0, stream,
                     (const u16*)x, (const int*)rows, (const float*)g,
                     (u16*)parts, K, eps);
  hipLaunchKernelGGL(k_head_rows, dim3((N + HR_TN * 16 - 1) / (HR_TN * 16)),
                     dim3(64 * HR_NW), 0, stream, (const uint8_t*)w,
                     (const float*)ws, (const u16*)parts, (float*)y, M, N, K,
                     softcap);
  return hipGetLastError();
}
