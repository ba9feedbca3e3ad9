// row_gemm.hip — linears of few rows: Y[M,N] = X[M,K] W[N,K]^T, up to 16 rows.
//
// Bound by streaming W once.  X (its RMSNorm taken on the way) waits in LDS
// while a block walks tiles of 16 outputs; its eight waves share out K, so
// W goes from memory to the MFMA operand with no LDS and no barrier between,
// the next slabs already in flight, and the partial sums meet in LDS once a
// tile.  Deep or narrow products split K over blocks as well; the last block
// of a column group to arrive adds the parts in their order.  What used to
// be a launch of its own rides along: norm, gate activation (gate and up
// rows of W belong to the same tile), bias, soft cap, residual.
//
// A wave's load takes 8 rows x 128 bytes of W (whole lines: 6.9 TB/s; 16
// rows x 64 bytes reach 5.7), which leaves lane l with row l&7 and 16-byte
// chunk l>>3 of it.  Two such loads (rows 0-7, 8-15) and an exchange with
// lane l^8 put row l&15 with chunks 2(l>>4) and 2(l>>4)+1 into every lane:
// the MFMA operand, since the order of k is free as long as X agrees.
// MXFP4 weights are widened to bf16 in registers (exact) beside a bf16 X;
// e4m3 weights meet rows of X rounded to e4m3, as in the prompt's products.
#include "common.h"

typedef __bf16 rg_b8 __attribute__((ext_vector_type(8)));
typedef __bf16 rg_b2 __attribute__((ext_vector_type(2)));

struct RgArgs {
  const void* x;       // [M, ldx] bf16; e4m3 beside e4m3 weights and no norm
  const float* sx;     // e4m3 x: scale of a row
  const void* w;       // [N, K] (with an activation [2N, K]: gate, then up)
  const float* ws;     // e4m3: scale of a row
  const uint8_t* we;   // MXFP4: exponents [rows, K/32]
  const float* g;      // RMSNorm weights [K]
  const u16* bias;     // [N]
  const u16* res;      // [M, ldr]
  void* y;             // [M, ldy]
  float* part;         // split K: sums of a tile, [tile, split, ...]
  int* cnt;            // split K: blocks of a column group that are done
  int M, N, K, ldx, ldr, ldy, act, out_f32, kr;
  float eps, softcap;
};

enum { RG_BF16 = 0, RG_FP8 = 1, RG_FP4 = 2 };
template <int WT> struct RgT;
template <> struct RgT<RG_BF16> { static constexpr int E = 8; };
template <> struct RgT<RG_FP8> { static constexpr int E = 16; };
template <> struct RgT<RG_FP4> { static constexpr int E = 32; };

// elements 8f..8f+7 of a 16-byte chunk, times 8 of X
template <int WT>
DEVINL f4v rg_mma(u4v_ x, u4v_ c, int f, uint32_t e8, f4v acc) {
  if constexpr (WT == RG_FP8) {
    union { u4v_ u; long l[2]; } a, b;
    a.u = x;
    b.u = c;
    return __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(a.l[f], b.l[f], acc, 0,
                                                      0, 0);
  } else {
    union { rg_b2 p[4]; rg_b8 v; u4v_ u; } a, b;
    a.u = x;
    if constexpr (WT == RG_BF16) {
      b.u = c;
    } else {
      const float s = __uint_as_float(e8 << 23);
      b.p[0] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(c[f], s, 0);
      b.p[1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(c[f], s, 1);
      b.p[2] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(c[f], s, 2);
      b.p[3] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(c[f], s, 3);
    }
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, acc, 0, 0, 0);
  }
}

DEVINL uint32_t swap8(uint32_t v) {        // the value of lane l^8
  return __builtin_amdgcn_update_dpp(0, v, 0x128, 0xf, 0xf, true);
}

DEVINL float rg_act(float x, int act) {
  if (act == 0) return x / (1.f + __expf(-x));
  const float c = 0.7978845608028654f * (x + 0.044715f * x * x * x);
  return 0.5f * x * (1.f + tanhf(c));
}

#define RG_NW 8
#define RG_NORM_K 4096     // the longest row that is normed on the way

// NB: outputs of a tile (8: half of an MFMA tile).
template <int WT, int NB, bool GLU, bool NORM>
__global__ void __launch_bounds__(64 * RG_NW) k_row_gemm(RgArgs a) {
  constexpr int E = RgT<WT>::E, SE = 8 * E;  // elements of a chunk, a slab
  constexpr int XF = E / 8;                  // fragments of a chunk
  constexpr int XB = WT == RG_FP8 ? 1 : 2;   // bytes of an x in LDS
  constexpr int P = GLU ? 2 : 1;             // weight rows of an output
  constexpr int R = NB / 8;                  // loads of a slab and matrix
  constexpr int U = 8 / (P * R);             // slabs of a group: 8 loads
  __shared__ __attribute__((aligned(16))) float red[RG_NW][P][256];
  __shared__ float sx[16];
  __shared__ int last_flag;
  extern __shared__ __attribute__((aligned(16))) char xs[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, gq = lane >> 4;
  const int r8 = lane & 7, c8 = lane >> 3;
  const bool low = lr < 8;
  const int KS = gridDim.y;
  const int k0 = blockIdx.y * a.kr;
  const int kn = min(a.kr, a.K - k0);        // elements of this block
  const int nslab = (kn + SE - 1) / SE;
  const int spw = (nslab + RG_NW - 1) / RG_NW;
  const int s_lo = min(wave * spw, nslab), s_hi = min(s_lo + spw, nslab);
  const int ngrp = (spw + U - 1) / U;        // alike in all waves
  const int ntile = (a.N + NB - 1) / NB;
  const int xstride = nslab * SE * XB + 16;  // bytes: rows on other banks

  u4v_ wc[U][P * R], wn[U][P * R];
  uint32_t ec[U][P], en[U][P];
  auto load = [&](u4v_ (&w)[U][P * R], uint32_t (&ex)[U][P], int tile,
                  int grp) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int s = s_lo + grp * U + u;
      if (s < s_hi) {
        const int ke = k0 + s * SE + c8 * E;
        const bool in = SE == 64 || ke < a.K;   // K is a multiple of 64
#pragma unroll
        for (int p = 0; p < P; p++) {
#pragma unroll
          for (int r = 0; r < R; r++) {
            const size_t row = (size_t)p * a.N +
                               min(tile * NB + r * 8 + r8, a.N - 1);
            const char* q = (const char*)a.w + row * ((size_t)a.K * 16 / E) +
                            (size_t)(in ? ke : 0) * 16 / E;
            w[u][p * R + r] = __builtin_nontemporal_load((const u4v_*)q);
            if (!in) w[u][p * R + r] = u4v_{};
          }
          if constexpr (WT == RG_FP4) {
            // exponents of this lane's two chunks after the exchange
            const size_t row = (size_t)p * a.N +
                               min(tile * NB + (lr & (NB - 1)), a.N - 1);
            const int kb = (k0 + s * SE) / 32 + gq * 2;
            ex[u][p] = kb < a.K / 32
                           ? *(const u16*)(a.we + row * (a.K / 32) + kb)
                           : 0;
          }
        }
      }
    }
  };

  int tile = blockIdx.x;

  // X into LDS, zeros behind K.  Its loads go out ahead of W's: they come
  // from L2 and return first, and loads return in order.
  if constexpr (NORM) {
    s8v v[2][RG_NORM_K / 512];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < RG_NORM_K / 512; j++) {
        const int row = i * RG_NW + wave, k = j * 512 + lane * 8;
        v[i][j] = s8v{};
        if (row < a.M && k < kn)
          v[i][j] = *(const s8v*)((const u16*)a.x + (size_t)row * a.ldx + k);
      }
    load(wc, ec, tile, 0);
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int row = i * RG_NW + wave;
      if (row >= a.M) break;
      float ss = 0.f;
#pragma unroll
      for (int j = 0; j < RG_NORM_K / 512; j++)
#pragma unroll
        for (int q = 0; q < 8; q++) {
          const float f = b2f(((u16*)&v[i][j])[q]);
          ss += f * f;
        }
      const float rn = rsqrtf(wave_reduce_sum(ss) / (float)a.K + a.eps);
      auto normed = [&](int j, int q) {
        return b2f(((u16*)&v[i][j])[q]) * rn * a.g[j * 512 + lane * 8 + q];
      };
      float am = 1.f;
      if constexpr (WT == RG_FP8) {          // rows rounded to e4m3
        am = 0.f;
#pragma unroll
        for (int j = 0; j < RG_NORM_K / 512; j++)
          if (j * 512 + lane * 8 < kn)
#pragma unroll
            for (int q = 0; q < 8; q++) am = fmaxf(am, fabsf(normed(j, q)));
#pragma unroll
        for (int w = 1; w < 64; w <<= 1) am = fmaxf(am, __shfl_xor(am, w));
        am = fmaxf(am, 1e-8f) / 448.0f;
        if (lane == 0) sx[row] = am;
      }
#pragma unroll
      for (int j = 0; j < RG_NORM_K / 512; j++) {
        const int k = j * 512 + lane * 8;
        if (k < nslab * SE) {
          float f[8] = {};
          if (k < kn) {
#pragma unroll
            for (int q = 0; q < 8; q++) f[q] = normed(j, q);
          }
          if constexpr (WT == RG_FP8) {
            *(unsigned long long*)(xs + row * xstride + k) =
                f32x8_to_fp8(f, 1.0f / am);
          } else {
            u16 o[8];
#pragma unroll
            for (int q = 0; q < 8; q++) o[q] = f2b(f[q]);
            *(s8v*)(xs + row * xstride + k * 2) = *(s8v*)o;
          }
        }
      }
    }
  } else {
    constexpr int NV = 12, VE = 16 / XB;     // 16-byte loads a thread
    const int per = nslab * SE / VE, all = a.M * per;
    u4v_ v[NV];
    auto get = [&](int e) {
      const int row = e / per, k = (e - row * per) * VE;
      u4v_ r{};
      if (e < all && k < kn)
        r = *(const u4v_*)((const char*)a.x +
                           ((size_t)row * a.ldx + k0 + k) * XB);
      return r;
    };
    auto put = [&](int e, u4v_ r) {
      const int row = e / per, k = (e - row * per) * VE;
      if (e < all) *(u4v_*)(xs + row * xstride + k * XB) = r;
    };
#pragma unroll
    for (int j = 0; j < NV; j++) v[j] = get(j * 64 * RG_NW + tid);
    load(wc, ec, tile, 0);
    if (WT == RG_FP8 && tid < a.M) sx[tid] = a.sx[tid];
#pragma unroll
    for (int j = 0; j < NV; j++) put(j * 64 * RG_NW + tid, v[j]);
    for (int e0 = NV * 64 * RG_NW; e0 < all; e0 += NV * 64 * RG_NW) {
#pragma unroll
      for (int j = 0; j < NV; j++) v[j] = get(e0 + j * 64 * RG_NW + tid);
#pragma unroll
      for (int j = 0; j < NV; j++) put(e0 + j * 64 * RG_NW + tid, v[j]);
    }
  }
  const char* xr = xs + min(lr, a.M - 1) * xstride + gq * 2 * E * XB;
  __syncthreads();

  // what an output needs besides its sum: loaded ahead of the next tile's W,
  // since loads return in order
  struct Rest { float s, s2, add; };
  auto rest = [&](int t) {
    const int row = (tid >> 4) & 15, cl = tid & 15, n = t * NB + cl;
    Rest o = {1.f, 1.f, 0.f};
    if (row >= a.M || n >= a.N || cl >= NB) return o;
    if (WT == RG_FP8) {
      o.s = a.ws[n];
      if (GLU) o.s2 = a.ws[a.N + n];
    }
    if (a.bias) o.add = b2f(a.bias[n]);
    if (a.res) o.add += b2f(a.res[(size_t)row * a.ldr + n]);
    return o;
  };
  auto finish = [&](int t, float v, float up, const Rest& o) {
    const int row = tid >> 4, cl = tid & 15, n = t * NB + cl;
    if (row >= a.M || n >= a.N || cl >= NB) return;
    if (WT == RG_FP8) {
      v *= sx[row] * o.s;
      up *= sx[row] * o.s2;
    }
    if (GLU) {
      if (WT == RG_FP8) {
        // to be rounded to e4m3 next: from bf16 halves, like the prompt's
        up = b2f(f2b(up));
        v = b2f(f2b(v));
      }
      v = rg_act(v, a.act) * up;
    }
    if (a.softcap > 0.f) v = a.softcap * tanhf(v / a.softcap);
    v += o.add;
    if (a.out_f32) ((float*)a.y)[(size_t)row * a.ldy + n] = v;
    else ((u16*)a.y)[(size_t)row * a.ldy + n] = f2b(v);
  };

  for (; tile < ntile; tile += gridDim.x) {
    f4v acc[P];
#pragma unroll
    for (int p = 0; p < P; p++) acc[p] = {0.f, 0.f, 0.f, 0.f};
    Rest ahead = {1.f, 1.f, 0.f};
    if (KS == 1 && tid < 256) ahead = rest(tile);

    for (int grp = 0; grp < ngrp; grp++) {
      const bool next = grp + 1 < ngrp;
      const int tn = next ? tile : tile + (int)gridDim.x;
      if (tn < ntile) load(wn, en, tn, next ? grp + 1 : 0);
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int s = s_lo + grp * U + u;
        if (s < s_hi) {
          // row lr, chunks 2gq and 2gq+1 of either matrix
          u4v_ ch[P][2];
#pragma unroll
          for (int p = 0; p < P; p++) {
            if constexpr (R == 1) {
              // rows 8-15 are not there: their outputs are dropped
              ch[p][0] = wc[u][p];
#pragma unroll
              for (int d = 0; d < 4; d++) ch[p][1][d] = swap8(wc[u][p][d]);
            } else {
#pragma unroll
              for (int d = 0; d < 4; d++) {
                const uint32_t a0 = wc[u][p * R][d], a1 = wc[u][p * R + 1][d];
                const uint32_t got = swap8(low ? a1 : a0);
                ch[p][0][d] = low ? a0 : got;
                ch[p][1][d] = low ? got : a1;
              }
            }
          }
#pragma unroll
          for (int q = 0; q < 2; q++)
#pragma unroll
            for (int f = 0; f < XF; f++) {
              // 8 elements of X: 16 bytes of bf16, half as much of e4m3
              const u4v_ xf = *(const u4v_*)(
                  xr + s * SE * XB + (q * XF + f) / (3 - XB) * 16);
#pragma unroll
              for (int p = 0; p < P; p++)
                acc[p] = rg_mma<WT>(xf, ch[p][q], f,
                                    WT == RG_FP4 ? (ec[u][p] >> (8 * q)) & 255
                                                 : 0, acc[p]);
            }
        }
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
#pragma unroll
        for (int j = 0; j < P * R; j++) wc[u][j] = wn[u][j];
#pragma unroll
        for (int p = 0; p < P; p++) ec[u][p] = en[u][p];
      }
    }

    // element r of acc: row gq*4 + r, output lr.  The barriers wait for LDS
    // only: the next tile's loads stay in flight.
    auto meet = [&] {
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };
#pragma unroll
    for (int p = 0; p < P; p++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        red[wave][p][(gq * 4 + r) * 16 + lr] = acc[p][r];
    meet();
    if (tid < 256) {
      float v = 0.f, up = 0.f;
#pragma unroll
      for (int q = 0; q < RG_NW; q++) {
        v += red[q][0][tid];
        if (GLU) up += red[q][P - 1][tid];
      }
      if (KS == 1) {
        finish(tile, v, up, ahead);
      } else {
        float* pp =
            a.part + ((size_t)tile * KS + blockIdx.y) * (P * 256) + tid;
        pp[0] = v;
        if (GLU) pp[256] = up;
      }
    }
    meet();
  }
  if (KS == 1) return;

  // the last of the blocks that share these columns adds the parts
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const int t = __hip_atomic_fetch_add(&a.cnt[blockIdx.x], 1,
                                         __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
    last_flag = t == KS - 1;
  }
  __syncthreads();
  if (!last_flag) return;
  if (tid == 0) {
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    a.cnt[blockIdx.x] = 0;                   // for the next launch
  }
  __syncthreads();
  if (tid >= 256) return;
  for (tile = blockIdx.x; tile < ntile; tile += gridDim.x) {
    const float* pp = a.part + (size_t)tile * KS * (P * 256) + tid;
    float v = 0.f, up = 0.f;
    for (int q = 0; q < KS; q++) {
      v += pp[(size_t)q * (P * 256)];
      if (GLU) up += pp[(size_t)q * (P * 256) + 256];
    }
    finish(tile, v, up, rest(tile));
  }
}

// LDS that X may take: all but the sums
template <bool GLU> constexpr int rg_room() {
  return (160 - RG_NW * (GLU ? 2 : 1) - 1) * 1024;
}

template <int WT, int NB, bool GLU, bool NORM>
static void rg_go(const RgArgs& a, dim3 grid, size_t lds, hipStream_t s) {
  static const hipError_t raised = hipFuncSetAttribute(
      (const void*)&k_row_gemm<WT, NB, GLU, NORM>,
      hipFuncAttributeMaxDynamicSharedMemorySize, rg_room<GLU>());
  (void)raised;
  hipLaunchKernelGGL((k_row_gemm<WT, NB, GLU, NORM>), grid, dim3(64 * RG_NW),
                     lds, s, a);
}

template <int WT, bool GLU>
static hipError_t rg_run(RgArgs a, long part_floats, int ncnt,
                         hipStream_t s) {
  constexpr int SE = 8 * RgT<WT>::E, P = GLU ? 2 : 1;
  // K per block for a split, whole slabs
  auto part_k = [&](int ks) {
    return ((a.K + ks - 1) / ks + SE - 1) / SE * SE;
  };
  auto lds_of = [&](int ks) {
    return (long)a.M * (part_k(ks) * (WT == RG_FP8 ? 1 : 2) + 16);
  };
  auto fits = [&](int ks, int nb) {
    const long nt = (a.N + nb - 1) / nb;
    return lds_of(ks) <= rg_room<GLU>() &&
           (ks == 1 || (!a.g && nt * ks * P * 256 <= part_floats &&
                        (nt < 256 ? nt : 256) <= ncnt));
  };
  // as many parts of K as it takes for X to fit
  int ks = 1, nb = 16;
  while (ks < 64 && !fits(ks, nb)) ks++;
  // Narrow products: half tiles and more parts until the 256 CUs have a
  // block each, or a part is down to 512.  (5 rows, 2048x8192: 128 blocks
  // 12.0 us, 256 of half tiles 10.1.)
  if ((a.N + 15) / 16 * ks < 192) {
    nb = 8;
    while (ks < 16 && (a.N + 7) / 8 * ks < 192 && a.K / (ks + 1) >= 512 &&
           fits(ks + 1, nb)) ks++;
  }
  if (!fits(ks, nb)) return hipErrorInvalidValue;
  a.kr = part_k(ks);
  ks = (a.K + a.kr - 1) / a.kr;
  // A block a CU, walking tiles with X in place: two a CU read X twice and
  // run no faster (5 rows, 2x8192x2048: 16.9 us, 512 blocks 21.1; 32768x3072
  // 38.9 and 43.9).
  const int nt = (a.N + nb - 1) / nb;
  int ng = 256 / ks > 1 ? 256 / ks : 1;
  if (ng > nt) ng = nt;
  dim3 grid(ng, ks);
  const size_t lds = lds_of(ks);
  if (a.g) {
    if (nb == 8) rg_go<WT, 8, GLU, true>(a, grid, lds, s);
    else rg_go<WT, 16, GLU, true>(a, grid, lds, s);
  } else {
    if (nb == 8) rg_go<WT, 8, GLU, false>(a, grid, lds, s);
    else rg_go<WT, 16, GLU, false>(a, grid, lds, s);
  }
  return hipGetLastError();
}

// wt: 0 bf16, 1 e4m3 with ws, 2 MXFP4 with we.  act < 0: no gate.
extern "C" hipError_t launch_row_gemm(
    const void* x, const void* sx, const void* w, const void* ws,
    const void* we, const void* g, const void* bias, const void* res, void* y, void* part,
    void* cnt, long part_floats, int ncnt, int wt, int M, int N, int K,
    int ldx, int ldr, int ldy, int act, int out_f32, float eps,
    float softcap, hipStream_t stream) {
  if (M < 1 || M > 16 || N < 1 || K < 64 || K % 64 || ldx < K || ldx % (wt == RG_FP8 && !g ? 16 : 8) ||
      ldy < N || (res && ldr < N) || (g && K > RG_NORM_K) ||
      (wt == RG_FP8 && (!ws || (!g && !sx))) || (wt == RG_FP4 && !we))
    return hipErrorInvalidValue;
  RgArgs a = {x, (const float*)sx, w, (const float*)ws, (const uint8_t*)we,
              (const float*)g, (const u16*)bias, (const u16*)res, y,
              (float*)part, (int*)cnt, M, N, K, ldx, ldr, ldy, act, out_f32,
              0, eps, softcap};
  if (!part || !cnt) part_floats = 0;
#define RG_CASE(WTV)                                                         \
  return act >= 0 ? rg_run<WTV, true>(a, part_floats, ncnt, stream)          \
                  : rg_run<WTV, false>(a, part_floats, ncnt, stream)
  if (wt == RG_BF16) RG_CASE(RG_BF16);
  if (wt == RG_FP8) RG_CASE(RG_FP8);
  if (wt == RG_FP4) RG_CASE(RG_FP4);
#undef RG_CASE
  return hipErrorInvalidValue;
}
