// row_gemm.hip — linears of few rows: Y[M,N] = X[M,K] W[N,K]^T, up to 16 rows.
//
// Bound by streaming W once.  X (its RMSNorm taken on the way) waits in LDS
// while a block takes its share of the outputs, alike for all blocks, in tiles
// of 16 (of 8 where a share is small); W goes from memory to the MFMA operand
// with no LDS and no barrier between.  The slabs of all its tiles are one list
// that the eight waves share out evenly, the next group always in flight:
// every load is taken, at a place that stays at the list's end, for the
// compiler counts those behind a load that it waits for only where no branch
// and no use of a value stands between.  What a wave has of a tile goes to
// LDS, and the waves meet once.
// us, by tiles dealt out whole, a meeting each, and a choice of value or zero
// right behind each e4m3 and MXFP4 load -> here:
//   16 rows e4m3  2x14336x3584 34.4 -> 22.6 (4.5 TB/s), with the norm 40.5 ->
//                 27.5; 3584x14336 25.7 -> 19.1; 32768x3584 43.8 -> 29.9
//   4 rows e4m3   8192x3584 14.7 -> 9.6, 3584x14336 19.0 -> 14.0
//   3 rows bf16   4608x3584 14.8 -> 11.6, 2x18944x3584 55.4 -> 51.0 (5.3 TB/s)
//   4 rows MXFP4  2x8192x3072 14.1 -> 11.8
// Left: two us of launch, the norm of 16 rows in each block (5 us), and the
// meeting of parts where K is split.
// Deep or narrow products split K over blocks as well; the last block of a
// column group to arrive adds the parts in their order.  What used to be a
// launch of its own rides along: norm, gate activation (gate and up rows of W
// belong to the same tile), bias, soft cap, residual.
//
// A wave's load takes 8 rows x 128 bytes of W (whole lines: 6.9 TB/s; 16
// rows x 64 bytes reach 5.7), which leaves lane l with row l&7 and 16-byte
// chunk l>>3 of it.  Two such loads (rows 0-7, 8-15) and an exchange with
// lane l^8 put row l&15 with chunks 2(l>>4) and 2(l>>4)+1 into every lane:
// the MFMA operand, since the order of k is free as long as X agrees.
// MXFP4 weights are widened to bf16 in registers (exact) beside a bf16 X;
// e4m3 weights meet rows of X rounded to e4m3, as in the prompt's products.
#include <type_traits>

#include "common.h"
#include "mid_gemm.h"

typedef __bf16 rg_b8 __attribute__((ext_vector_type(8)));
typedef __bf16 rg_b2 __attribute__((ext_vector_type(2)));
typedef float rg_f4 __attribute__((ext_vector_type(4), aligned(4)));

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
  int rpb;             // outputs of a block
  int n16;             // NORM 2
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

#define RG_NW 8
#define RG_NORM_K 4096     // the longest row that is normed on the way

// NB: outputs of a tile (8: half of an MFMA tile).  NORM 2: to bf16 before
// e4m3, like a prompt's rows (a choice in the loop cost 16 rows 2 us).
template <int WT, int NB, bool GLU, int NORM>
__global__ void __launch_bounds__(64 * RG_NW) k_row_gemm(RgArgs a) {
  constexpr int E = RgT<WT>::E, SE = 8 * E;  // elements of a chunk, a slab
  constexpr int XF = E / 8;                  // fragments of a chunk
  constexpr int XB = WT == RG_FP8 ? 1 : 2;   // bytes of an x in LDS
  constexpr int P = GLU ? 2 : 1;             // weight rows of an output
  constexpr int R = NB / 8;                  // loads of a slab and matrix
  constexpr int U = 8 / (P * R);             // slabs of a group: 8 loads
  __shared__ float sx[16];
  __shared__ int last_flag;
  // X, then what the waves have of the tiles: of tile t wave w's is w + t,
  // since a wave starts where the one before ends
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
  const int n0 = blockIdx.x * a.rpb, n1 = min(n0 + a.rpb, a.N);
  const int ntile = (n1 - n0 + NB - 1) / NB;
  const int xstride = nslab * SE * XB + 16;  // bytes: rows on other banks

  // a wave's place in the list: slabs still to come, the next one's tile, slab
  struct Place { int left, t, s; };
  const int steps = ntile * nslab, per = (steps + RG_NW - 1) / RG_NW;
  float* red = (float*)(xs + a.M * xstride);
  Place at;                                  // a wave without slabs: left 0
  {
    const int lo = min(wave * per, steps), l = min(lo, steps - 1);
    at.left = min(per, steps - lo);
    at.t = l / nslab;
    at.s = l % nslab;
  }
  auto step = [&](Place& p, int by) {        // by 1 or 0, without a branch
    p.left -= by;
    p.s += by;
    const int over = p.s == nslab;
    p.s -= over ? nslab : 0;
    p.t += over;
  };

  u4v_ wa[U][P * R], wb[U][P * R];
  uint32_t ea[U][P], eb[U][P];
  Place ahead = at;
  auto load = [&](u4v_ (&w)[U][P * R], uint32_t (&ex)[U][P]) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      // behind K (e4m3, MXFP4: half a slab) X is zero, whatever W is
      const int ke = k0 + ahead.s * SE + c8 * E;
      const size_t kb = (size_t)(SE == 64 || ke < a.K ? ke : 0) * 16 / E;
#pragma unroll
      for (int m = 0; m < P; m++) {
#pragma unroll
        for (int r = 0; r < R; r++) {
          const size_t row = (size_t)m * a.N +
                             min(n0 + ahead.t * NB + r * 8 + r8, n1 - 1);
          w[u][m * R + r] = __builtin_nontemporal_load(
              (const u4v_*)((const char*)a.w +
                            row * ((size_t)a.K * 16 / E) + kb));
        }
        if constexpr (WT == RG_FP4) {
          // exponents of this lane's two chunks after the exchange
          const size_t row = (size_t)m * a.N +
                             min(n0 + ahead.t * NB + (lr & (NB - 1)), n1 - 1);
          const int k2 = min((k0 + ahead.s * SE) / 32 + gq * 2, a.K / 32 - 2);
          ex[u][m] = *(const u16*)(a.we + row * (a.K / 32) + k2);
        }
      }
      step(ahead, ahead.left > 1);
    }
  };

  // what an output needs besides its sum: of a thread's first ones ahead of
  // all else
  struct Rest { float s, s2, add; };
  auto rest = [&](int e) {
    const int row = (e >> 4) & 15, cl = e & 15, n = n0 + (e >> 8) * NB + cl;
    Rest o = {1.f, 1.f, 0.f};
    if (row >= a.M || n >= n1 || cl >= NB) return o;
    if (WT == RG_FP8) {
      o.s = a.ws[n];
      if (GLU) o.s2 = a.ws[a.N + n];
    }
    if (a.bias) o.add = b2f(a.bias[n]);
    if (a.res) o.add += b2f(a.res[(size_t)row * a.ldr + n]);
    return o;
  };
  constexpr int NT = 64 * RG_NW, J = 2;
  Rest o[J];
#pragma unroll
  for (int j = 0; j < J; j++)
    if (KS == 1) o[j] = rest(tid + j * NT);

  // X into LDS, zeros behind K.  Its loads go out ahead of W's: they come
  // from L2 and return first, and loads return in order.
  if constexpr (NORM > 0) {
    s8v v[2][RG_NORM_K / 512];
    rg_f4 g[RG_NORM_K / 512][2];
#pragma unroll
    for (int j = 0; j < RG_NORM_K / 512; j++)
      if (j * 512 < kn) {
        const int k = min(j * 512 + lane * 8, kn - 8);
        g[j][0] = *(const rg_f4*)(a.g + k);
        g[j][1] = *(const rg_f4*)(a.g + k + 4);
#pragma unroll
        for (int i = 0; i < 2; i++) {
          const int row = i * RG_NW + wave;
          if (row < a.M)
            v[i][j] = *(const s8v*)((const u16*)a.x + (size_t)row * a.ldx + k);
        }
      }
    load(wa, ea);
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int row = i * RG_NW + wave;
      if (row >= a.M) break;
      float ss = 0.f;
#pragma unroll
      for (int j = 0; j < RG_NORM_K / 512; j++)
        if (j * 512 + lane * 8 < kn)
#pragma unroll
          for (int q = 0; q < 8; q++) {
            const float f = b2f(((u16*)&v[i][j])[q]);
            ss += f * f;
          }
      const float rn = rsqrtf(wave_reduce_sum(ss) / (float)a.K + a.eps);
      auto normed = [&](int j, int q) {
        const float f = b2f(((u16*)&v[i][j])[q]) * rn * g[j][q / 4][q % 4];
        return NORM == 2 ? b2f(f2b(f)) : f;
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
    const float rper = 1.f / per;            // e / per: exact below 2^20
    u4v_ v[NV];
    auto get = [&](int e) {
      const int row = (int)((e + 0.5f) * rper), k = (e - row * per) * VE;
      u4v_ r{};
      if (e < all && k < kn)
        r = *(const u4v_*)((const char*)a.x +
                           ((size_t)row * a.ldx + k0 + k) * XB);
      return r;
    };
    auto put = [&](int e, u4v_ r) {
      const int row = (int)((e + 0.5f) * rper), k = (e - row * per) * VE;
      if (e < all) *(u4v_*)(xs + row * xstride + k * XB) = r;
    };
#pragma unroll
    for (int j = 0; j < NV; j++)
      if (j * NT < all) v[j] = get(j * NT + tid);
    const float sr = WT == RG_FP8 ? a.sx[min(tid, a.M - 1)] : 0.f;
    load(wa, ea);
    if (WT == RG_FP8 && tid < a.M) sx[tid] = sr;
#pragma unroll
    for (int j = 0; j < NV; j++)
      if (j * NT < all) put(j * NT + tid, v[j]);
    for (int e0 = NV * NT; e0 < all; e0 += NV * NT) {
#pragma unroll
      for (int j = 0; j < NV; j++) v[j] = get(e0 + j * NT + tid);
#pragma unroll
      for (int j = 0; j < NV; j++) put(e0 + j * NT + tid, v[j]);
    }
  }
  const char* xr = xs + min(lr, a.M - 1) * xstride + gq * 2 * E * XB;
  __syncthreads();

  auto finish = [&](int e, float v, float up, const Rest& o) {
    const int row = (e >> 4) & 15, cl = e & 15, n = n0 + (e >> 8) * NB + cl;
    if (row >= a.M || n >= n1 || cl >= NB) return;
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
      v = gate_act(v, a.act) * up;
    }
    if (a.softcap > 0.f) v = a.softcap * tanhf(v / a.softcap);
    v += o.add;
    if (a.out_f32) ((float*)a.y)[(size_t)row * a.ldy + n] = v;
    else ((u16*)a.y)[(size_t)row * a.ldy + n] = f2b(v);
  };

  f4v acc[P];
#pragma unroll
  for (int p = 0; p < P; p++) acc[p] = {0.f, 0.f, 0.f, 0.f};
  auto group = [&](u4v_ (&w)[U][P * R], uint32_t (&ex)[U][P]) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      // row lr, chunks 2gq and 2gq+1 of either matrix
      u4v_ ch[P][2];
#pragma unroll
      for (int p = 0; p < P; p++) {
        if constexpr (R == 1) {
          // rows 8-15 are not there: their outputs are dropped
          ch[p][0] = w[u][p];
#pragma unroll
          for (int d = 0; d < 4; d++) ch[p][1][d] = swap8(w[u][p][d]);
        } else {
#pragma unroll
          for (int d = 0; d < 4; d++) {
            const uint32_t a0 = w[u][p * R][d], a1 = w[u][p * R + 1][d];
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
              xr + at.s * SE * XB + (q * XF + f) / (3 - XB) * 16);
#pragma unroll
          for (int p = 0; p < P; p++)
            acc[p] = rg_mma<WT>(xf, ch[p][q], f,
                                WT == RG_FP4 ? (ex[u][p] >> (8 * q)) & 255
                                             : 0, acc[p]);
        }
      // sums behind the list's end are not put anywhere
      const int t = at.t;
      step(at, 1);
      if (at.left >= 0 && (at.s == 0 || at.left == 0)) {
        // element r of acc: row gq*4 + r, output lr
#pragma unroll
        for (int p = 0; p < P; p++) {
#pragma unroll
          for (int r = 0; r < 4; r++)
            red[((wave + t) * P + p) * 256 + (gq * 4 + r) * 16 + lr] =
                acc[p][r];
          acc[p] = {0.f, 0.f, 0.f, 0.f};
        }
      }
    }
  };
  // the last group by itself: no loads behind it
  for (int todo = at.left - U;;) {
    if (todo <= 0) {
      group(wa, ea);
      break;
    }
    load(wb, eb);
    todo -= U;
    group(wa, ea);
    if (todo <= 0) {
      group(wb, eb);
      break;
    }
    load(wa, ea);
    todo -= U;
    group(wb, eb);
  }

  // outputs of four tiles at a time, two a thread
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  const int tiles = (a.rpb + NB - 1) / NB;   // of a full block
  float* parts = a.part + (size_t)blockIdx.x * tiles * KS * (P * 256);
  const float rper = 1.f / per;
  for (int e0 = tid; e0 < ntile * 256; e0 += NT * J) {
    if (KS == 1 && e0 != tid)
#pragma unroll
      for (int j = 0; j < J; j++) o[j] = rest(e0 + j * NT);
#pragma unroll
    for (int j = 0; j < J; j++) {
      const int e = e0 + j * NT, t = e >> 8;
      if (t >= ntile || ((e >> 4) & 15) >= a.M) continue;
      // waves that have slabs of it; exact for less than 2^20 slabs
      const int lo = (int)((t * nslab + 0.5f) * rper);
      const int hi = (int)((t * nslab + nslab - 0.5f) * rper);
      float v = 0.f, up = 0.f;
      for (int q = lo; q <= hi; q++) {
        v += red[(q + t) * P * 256 + (e & 255)];
        if (GLU) up += red[((q + t) * P + P - 1) * 256 + (e & 255)];
      }
      if (KS == 1) {
        finish(e, v, up, o[j]);
      } else {
        float* pp = parts + ((size_t)t * KS + blockIdx.y) * (P * 256) + (e & 255);
        part_put(pp, v);
        if (GLU) part_put(pp + 256, up);
      }
    }
  }
  if (KS == 1) return;

  // the last of the blocks that share these columns adds the parts
  if (!last_block(&a.cnt[blockIdx.x], KS, &last_flag)) return;
  for (int e = tid; e < ntile * 256; e += 64 * RG_NW) {
    if (((e >> 4) & 15) >= a.M) continue;
    const float* pp = parts + (size_t)(e >> 8) * KS * (P * 256) + (e & 255);
    const Rest o = rest(e);
    float v = 0.f, up = 0.f;
    for (int q0 = 0; q0 < KS; q0 += 8) {     // eight parts a trip
      float x[8], y[8];
#pragma unroll
      for (int q = 0; q < 8; q++) {
        const float* at = pp + (size_t)min(q0 + q, KS - 1) * (P * 256);
        x[q] = part_get(at);
        if (GLU) y[q] = part_get(at + 256);
      }
#pragma unroll
      for (int q = 0; q < 8; q++)
        if (q0 + q < KS) {
          v += x[q];
          if (GLU) up += y[q];
        }
    }
    finish(e, v, up, o);
  }
}

#define RG_ROOM (159 * 1024)     // LDS of a block: X and the sums

template <int WT, int NB, bool GLU, int NORM>
static void rg_go(const RgArgs& a, dim3 grid, size_t lds, hipStream_t s) {
  static const hipError_t raised = hipFuncSetAttribute(
      (const void*)&k_row_gemm<WT, NB, GLU, NORM>,
      hipFuncAttributeMaxDynamicSharedMemorySize, RG_ROOM);
  (void)raised;
  hipLaunchKernelGGL((k_row_gemm<WT, NB, GLU, NORM>), grid, dim3(64 * RG_NW),
                     lds, s, a);
}

// How a product goes: m rows a launch, K in ks parts of kr, rpb outputs a
// block in tiles of nb, ng blocks a part; LDS of a block, floats of `part`.
struct RgPlan { int m, ks, kr, rpb, nb, ng; long lds, floats; };

static int rg_up(int a, int b) { return (a + b - 1) / b; }

static bool rg_plan_rows(RgPlan& p, int wt, bool glu, bool norm, int M, int N,
                         int K, long part_floats, int ncnt) {
  const int P = glu ? 2 : 1, XB = wt == RG_FP8 ? 1 : 2;
  const int SE = wt == RG_BF16 ? 64 : wt == RG_FP8 ? 128 : 256;
  // A block a CU, with X in place for all its outputs: two a CU read X twice
  // and run no faster (5 rows, 2x8192x2048: 16.9 us, 512 blocks 21.1;
  // 32768x3072 38.9 and 43.9).  Less than eight outputs a block gain nothing;
  // more than LDS has room for the sums of are left to blocks of a next round.
  auto plan = [&](int ks) {
    RgPlan q = {M, ks, rg_up(rg_up(K, ks), SE) * SE, 0, 16, 0, 0, 0};
    q.lds = (long)M * (q.kr * XB + 16);
    const int r = rg_up(N, 256 / ks > 1 ? 256 / ks : 1);
    const long most = (RG_ROOM - q.lds) / (P * 1024) - (RG_NW - 1);
    if (most < 1) return q;                  // ng 0: X does not fit
    q.rpb = r < 8 ? 8 : r < most * 16 ? r : (int)most * 16;
    if (q.rpb <= 24 && (q.rpb - 1) % 16 < 8 && rg_up(q.rpb, 8) <= most)
      q.nb = 8;
    q.ng = rg_up(N, q.rpb);
    const int tiles = rg_up(q.rpb, q.nb);
    q.lds += (long)(tiles + RG_NW - 1) * P * 1024;
    if (ks > 1) q.floats = (long)q.ng * tiles * ks * P * 256;
    return q;
  };
  auto fits = [&](const RgPlan& q) {
    return q.ng && (q.ks == 1 || (!norm && q.floats <= part_floats &&
                                  q.ng <= ncnt));
  };
  // the next number of parts that has slabs for all of them
  auto after = [&](int ks) {
    do ks++;
    while (ks < 64 && rg_up(K, rg_up(rg_up(K, ks), SE) * SE) != ks);
    return ks;
  };
  // as many parts of K as it takes for X to fit
  p = plan(1);
  for (int ks = after(1); ks < 64 && !fits(p); ks = after(ks)) p = plan(ks);
  if (!fits(p)) return false;
  // Narrow products: more parts until the 256 CUs have a block each, or a
  // part is down to 512.  (5 rows, 2048x8192: 128 blocks 12.0 us, 256 of half
  // tiles 10.1.)
  while (p.ng * p.ks < 192) {
    const int ks = after(p.ks);
    if (ks > 16 || K / ks < 512) break;
    const RgPlan q = plan(ks);
    if (!fits(q)) break;
    p = q;
  }
  return true;
}

// Where the room for parts is too small for the rows' X, fewer rows a launch.
static bool rg_plan(RgPlan& p, int wt, bool glu, bool norm, int M, int N,
                    int K, long part_floats, int ncnt) {
  for (int m = M; m > 0; m = m > 1 ? (m + 1) / 2 : 0)
    if (rg_plan_rows(p, wt, glu, norm, m, N, K, part_floats, ncnt))
      return true;
  return false;
}

template <int WT, bool GLU>
static hipError_t rg_run(RgArgs a, long part_floats, int ncnt,
                         hipStream_t s) {
  RgPlan p;
  if (!rg_plan(p, WT, GLU, a.g, a.M, a.N, a.K, part_floats, ncnt))
    return hipErrorInvalidValue;
  a.kr = p.kr;
  a.rpb = p.rpb;
  const dim3 grid(p.ng, p.ks);
  auto go = [&](auto norm) {
    if (p.nb == 8) rg_go<WT, 8, GLU, decltype(norm)::value>(a, grid, p.lds, s);
    else rg_go<WT, 16, GLU, decltype(norm)::value>(a, grid, p.lds, s);
  };
  const RgArgs all = a;
  for (int r = 0; r < all.M; r += p.m) {
    a.M = all.M - r < p.m ? all.M - r : p.m;
    a.x = (const char*)all.x +
          (size_t)r * a.ldx * (WT == RG_FP8 && !a.g ? 1 : 2);
    if (a.sx) a.sx = all.sx + r;
    if (a.res) a.res = all.res + (size_t)r * a.ldr;
    a.y = (char*)all.y + (size_t)r * a.ldy * (a.out_f32 ? 4 : 2);
    if (!a.g) go(std::integral_constant<int, 0>());
    else if (WT != RG_FP8 || !a.n16) go(std::integral_constant<int, 1>());
    else go(std::integral_constant<int, WT == RG_FP8 ? 2 : 1>());
  }
  return hipGetLastError();
}

// The plan of a product as numbers (m, ks, kr, rpb, nb, ng), its LDS and the
// floats of `part` that it takes; what it would take where there is room
// enough says how much to allocate.
extern "C" hipError_t row_gemm_plan(int wt, int glu, int norm, int M, int N,
                                    int K, long part_floats, int ncnt,
                                    long* out) {
  RgPlan p;
  if (wt < 0 || wt > RG_FP4 || M < 1 || M > 16 || N < 1 || K < 64 || K % 64 ||
      !rg_plan(p, wt, glu, norm, M, N, K, part_floats, ncnt))
    return hipErrorInvalidValue;
  const long v[8] = {p.m, p.ks, p.kr, p.rpb, p.nb, p.ng, p.lds, p.floats};
  for (int i = 0; i < 8; i++) out[i] = v[i];
  return hipSuccess;
}

// wt: 0 bf16, 1 e4m3 with ws, 2 MXFP4 with we.  act < 0: no gate.
extern "C" hipError_t launch_row_gemm(
    const void* x, const void* sx, const void* w, const void* ws,
    const void* we, const void* g, const void* bias, const void* res, void* y, void* part,
    void* cnt, long part_floats, int ncnt, int wt, int M, int N, int K,
    int ldx, int ldr, int ldy, int act, int out_f32, int n16, float eps,
    float softcap, hipStream_t stream) {
  if (M < 1 || M > 16 || N < 1 || K < 64 || K % 64 || ldx < K || ldx % (wt == RG_FP8 && !g ? 16 : 8) ||
      ldy < N || (res && ldr < N) || (g && K > RG_NORM_K) ||
      (wt == RG_FP8 && (!ws || (!g && !sx))) || (wt == RG_FP4 && !we))
    return hipErrorInvalidValue;
  RgArgs a = {x, (const float*)sx, w, (const float*)ws, (const uint8_t*)we,
              (const float*)g, (const u16*)bias, (const u16*)res, y,
              (float*)part, (int*)cnt, M, N, K, ldx, ldr, ldy, act, out_f32,
              0, 0, n16, eps, softcap};
  if (!part || !cnt) part_floats = 0;
  if (!g && wt != RG_FP4 && act < 0 && mid_takes(wt == RG_FP8, M, N, K, false))
    return launch_mid_gemm(x, w, wt == RG_FP8 ? sx : nullptr, ws, res, bias,
                           y, part, cnt, part_floats, ncnt, M, N, K, ldx, ldr,
                           ldy, act, out_f32, softcap, stream);
#define RG_CASE(WTV)                                                         \
  return act >= 0 ? rg_run<WTV, true>(a, part_floats, ncnt, stream)          \
                  : rg_run<WTV, false>(a, part_floats, ncnt, stream)
  if (wt == RG_BF16) RG_CASE(RG_BF16);
  if (wt == RG_FP8) RG_CASE(RG_FP8);
  if (wt == RG_FP4) RG_CASE(RG_FP4);
#undef RG_CASE
  return hipErrorInvalidValue;
}
