// gemm_prompt.hip — linears of many rows: Y[M,N] = X[M,K] W[N,K]^T, bf16 or
// e4m3 with row scales, or bf16 rows beside MXFP4 weights; fp32 sums, bf16
// out.
//
// Slabs of 128 bytes a row (64 bf16, 128 e4m3) go straight into LDS.  What
// bounds these products is the way there: a slab is back from L2 or memory
// after one to two microseconds, the matrix cores want one a microsecond, and
// a CU gets 45 to 55 GB/s from its L2 and what is behind it.  So tiles are as
// large as fits, and loads stay in flight across the barriers.  Tiles 256 wide
// are k_gemm_wide's; the others have two to six buffers and one barrier a slab
// that waits for the next slab only.
//
// Rows are XOR-swizzled by 16-byte slots; the DMA writes lane-linear, so the
// swizzle sits in the address that a lane reads and in the fragment reads.
// The order of k inside a slab is free as long as X and W agree: a lane's two
// slots are two bf16 operands or one e4m3 operand of the 128-deep MFMA.  W is
// the first operand, so a lane ends with four neighbouring outputs of one row
// and stores them at once.
//
// Blocks of one XCD take neighbouring tiles, rows fastest, so that its L2
// holds the few panels of W they share.  Gate and up rows of W alternate by
// 16 in a tile (GLU): a lane has both halves of its outputs and stores
// act(gate) * up, half the bytes and one launch instead of three.
//
// MXFP4 weights are widened to bf16 (exact) on their way into LDS, once a
// block, between the operands of the next products and the products at hand.
// A thread asks for its piece of a slab as many slabs ahead as there are
// buffers: two ahead, and put down before the operands are read, 2048 rows of
// 37888x3584 with the gate took 881 us, so 605.  With double-buffered tiles of
// 128x128 alone, a wait for all each slab, parts of K that were added by
// atomics to zeroed sums and a launch for each half of a gate it was 911; 130
// rows 194 us, here 91; 600 rows of 3584x18944 266, 130.  The halves of a gate
// are not rounded to bf16 any more on their way to it.
//
// With few tiles K is split over blocks; the last block of a tile to arrive
// adds the parts in their order (the result does not depend on timing).
#include <type_traits>

#include "common.h"
#include "mid_gemm.h"

typedef short gp_s8 __attribute__((ext_vector_type(8)));
typedef int gp_i8 __attribute__((ext_vector_type(8)));
typedef __bf16 gp_b2 __attribute__((ext_vector_type(2)));

struct GpArgs {
  const void* x;       // [M, K]
  const void* w;       // [N, K], GLU: [2N, K] gate then up
  const float* sx;     // e4m3: row scales
  const float* sw;
  const uint8_t* we;   // MXFP4: exponents [rows of w, K/32]
  const u16* res;      // [M, N]
  const u16* bias;     // [N]
  u16* y;              // [M, N]
  float* part;         // split K: [tile, split, BM*BN]
  int* cnt;            // split K: blocks of a tile that are done
  int M, N, K, act, tm, tn, band;
  // Routed experts: a row tile has n[t] rows of expert e[t]; row r of it is
  // pair perm[row0[t] + r].  x by token (a pair / top) and y in that order
  // (gather), or x in that order and y by pair.
  const int *perm, *tile_e, *tile_row0, *tile_n;
  int top, gather;
};

// Row and column of a tile: bands of rows of tiles, rows fastest in each.
struct GpAt { int row, col; };
DEVINL GpAt gp_at(const GpArgs& a, int tile) {
  const int all = a.band * a.tn, b = tile / all, r = tile - b * all;
  const int h = min(a.band, a.tm - b * a.band);
  return {b * a.band + r % h, r / h};
}

// gate_act with tanh by exp: an epilogue has some hundred of them a lane
DEVINL float gp_act(float x, int act) {
  if (act == 0) return x / (1.f + __expf(-x));
  const float c = 0.7978845608028654f * (x + 0.044715f * x * x * x);
  return x * (1.f - 1.f / (__expf(2.f * c) + 1.f));
}

// Barrier after the wave's LDS reads and all but its last N DMA loads.  The
// builtin tells the compiler which of them are over; it would wait for all
// of them before the next read otherwise.
template <int N> DEVINL void gp_meet() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | (N >> 4 << 14) | 7 << 4);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// The sums of a tile on their way out: parts of K meet, scales, the gate, bias,
// residual.  Fragment (i, j) of a wave holds rows row_of(i) + (lane & 15) and
// outputs col_of(j) + (lane >> 4) * 4 + 0..3 of the tile.
template <bool F8, int BM, int BN, int NW, int FM, int FN, bool GLU, bool MOE,
          bool SPLIT, class RowOf, class ColOf, class XRow>
DEVINL void gp_finish(const GpArgs& a, f4v (&acc)[FM][FN], int tile, int part,
                      int SK, int bm, int bn, int rows, int first, const int* perm, size_t w0,
                      int* last_flag, RowOf row_of, ColOf col_of, XRow x_row) {
  const int tid = threadIdx.x, lane = tid & 63, fr = lane & 15, fk = lane >> 4;
  if (SPLIT && SK > 1) {
    // fragments as they lie in registers: the last block reads them alike
    float* pp = a.part + (size_t)tile * SK * (BM * BN) + tid * 2;
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
      for (int j = 0; j < FN; j++)
        part_put4(pp + (size_t)part * (BM * BN) +
                  (i * FN + j) * (NW * 256), NW * 128, acc[i][j]);
    if (!last_block(&a.cnt[tile], SK, last_flag)) return;
    // up to 16 fragments of a part on the way at a time: a part a trip, not
    // a fragment of one
    constexpr int G = FM * FN > 16 ? 16 / FN : FM;
#pragma unroll
    for (int i0 = 0; i0 < FM; i0 += G) {
#pragma unroll
      for (int i = 0; i < G; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) acc[i0 + i][j] = {0.f, 0.f, 0.f, 0.f};
      for (int q = 0; q < SK; q++) {
        f4v t[G][FN];
#pragma unroll
        for (int i = 0; i < G; i++)
#pragma unroll
          for (int j = 0; j < FN; j++)
            t[i][j] = part_get4(pp + (size_t)q * (BM * BN) +
                                ((i0 + i) * FN + j) * (NW * 256), NW * 128);
#pragma unroll
        for (int i = 0; i < G; i++)
#pragma unroll
          for (int j = 0; j < FN; j++) acc[i0 + i][j] += t[i][j];
      }
    }
  }

  constexpr int P = GLU ? 2 : 1;
  const bool wide = a.N % 4 == 0;
  // e4m3 scales, all asked for ahead of the stores, behind which each would
  // be waited for (2048x14336x3584 with a gate 285 us, so 273)
  [[maybe_unused]] float sx[FM], sv[FN / P][4], su[FN / P][4];
  if constexpr (F8) {
#pragma unroll
    for (int i = 0; i < FM; i++)
      sx[i] = a.sx[x_row(min(bm + row_of(i) + fr, rows - 1))];
#pragma unroll
    for (int j = 0; j < FN / P; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int n = min(bn + col_of(j * P) / P + fk * 4 + r, a.N - 1);
        sv[j][r] = a.sw[w0 + n];
        if (GLU) su[j][r] = a.sw[w0 + a.N + n];
      }
  }
#pragma unroll
  for (int i = 0; i < FM; i++) {
    const int r_in = bm + row_of(i) + fr;
    if (r_in >= rows) continue;
    const int row = !MOE ? r_in : a.gather ? first + r_in : perm[r_in];
#pragma unroll
    for (int j = 0; j < FN; j += P) {
      const int n = bn + col_of(j) / P + fk * 4;
      if (n >= a.N) continue;
      f4v v = acc[i][j];
      if (F8) {
#pragma unroll
        for (int r = 0; r < 4; r++) v[r] *= sx[i] * sv[j / P][r];
      }
      if constexpr (GLU) {
        f4v u = acc[i][j + 1];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          if (F8) {
            // to be rounded to e4m3 next, where a value's last bits decide
            // which of two it takes: from bf16 halves, as by single launches
            u[r] = (float)(__bf16)(u[r] * sx[i] * su[j / P][r]);
            v[r] = (float)(__bf16)v[r];
          }
          v[r] = gp_act(v[r], a.act) * u[r];
        }
      }
      const size_t at = (size_t)row * a.N + n;
      if (wide) {
        union { gp_b2 b[2]; u16 h[4]; unsigned long long q; } o;
        if (a.bias) {
          o.q = *(const unsigned long long*)(a.bias + n);
#pragma unroll
          for (int r = 0; r < 4; r++) v[r] += b2f(o.h[r]);
        }
        if (a.res) {
          o.q = *(const unsigned long long*)(a.res + at);
#pragma unroll
          for (int r = 0; r < 4; r++) v[r] += b2f(o.h[r]);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) o.b[r / 2][r % 2] = (__bf16)v[r];
        *(unsigned long long*)(a.y + at) = o.q;
      } else {
        for (int r = 0; r < 4 && n + r < a.N; r++) {
          float f = v[r];
          if (a.bias) f += b2f(a.bias[n + r]);
          if (a.res) f += b2f(a.res[at + r]);
          a.y[at + r] = f2b(f);
        }
      }
    }
  }
}

// Two waves a SIMD, of one block or of two: left to itself, 128x128 by four waves
// took 264 registers beside MXFP4, so that one block fitted a CU
// (1974x14336x128 with a gate 48 us, then 87).
template <bool F8, int BM, int BN, int WM, int WN, int NS, bool GLU,
          bool MOE = false, bool W4 = false, bool FAR = false, bool NT = false>
__global__ void __launch_bounds__(64 * WM * WN, 2) k_gemm_prompt(GpArgs a) {
  constexpr int NW = WM * WN;
  constexpr int FM = BM / WM / 16, FN = BN / WN / 16;   // fragments of a wave
  constexpr int AI = BM / 8 / NW, BI = BN / 8 / NW;     // DMA of a wave
  static_assert(AI > 0 && BI > 0 && FM > 0 && FN % (GLU ? 2 : 1) == 0);
  // loads of a wave for a slab (MXFP4: a piece of W and its exponent)
  constexpr int PS = W4 ? AI + 2 : AI + BI;
  // An array a buffer, and the loop unrolled over them: the compiler sees
  // that a DMA into one does not touch what is read from another, and puts
  // no wait for it before the reads.
  constexpr int ZA = BM * 128, ZB = BN * 128;
#define GP_BUF(i)                                                            \
  __shared__ __attribute__((aligned(16))) char A##i[NS > i ? ZA : 16],       \
      B##i[NS > i ? ZB : 16];
  GP_BUF(0) GP_BUF(1) GP_BUF(2) GP_BUF(3) GP_BUF(4) GP_BUF(5)
#undef GP_BUF
  char* const A[6] = {A0, A1, A2, A3, A4, A5};
  char* const B[6] = {B0, B1, B2, B3, B4, B5};
  [[maybe_unused]] __shared__ int last_flag;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  // tiles of an XCD (block id modulo 8) are neighbours
  const int tiles = a.tm * a.tn, chunk = (tiles + 7) / 8;
  const int tile = (blockIdx.x & 7) * chunk + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= chunk || tile >= tiles) return;
  const GpAt at = MOE ? GpAt{tile % a.tm, tile / a.tm} : gp_at(a, tile);
  const int bm = MOE ? 0 : at.row * BM;
  const int bn = at.col * (GLU ? BN / 2 : BN);
  // the rows of a tile that are there
  const int rows = MOE ? a.tile_n[at.row] : a.M;
  if (MOE && rows == 0) return;
  const int* perm = MOE ? a.perm + a.tile_row0[at.row] : nullptr;
  const int first = MOE ? a.tile_row0[at.row] : 0;
  const size_t w0 = MOE ? (size_t)a.tile_e[at.row] * (GLU ? 2 : 1) * a.N
                        : 0;                 // first row of the expert's W
  auto x_row = [&](int r) {
    if (!MOE) return r;
    return a.gather ? perm[r] / a.top : first + r;
  };

  const size_t rowb = (size_t)a.K * (F8 ? 1 : 2);       // bytes of a row
  const int slabs = (int)((rowb + 127) / 128);
  const int SK = gridDim.y, per = (slabs + SK - 1) / SK;
  const int s_lo = blockIdx.y * per, s_hi = min(s_lo + per, slabs);
  // e4m3 rows of 64 * odd: the last slab is half a slab
  const bool half = F8 && (rowb & 127) && s_hi == slabs;

  const int g_r = lane >> 3, g_s = lane & 7;
  // Where a lane's rows lie behind the tile's first: 32 bits beside a base in
  // scalar registers (an expert's rows of x are anywhere; beside MXFP4 weights
  // a launch takes 0.35 us longer so).  FAR: rows so long that 32 bits are not
  // enough.
  typedef typename std::conditional<MOE || W4 || FAR, size_t, uint32_t>::type
      Off;
  const char* const x_at = (const char*)a.x + (MOE ? 0 : (size_t)bm * rowb);
  const char* const w_at = (const char*)a.w + (w0 + bn) * rowb;
  Off pa[AI];
  [[maybe_unused]] Off pb[BI];
#pragma unroll
  for (int i = 0; i < AI; i++) {
    const int r = min(bm + (wave * AI + i) * 8 + g_r, rows - 1);
    pa[i] = MOE ? (Off)x_row(r) * (Off)rowb : (Off)(r - bm) * (Off)rowb;
  }
  auto w_out = [&](int r) {                  // output of row r of the tile
    return min(bn + (GLU ? (r >> 5) * 16 + (r & 15) : r), a.N - 1);
  };
  if constexpr (!W4)
#pragma unroll
    for (int i = 0; i < BI; i++)
      pb[i] = (Off)(w_out((wave * BI + i) * 8 + g_r) - bn) * (Off)rowb;
  // MXFP4: a thread's piece of a slab, 32 or 16 values of a row
  constexpr int WB = W4 ? BN * 32 / (64 * NW) : 16, WT = 32 / WB;
  static_assert(WB == 16 || WB == 8);
  const int w_r = tid / WT, w_p = tid % WT;
  [[maybe_unused]] const uint8_t *p4 = nullptr, *pe = nullptr;
  if constexpr (W4) {
    const size_t row = (GLU && ((w_r >> 4) & 1) ? a.N : 0) + (size_t)w_out(w_r);
    p4 = (const uint8_t*)a.w + row * (a.K / 2) + w_p * WB;
    pe = a.we + row * (a.K / 32) + w_p * WB / 16;
  }
  [[maybe_unused]] uint32_t raw[NS][WB / 4], rexp[NS];
  auto ask = [&](int b, int s) {             // the piece of slab s
    s = min(s, s_hi - 1);
    if constexpr (WB == 16) *(u4v_*)raw[b] = *(const u4v_*)(p4 + s * 32);
    else *(uint2*)raw[b] = *(const uint2*)(p4 + s * 32);
    rexp[b] = pe[s * 2];
  };
  auto widen = [&](int b, char* B) {         // and into LDS
    const float sc = __uint_as_float(rexp[b] << 23);
#pragma unroll
    for (int d = 0; d < WB / 4; d++) {
      union { gp_b2 p[4]; u4v_ u; } o;
      o.p[0] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(raw[b][d], sc, 0);
      o.p[1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(raw[b][d], sc, 1);
      o.p[2] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(raw[b][d], sc, 2);
      o.p[3] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(raw[b][d], sc, 3);
      const int slot = (w_p * (WB / 4) + d) ^ ((w_r >> 1) & 7);
      *(u4v_*)(B + w_r * 128 + slot * 16) = o.u;
    }
  };
  auto put = [&](int b, char* B, int s) {
    widen(b, B);
    ask(b, s + NS);
    asm volatile("" ::: "memory");
  };
  // row r of a tile keeps slot q at q ^ ((r >> 1) & 7)
  const int src0 = (g_s ^ (g_r >> 1)) * 16, src1 = src0 ^ 64;
  auto stage = [&](char* A, char* B, int s) {
    int o0 = src0, o1 = src1;
    if (F8 && half && s == slabs - 1) o0 &= 63, o1 &= 63;   // stay in the row
    const char* const xs = x_at + (size_t)s * 128;
#pragma unroll
    for (int i = 0; i < AI; i++)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) uint32_t*)(
              xs + (Off)(pa[i] + (((wave * AI + i) & 1) ? o1 : o0))),
          (__attribute__((address_space(3))) uint32_t*)(
              A + (wave * AI + i) * 1024), 16, 0, 0);
    if constexpr (W4) {
      asm volatile("" ::: "memory");       // the waits count loads in order
      return;
    }
#pragma unroll
    for (int i = 0; i < BI; i++) {
      // 16 rows of the gate, 16 of what it gates
      const char* const ws = w_at + (size_t)s * 128 +
          (GLU && (((wave * BI + i) >> 1) & 1) ? (size_t)a.N * rowb : 0);
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) uint32_t*)(
              ws + (Off)(pb[i] + (((wave * BI + i) & 1) ? o1 : o0))),
          (__attribute__((address_space(3))) uint32_t*)(
              B + (wave * BI + i) * 1024), 16, 0, NT ? 2 : 0);
    }
  };

  f4v acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; i++)
#pragma unroll
    for (int j = 0; j < FN; j++) acc[i][j] = {0.f, 0.f, 0.f, 0.f};

  const int fr = lane & 15, fk = lane >> 4;
  const int x0 = (fk ^ (fr >> 1)) * 16, x1 = x0 ^ 64;
  const int la = (wm * FM * 16 + fr) * 128, lb = (wn * FN * 16 + fr) * 128;

  // A slab ends with a meeting that hands over the next one: its DMA is
  // over, that of the NS - 2 behind it stays in flight.  The loop is free of
  // conditions while there are slabs to ask for; the last few wait for all.
  int s = s_lo;
  if (s_lo < s_hi) {
    if constexpr (W4)
#pragma unroll
      for (int u = 0; u < NS; u++) ask(u, s_lo + u);
#pragma unroll
    for (int u = 0; u < NS; u++) {
      if (s_lo + u < s_hi) stage(A[u], B[u], s_lo + u);
      if constexpr (W4) put(u, B[u], s_lo + u);
    }
    // all but the first may still be in flight
    if (s_lo + NS <= s_hi) gp_meet<PS * (NS - 1)>();
    else gp_meet<0>();
    if constexpr (F8) {
      auto slab = [&](char* A, char* B, int s, bool steady) {
        const char *ca = A + la, *cb = B + lb;
        if (steady || !(half && s == slabs - 1)) {
          union { u4v_ q[2]; gp_i8 v; } wb[FN];
#pragma unroll
          for (int j = 0; j < FN; j++) {
            wb[j].q[0] = *(const u4v_*)(cb + j * 2048 + x0);
            wb[j].q[1] = *(const u4v_*)(cb + j * 2048 + x1);
          }
          // no block scales: the row scales come at the end
#pragma unroll
          for (int i = 0; i < FM; i++) {
            union { u4v_ q[2]; gp_i8 v; } xa;
            xa.q[0] = *(const u4v_*)(ca + i * 2048 + x0);
            xa.q[1] = *(const u4v_*)(ca + i * 2048 + x1);
#pragma unroll
            for (int j = 0; j < FN; j++)
              acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                  wb[j].v, xa.v, acc[i][j], 0, 0, 0, 0, 0, 0);
          }
        } else {
#pragma unroll
          for (int i = 0; i < FM; i++) {
            union { u4v_ q; long l[2]; } xa, wb;
            xa.q = *(const u4v_*)(ca + i * 2048 + x0);
#pragma unroll
            for (int j = 0; j < FN; j++) {
              wb.q = *(const u4v_*)(cb + j * 2048 + x0);
#pragma unroll
              for (int h = 0; h < 2; h++)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
                    wb.l[h], xa.l[h], acc[i][j], 0, 0, 0);
            }
          }
        }
        if (steady) {
          gp_meet<PS * (NS - 2)>();
          stage(A, B, s + NS);
        } else if (s + 1 < s_hi) {
          gp_meet<0>();
          if (s + NS < s_hi) stage(A, B, s + NS);
        }
      };
      for (; s + 2 * NS <= s_hi; s += NS) {
#pragma unroll
        for (int u = 0; u < NS; u++) slab(A[u], B[u], s + u, true);
      }
      for (; s < s_hi; s += NS) {
#pragma unroll
        for (int u = 0; u < NS; u++)
          if (s + u < s_hi) slab(A[u], B[u], s + u, false);
      }
    } else {
      // Half a slab of fragments ahead: the hand-over stands between two
      // halves' products, when the second half is in registers already.
      union Frag { u4v_ q; gp_s8 v; };
      Frag xa[2][FM], wb[2][FN];
      auto fetch = [&](int h, const char* A, const char* B) {
        const char *ca = A + la + (h ? x1 : x0), *cb = B + lb + (h ? x1 : x0);
#pragma unroll
        for (int j = 0; j < FN; j++)
          wb[h][j].q = *(const u4v_*)(cb + j * 2048);
#pragma unroll
        for (int i = 0; i < FM; i++)
          xa[h][i].q = *(const u4v_*)(ca + i * 2048);
        __builtin_amdgcn_sched_barrier(0);
      };
      auto mma = [&](int h) {
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
          for (int j = 0; j < FN; j++)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                wb[h][j].v, xa[h][i].v, acc[i][j], 0, 0, 0);
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
      };
      auto slab = [&](char* A, char* B, const char* An, const char* Bn,
                      int s, int u, bool steady) {
        fetch(1, A, B);
        mma(0);
        if (steady) {
          gp_meet<PS * (NS - 2)>();
          stage(A, B, s + NS);
          fetch(0, An, Bn);
        } else if (s + 1 < s_hi) {
          gp_meet<0>();
          if (s + NS < s_hi) stage(A, B, s + NS);
          fetch(0, An, Bn);
        }
        if constexpr (W4)
          if (steady || s + NS < s_hi) put(u, B, s + NS);
        mma(1);
      };
      fetch(0, A[0], B[0]);
      for (; s + 2 * NS <= s_hi; s += NS) {
#pragma unroll
        for (int u = 0; u < NS; u++)
          slab(A[u], B[u], A[(u + 1) % NS], B[(u + 1) % NS], s + u, u,
               true);
      }
      for (; s < s_hi; s += NS) {
#pragma unroll
        for (int u = 0; u < NS; u++)
          if (s + u < s_hi)
            slab(A[u], B[u], A[(u + 1) % NS], B[(u + 1) % NS], s + u, u,
                 false);
      }
    }
  }

  gp_finish<F8, BM, BN, NW, FM, FN, GLU, MOE, true>(
      a, acc, tile, blockIdx.y, SK, bm, bn, rows, first, perm, w0, &last_flag,
      [&](int i) { return (wm * FM + i) * 16; },
      [&](int j) { return (wn * FN + j) * 16; }, x_row);
}

// Tiles 256 wide, by two groups of four waves that take turns: while one has
// the matrix cores, the other brings its next operands from LDS and asks for
// slabs to come.
//
// A slab comes in pieces of 128 rows of 128 bytes: two of W (B0, B1) and HA of
// X (A0, A1), read and asked for in the order B0, A0, B1, A1.  Pieces lie in a
// ring of nine.  A turn is 64 rows by 32 outputs of a wave's tile, 16
// products: it brings what the next products need, asks for pieces where both
// groups have theirs in registers, waits for the pieces that the turn after it
// reads, with all those behind them still in flight, and meets the others
// twice, ahead of its products and behind them.  The groups are one meeting
// apart.
//
// A block takes tile after tile, and the pieces that are asked for are those
// of the next tile where a tile ends: none waits for its first slabs but the
// first.  Behind the last one loads go on, to one line, so that the waits
// count alike.
//
// Of routed experts (MOE) the blocks share the row tiles that have rows: with
// the empty ones left in place some had a tile more than others (1100 rows, 8
// experts, 2048->2x4096: 130 us, so 107).
#define GW_RING 9
// 64 lanes of 16 bytes to lds and behind it.  By asm: ahead of a builtin's load
// the compiler would wait for those in flight.  m0 is named, so that one that it
// sets for a builtin is set again behind this; it warns that it keeps m0 itself.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
template <bool NT = false>
DEVINL void gw_load(const char* base, uint32_t off, uint32_t lds) {
  if constexpr (NT)
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\t"
                 "global_load_lds_dwordx4 %1, %0 nt"
                 :: "s"(base), "v"(off), "s"(lds) : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\t"
                 "global_load_lds_dwordx4 %1, %0"
                 :: "s"(base), "v"(off), "s"(lds) : "memory", "m0");
}
#pragma clang diagnostic pop
DEVINL void gw_meet() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
// LDS reads are over, and all loads but the last N
template <int N> DEVINL void gw_wait() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | (N >> 4 << 14) | 7 << 4);
  asm volatile("" ::: "memory");
}

template <bool F8, int HA, bool GLU, bool NT, bool MOE = false>
__global__ void __launch_bounds__(512) k_gemm_wide(GpArgs a, int SK) {
  constexpr int BM = 128 * HA, BN = 256, FM = 4 * HA, FN = 4;
  __shared__ __attribute__((aligned(16))) char ring[GW_RING * 16384];
  __shared__ int last_flag;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  if constexpr (MOE) {
    // row tiles that have rows: the last E of those counted on may have none
    const int t = a.tm - 1 - lane;
    a.tm -= __popcll(__ballot(t >= 0 && a.tile_n[max(t, 0)] == 0));
    a.band = a.tm;
  }
  // Work of an XCD (block id modulo 8): neighbouring tiles, rows fastest, in
  // each part of K.  A block takes every step-th item of it.
  const int tiles = a.tm * a.tn, chunk = (tiles + 7) / 8, items = chunk * SK;
  const int step = gridDim.x >> 3, t0 = (blockIdx.x & 7) * chunk;
  auto there = [&](int k) {                  // the next item from k on
    while (k < items && t0 + k % chunk >= tiles) k += step;
    return k;
  };
  int item = there(blockIdx.x >> 3);
  if (item >= items) return;

  const size_t rowb = (size_t)a.K * (F8 ? 1 : 2);       // bytes of a row
  const int slabs = (int)((rowb + 127) / 128), per = (slabs + SK - 1) / SK;

  // ---- what is asked for: a slab of an item, then the next one ----
  const int g_r = lane >> 3, g_s = lane & 7;
  // row r of a piece keeps slot q at q ^ ((r >> 1) & 7)
  const uint32_t src = (g_s ^ (g_r >> 1)) * 16;
  const char *xp, *wp;
  uint32_t pa[HA][2], pb[2][2];
  int ahead = item, left, adv = 128;
  auto aim = [&] {
    left = 1 << 30;
    if (ahead >= items) {                    // no more: one line of each
      adv = 0;
      xp = (const char*)a.x;
      wp = (const char*)a.w;
#pragma unroll
      for (int t = 0; t < 2; t++) {
#pragma unroll
        for (int h = 0; h < HA; h++) pa[h][t] = 0;
#pragma unroll
        for (int h = 0; h < 2; h++) pb[h][t] = 0;
      }
      return;
    }
    const int tile = t0 + ahead % chunk, lo = ahead / chunk * per;
    left = min(per, slabs - lo);
    const GpAt at = gp_at(a, tile);
    const int bm = MOE ? 0 : at.row * BM, bn = at.col * (GLU ? BN / 2 : BN);
    const int rows = MOE ? a.tile_n[at.row] : a.M - bm;
    const int first = MOE ? a.tile_row0[at.row] : 0;
    xp = (const char*)a.x + (size_t)bm * rowb + (size_t)lo * 128;
    // 16 rows of the gate, 16 of what it gates
    wp = (const char*)a.w + (size_t)bn * rowb + (size_t)lo * 128 +
         (GLU && (wave & 1) ? (size_t)a.N * rowb : 0);
    if (MOE)
      wp += (size_t)__builtin_amdgcn_readfirstlane(a.tile_e[at.row]) *
            (GLU ? 2 : 1) * a.N * rowb;
#pragma unroll
    for (int t = 0; t < 2; t++) {
      const int r = (wave * 2 + t) * 8 + g_r;
      const uint32_t o = t ? src ^ 64 : src;
#pragma unroll
      for (int h = 0; h < HA; h++) {
        int x = min(h * 128 + r, rows - 1);
        if (MOE) x = a.gather ? a.perm[first + x] / a.top : first + x;
        pa[h][t] = (uint32_t)x * (uint32_t)rowb + o;
      }
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int c = h * 128 + r;
        pb[h][t] = (uint32_t)min(GLU ? (c >> 5) * 16 + (c & 15) : c,
                                 a.N - 1 - bn) * (uint32_t)rowb + o;
      }
    }
  };
  const uint32_t ring0 = __builtin_amdgcn_readfirstlane(
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)ring +
      wave * 2048);
  uint32_t put = 0, get = 0;
  auto turned = [](uint32_t at) {
    return at == (GW_RING - 1) * 16384 ? 0 : at + 16384;
  };
  auto ask = [&](auto nt, const char* base, const uint32_t (&off)[2]) {
#pragma unroll
    for (int t = 0; t < 2; t++)
      gw_load<decltype(nt)::value>(base, off[t], ring0 + put + t * 1024);
    put = turned(put);
  };
  // piece 0: B0, 1: A0, 2: B1, 3: A1
  auto ask_piece = [&](int u) {
    if (u & 1) ask(std::false_type(), xp, pa[HA == 2 ? u >> 1 : 0]);
    else ask(std::integral_constant<bool, NT>(), wp, pb[u >> 1]);
    if (u == HA + 1) {                       // the slab's last
      xp += adv;
      wp += adv;
      if (--left == 0) {
        ahead = there(ahead + step);
        aim();
      }
    }
  };

  // ---- products ----
  f4v acc[FM][FN];
  const int fr = lane & 15, fk = lane >> 4;
  const int x0 = (fk ^ (fr >> 1)) * 16, x1 = x0 ^ 64;
  const int la = (wm * 64 + fr) * 128, lb = (wn * 32 + fr) * 128;
  union Frag { u4v_ q[2]; gp_i8 v; gp_s8 h[2]; };
  Frag xa[4], wb[2][2];
  auto get_a = [&] {
    const char* const c = ring + get + la;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      xa[i].q[0] = *(const u4v_*)(c + i * 2048 + x0);
      xa[i].q[1] = *(const u4v_*)(c + i * 2048 + x1);
    }
    get = turned(get);
  };
  auto get_b = [&](int h) {
    const char* const c = ring + get + lb;
#pragma unroll
    for (int j = 0; j < 2; j++) {
      wb[h][j].q[0] = *(const u4v_*)(c + j * 2048 + x0);
      wb[h][j].q[1] = *(const u4v_*)(c + j * 2048 + x1);
    }
    get = turned(get);
  };
  auto mma = [&](int ha, int hb) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int k = 0; k < (F8 ? 1 : 2); k++)
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
          f4v& c = acc[ha * 4 + i][hb * 2 + j];
          // e4m3: without block scales, which would take an instruction more
          // each (2048x16384x8192 270 us, so 239); row scales at the end
          if constexpr (F8)
            c = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                wb[hb][j].v, xa[i].v, c, 0, 0, 0, 0, 0, 0);
          else
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                wb[hb][j].h[k], xa[i].h[k], c, 0, 0, 0);
        }
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
  };

  aim();
  // the slabs that fit in the ring, as if turns before had asked for them
  constexpr int P = HA == 2 ? GW_RING : GW_RING - 1;
#pragma unroll
  for (int n = 0; n < P; n++) ask_piece(n % (HA + 2));
  gw_wait<2 * (P - 2)>();
  gw_meet();
  get_b(0);
  gw_wait<2 * (P - 2)>();
  gw_meet();
  for (;;) {
    const int tile = t0 + item % chunk, part = item / chunk;
    const GpAt at = gp_at(a, tile);
    const int bm = MOE ? 0 : at.row * BM, bn = at.col * (GLU ? BN / 2 : BN);
    const int rows = MOE ? a.tile_n[at.row] : a.M;
    const int first = MOE ? a.tile_row0[at.row] : 0;
    const int* const perm = MOE ? a.perm + first : nullptr;
    const size_t w0 =
        MOE ? (size_t)a.tile_e[at.row] * (GLU ? 2 : 1) * a.N : 0;
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
      for (int j = 0; j < FN; j++) acc[i][j] = {0.f, 0.f, 0.f, 0.f};
    if (wm) gw_meet();
    for (int n = min(per, slabs - part * per); n > 0; n--) {
      if constexpr (HA == 2) {
        constexpr int N = 2 * (GW_RING - 2);
        get_a();
        ask_piece(1);
        gw_wait<N>();
        gw_meet();
        mma(0, 0);
        gw_meet();
        get_b(1);
        ask_piece(2);
        gw_wait<N>();
        gw_meet();
        mma(0, 1);
        gw_meet();
        get_a();
        ask_piece(3);
        gw_wait<N>();
        gw_meet();
        mma(1, 0);
        gw_meet();
        get_b(0);                            // of the next slab
        ask_piece(0);
        gw_wait<N>();
        gw_meet();
        mma(1, 1);
        gw_meet();
      } else {
        constexpr int N = 2 * (GW_RING - 3);
        get_a();
        ask_piece(2);
        ask_piece(0);
        gw_wait<N>();
        gw_meet();
        mma(0, 0);
        gw_meet();
        get_b(1);
        get_b(0);                            // of the next slab
        ask_piece(1);
        gw_wait<N>();
        gw_meet();
        mma(0, 1);
        gw_meet();
      }
    }
    if (!wm) gw_meet();
    item = there(item + step);
    gp_finish<F8, BM, BN, 8, FM, FN, GLU, MOE, HA == 1 && !MOE>(
        a, acc, tile, part, SK, bm, bn, rows, first, perm, w0, &last_flag,
        [&](int i) { return (i >> 2) * 128 + wm * 64 + (i & 3) * 16; },
        [&](int j) { return (j >> 1) * 128 + wn * 32 + (j & 1) * 16; },
        [&](int r) {
          return !MOE ? r : a.gather ? perm[r] / a.top : first + r;
        });
    if (item >= items) break;
  }
  gw_wait<0>();
}

enum { GP_BF16, GP_E4M3, GP_MXFP4 };           // of W
#define GP_FAR (1 << 23)       // K up to which 32 bits reach all rows of a tile

// Tiles, in bands of rows that are about as high as what the CUs of an XCD work
// on is wide: its L2 then misses least (2048x4096x14336 in 128x256 207 -> 202
// us, e4m3 125 -> 119; 1999x2048x8192 in 128x128 76 -> 72; no difference from
// 4 to 8 rows of tiles).  256x256 is best in one band of 2048 rows.
static void gp_tiling(GpArgs& a, int bm, int wide) {
  a.tm = (a.M + bm - 1) / bm;
  a.tn = (a.N + wide - 1) / wide;
  const int most = bm == 256 ? 8 : 1024 / bm, bands = (a.tm + most - 1) / most;
  a.band = (a.tm + bands - 1) / bands;
}

// One row of tiles reads W once: past the caches, where there is much of it
// (us, W of 16 to 155 MB, in them -> past: 64 rows of 28672x4096 54.0 -> 47.1,
// of 16384x2048 17.4 -> 16.9, 128 rows of 28672x4096 by 128x128 58.9 -> 51.5;
// 6144x2304 of 28 MB 17.8 -> 18.1, and e4m3 3072x2048 of 6 MB, which the last
// level may still hold, 10.9 -> 13.0).
template <int T> static bool gp_once(const GpArgs& a) {
  return a.tm == 1 && (a.act >= 0 ? 2.f : 1.f) * a.N * a.K *
                              (T == GP_E4M3 ? 1 : 2) >= 32 << 20;
}

template <int T, int BM, int BN, int WM, int WN, int NS, bool FAR = false>
static hipError_t gp_go(GpArgs a, int sk, hipStream_t s) {
  constexpr bool F8 = T == GP_E4M3, W4 = T == GP_MXFP4;
  const bool glu = a.act >= 0;
  const int wide = glu ? BN / 2 : BN;
  gp_tiling(a, BM, wide);
  const dim3 grid((a.tm * a.tn + 7) / 8 * 8, sk), nt(64 * WM * WN);
#define GP_GO(GLU, NT)                                                       \
  hipLaunchKernelGGL((k_gemm_prompt<F8, BM, BN, WM, WN, NS, GLU, false, W4,  \
                                    FAR, NT>), grid, nt, 0, s, a)
  if constexpr (!W4 && !FAR) {
    if (gp_once<T>(a)) {
      if (glu) GP_GO(true, true);
      else GP_GO(false, true);
      return hipGetLastError();
    }
  }
  if (glu) GP_GO(true, false);
  else GP_GO(false, false);
#undef GP_GO
  return hipGetLastError();
}

// of parts of K as many as have slabs
template <int T> static int gw_parts(int K, int sk) {
  const int slabs = (int)((long)K * (T == GP_E4M3 ? 1 : 2) / 128);
  const int per = (slabs + sk - 1) / sk;
  return (slabs + per - 1) / per;
}

// by k_gemm_wide; e4m3 rows of whole slabs
template <int T, int HA>
static hipError_t gp_go_wide(GpArgs a, int sk, hipStream_t s) {
  constexpr bool F8 = T == GP_E4M3;
  const bool glu = a.act >= 0;
  gp_tiling(a, 128 * HA, glu ? 128 : 256);
  sk = gw_parts<T>(a.K, sk);
  const int share = (a.tm * a.tn + 7) / 8 * sk;          // of an XCD
  const dim3 grid(8 * (share < 32 ? share : 32));        // a block a CU
#define GW_GO(GLU, NT)                                                       \
  hipLaunchKernelGGL((k_gemm_wide<F8, HA, GLU, NT>), grid, dim3(512), 0, s,  \
                     a, sk)
  if constexpr (HA == 1) {
    if (gp_once<T>(a)) {
      if (glu) GW_GO(true, true);
      else GW_GO(false, true);
      return hipGetLastError();
    }
  }
  if (glu) GW_GO(true, false);
  else GW_GO(false, false);
#undef GW_GO
  return hipGetLastError();
}

// Large tiles ask L2 for the fewest bytes a product: 128x128 by four waves
// wants 64 bytes a clock, all that a CU gets.  They win where there are rounds
// of them; where tiles are fewer than the chip has CUs a smaller one that is
// deep in flight does.  256x256 is never split (1999x2048x8192 in four parts
// 85 us, 128x128 72: its parts cost most) and not for MXFP4 (W on its way to
// LDS spills: 467 TFLOP/s at 2048x37888x3584, 128x128 944).  The second 128x128
// has eight waves and four buffers.
struct GpTile { int bm, bn, occ; };              // occ: blocks that fit on a CU
static const GpTile gp_tiles[8] = {
    {256, 256, 1}, {128, 256, 1}, {128, 128, 2}, {128, 128, 1},
    {64, 128, 2},  {128, 64, 2},  {64, 64, 2},   {32, 64, 2}};

// What a slab of each tile costs a CU with one block and with as many as fit,
// a round besides (first slabs, epilogue); the second block on some CUs, the
// first on few; K in parts, and each of their floats; a round where outputs are
// no multiple of four and leave one by one.  0: not for that type (e4m3 in
// 128x128 by four waves: no product of the fits chose it).
// The numbers are about us, but fitted to what they choose: the times of every
// likely tile and split (1 to 8 parts), W from memory, of 26250 products of 17
// to 2048 rows, 29 and 12 (with a gate) shapes of models and others of 64 to
// 24000 outputs and K of 128 to 19200, so that few take longer than by the
// numbers and kernels before k_gemm_wide and tiles of eight waves.  Above the
// best of the times, and how many took 4% longer than by those kernels, by
// numbers fitted to K from 2048 on -> now, half of the products, which were not
// fitted (outputs a multiple of four):
//   bf16 2.4% -> 1.6%, 53 -> 27 of 1959; with a gate 2.0% -> 1.0%, 17 -> 2 of 1026
//   e4m3 2.4%, 21 of 1240, as it was: beside e4m3 rounding parts of K elsewhere
//       are other values; with a gate 1.4% -> 1.0%, 21 -> 7 of 678
//   e4m3 rows of half a slab, which k_gemm_wide does not take, by numbers of
//       their own 3.2% -> 1.7%, 57 -> 30 of 1647; with a gate 2.0% -> 0.9%,
//       61 -> 14 of 1067
// (us: 1883x1152x896 17.2 -> 13.8; 789x1536x576 with a gate 12.6 -> 9.2; e4m3
// 1792x4786x704 63.5 -> 41.9.)  MXFP4 is fitted to 64, 130, 600 and 2048 rows of
// five shapes (2.2%).
struct GpCost {
  float one[8], full[8], round[8], second, first, split, part, off;
};
static const GpCost gp_cost[7] = {
    {// bf16
     {1.4f, 0.864f, 0.807f, 0.608f, 2.27f, 0.463f, 0.305f, 0.26f},
     {1.4f, 0.864f, 1.66f, 0.608f, 4.51f, 0.729f, 0.536f, 0.518f},
     {13.9f, 6.96f, 4.85f, 4.27f, 2.55f, 3.19f, 2.01f, 1.77f},
     0.904f, 0.846f, 1.43f, 4.03e-6f, 2.92f},
    {// bf16 with a gate
     {1.17f, 0.775f, 1.85f, 0.523f, 0.556f, 0.507f, 0.317f, 0.262f},
     {1.17f, 0.775f, 4.01f, 0.523f, 0.914f, 0.66f, 0.556f, 0.576f},
     {20.f, 11.9f, 4.6f, 8.12f, 4.74f, 5.17f, 3.97f, 3.58f},
     1.f, 0.854f, 2.25f, 3.92e-6f, 1.f},
    {// e4m3
     {1.76f, 0.954f, 0.f, 0.752f, 0.633f, 0.892f, 0.405f, 0.286f},
     {1.76f, 0.954f, 0.f, 0.752f, 0.817f, 0.892f, 0.556f, 0.449f},
     {6.f, 3.81f, 0.f, 2.16f, 2.07f, 2.84f, 1.14f, 1.21f},
     0.626f, 0.952f, 0.273f, 5.43e-6f, 1.f},
    {// e4m3 with a gate
     {2.43f, 1.66f, 0.f, 1.04f, 0.897f, 0.775f, 0.439f, 0.299f},
     {2.43f, 1.66f, 0.f, 1.04f, 1.36f, 1.15f, 0.717f, 0.505f},
     {6.56f, 3.27f, 0.f, 2.88f, 0.546f, 0.677f, 0.926f, 1.05f},
     0.656f, 1.f, 1.06f, 3.35e-6f, 1.f},
    {// e4m3, half a slab at the end of a row
     {0.f, 1.84f, 0.f, 1.03f, 0.903f, 0.842f, 0.589f, 0.374f},
     {0.f, 1.84f, 0.f, 1.03f, 1.29f, 1.22f, 0.836f, 0.618f},
     {0.f, 3.41f, 0.f, 6.f, 2.52f, 1.29f, 0.647f, 0.626f},
     0.824f, 0.852f, 1.27f, 4.33e-6f, 1.98f},
    {// the same with a gate
     {0.f, 1.18f, 0.f, 0.739f, 0.648f, 0.555f, 0.38f, 0.217f},
     {0.f, 1.18f, 0.f, 0.739f, 0.891f, 0.8f, 0.511f, 0.387f},
     {0.f, 3.87f, 0.f, 2.18f, 1.64f, 1.16f, 1.11f, 1.34f},
     0.99f, 0.856f, 0.944f, 2.79e-6f, 1.f},
    {// MXFP4
     {0.f, 0.96f, 0.654f, 0.562f, 0.44f, 0.f, 0.292f, 0.f},
     {0.f, 0.96f, 1.08f, 0.562f, 0.773f, 0.f, 0.538f, 0.f},
     {0.f, 4.f, 3.2f, 3.4f, 1.8f, 0.f, 1.4f, 0.f},
     0.42f, 0.96f, 2.1f, 5e-6f, 1.f}};

// the tile and split of a product, and what it takes by the numbers
struct GpPick { int tile, sk; float time; };

template <int T>
static GpPick gp_pick(const GpArgs& a, long part_floats, int ncnt) {
  const int width = a.act >= 0 ? 2 * a.N : a.N;
  const int slabs = (int)(((long)a.K * (T == GP_E4M3 ? 1 : 2) + 127) / 128);
  const bool half = T == GP_E4M3 && a.K % 128;
  const GpCost& k = gp_cost[T == GP_MXFP4 ? 6 : (half ? 4 : T * 2) + (a.act >= 0)];
  const bool far = T != GP_MXFP4 && a.K > GP_FAR;        // 64x64 alone
  int best = -1, best_sk = 1;
  float best_t = 0.f;
  for (int c = 0; c < 8; c++) {
    const GpTile& g = gp_tiles[c];
    const float one = k.one[c], full = k.full[c];
    if (one == 0.f || (far && c != 6)) continue;
    const float round = k.round[c] * (a.N % 4 ? k.off : 1.f);
    const long tiles = (long)((a.M + g.bm - 1) / g.bm) *
                       ((width + g.bn - 1) / g.bn);
    for (int sk = 1; sk <= 8; sk++) {
      const double parts = (double)tiles * sk * g.bm * g.bn;
      if (sk > 1 && (c == 0 || tiles > ncnt || tiles * sk > 700 ||
                     parts > part_floats || slabs / sk < 4))
        break;
      // Full rounds and a rest.  A few CUs with two blocks set the time for
      // all: blocks are counted on the XCD that has most, 32 CUs of it (three
      // parts of 84 tiles are 252 blocks, but 33 on four of the XCDs:
      // 130x3584x18944 MXFP4 80 us; in parts of four 68).
      const float x = (float)((tiles + 7) / 8 * sk) / 32.f;   // of a CU
      const int rounds = (int)(x / g.occ);
      const float rest = x - rounds * g.occ;
      float t = rounds * full;
      if (rest > 1.f)
        t += one + (full - one) * (k.second + (1.f - k.second) * (rest - 1.f));
      else if (rest > 0.f)
        t += one * (k.first + (1.f - k.first) * rest);
      t = t * ((slabs + sk - 1) / sk) + (rounds + (rest > 0.f)) * round;
      // parts written and read, and a trip for each
      if (sk > 1) t += k.split + (float)(parts * k.part);
      if (best < 0 || t < best_t) {
        best = c;
        best_sk = sk;
        best_t = t;
      }
    }
  }
  return {best, best_sk, best_t};
}

template <int T>
static hipError_t gp_run(const GpArgs& a, long part_floats, int ncnt,
                         hipStream_t s) {
  const bool far = T != GP_MXFP4 && a.K > GP_FAR;        // 64x64 alone
  const bool odd = T == GP_E4M3 && a.K % 128;            // half a slab
  const GpPick pick = gp_pick<T>(a, part_floats, ncnt);
  const int best_sk = pick.sk;
  // eight waves, four beside MXFP4, whose pieces of W a thread would be halves
  constexpr int WM = T == GP_MXFP4 ? 2 : 4;
  switch (pick.tile) {
    case 0:
      if constexpr (T != GP_MXFP4) return gp_go_wide<T, 2>(a, best_sk, s);
      break;
    case 1:
      if constexpr (T != GP_MXFP4)
        if (!odd) return gp_go_wide<T, 1>(a, best_sk, s);
      if constexpr (T != GP_BF16)
        return gp_go<T, 128, 256, 2, 4, 3>(a, best_sk, s);
      break;
    case 2:
      if constexpr (T != GP_E4M3)
        return gp_go<T, 128, 128, 2, 2, 2>(a, best_sk, s);
      break;
    case 3: return gp_go<T, 128, 128, 2, 4, 4>(a, best_sk, s);
    case 4: return gp_go<T, 64, 128, WM, 2, 3>(a, best_sk, s);
    case 5:
      if constexpr (T != GP_MXFP4)
        return gp_go<T, 128, 64, WM, 2, 3>(a, best_sk, s);
      break;
    case 6:
      if constexpr (T != GP_MXFP4)
        if (far) return gp_go<T, 64, 64, WM, 2, 4, true>(a, best_sk, s);
      return gp_go<T, 64, 64, WM, 2, 4>(a, best_sk, s);
    case 7:
      if constexpr (T != GP_MXFP4)
        return gp_go<T, 32, 64, 2, 2, 6>(a, best_sk, s);
      break;
  }
  return hipErrorInvalidValue;
}

// sx, sw: row scales of e4m3 x and w.  act < 0: no gate.  part and cnt (zero,
// left zero) let K be split.
extern "C" hipError_t launch_gemm_prompt(
    const void* x, const void* w, const void* sx, const void* sw,
    const void* res, const void* bias, void* y, void* part, void* cnt,
    long part_floats, int ncnt, int M, int N, int K, int act,
    hipStream_t stream) {
  if (M < 1 || N < 1 || K < 64 || K % 64 || (!sx != !sw))
    return hipErrorInvalidValue;
  GpArgs a = {x, w, (const float*)sx, (const float*)sw, nullptr,
              (const u16*)res, (const u16*)bias, (u16*)y, (float*)part,
              (int*)cnt, M, N, K, act, 0, 0, 0, nullptr, nullptr, nullptr, nullptr, 1, 0};
  if (!part || !cnt) part_floats = 0;
  if (mid_takes(sx, M, N, K, act >= 0))
    return launch_mid_gemm(x, w, sx, sw, res, bias, y, part, cnt, part_floats,
                           ncnt, M, N, K, K, res ? N : 0, N, act, 0, 0.f,
                           stream);
  return sx ? gp_run<GP_E4M3>(a, part_floats, ncnt, stream)
            : gp_run<GP_BF16>(a, part_floats, ncnt, stream);
}

// The same of bf16 rows and MXFP4 weights: w [N, K/2], we [N, K/32]
extern "C" hipError_t launch_gemm_fp4w(
    const void* x, const void* w, const void* we, const void* res,
    const void* bias, void* y, void* part, void* cnt, long part_floats,
    int ncnt, int M, int N, int K, int act, hipStream_t stream) {
  if (M < 1 || N < 1 || K < 64 || K % 64 || !we)
    return hipErrorInvalidValue;
  GpArgs a = {x, w, nullptr, nullptr, (const uint8_t*)we, (const u16*)res,
              (const u16*)bias, (u16*)y, (float*)part, (int*)cnt, M, N, K,
              act, 0, 0, 0, nullptr, nullptr, nullptr, nullptr, 1, 0};
  return gp_run<GP_MXFP4>(a, part && cnt ? part_floats : 0, ncnt, stream);
}

// About what a product of bf16 rows takes, us, W bf16 or MXFP4
extern "C" float gemm_prompt_time(int fp4, int M, int N, int K, int act,
                                  long part_floats, int ncnt) {
  GpArgs a = {};
  a.M = M;
  a.N = N;
  a.K = K;
  a.act = act;
  return fp4 ? gp_pick<GP_MXFP4>(a, part_floats, ncnt).time
             : gp_pick<GP_BF16>(a, part_floats, ncnt).time;
}

// What a product runs by, on the host alone: rows and outputs of a tile, parts of
// K, whether by k_gemm_wide, whether W goes past the caches, waves of a block.
// kind: GP_BF16 ..; all 0: by launch_mid_gemm.
template <int T>
static void gp_plan(GpArgs& a, long part_floats, int ncnt, int* out) {
  const GpPick p = gp_pick<T>(a, part_floats, ncnt);
  const GpTile& g = gp_tiles[p.tile];
  const bool far = T != GP_MXFP4 && a.K > GP_FAR;
  gp_tiling(a, g.bm, a.act >= 0 ? g.bn / 2 : g.bn);
  out[0] = g.bm;
  out[1] = g.bn;
  out[3] = T != GP_MXFP4 && p.tile < 2 && !(T == GP_E4M3 && a.K % 128);
  out[2] = out[3] ? gw_parts<T>(a.K, p.sk) : p.sk;
  out[4] = T != GP_MXFP4 && !far && p.tile > 0 && gp_once<T>(a);
  out[5] = p.tile == 2 || p.tile == 7 || (T == GP_MXFP4 && p.tile > 3) ? 4 : 8;
}

extern "C" int gemm_prompt_plan(int kind, int M, int N, int K, int act,
                                long part_floats, int ncnt, int* out) {
  if (M < 1 || N < 1 || K < 64 || K % 64 || kind < GP_BF16 || kind > GP_MXFP4)
    return 1;
  GpArgs a = {};
  a.M = M;
  a.N = N;
  a.K = K;
  a.act = act;
  for (int i = 0; i < 6; i++) out[i] = 0;
  if (kind == GP_MXFP4) gp_plan<GP_MXFP4>(a, part_floats, ncnt, out);
  else if (mid_takes(kind == GP_E4M3, M, N, K, act >= 0)) return 0;
  else if (kind == GP_E4M3) gp_plan<GP_E4M3>(a, part_floats, ncnt, out);
  else gp_plan<GP_BF16>(a, part_floats, ncnt, out);
  return 0;
}

// ---- routed experts --------------------------------------------------------
// Every expert used to take all rows, E/top times the work, with a launch a
// product and one to add: 16 products and 8 sums a layer for eight experts.
// Here the pairs of a row and a choice are sorted by expert on the device, a
// row tile belongs to one expert, and each product is one launch (a tile more
// than there may be an expert is launched and leaves).  1100 rows, eight
// experts of 2x4096x2048, two a row, and 24 steps: 5.17 -> 4.00 ms.
//
// One block: pairs (token, choice) by expert, and the row tiles of each.
// Pairs of an expert may come in any order: a row's result does not depend on
// its place.
__global__ void __launch_bounds__(1024)
k_expert_sort(const int* __restrict__ idx, int* __restrict__ perm,
              int* __restrict__ tile_e, int* __restrict__ tile_row0,
              int* __restrict__ tile_n, int pairs, int E, int bm,
              int maxtiles) {
  __shared__ int cnt[64], start[65], tile0[65];
  const int tid = threadIdx.x;
  if (tid < E) cnt[tid] = 0;
  __syncthreads();
  for (int p = tid; p < pairs; p += 1024) atomicAdd(&cnt[idx[p]], 1);
  __syncthreads();
  if (tid == 0) {
    int s = 0, t = 0;
    for (int e = 0; e < E; e++) {
      start[e] = s;
      tile0[e] = t;
      s += cnt[e];
      t += (cnt[e] + bm - 1) / bm;
    }
    start[E] = s;
    tile0[E] = t;
  }
  __syncthreads();
  for (int t = tid; t < maxtiles; t += 1024) {
    int e = 0, n = 0, r0 = 0;
    if (t < tile0[E]) {
      while (t >= tile0[e + 1]) e++;
      r0 = start[e] + (t - tile0[e]) * bm;
      n = min(bm, start[e + 1] - r0);
    }
    tile_e[t] = e;
    tile_row0[t] = r0;
    tile_n[t] = n;
  }
  __syncthreads();
  if (tid < E) cnt[tid] = 0;
  __syncthreads();
  for (int p = tid; p < pairs; p += 1024) {
    const int e = idx[p];
    perm[start[e] + atomicAdd(&cnt[e], 1)] = p;
  }
}

// h[t] += w[t, j] y[t, j], 8 elements a thread: one expert after the other, h
// bf16 between them, as when each expert's result was a launch of its own
__global__ void __launch_bounds__(256)
k_expert_sum(const u16* __restrict__ y, const float* __restrict__ w,
             const int* __restrict__ idx, u16* __restrict__ h, int top,
             int H) {
  const int t = blockIdx.y, i = (blockIdx.x * 256 + threadIdx.x) * 8;
  if (i >= H) return;
  const size_t p0 = (size_t)t * top;
  s8v hv = *(const s8v*)(h + (size_t)t * H + i);
  for (int n = 0, last = -1; n < top; n++) {
    int j = -1;                              // the next expert
    for (int q = 0; q < top; q++)
      if (idx[p0 + q] > last && (j < 0 || idx[p0 + q] < idx[p0 + j])) j = q;
    if (j < 0) break;
    last = idx[p0 + j];
    const s8v v = *(const s8v*)(y + (p0 + j) * H + i);
    const float s = w[p0 + j];
#pragma unroll
    for (int k = 0; k < 8; k++)
      ((u16*)&hv)[k] = f2b(b2f(((u16*)&hv)[k]) + s * b2f(((u16*)&v)[k]));
  }
  *(s8v*)(h + (size_t)t * H + i) = hv;
}

// rows of a tile: what an expert gets on average, or more (278 rows each:
// 128; with 64 W is read twice as often)
static int expert_bm(int pairs, int E) {
  const int mean = pairs / E;
  return mean >= 96 ? 128 : mean >= 24 ? 64 : 32;
}

extern "C" hipError_t launch_expert_sort(const void* idx, void* sorted,
                                         int pairs, int E, long room,
                                         hipStream_t stream) {
  const int bm = expert_bm(pairs, E), tiles = pairs / bm + E;
  if (pairs < 1 || E < 1 || E > 64 || room < pairs + 3L * tiles)
    return hipErrorInvalidValue;
  int* p = (int*)sorted;
  hipLaunchKernelGGL(k_expert_sort, dim3(1), dim3(1024), 0, stream,
                     (const int*)idx, p, p + pairs, p + pairs + tiles,
                     p + pairs + 2 * tiles, pairs, E, bm, tiles);
  return hipGetLastError();
}

template <bool F8, int BM, int BN, int WM, int WN, int NS>
static hipError_t gp_experts(GpArgs a, hipStream_t s) {
  const int wide = a.act >= 0 ? BN / 2 : BN;
  a.tn = (a.N + wide - 1) / wide;
  const dim3 grid((a.tm * a.tn + 7) / 8 * 8), nt(64 * WM * WN);
  if (a.act >= 0)
    hipLaunchKernelGGL((k_gemm_prompt<F8, BM, BN, WM, WN, NS, true, true>),
                       grid, nt, 0, s, a);
  else
    hipLaunchKernelGGL((k_gemm_prompt<F8, BM, BN, WM, WN, NS, false, true>),
                       grid, nt, 0, s, a);
  return hipGetLastError();
}

// Whether routed experts go by k_gemm_wide: 128x256 tiles in turns with more than
// a 128x128 tile a CU to do (8 experts, 1100 rows, 2 each, 2048->2x4096 143 us, so
// 107, e4m3 101, 69; 4096->2048 80, 64; 700 rows 4096->2x14336 594, 478; 16 experts
// of 1024 30, 21).  With a tile a CU or less the small ones end sooner: 700 rows
// 4096->2048 46, 60.  Row offsets have 32 bits.
//
// The host does not know what the router chose.  It counts on half a row tile an
// expert for the last of its rows, but on no more than if all had as many: eight
// of 212 rows each have 16 tiles, not 17 (848 rows, 2 each, 4096->2048 47 us by
// small tiles, 64 by wide ones).  Of 17900 products 4% slower than by small tiles
// as they were 461 without that bound, 248 with it.
static bool expert_wide(bool f8, int pairs, int E, int N, int K, int act) {
  const int glu = act >= 0 ? 2 : 1, even = E * ((pairs / E + 127) / 128);
  const float tiles = fminf(pairs / 128.f + E / 2.f, even);
  return expert_bm(pairs, E) == 128 && !(f8 && K % 128) &&
         (size_t)pairs * K * (f8 ? 1 : 2) <= UINT32_MAX &&
         tiles * ((N * glu + 127) / 128) > 256.f;
}

// Rows of a tile and whether by k_gemm_wide, on the host alone
extern "C" int expert_gemm_plan(int f8, int pairs, int E, int N, int K, int act,
                                int* out) {
  if (pairs < 1 || E < 1 || E > 64 || N < 1 || K < 64 || K % 64) return 1;
  out[0] = expert_bm(pairs, E);
  out[1] = expert_wide(f8, pairs, E, N, K, act);
  return 0;
}

// y = x W^T of each pair's expert.  sorted: of launch_expert_sort.  gather: x
// by token, y in the sorted order; else x in that order, y by pair.
extern "C" hipError_t launch_expert_gemm(
    const void* x, const void* w, const void* sx, const void* sw, void* y,
    const void* sorted, int pairs, int E, int top, int gather, int N, int K,
    int act, hipStream_t stream) {
  if (pairs < 1 || E < 1 || E > 64 || top < 1 || pairs % top || N < 1 ||
      K < 64 || K % 64 || (!sx != !sw))
    return hipErrorInvalidValue;
  const int bm = expert_bm(pairs, E), tiles = pairs / bm + E;
  const int* p = (const int*)sorted;
  GpArgs a = {x, w, (const float*)sx, (const float*)sw, nullptr, nullptr,
              nullptr, (u16*)y, nullptr, nullptr, pairs, N, K, act, tiles, 0, tiles,
              p, p + pairs, p + pairs + tiles, p + pairs + 2 * tiles, top,
              gather};
  if (expert_wide(sx, pairs, E, N, K, act)) {
    a.tn = (N * (act >= 0 ? 2 : 1) + 255) / 256;
    const int share = (tiles * a.tn + 7) / 8;
    const dim3 grid(8 * (share < 32 ? share : 32)), nt(512);
#define WIDE(F8, GLU)                                                        \
  hipLaunchKernelGGL((k_gemm_wide<F8, 1, GLU, false, true>), grid, nt, 0,    \
                     stream, a, 1)
    if (sx && act >= 0) WIDE(true, true);
    else if (sx) WIDE(true, false);
    else if (act >= 0) WIDE(false, true);
    else WIDE(false, false);
#undef WIDE
    return hipGetLastError();
  }
#define EXPERTS(F8)                                                          \
  return bm == 128  ? gp_experts<F8, 128, 128, 2, 4, 4>(a, stream)           \
         : bm == 64 ? gp_experts<F8, 64, 64, 4, 2, 4>(a, stream)             \
                    : gp_experts<F8, 32, 64, 2, 2, 6>(a, stream)
  if (sx) EXPERTS(true);
  EXPERTS(false);
#undef EXPERTS
}

extern "C" hipError_t launch_expert_sum(const void* y, const void* w,
                                        const void* idx, void* h, int M,
                                        int top, int H, hipStream_t stream) {
  if (M < 1 || top < 1 || H < 8 || H % 8) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_expert_sum, dim3((H / 8 + 255) / 256, M), dim3(256), 0,
                     stream, (const u16*)y, (const float*)w, (const int*)idx, (u16*)h, top,
                     H);
  return hipGetLastError();
}
