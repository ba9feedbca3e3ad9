// mid_gemm.hip — linears of some rows: Y[M,N] = X[M,K] W[N,K]^T, up to 64
// rows, bf16 or e4m3 with row scales, fp32 sums, bf16 out.
//
// Bound by streaming W once.  The eight waves of a block share out its K,
// slab by slab, and each takes all rows of X and all columns of the block
// over its own slabs: what a wave wants of X no other wave of the block does,
// so there is no barrier ahead of the sums, which meet in LDS once.  Blocks
// are narrow (16 or 32 rows of W), so there are some for every CU; where there
// are not, K is split over blocks as well, and the last one of a column group
// to arrive adds the parts in their order.
// us, by tiles of 32x64 (six buffers, 64 to 256 blocks) -> here, bf16: 37 rows
// 3072x2048 11.4 -> 7.4, 2048x2048 9.5 -> 7.2, 2048x8192 15.2 -> 13.0 (2.6
// TB/s); e4m3: 33 rows 3584x3584 13.1 -> 7.4, 3072x8192 22.5 -> 11.5.  Left:
// two us of launch, the first loads, and X, read by every block.
//
// X goes by DMA into a stretch of LDS of each wave, whole lines at a time
// (straight into operands, 16 rows a line apart at once, a CU takes 15 bytes
// a clock: 64x2048x8192 17.4 us, 15.0 so).
// A load takes 8 rows x 128 bytes of W (whole lines), and an exchange with
// lane l^8 makes operands of two of them: row l&15, 16-byte chunks 2(l>>4)
// and 2(l>>4)+1.  X is read in that order.  W is the first operand, so a lane
// ends with four neighbouring outputs of one row.
#include "common.h"
#include "mid_gemm.h"

typedef short mg_s8 __attribute__((ext_vector_type(8)));
typedef int mg_i8 __attribute__((ext_vector_type(8)));

struct MgArgs {
  const void* x;       // [M, ldx]
  const void* w;       // [N, K], GLU: [2N, K] gate then up
  const float* sx;     // e4m3: row scales
  const float* sw;
  const u16* res;      // [M, ldr]
  const u16* bias;     // [N]
  void* y;             // [M, ldy]
  float* part;         // split K: [group, split, items * 4]
  int* cnt;            // split K: blocks of a group that are done
  int M, N, K, act, per;                   // per: slabs of a part
  int ldx, ldr, ldy;                       // elements from row to row
  int out_f32, wide;                       // wide: outputs four at a time
  float softcap;
};

DEVINL uint32_t mg_swap8(uint32_t v) {     // the value of lane l^8
  return __builtin_amdgcn_update_dpp(0, v, 0x128, 0xf, 0xf, true);
}

#define MG_NW 8

// MT tiles of 16 rows, NT of 16 rows of W (GLU: gate, up)
template <bool F8, int MT, int NT, bool GLU>
__global__ void __launch_bounds__(64 * MG_NW) k_mid_gemm(MgArgs a) {
  static_assert(!GLU || NT == 2);
  constexpr int OUT = GLU ? 16 : NT * 16;  // outputs of a block
  constexpr int ITEMS = MT * NT * 64;      // lanes' four sums
  // X of a slab, 128 bytes a row: each wave's own, two of them in arrays of
  // their own, so that the compiler sees that what is on the way into one is
  // not read from the other.  The sums of a wave go where its X was.
  constexpr int ZX = MT * 2048;
  __shared__ __attribute__((aligned(16))) char X0[MG_NW * ZX], X1[MG_NW * ZX];
  __shared__ int last_flag;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, gq = lane >> 4, r8 = lane & 7, c8 = lane >> 3;
  const bool low = lr < 8;
  const int n0 = blockIdx.x * OUT;
  const size_t rowb = (size_t)a.K * (F8 ? 1 : 2);
  const int slabs = (int)((rowb + 127) / 128);
  const int s0 = blockIdx.y * a.per, s1 = min(s0 + a.per, slabs);
  // slabs s0 + wave, s0 + wave + 8, ..
  const int n = max(0, (s1 - s0 - wave + MG_NW - 1) / MG_NW);

  const char* pw[NT][2];
#pragma unroll
  for (int t = 0; t < NT; t++)
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int r = h * 8 + r8;
      const size_t row = GLU ? (size_t)t * a.N + min(n0 + r, a.N - 1)
                             : (size_t)min(n0 + t * 16 + r, a.N - 1);
      pw[t][h] = (const char*)a.w + row * rowb;
    }
  // row r of a slab keeps chunk c at c ^ (r & 7)
  const int xr = lane >> 3, xc = ((lane & 7) ^ xr) * 16;
  const char* px[MT * 2];
#pragma unroll
  for (int i = 0; i < MT * 2; i++)
    px[i] = (const char*)a.x +
            (size_t)min(i * 8 + xr, a.M - 1) * a.ldx * (F8 ? 1 : 2);
  const int at0 = lr * 128 + ((gq * 2) ^ r8) * 16;      // r8 = lr & 7

  f4v acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int t = 0; t < NT; t++) acc[i][t] = {0.f, 0.f, 0.f, 0.f};

  struct Slab { u4v_ w[NT][2]; };
  const int rot = n > 0 ? blockIdx.x % n : 0;
  auto slab = [&](int i) {
    const int j = i + rot;
    return s0 + wave + (j < n ? j : j - n) * MG_NW;
  };
  auto load = [&](Slab& d, char* X, int i) {
    __builtin_amdgcn_sched_barrier(0);     // not ahead of what d held before
    const size_t k = (size_t)slab(i) * 128;
    // e4m3 rows of 64 * odd: what is behind the end is read inside the row
    // and multiplied by nothing
    const size_t kw = k + c8 * 16, kx = k + xc;
    const size_t cw = F8 && kw >= rowb ? 0 : kw;
    const size_t cx = F8 && kx >= rowb ? 0 : kx;
#pragma unroll
    for (int j = 0; j < MT * 2; j++)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) uint32_t*)(px[j] + cx),
          (__attribute__((address_space(3))) uint32_t*)(
              X + wave * ZX + j * 1024), 16, 0, 0);
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int h = 0; h < 2; h++)
        d.w[t][h] = __builtin_nontemporal_load((const u4v_*)(pw[t][h] + cw));
    __builtin_amdgcn_sched_barrier(0);
  };
  auto mul = [&](Slab& d, const char* X, int i) {
    const size_t kx = (size_t)slab(i) * 128 + gq * 32;
    const bool out = F8 && kx >= rowb;
    union Op { u4v_ q[2]; mg_i8 v; mg_s8 s[2]; };
    Op w[NT];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const uint32_t a0 = d.w[t][0][e], a1 = d.w[t][1][e];
        const uint32_t got = mg_swap8(low ? a1 : a0);
        w[t].q[0][e] = low ? a0 : got;
        w[t].q[1][e] = low ? got : a1;
      }
#pragma unroll
    for (int i = 0; i < MT; i++) {
      Op x;
#pragma unroll
      for (int h = 0; h < 2; h++) {
        x.q[h] = *(const u4v_*)(X + wave * ZX + i * 2048 + (at0 ^ h * 16));
        if (F8 && out) x.q[h] = u4v_{0, 0, 0, 0};
      }
#pragma unroll
      for (int t = 0; t < NT; t++) {
        if constexpr (F8) {
          // block scales of one (e8m0 127): the row scales come at the end
          // (as exact as the 32-deep instruction: the same errors to five
          // places)
          acc[i][t] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
              w[t].v, x.v, acc[i][t], 0, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f);
        } else {
#pragma unroll
          for (int h = 0; h < 2; h++)
            acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                w[t].s[h], x.s[h], acc[i][t], 0, 0, 0);
        }
      }
    }
  };
  // Two slabs in flight.  No branch stands between a load and its use (the
  // compiler would wait for all loads there): of an odd number the last is
  // asked for twice.
  if (n > 0) {
    Slab p, q;
    load(p, X0, 0);
    load(q, X1, min(1, n - 1));
    int i = 0;
    for (; i + 2 < n; i += 2) {
      mul(p, X0, i);
      load(p, X0, i + 2);
      mul(q, X1, i + 1);
      load(q, X1, min(i + 3, n - 1));
    }
    mul(p, X0, i);
    if (i + 1 < n) mul(q, X1, i + 1);
    // nothing is on its way into LDS when the block ends
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  f4v* const sums = (f4v*)X0;
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int t = 0; t < NT; t++)
      sums[(wave * 2 * MT + i * NT + t) * 64 + lane] = acc[i][t];
  __syncthreads();

  // outputs n..n+3 of a row, with a gate of the same places of both tiles
  constexpr int P = GLU ? 2 : 1, DONE = ITEMS / P;

  auto finish = [&](int e, f4v v, f4v u) {
    const int i = e / (NT / P * 64), t = e / 64 % (NT / P), l = e & 63;
    const int row = i * 16 + (l & 15), n = n0 + t * 16 + (l >> 4) * 4;
    if (row >= a.M || n >= a.N) return;
    if (F8) {
      const float sx = a.sx[row];
#pragma unroll
      for (int r = 0; r < 4; r++) {
        v[r] *= sx * a.sw[min(n + r, a.N - 1)];
        if (GLU) {
          // to be rounded to e4m3 next: from bf16 halves, like more rows'
          u[r] = b2f(f2b(u[r] * sx * a.sw[a.N + min(n + r, a.N - 1)]));
          v[r] = b2f(f2b(v[r]));
        }
      }
    }
    if (GLU)
#pragma unroll
      for (int r = 0; r < 4; r++) v[r] = gate_act(v[r], a.act) * u[r];
    if (a.softcap > 0.f)
#pragma unroll
      for (int r = 0; r < 4; r++) v[r] = a.softcap * tanhf(v[r] / a.softcap);
    const size_t at = (size_t)row * a.ldy + n;
    const u16* res = a.res ? a.res + (size_t)row * a.ldr + n : nullptr;
    if (a.wide) {
      union { u16 h[4]; unsigned long long q; } o;
      if (a.bias) {
        o.q = *(const unsigned long long*)(a.bias + n);
#pragma unroll
        for (int r = 0; r < 4; r++) v[r] += b2f(o.h[r]);
      }
      if (res) {
        o.q = *(const unsigned long long*)res;
#pragma unroll
        for (int r = 0; r < 4; r++) v[r] += b2f(o.h[r]);
      }
      if (a.out_f32) {
        *(f4v*)((float*)a.y + at) = v;
      } else {
#pragma unroll
        for (int r = 0; r < 4; r++) o.h[r] = f2b(v[r]);
        *(unsigned long long*)((u16*)a.y + at) = o.q;
      }
    } else {
      for (int r = 0; r < 4 && n + r < a.N; r++) {
        float f = v[r];
        if (a.bias) f += b2f(a.bias[n + r]);
        if (res) f += b2f(res[r]);
        if (a.out_f32) ((float*)a.y)[at + r] = f;
        else ((u16*)a.y)[at + r] = f2b(f);
      }
    }
  };
  // the first of a gate's pair of sums, the second 64 behind it
  auto place = [&](int e) { return GLU ? e / 64 * 128 + (e & 63) : e; };
  auto meet = [&](int at) {
    f4v v = sums[at];
#pragma unroll
    for (int k = 1; k < MG_NW; k++) v += sums[k * (MT * 128) + at];
    return v;
  };
  const int KS = gridDim.y;
  if (KS == 1) {
    for (int e = tid; e < DONE; e += 64 * MG_NW) {
      const int at = place(e);
      finish(e, meet(at), GLU ? meet(at + 64) : f4v{});
    }
    return;
  }
  float* part = a.part + (size_t)blockIdx.x * KS * ITEMS * 4;
  for (int e = tid; e < ITEMS; e += 64 * MG_NW)
    part_put4(part + (size_t)blockIdx.y * ITEMS * 4 + e * 2, ITEMS * 2,
              meet(e));
  if (!last_block(&a.cnt[blockIdx.x], KS, &last_flag)) return;
  // four parts on the way at a time (one after the other, and in halves of
  // lines: 37x2048x8192 12.7 us, so 12.2)
  auto parts = [&](int at) {
    f4v v, t[4];
    for (int k = 0; k < KS; k += 4) {
#pragma unroll
      for (int q = 0; q < 4; q++)
        t[q] = part_get4(part + (size_t)min(k + q, KS - 1) * ITEMS * 4 +
                             at * 2, ITEMS * 2);
#pragma unroll
      for (int q = 0; q < 4; q++)
        if (k + q < KS) v = k + q ? v + t[q] : t[q];
    }
    return v;
  };
  for (int e = tid; e < DONE; e += 64 * MG_NW) {
    const int at = place(e);
    finish(e, parts(at), GLU ? parts(at + 64) : f4v{});
  }
}

// How a product goes: nt tiles of W a block, K in ks parts of per slabs.
struct MgPlan { int nt, ks, per, groups; };

// us of 16 and 37 rows, by blocks of 16 and of 32 rows of W:
//   rows of up to 8 KB  2048x2048 5.7 and 7.3, 7.3 and 9.4 (32, K in two: 6.9
//     and 8.0); 3584x3584 8.6 and 12.1, 11.9 and 15.6; more than 256 blocks of
//     16 read X too often: 4608x3584 14.0 and 21.4, 12.1 and 15.7
//   longer  2048x8192 11.7 and 16.7 (K in four), 10.6 and 13.1 (in four);
//     3072x8192 15.0 and 23.0 (in four), 14.3 and 18.5 (in two)
static MgPlan mg_plan(bool f8, int M, int N, int K, bool glu,
                      long part_floats, int ncnt) {
  const long rowb = (long)K * (f8 ? 1 : 2);
  const int slabs = (int)((rowb + 127) / 128), mt = (M + 15) / 16;
  MgPlan p = {1, 1, slabs, (N + 15) / 16};
  if (glu) {
    p.nt = 2;
    return p;
  }
  if (rowb > 8192 || p.groups > 256) {
    p.nt = 2;
    p.groups = (N + 31) / 32;
    // a block for each CU, two slabs at least for each of its waves
    while (p.groups * (p.ks + 1) <= 256 &&
           slabs / (p.ks + 1) >= 2 * MG_NW && p.groups <= ncnt &&
           (long)p.groups * (p.ks + 1) * mt * p.nt * 256 <= part_floats)
      p.ks++;
  }
  p.per = (slabs + p.ks - 1) / p.ks;
  p.ks = (slabs + p.per - 1) / p.per;
  return p;
}

// us, row_gemm / here, W from memory (15 widths by 11 lengths at 12 numbers of
// rows each):
//   bf16  up to 4096 columns: 2048x2048 5 rows 7.5/6.7, 3584x3584 9.7/9.1; where
//       rows are 6 to 8 KB and blocks neither few, as row_gemm has it then
//       (1024x4096 10.2/8.8), nor one for most CUs, K in one stretch a block is
//       too long (2048x3584 7.9/8.8)
//     longer rows  row_gemm stages more than eight rows of X in parts
//       (2304x14336 5 rows 16.9/17.0, 9 21.3/17.4), but not beside few columns
//       (9x512x14336 12.2/13.1); 16 KB apart they stand in each other's way
//       here (9x4096x8192 17.3/20.4)
//   e4m3  2048x2048 7.5/5.6, 8192x3584 8 rows 10.1/9.4; 2048x8192 5 rows
//       8.7/9.1, 16 10.7/9.7; many rows not 4 and 8 KB apart (5x8192x4096
//       10.4/11.1, 9x4608x8192 13.1/14.2)
static bool mid_takes_few(bool f8, int M, int N, int K) {
  if (N > (f8 ? 8192 : 4096) || (K > 4096 && M <= 8)) return false;
  if (f8)
    return N <= 4096 || (K % 8192 && (K % 4096 || N <= 6144) &&
                         (K <= 16384 || N > 7168));
  if (K <= 4096)
    return K <= 2304 || M > 12 || N <= 1024 || N > (K <= 3072 ? 2048 : 2560);
  if (K > 8192 && N < 1024) return false;
  return K % 8192 || N <= (M > 12 ? 3584 : 2560);
}

// More rows and gates: us, the best tile / here, W from memory:
//   bf16  rows of up to 4.5 KB  2304x2048 17 rows 8.5/6.0, 64 8.8/7.7; 6144x2048
//       48 11.7/10.6, 64 12.3/11.5
//     up to 8 KB  17x3584x3584 12.0/9.2, 48 13.2/12.1; the more rows of X, the
//       more columns it takes to be worth their way (48x1024x4096 9.2/10.0,
//       48x3072x4096 12.4/11.9, 64x3072x4096 12.9/13.4), and 4608 make 144
//       blocks of 32, too few (33x4608x3584 13.9/14.9)
//     longer  3072x8192 24 rows 15.5/15.9, 48 17.3/19.6; 3584x14336 17
//       22.7/23.5, 32 23.8/26.7; 17x4608x14336 27.0/38.1
//   e4m3  4096x4096 17 10.6/6.7, 64 11.0/8.6; 3584x14336 17 16.5/15.7, 64
//       20.0/20.6; 512x8192 64 9.6/11.4
//   gate  8192x2048 17 16.7/14.7, 32 16.6/16.5; 17x8192x3584 21.7/25.0; e4m3
//       8192x2048 17 10.8/9.6, 6144x1024 32 6.4/8.7
// The lines lie where they did beside tiles of four waves, to which most of
// this was further ahead.  By times of 5200 products without a gate and 1060
// with one: of the 4119 and 352 that are taken a tile is 4 and 5% faster for 309
// and 121 (bf16 of more than 8 KB a row, 32 rows with a gate), of those left 191
// and 92 are slower by tiles.
bool mid_takes(bool f8, int M, int N, int K, bool glu) {
  if (glu)
    return M > 16 && M <= 32 && N <= 8192 && K <= 2048 &&
           !(f8 && K <= 1024 && N > 4096);
  if (M <= 16) return mid_takes_few(f8, M, N, K);
  if (M > 64 || N > 8192) return false;
  if (f8) return K <= 7168 || K > 8192 || N > 1024 || M < 48;
  if (K <= 2304) return N <= 4096 || M <= 48;
  if (K > 8192) return M <= 24 && (N <= 4096 || N >= 7168);
  if (M > 48 || (N > 4096 && N < 5120)) return false;
  return K > 4096 || M <= 32 || N >= 48 * M;
}

// Y [M, N], M up to 64 (32 with a gate); sx, sw: row scales of e4m3 x and w.
// act < 0: no gate.  part and cnt (zero, left zero) let K be split.
extern "C" hipError_t launch_mid_gemm(
    const void* x, const void* w, const void* sx, const void* sw,
    const void* res, const void* bias, void* y, void* part, void* cnt,
    long part_floats, int ncnt, int M, int N, int K, int ldx, int ldr,
    int ldy, int act, int out_f32, float softcap, hipStream_t stream) {
  if (M < 1 || M > 64 || N < 1 || K < 64 || K % 64 || (!sx != !sw) ||
      ldx < K || ldx % (sx ? 16 : 8) || ldy < N || (res && ldr < N) ||
      (act >= 0 && M > 32))
    return hipErrorInvalidValue;
  const bool glu = act >= 0;
  const int wide = (N | ldy | (res ? ldr : 0)) % 4 == 0 &&
                   (size_t)y % 16 == 0 &&
                   ((size_t)res | (size_t)bias) % 8 == 0;
  if (!part || !cnt) part_floats = 0;
  const MgPlan p = mg_plan(sx, M, N, K, glu, part_floats, ncnt);
  const MgArgs a = {x, w, (const float*)sx, (const float*)sw,
                    (const u16*)res, (const u16*)bias, y, (float*)part,
                    (int*)cnt, M, N, K, act, p.per, ldx, ldr, ldy, out_f32,
                    wide, softcap};
  const dim3 grid(p.groups, p.ks), nt(64 * MG_NW);
#define MG_GO(F8, MT, NT, GLU)                                               \
  hipLaunchKernelGGL((k_mid_gemm<F8, MT, NT, GLU>), grid, nt, 0, stream, a)
#define MG_ROWS(F8, NT, GLU)                                                 \
  switch ((M + 15) / 16) {                                                   \
    case 1: MG_GO(F8, 1, NT, GLU); break;                                    \
    case 2: MG_GO(F8, 2, NT, GLU); break;                                    \
    case 3: MG_GO(F8, 3, NT, GLU); break;                                    \
    default: MG_GO(F8, 4, NT, GLU);                                          \
  }
#define MG_KIND(F8)                                                          \
  if (glu) MG_GO(F8, 2, 2, true);                                            \
  else if (p.nt == 2) MG_ROWS(F8, 2, false)                                  \
  else MG_ROWS(F8, 1, false)
  if (sx) { MG_KIND(true) } else { MG_KIND(false) }
#undef MG_KIND
#undef MG_ROWS
#undef MG_GO
  return hipGetLastError();
}
