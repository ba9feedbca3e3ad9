// attn_prefill.hip — flash attention of prompt rows over the KV pool.
//
// One wave holds 32 query rows and walks the keys in tiles of 32; a block
// of four waves shares the tiles through LDS.  The rows of a block are
// (position, head) pairs of ONE kv head, so a K/V tile is read once for
// all heads of its group and a check of five proposed tokens fills half a
// tile instead of five heads' own.
//
// S^T = K Q^T puts a query in a lane (column lane&31 of
// mfma_f32_32x32x16), so maximum, sum and rescaling never leave the lane
// pair (l, l+32).  The 16 scores a lane then holds are, in register order,
// the k elements of the second product's B operand for keys
// {0-3,8-11} + 4*half of a 16-key slab, so P goes from accumulator to
// operand without moving between lanes; V^T comes out of LDS in that same
// key order with ds_read_b64_tr_b16, which turns a 4-key x 16-dim tile so
// that a lane holds one dim's four keys.
//
// What bounds it: head_dim 128 spends 512 MFMA cycles and about 450 VALU
// cycles on 32 keys x 32 rows; two blocks of 64 KB LDS on a CU overlap them.
// Measured (32/8 heads of 128, 2048 rows behind 6139 keys): 270 us,
// 890 TFLOP/s; a wave per head and 16 queries took 1422 us.  (With both
// buffers in one array the DMA drained ahead of every tile's reads: 314 us.)
// 5 rows of 24/8 heads over 906 keys, split: 11 us, unsplit per-head waves
// 74 us.  Head dim 256 at two waves a SIMD just fits the registers where LDS
// addresses are made again for each tile (2048 rows of 16/8 heads behind 2048
// keys with a soft cap 181 us, so 177); beside an e4m3 pool it spills 28, with a
// cap 29 (6 where one wave has all rows).  One wave a SIMD without spills was
// slower.  Of the others 64 dims by two groups of waves without a cap spills one.
//
// Where a block's own keys are what takes long (the last rows of a prompt see
// all of them, and a block goes through its tiles one after the other), two
// groups of four waves take its tiles in turn and meet in LDS at the end: a
// chain half as long and nothing past the L2, where ranges of keys leave parts
// of every row.  us, ranges or one block as before -> two groups:
//   64 dims   32/8 heads  611 rows 22.8 -> 12.7, 1000 34.9 -> 17.1, 1999 34.1 ->
//             29.9; 700 behind 1300 keys 37.5 -> 27.6
//   128 dims  32/8 1000 rows 40.5 -> 24.4, 1999 54.1 -> 49.6; 24/8 1999 52.7 ->
//             40.8; 16/4 1999 51.6 -> 39.7
// Of 256 dims a CU is bound by its LDS (each wave reads all of K and V for 32
// rows of its own): 1999 rows of 8/4 heads 111.7 by one group and by two.
//
// Rows of several sequences (a group's prompts in one batch) bring a table:
// which rows, position and pool a block's tile belongs to, the ones with the
// most keys first.  A scalar load a block; nothing else differs.
#include "common.h"
#include "attn_prefill.h"

typedef short ap_s4 __attribute__((ext_vector_type(4)));
typedef __bf16 ap_b8 __attribute__((ext_vector_type(8)));
typedef __bf16 ap_b2 __attribute__((ext_vector_type(2)));
typedef float ap_f16 __attribute__((ext_vector_type(16)));

#define LOG2E 1.4426950408889634f

// tanh by exp2: |error| below 2e-7, exact limits at +-inf
DEVINL float ap_tanh(float x) {
  const float e = __builtin_amdgcn_exp2f(x * (2.f * LOG2E));
  return 1.f - 2.f * __builtin_amdgcn_rcpf(e + 1.f);
}

// LDS rows are `HD` bf16.  K: 16-byte slots swizzled by the row (a b128
// fragment read takes one slot of 32 rows); V: 64-byte chunks swizzled (a
// transposed read takes one chunk of 8 rows).
template <int HD> DEVINL int k_slot(int row, int slot) {
  return slot ^ (row & (HD / 8 < 16 ? 7 : 15));
}
template <int HD> DEVINL int v_slot(int row, int slot) {
  const int x = HD == 64 ? (row >> 1) & 1 : row & 3;
  return slot ^ (x << 2);
}

// A kv head's part of a range of keys, in the (HD + 4) floats a row that it has.
// Row by row, or (in lines) four dims of all rows, the next four, .., then
// maxima, then sums.  Where that leaves room, rows are counted up to whole lines
// and parts begin with one.
struct ApPart { uint32_t rows; size_t size; };
template <int HD> DEVINL ApPart ap_part(uint32_t rows) {
  const size_t size = (size_t)rows * (HD + 4);
  if (rows < 4 * (HD + 2)) return {rows, size};
  return {(rows + 7) / 8 * 8, size / 32 * 32};
}

template <int HD, int BKV, int NW, int KG, bool KV8, bool CAP>
__global__ void __launch_bounds__(64 * NW * KG, KG == 2 && HD == 64 ? 4 : 2)
k_attn_rows(ApArgs a) {
  constexpr int RB = HD * 2;                 // LDS bytes of a row
  constexpr int TILE = BKV * RB;
  constexpr int SLOTS = HD / 8;              // 16-byte slots of a row
  constexpr int NS = BKV / 32;               // 32-key parts of a tile
  constexpr int NT = 64 * NW;
  constexpr bool RAW = !CAP && !KV8;
  // an array a buffer, and the loop unrolled over the two: the compiler sees
  // that the DMA into one does not touch what is read from the other, and
  // does not wait for it before the reads
  __shared__ __attribute__((aligned(16))) char KA[KG * TILE], KB[KG * TILE];
  __shared__ __attribute__((aligned(16))) char VA[KG * TILE], VB[KG * TILE];
  __shared__ __attribute__((aligned(16))) float SA[KG][2][KV8 ? BKV : 4],
      SB[KG][2][KV8 ? BKV : 4];

  const int tid = KG == 1 ? threadIdx.x : threadIdx.x & (NT - 1);
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // tiles of keys go to the groups of waves in turn
  const int kg = KG == 1 ? 0
                         : __builtin_amdgcn_readfirstlane(threadIdx.x / NT);
  char *const K0 = KA + kg * TILE, *const K1 = KB + kg * TILE;
  char *const V0 = VA + kg * TILE, *const V1 = VB + kg * TILE;
  float(*const S0)[KV8 ? BKV : 4] = SA[kg], (*const S1)[KV8 ? BKV : 4] = SB[kg];
  const int hh = lane >> 5, col = lane & 31;
  const int grp = a.nh / a.kvh;
  // heads vary fastest, so that with a multiple of eight of them the
  // blocks of a kv head land on one XCD and share its L2
  const int kvhead = blockIdx.x;
  const int nq = gridDim.y;
  // longest rows first; where two blocks a CU hold the whole grid, the second
  // of a CU come shortest first
  int qt = nq - 1 - (int)blockIdx.y;
  if ((int)blockIdx.y >= a.fold) qt = (int)blockIdx.y - a.fold;

  int base = 0, M = a.M, pool = 0, pos0;
  if (a.tiles) {
    const int* t = a.tiles + blockIdx.y * 5;
    qt = t[0];
    base = t[1];
    M = t[2];
    pos0 = t[3];
    pool = t[4];
  } else {
    pos0 = *a.len_ptr;
  }
  const int nrows = M * grp;
  const int row0 = (qt * NW + wave) * 32;
  const int row = row0 + col;
  const int rowc = min(row, nrows - 1);
  const int my_m = rowc / grp, my_g = rowc % grp;
  const int qpos = pos0 + my_m;
  // positions of the wave's first and last row, and of the block's last
  const int q_lo = pos0 + min(row0, nrows - 1) / grp;
  const int q_hi = pos0 + min(row0 + 31, nrows - 1) / grp;
  const int b_lo = pos0 + min(qt * NW * 32, nrows - 1) / grp;
  const int b_hi = pos0 + min(qt * NW * 32 + NW * 32 - 1, nrows - 1) / grp;
  const bool live = row0 < nrows;

  // keys [k_lo, k_hi) of this block
  int k_lo = 0, k_hi = b_hi + 1;
  if (a.window > 0) k_lo = max(0, b_lo + 1 - a.window);
  if (gridDim.z > 1) {
    const int tiles = (k_hi - k_lo + BKV - 1) / BKV;
    const int per = (tiles + gridDim.z - 1) / gridDim.z;
    const int lo = k_lo + (int)blockIdx.z * per * BKV;
    k_hi = min(k_hi, lo + per * BKV);
    k_lo = lo;
  }
  const int t_last = b_hi;                   // last key that may be read

  // Q: B operand, column = row of the tile, 8 dims at 16*c + 8*hh
  ap_b8 qf[HD / 16];
  {
    const u16* qp = a.q + (size_t)(base + my_m) * a.ldq +
                    (size_t)(kvhead * grp + my_g) * HD + hh * 8;
#pragma unroll
    for (int c = 0; c < HD / 16; c++) qf[c] = *(const ap_b8*)(qp + c * 16);
  }

  const size_t head = ((size_t)pool * a.kvh + kvhead) * a.S;   // first key's
  const char* Kg = (const char*)a.kc + head * HD * (KV8 ? 1 : 2);
  const char* Vg = (const char*)a.vc + head * HD * (KV8 ? 1 : 2);
  const float* kS = KV8 ? a.kS + head : nullptr;
  const float* vS = KV8 ? a.vS + head : nullptr;

  // bf16 pool: straight into LDS.  A wave's instruction fills 1 KB, lane by
  // lane; the swizzle sits in the address that the lane reads.
  constexpr int RPI = 1024 / RB;             // rows an instruction fills
  auto stage16 = [&](char* Ks, char* Vs, int t0) {
#pragma unroll
    for (int i = 0; i < BKV / RPI / NW; i++) {
      const int r0 = (i * NW + wave) * RPI;
      const int r = r0 + lane / SLOTS, s = lane % SLOTS;
      const size_t t = min(t0 + r, t_last);
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) uint32_t*)(
              Kg + t * RB + k_slot<HD>(r, s) * 16),
          (__attribute__((address_space(3))) uint32_t*)(Ks + r0 * RB),
          16, 0, 0);
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) uint32_t*)(
              Vg + t * RB + v_slot<HD>(r, s) * 16),
          (__attribute__((address_space(3))) uint32_t*)(Vs + r0 * RB),
          16, 0, 0);
    }
  };
  // fp8 pool: through registers, widened to bf16 (exact) on the way in;
  // the scale of a key stays out of the rounding: it multiplies the fp32
  // score, the one of a value the fp32 probability.
  constexpr int L8 = KV8 ? BKV * HD / 16 / NT : 1;   // 16-byte loads a thread
  u4v_ kr[L8], vr[L8];
  constexpr int NSC = (2 * BKV + NT - 1) / NT;
  float scr[NSC];
  auto load8 = [&](int t0) {
    if constexpr (KV8) {
#pragma unroll
      for (int i = 0; i < L8; i++) {
        const int e = i * NT + tid, r = e / (HD / 16), s = e % (HD / 16);
        const size_t t = min(t0 + r, t_last);
        kr[i] = *(const u4v_*)(Kg + t * HD + s * 16);
        vr[i] = *(const u4v_*)(Vg + t * HD + s * 16);
      }
#pragma unroll
      for (int i = 0; i < NSC; i++) {
        const int e = i * NT + tid;
        if (e < 2 * BKV)
          scr[i] = (e < BKV ? kS : vS)[min(t0 + e % BKV, t_last)];
      }
    }
  };
  auto store8 = [&](char* Ks, char* Vs, float (*Sc)[KV8 ? BKV : 4]) {
    if constexpr (KV8) {
#pragma unroll
      for (int i = 0; i < L8; i++) {
        const int e = i * NT + tid, r = e / (HD / 16), s = e % (HD / 16);
#pragma unroll
        for (int h = 0; h < 2; h++) {
          union { ap_b2 b[4]; s8v v; } ko, vo;
#pragma unroll
          for (int d = 0; d < 2; d++) {
            ko.b[d * 2] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(
                kr[i][h * 2 + d], 1.0f, false);
            ko.b[d * 2 + 1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(
                kr[i][h * 2 + d], 1.0f, true);
            vo.b[d * 2] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(
                vr[i][h * 2 + d], 1.0f, false);
            vo.b[d * 2 + 1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(
                vr[i][h * 2 + d], 1.0f, true);
          }
          const int sl = s * 2 + h;
          *(s8v*)(Ks + r * RB + k_slot<HD>(r, sl) * 16) = ko.v;
          *(s8v*)(Vs + r * RB + v_slot<HD>(r, sl) * 16) = vo.v;
        }
      }
#pragma unroll
      for (int i = 0; i < NSC; i++) {
        const int e = i * NT + tid;
        if (e < 2 * BKV) Sc[e / BKV][e % BKV] = scr[i];
      }
    }
  };

  // LDS offsets of fragments that the swizzle makes differ by more than a
  // constant: 8 of K (16-byte slots of a row), 4 of V (64-byte chunks).  Of 256
  // dims, where registers are short, they are made for each tile of the first
  // ones: kept, some were spilled, and their way back waited for the next
  // tile's DMA (1792 rows of 8/4 heads with a cap, parts
  // left as they are now: 54.9 us, so 50.4).
  constexpr int KC = HD / 16 < 8 ? HD / 16 : 8, VD = HD / 32 < 4 ? HD / 32 : 4;
  constexpr bool FEW = HD == 256;
  const int vrow = hh * 4 + ((lane & 15) >> 2);
  const int vcol = ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
  int kb[FEW ? 1 : KC], vb[FEW ? 1 : VD];
#pragma unroll
  for (int c = 0; c < (FEW ? 1 : KC); c++)
    kb[c] = col * RB + k_slot<HD>(col, c * 2 + hh) * 16;
#pragma unroll
  for (int d = 0; d < (FEW ? 1 : VD); d++)
    vb[d] = vrow * RB + v_slot<HD>(vrow, d * 4 + (vcol >> 3)) * 16 +
            (vcol & 7) * 2;

  float m = -INFINITY, l = 0.f;     // m in units of log2
  ap_f16 o[HD / 32];
#pragma unroll
  for (int d = 0; d < HD / 32; d++)
#pragma unroll
    for (int r = 0; r < 16; r++) o[d][r] = 0.f;
  const float c1 = CAP ? a.scale / a.softcap : a.scale * LOG2E;
  const float c2 = CAP ? a.softcap * LOG2E : 1.f;

  auto tile = [&](char* Ks, char* Vs, float (*Sc)[KV8 ? BKV : 4], char* Kn,
                  char* Vn, float (*Sn)[KV8 ? BKV : 4], int t0) {
    const bool more = t0 + KG * BKV < k_hi;
    if (more) {
      if constexpr (KV8) load8(t0 + KG * BKV);
      else stage16(Kn, Vn, t0 + KG * BKV);
    }
    const bool some = live && t0 <= q_hi && (KG == 1 || t0 < k_hi) &&
                      (a.window <= 0 || t0 + BKV > q_lo - a.window);
    if (some) {
      int k0 = kb[0], v0 = vb[0];
      if constexpr (FEW) asm volatile("" : "+v"(k0), "+v"(v0));
      auto k_at = [&](int c) { return FEW ? k0 ^ c % KC << 5 : kb[FEW ? 0 : c % KC]; };
      auto v_at = [&](int d) { return FEW ? v0 ^ d % VD << 6 : vb[FEW ? 0 : d % VD]; };
      ap_f16 s[NS];
#pragma unroll
      for (int n = 0; n < NS; n++) {
#pragma unroll
        for (int r = 0; r < 16; r++) s[n][r] = 0.f;
#pragma unroll
        for (int c = 0; c < HD / 16; c++) {
          const ap_b8 kf = *(const ap_b8*)(
              Ks + k_at(c) + c / KC * 256 + n * 32 * RB);
          s[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[c], s[n], 0,
                                                         0, 0);
        }
      }
      // keys t0 + 32n + 8(r/4) + 4hh + r%4
      const bool edge = t0 + BKV - 1 > q_lo || t0 + BKV > k_hi ||
                        (a.window > 0 && t0 <= q_hi - a.window);
      // Plain scores stay as they are: their scale rides in the exponent.
      if constexpr (!RAW) {
#pragma unroll
        for (int n = 0; n < NS; n++)
#pragma unroll
          for (int q4 = 0; q4 < 4; q4++) {
            f4v ks = {1.f, 1.f, 1.f, 1.f};
            if constexpr (KV8)
              ks = *(const f4v*)(&Sc[0][n * 32 + q4 * 8 + hh * 4]);
#pragma unroll
            for (int j = 0; j < 4; j++) {
              float v = s[n][q4 * 4 + j] * c1;
              if constexpr (KV8) v *= ks[j];
              if constexpr (CAP) v = c2 * ap_tanh(v);
              s[n][q4 * 4 + j] = v;
            }
          }
      }
      if (edge) {
#pragma unroll
        for (int n = 0; n < NS; n++)
#pragma unroll
          for (int r = 0; r < 16; r++) {
            const int t = t0 + n * 32 + (r >> 2) * 8 + hh * 4 + (r & 3);
            const bool bad = (t > qpos) | (t >= k_hi) |
                             ((a.window > 0) & (t <= qpos - a.window));
            s[n][r] = bad ? -INFINITY : s[n][r];
          }
      }
      float mx = -INFINITY;
#pragma unroll
      for (int n = 0; n < NS; n++)
#pragma unroll
        for (int r = 0; r < 16; r++) mx = fmaxf(mx, s[n][r]);
      if constexpr (RAW) mx *= c1;
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      const float mn = fmaxf(m, mx);
      const float mu = mn == -INFINITY ? 0.f : mn;
      if (__any(mn > m)) {
        const float al = __builtin_amdgcn_exp2f(m - mu);
        l *= al;
#pragma unroll
        for (int d = 0; d < HD / 32; d++)
#pragma unroll
          for (int r = 0; r < 16; r++) o[d][r] *= al;
        m = mn;
      }
#pragma unroll
      for (int n = 0; n < NS; n++) {
#pragma unroll
        for (int sl = 0; sl < 2; sl++) {
          float p[8];
#pragma unroll
          for (int j = 0; j < 8; j++) {
            p[j] = __builtin_amdgcn_exp2f(
                RAW ? fmaf(s[n][sl * 8 + j], c1, -mu) : s[n][sl * 8 + j] - mu);
            l += p[j];
          }
          if constexpr (KV8) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
              const f4v vs = *(const f4v*)(
                  &Sc[1][n * 32 + sl * 16 + h * 8 + hh * 4]);
#pragma unroll
              for (int j = 0; j < 4; j++) p[h * 4 + j] *= vs[j];
            }
          }
          union { ap_b2 b[4]; ap_b8 v; } pf;
#pragma unroll
          for (int j = 0; j < 4; j++) {
            pf.b[j][0] = (__bf16)p[j * 2];
            pf.b[j][1] = (__bf16)p[j * 2 + 1];
          }
          // V^T: dims 32d + col, keys as above; a lane of the read points
          // at 4 dims of key (lane/4)%4 of its 16-lane group's tile
#pragma unroll
          for (int d = 0; d < HD / 32; d++) {
            union { ap_s4 h[2]; ap_b8 v; } vf;
#pragma unroll
            for (int h = 0; h < 2; h++)
              vf.h[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                  (__attribute__((address_space(3))) ap_s4*)(
                      Vs + v_at(d) + d / VD * 256 +
                      (n * 32 + sl * 16 + h * 8) * RB));
            o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf.v, pf.v, o[d],
                                                           0, 0, 0);
          }
        }
      }
    }
    if constexpr (KV8) { if (more) store8(Kn, Vn, Sn); }
    __syncthreads();
  };
  const int first = k_lo + kg * BKV;         // of the group
  if (first < k_hi) {
    if constexpr (KV8) { load8(first); store8(K0, V0, S0); }
    else stage16(K0, V0, first);
  }
  __syncthreads();
  for (int t0 = k_lo; t0 < k_hi; t0 += 2 * KG * BKV) {
    tile(K0, V0, S0, K1, V1, S1, t0 + kg * BKV);
    if (t0 + KG * BKV < k_hi)
      tile(K1, V1, S1, K0, V0, S0, t0 + (KG + kg) * BKV);
  }

  l += __shfl_xor(l, 32);
  if constexpr (KG == 2) {
    // what the second group has, through the LDS that held the keys; lanes of
    // a wave beside each other
    static_assert(NW == 4 && 32 * HD * 4 <= KG * TILE);
    __shared__ float ml[NW][2][64];
    char* const to = wave == 0 ? KA : wave == 1 ? KB : wave == 2 ? VA : VB;
    float* const at = (float*)to + lane * 4;
    if (kg == 1) {
#pragma unroll
      for (int d = 0; d < HD / 32; d++)
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++)
          *(f4v*)(at + (d * 4 + q4) * 256) =
              f4v{o[d][q4 * 4], o[d][q4 * 4 + 1], o[d][q4 * 4 + 2],
                  o[d][q4 * 4 + 3]};
      ml[wave][0][lane] = m;
      ml[wave][1][lane] = l;
    }
    __syncthreads();
    if (kg == 1) return;
    const float m1 = ml[wave][0][lane], l1 = ml[wave][1][lane];
    const float mt = fmaxf(m, m1);
    const float w0 = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mt);
    const float w1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m1 - mt);
#pragma unroll
    for (int d = 0; d < HD / 32; d++)
#pragma unroll
      for (int q4 = 0; q4 < 4; q4++) {
        const f4v v = *(const f4v*)(at + (d * 4 + q4) * 256);
#pragma unroll
        for (int j = 0; j < 4; j++)
          o[d][q4 * 4 + j] = o[d][q4 * 4 + j] * w0 + v[j] * w1;
      }
    l = l * w0 + l1 * w1;
    m = mt;
  }
  if (row >= nrows) return;
  if (gridDim.z == 1) {
    const float inv = 1.f / l;
    u16* op = a.out +
              ((size_t)(base + my_m) * a.nh + kvhead * grp + my_g) * HD;
#pragma unroll
    for (int d = 0; d < HD / 32; d++)
#pragma unroll
      for (int q4 = 0; q4 < 4; q4++) {
        union { ap_b2 b[2]; unsigned long long u; } w;
#pragma unroll
        for (int j = 0; j < 4; j++)
          w.b[j / 2][j % 2] = (__bf16)(o[d][q4 * 4 + j] * inv);
        *(unsigned long long*)(op + d * 32 + q4 * 8 + hh * 4) = w.u;
      }
  } else if (NW == 1 || a.by_row) {
    // unnormalised part of this key range: HD values, maximum, sum
    float* pp = a.part + (((size_t)blockIdx.z * a.kvh + kvhead) * a.M * grp +
                          base * grp + row) * (HD + 4);
#pragma unroll
    for (int d = 0; d < HD / 32; d++)
#pragma unroll
      for (int q4 = 0; q4 < 4; q4++)
        *(f4v*)(pp + d * 32 + q4 * 8 + hh * 4) =
            f4v{o[d][q4 * 4], o[d][q4 * 4 + 1], o[d][q4 * 4 + 2],
                o[d][q4 * 4 + 3]};
    if (hh == 0) { pp[HD] = m; pp[HD + 1] = l; }
  } else {
    // Unnormalised part of this key range: the lanes of a store, which are
    // rows, leave whole lines (each row for itself, 16 bytes a lane: 1000 rows of
    // 32/8 heads of 64 in two ranges 35.2 us, so 26.7, of 128 40.7, 35.7).
    const ApPart part = ap_part<HD>(a.M * grp);
    const uint32_t nr = part.rows, at = base * grp + row;
    float* pp = a.part + ((size_t)blockIdx.z * a.kvh + kvhead) * part.size;
    float* to = pp + ((size_t)hh * nr + at) * 4;
#pragma unroll
    for (int d = 0; d < HD / 32; d++)
#pragma unroll
      for (int q4 = 0; q4 < 4; q4++) {
        *(f4v*)to = f4v{o[d][q4 * 4], o[d][q4 * 4 + 1], o[d][q4 * 4 + 2],
                        o[d][q4 * 4 + 3]};
        to += (size_t)nr * 8;
      }
    if (hh == 0) {
      pp[(size_t)HD * nr + at] = m;
      pp[(size_t)(HD + 1) * nr + at] = l;
    }
  }
}

#define AP_MAX_SPLIT 64
// the parts of a row, one wave a row
template <int HD>
__global__ void __launch_bounds__(256) k_attn_rows_merge(ApArgs a, int split) {
  const int lane = threadIdx.x & 63, grp = a.nh / a.kvh;
  const int nrows = a.M * grp;
  const int w = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (w >= nrows * a.kvh) return;
  const int kvhead = w / nrows, row = w % nrows;
  const size_t stride = (size_t)a.kvh * nrows * (HD + 4);
  const float* p = a.part + ((size_t)kvhead * nrows + row) * (HD + 4);
  // a lane a part: all maxima and sums in one trip, then eight parts a trip
  const int zl = min(lane, split - 1);
  const float mz = lane < split ? p[zl * stride + HD] : -INFINITY;
  const float lz = p[zl * stride + HD + 1];
  float m = mz;
#pragma unroll
  for (int w = 1; w < 64; w <<= 1) m = fmaxf(m, __shfl_xor(m, w));
  // a part without keys of this row holds nothing, one that weighs nothing
  // may hold values without a number
  const float al = mz == -INFINITY ? -1.f : __builtin_amdgcn_exp2f(mz - m);
  const float l = wave_reduce_sum(mz == -INFINITY ? 0.f : lz * al);
  float v[HD / 64];
#pragma unroll
  for (int i = 0; i < HD / 64; i++) v[i] = 0.f;
  for (int z0 = 0; z0 < split; z0 += 8) {
    float x[8][HD / 64];
#pragma unroll
    for (int z = 0; z < 8; z++)
#pragma unroll
      for (int i = 0; i < HD / 64; i++)
        x[z][i] = p[min(z0 + z, split - 1) * stride + i * 64 + lane];
#pragma unroll
    for (int z = 0; z < 8; z++) {
      const float w = __shfl(al, min(z0 + z, 63));
      if (z0 + z < split && !(w < 0.f))
#pragma unroll
        for (int i = 0; i < HD / 64; i++) v[i] += x[z][i] * w;
    }
  }
  u16* op = a.out + ((size_t)(row / grp) * a.nh + kvhead * grp + row % grp) * HD;
#pragma unroll
  for (int i = 0; i < HD / 64; i++) op[i * 64 + lane] = f2b(v[i] / l);
}

// The same of parts in lines: 16 rows of a kv head a block, a thread takes ND
// times four dims of a row.  All maxima and sums and the first eight parts are
// on the way together.
template <int HD>
__global__ void __launch_bounds__(256) k_attn_rows_merge_many(ApArgs a, int split) {
  constexpr int R = 16, ND = HD / 64, NG = 16;
  __shared__ float ms[AP_MAX_SPLIT][R], ls[AP_MAX_SPLIT][R];
  const int tid = threadIdx.x, r = tid % R, g = tid / R;
  const int grp = a.nh / a.kvh, kvhead = blockIdx.y, all = a.M * grp;
  const int row = blockIdx.x * R + r, at = min(row, all - 1);
  const ApPart part = ap_part<HD>(all);
  const size_t nr = part.rows, stride = a.kvh * part.size;
  const float* p = a.part + kvhead * part.size;
  for (int z = g; z < split; z += NG) {
    ms[z][r] = p[z * stride + HD * nr + at];
    ls[z][r] = p[z * stride + (HD + 1) * nr + at];
  }
  f4v x[8][ND], v[ND];
  auto ask = [&](int z0) {
#pragma unroll
    for (int z = 0; z < 8; z++)
#pragma unroll
      for (int i = 0; i < ND; i++)
        x[z][i] = *(const f4v*)(p + min(z0 + z, split - 1) * stride +
                                ((g + i * NG) * nr + at) * 4);
  };
  ask(0);
  __syncthreads();
  float m = -INFINITY, l = 0.f;
  for (int z0 = 0; z0 < split; z0 += 8)
#pragma unroll
    for (int z = 0; z < 8; z++) m = fmaxf(m, ms[min(z0 + z, split - 1)][r]);
#pragma unroll
  for (int i = 0; i < ND; i++) v[i] = {0.f, 0.f, 0.f, 0.f};
  for (int z0 = 0; z0 < split; z0 += 8) {
    if (z0) ask(z0);
#pragma unroll
    for (int z = 0; z < 8; z++) {
      // a part without keys of this row holds nothing, one that weighs nothing
      // may hold values without a number
      const float mz = ms[min(z0 + z, split - 1)][r];
      const float lz = ls[min(z0 + z, split - 1)][r];
      if (z0 + z >= split || mz == -INFINITY) continue;
      const float w = __builtin_amdgcn_exp2f(mz - m);
      l += lz * w;
#pragma unroll
      for (int i = 0; i < ND; i++) v[i] += x[z][i] * w;
    }
  }
  if (row >= all) return;
  u16* op = a.out + ((size_t)(row / grp) * a.nh + kvhead * grp + row % grp) * HD;
#pragma unroll
  for (int i = 0; i < ND; i++) {
    union { ap_b2 b[2]; unsigned long long u; } o;
#pragma unroll
    for (int j = 0; j < 4; j++) o.b[j / 2][j % 2] = (__bf16)(v[i][j] / l);
    *(unsigned long long*)(op + (g + i * NG) * 4) = o.u;
  }
}

template <int HD, int BKV, int NW, int KG, bool KV8>
static void ap_go(const ApArgs& a, dim3 grid, hipStream_t s) {
  if (a.softcap > 0.f)
    hipLaunchKernelGGL((k_attn_rows<HD, BKV, NW, KG, KV8, true>), grid,
                       dim3(64 * NW * KG), 0, s, a);
  else
    hipLaunchKernelGGL((k_attn_rows<HD, BKV, NW, KG, KV8, false>), grid,
                       dim3(64 * NW * KG), 0, s, a);
}

// Into how many ranges the keys are split where blocks are too few for 256
// CUs of two each (four of one wave).  A range more takes tiles off the
// longest block, and writes and reads a part more of every row; blocks that
// share a CU slow each other down.  The numbers are fitted to the times of
// 3660 calls at up to 16 splits each (11 head layouts, both pools, 1 to 1400
// rows behind 0 to 20000 keys, from memory).  Above each call's best split, on
// average where more rows than a tile make up to 64 blocks: 1.1% here, by four
// tiles a block at least, as it once was, or by one, 8.2% and 8.4%, since many
// rows' parts cost more than they save.  us by four tiles, by one tile, here:
//   head dim 128   5 rows of 24/8 heads over 905 keys  18.0 12.5 12.5
//     120 of 28/4 over 1020                            20.5 24.6 19.5
//     300 of 24/8 over 300                             14.2 20.0 14.2
//   256  300 of 16/8 over 430                          27.2 34.2 27.2
//   64   200 of 4/1 over 4200                          24.1 21.7 15.0
template <int HD, int BKV>
static int ap_split(const ApArgs& a, int kv8, int keys, long part_floats,
                    int most, int nw, int blocks) {
  const int want = nw == 1 ? 1024 : 512;
  if (blocks * 2 > want || !a.part) return 1;
  const int span = a.window > 0 && a.window + most < keys ? a.window + most
                                                          : keys;
  const int tiles = (span + BKV - 1) / BKV;
  const long each = (long)a.kvh * a.M * (a.nh / a.kvh) * (HD + 4);
  int cap = want / blocks < AP_MAX_SPLIT ? want / blocks : AP_MAX_SPLIT;
  if (cap > tiles) cap = tiles;
  if (cap > part_floats / each) cap = (int)(part_floats / each);
  // Where neither was slower before, it stays: beside e4m3 rounding parts of
  // other lengths are other values.  Few rows, a tile of them a kv head: a tile
  // of keys a block from four on.  More blocks: four tiles at least.
  if (blocks == a.kvh || blocks > 64) {
    int s = span / BKV;
    if (blocks > 64) s /= 4;
    else if (s < 4) s = 1;
    if (s > cap) s = cap;
    return s < 1 ? 1 : s;
  }
  // us of a tile, by one wave and by four, and how much longer with another
  // block on the CU; of a part that is a block's, and of a MB of them
  const float one = HD == 64 ? 0.76f : HD == 128 ? 2.58f : 1.73f;
  const float four = HD == 64 ? 0.82f : HD == 128 ? 1.04f : 0.95f;
  const float tile = (nw == 1 ? one : four) * (kv8 ? 1.78f : 1.f);
  const float more = nw == 1 ? 0.40f : 0.20f;
  const float mb = HD == 64 ? 0.50f : HD == 128 ? 0.30f : 0.20f;
  const float part = 0.042f + mb * (float)each * 4e-6f;
  int split = 1, last = 0;
  float best = 0.f;
  for (int s = 1; s == 1 || s <= cap; s++) {
    const int per = (tiles + s - 1) / s;
    if (per == last) continue;
    last = per;
    float t = per * tile * (1.f + more * ((blocks * s + 255) / 256 - 1));
    if (s > 1) t += 2.43f + part * s;
    if (s == 1 || t < best) {
      best = t;
      split = s;
    }
  }
  return split;
}

// Whether two groups of waves share a block's keys, rather than `split` ranges
// or one group alone.  By the tiles that the longest block goes through (under a
// window those of a block's rows and of the window) and by how many a CU gets,
// fitted to 26700 calls timed both ways: 17 head layouts, 65 to 512 blocks, 40
// to 2048 rows behind 0 to 8000 keys, windows, and two to eight sequences, a
// part of them behind keys of their own.  Above the better way 0.9% on average
// (never two groups 10.7%); 176 calls take 4% longer than by ranges whose parts
// were left row by row, the others up to 3.4 times less.
//   More blocks than CUs: of 64 dims (two such blocks fit a CU) from eight tiles
// on (8 prompts of up to 40 rows, 64/64 heads, 6.2 us by one group, 7.6); of 128 (one does)
// where blocks differ in length enough that the short ones fill what the long
// ones leave: few keys ahead of the rows (32/8 heads, 1999 rows 54.1 -> 49.6,
// behind 2000 keys 114 -> 118), and of several sequences, which may be short but
// for one, where the longest is long (8 of up to 40 rows, 40/40 heads, 7.6 by one
// group, 12.8 by two).
//   Up to a block a CU by numbers for what two groups take more: of one sequence
// and of several; each of 64 dims, 128, 128 beside e4m3.
// 64 dims of e4m3 (which spill) and more than 512 blocks were not measured.
template <int HD, int BKV>
static bool ap_two(const ApArgs& a, int kv8, int keys, int most, int blocks,
                   int split, bool several) {
  if (HD == 256 || (HD == 64 && kv8) || blocks <= 64 || blocks > 512)
    return false;
  const int grp = a.nh / a.kvh, own = (128 + grp - 1) / grp;
  const int span = a.window > 0 && a.window + own < keys ? a.window + own
                                                         : keys;
  const int tiles = (span + BKV - 1) / BKV, per = (tiles + split - 1) / split;
  const float mean = fminf(keys - 0.5f * most, span);
  const float all = blocks * mean / BKV / 256;
  if (blocks > 256) {
    if (HD == 64) return tiles >= 8;
    if (several) return tiles >= (kv8 ? 8 : 11);
    if (kv8) return tiles - 0.8f * all > 1.6f;
    return tiles - all > 4.f && 2 * (keys - most) < most;
  }
  // parts of the rows, MB
  const float mb = split > 1 ? (float)a.M * a.nh * (HD + 4) * 4e-6f : 0.f;
  static const float fit[6][5] = {
      {0.646f, -0.329f, -0.907f, -0.518f, -0.39f},
      {0.563f, -0.0799f, -0.821f, -1.42f, -0.162f},
      {1.49f, -0.152f, -2.22f, -1.71f, -0.372f},
      {0.212f, 0.0593f, -0.421f, -0.567f, -0.158f},
      {0.186f, -0.0126f, -0.233f, -1.14f, -0.0603f},
      {0.397f, 0.121f, -0.842f, 0.397f, -0.133f}};
  const float* f = fit[several * 3 + (HD == 64 ? 0 : kv8 ? 2 : 1)];
  return 1.f + f[0] * tiles + f[1] * all + f[2] * per + f[3] * (split > 1) +
             f[4] * split * mb < 0.f;
}

// How a call runs: waves that share a tile of rows, such tiles, ranges of keys,
// whether two groups of waves share a block's.  most: rows of the longest
// sequence; ntiles: of several sequences.
struct ApPlan { int nw, tiles, split; bool two, by_row; };
template <int HD, int BKV>
static ApPlan ap_plan(const ApArgs& a, int kv8, int keys, long part_floats,
                      int most, int ntiles) {
  const int rows = a.M * (a.nh / a.kvh);
  // up to 32 rows are one wave's; more share their tiles among four
  const int nw = most * (a.nh / a.kvh) <= 32 ? 1 : 4;
  const int tiles = ntiles ? ntiles : (rows + nw * 32 - 1) / (nw * 32);
  const int split = ap_split<HD, BKV>(a, kv8, keys, part_floats, most, nw,
                                      tiles * a.kvh);
  const bool two = nw == 4 && ap_two<HD, BKV>(a, kv8, keys, most,
                                              tiles * a.kvh, split, ntiles);
  // Many parts of few rows lie row by row: a wave adds those of one row, where
  // 16 rows a block would leave most CUs without any (us, so / in lines: 64 dims,
  // 16 parts of 256 rows 13.6 / 16.1, 8 of 256 10.9 / 11.2, of 4096 -4%, 4 parts
  // of 256 -1%, of 4096 -6%; 8000 calls)
  return {nw, tiles, two ? 1 : split, two,
          nw == 1 || (split >= 8 && (long)rows * a.kvh < 128 * split)};
}

template <int HD, int BKV>
static hipError_t ap_run(ApArgs a, int kv8, const ApPlan& plan,
                         hipStream_t s) {
  const auto [nw, tiles, split, two, by_row] = plan;
  const int rows = a.M * (a.nh / a.kvh);
  a.by_row = by_row;
  // A block a CU, then the second of each (two groups of 128 dims have a CU to
  // themselves).  us, longest first -> so: 64 dims 1999 rows of 32/8 heads 32.4
  // -> 29.9, 2000 behind 2000 keys 72.3 -> 68.0; 128 dims 54.1 -> 52.3.
  a.fold = tiles;
  if (!a.tiles && split == 1 && tiles * a.kvh <= 512 && !(two && HD == 128))
    a.fold = a.kvh < 256 ? 256 / a.kvh : 1;
  dim3 grid(a.kvh, tiles, split);
  if (nw == 1) {
    if (kv8) ap_go<HD, BKV, 1, 1, true>(a, grid, s);
    else ap_go<HD, BKV, 1, 1, false>(a, grid, s);
  } else if (two) {
    if constexpr (HD == 128)
      if (kv8) ap_go<HD, BKV, 4, 2, true>(a, grid, s);
    if constexpr (HD <= 128)
      if (!kv8) ap_go<HD, BKV, 4, 2, false>(a, grid, s);
  } else {
    if (kv8) ap_go<HD, BKV, 4, 1, true>(a, grid, s);
    else ap_go<HD, BKV, 4, 1, false>(a, grid, s);
  }
  if (split > 1 && by_row)
    hipLaunchKernelGGL((k_attn_rows_merge<HD>), dim3((rows * a.kvh + 3) / 4),
                       dim3(256), 0, s, a, split);
  else if (split > 1)
    hipLaunchKernelGGL((k_attn_rows_merge_many<HD>),
                       dim3((rows + 15) / 16, a.kvh), dim3(256), 0, s, a,
                       split);
  return hipGetLastError();
}

// Counts that a call can have; heads, rows and their parts are divided by.
static bool ap_takes(int M, int nh, int kvh, bool several, int most,
                     int ntiles) {
  return M > 0 && nh > 0 && kvh > 0 && nh % kvh == 0 &&
         (!several || (ntiles > 0 && most > 0));
}

// keys: number of keys that the last row sees, as far as the host knows
// (a hint for the split; the kernel goes by *len_ptr).  tiles: M rows of
// several sequences, the longest of `most` rows; a tile has 32 rows times
// heads of a kv head where that is all of the longest, else 128.
extern "C" hipError_t launch_attn_prefill_mfma(
    const void* q, const void* kc, const void* vc, void* out,
    const void* len_ptr, const void* tiles, const void* kS, const void* vS,
    void* part,
    long part_floats, int kv8, int M, int nh, int kvh, int hd, int ldq,
    int S, int keys, int most, int ntiles, float scale, float softcap,
    int window, hipStream_t stream) {
  if (!ap_takes(M, nh, kvh, tiles, most, ntiles) || ldq < nh * hd || ldq % 8)
    return hipErrorInvalidValue;
  if (!tiles) {
    most = M;
    ntiles = 0;
  }
  ApArgs a = {(const u16*)q, kc, vc, (u16*)out, (const int*)len_ptr,
              (const int*)tiles,
              (const float*)kS, (const float*)vS, (float*)part, M, nh, kvh,
              ldq, S, 0, 0, scale, softcap, window};
  if (hd == 64)
    return ap_run<64, 64>(
        a, kv8, ap_plan<64, 64>(a, kv8, keys, part_floats, most, ntiles),
        stream);
  if (hd == 128)
    return ap_run<128, 64>(
        a, kv8, ap_plan<128, 64>(a, kv8, keys, part_floats, most, ntiles),
        stream);
  if (hd == 256)
    return ap_run<256, 32>(
        a, kv8, ap_plan<256, 32>(a, kv8, keys, part_floats, most, ntiles),
        stream);
  return hipErrorInvalidValue;
}

// How such a call runs, on the host alone: ranges of keys, whether two groups of
// waves share a block's, whether parts lie row by row.  1: counts or a head dim
// that the launch refuses.
extern "C" int attn_prefill_plan(int kv8, int M, int nh, int kvh, int hd,
                                 int keys, int most, int ntiles, int window,
                                 long part_floats, int* out) {
  if (!ap_takes(M, nh, kvh, ntiles, most, ntiles) ||
      (hd != 64 && hd != 128 && hd != 256))
    return 1;
  ApArgs a = {};
  a.M = M;
  a.nh = nh;
  a.kvh = kvh;
  a.window = window;
  a.part = part_floats > 0 ? (float*)out : nullptr;      // is there or not
  if (!ntiles) most = M;
  const ApPlan p =
      hd == 64 ? ap_plan<64, 64>(a, kv8, keys, part_floats, most, ntiles)
      : hd == 128 ? ap_plan<128, 64>(a, kv8, keys, part_floats, most, ntiles)
                  : ap_plan<256, 32>(a, kv8, keys, part_floats, most, ntiles);
  out[0] = p.split;
  out[1] = p.two;
  out[2] = p.by_row;
  return 0;
}
