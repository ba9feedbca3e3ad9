// chain.hip — the products between two attentions of one row in one launch:
// W_o, gate and up, W_down, and the next layer's q, k and v, or the head.
//
// A launch of its own costs each of them 3 to 4 us in which no weights move:
// the dispatch, x and its norm, the first loads, the last rows.  Here the
// weights never stop: a block's loader waves fill rings in LDS by DMA and run
// ahead into the next product while its x is still being computed, so what is
// left between two products is the way of x from block to block.
//
// A block of 12 waves on each CU:
//   4 that multiply: four rows at a time, a KB of each, off their ring; the
//     waves share out K, or rows, whichever leaves fewer rounds;
//   4 that load, one for each of these;
//   4 that bring x (the norm's weights on the way) and finish the outputs.
// They meet at counters in LDS.  A norm's factor is a number for all of x and
// comes in behind the product, so no one waits for a sum over x.
//
// From block to block there is neither a counter nor a fence (an arrival at a
// counter takes 25 ns, one after the other): outputs go past the L2 into
// memory that was filled with ones before the step, which no value is made
// of, and who needs them reads until none is left.  Every word is written
// once a step, so no reader meets an old one.
//
// All 256 blocks need not run at once.  Another stream's kernels may hold CUs,
// and a block that waits for one that cannot start would hold its own for
// nothing.  So each block has a word (`claims`) and marks there that it has
// started; waves that wait in vain for `limit` take over a block that has not,
// a quarter of its rows each, for all products (ch_unit), and it does nothing
// where it starts at last.  What has started waits for nothing that has not, so
// the launch ends whatever else holds CUs.  (Beside that, waves whose patience
// is at an end compute what is missing of anyone's.)
// It waits a while first, and as long as blocks still start or fewer than half
// have: CUs come free as others' blocks end, and of two launches of this kind
// that hold some each, one is to go on.  ms for 200 tokens of a 1B model, alone
// 117: beside prompts of 2000 rows on another stream 460 (each product in a
// launch of its own 555; where waves that waited computed whatever was missing,
// many of them the same, 3150), beside another model's decode 230 to 280 (198;
// 420 to 890).  With half of its blocks gone a launch of 26 us takes 150.
//
// Routed experts are products like the others, of weights that are known once
// the router has chosen: every block dots its x with the router as it brings
// it, and its loaders wait for the choice, not for a launch of the router's
// own.  Up to eight experts: their router rows stand in registers ahead of x.
// W_o, router, gate and up, down, q, k and v, five launches -> here, us:
//   2048 wide, two of 4096, bf16 39.5 -> 34.8, e4m3 35.1 -> 30.6
//   4096, two of 14336, bf16 144 -> 129, e4m3 90.2 -> 80.7
// (Of the first, x of both down products brought at once 34.6; x of one
// brought while the last is multiplied 35.3, as a read past the L2 takes 3 to
// 5 us while weights stream.)
//
// Behind the head, the largest logit of each wave's share goes to memory too,
// for a sampler that need not look for it (k_sample_pick).
//
// What is in flight is kept small: what x needs queues behind it.  us for a
// layer's four products, four launches -> here (weights cold):
//   2048 wide, 8192 in the middle, bf16        32.9 -> 25.7, e4m3 25.5 -> 20.5
//   3072, 8192, bf16                           47.3 -> 36.5, MXFP4 28.0 -> 24.3
//   4096, 14336, bf16 83.7 -> 76.3 (5.7 TB/s), e4m3 51.7 -> 46.5, MXFP4 39.3 -> 31.7
//   2304, 9216, bf16, two norms                40.2 -> 35.5
//   3584, 14336, e4m3, two norms               48.2 -> 43.6
//   3584, 18944, e4m3                          55.6 -> 50.5
// Of the first: two slots of a loader in flight ahead of the newest 28.1,
// weights kept in the caches 27.3, x read 8 bytes a lane 28.3, in copies for
// each die 29.1, eight waves that multiply 29.4.  With no x to wait for its
// weights alone take 17.3 (7 TB/s): a hand-over is 2 to 3 us from the last
// block's sums to the next product's first, and the rings hold 4 us.
//
// The waves that bring x have one way through: a return where others have the
// block's rows, out of their reads or ahead of an output, cost each launch 0.5
// us and 0.4 to 0.9; with the standing in in the same loop as the products it
// was 2 to 3, out of line 0.3 to 2.5.
#include <type_traits>

#include "common.h"
#include "gemv.h"

typedef unsigned long long ch_u8;
typedef __bf16 ch_b2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) uint32_t* ch_lp;
#define CH_LDS_OF(T) const __attribute__((address_space(3))) T
#define CH_VOL(T) volatile __attribute__((address_space(3))) T

enum { CH_RAW = 0, CH_NORM = 1, CH_NORM2 = 2 };
#define CH_MAX 6                           // products of a launch
#define CH_TOP 2                           // experts of a row, at most
#define CH_TOPS (CH_BLOCKS * CH_NS)
#define CH_EXPERTS 8                       // to choose from
#define CH_BLOCKS 256
#define CH_NC 4                            // waves: multiply, load, bring x
#define CH_NL CH_NC
#define CH_NS 4
#define CH_NT (64 * CH_NS)
// The longest row that is normed.  Its pieces are in registers until the sum of
// squares is there, with the norm's weights and, behind two norms, the stream's
// and theirs: two pieces a thread.  Four (4608, 8192 wide) were not built.
#define CH_NORM_K (2 * 8 * CH_NT)
#define CH_SLOTS 8                         // of a ring, at most
#define CH_MINOR 64                        // looks in vain while fewer than half have
#define CH_PATIENCE 1024                   // and of all
#define CH_QUIT (1 << 30)                  // in the counters of a block that ends
// A block's word, of which bits go as things happen: it has started; another
// has its rows; the host's own, its rows are for others.
#define CH_STARTED 1u
#define CH_GIVEN 2u
#define CH_ABSENT 4u
#define CH_LDS (160 * 1024 - 4096)         // 4 KB beside it

// A product as the caller gives it.  What is marked (*) is read until it is
// there; such words held ones before the step.
struct ChStage {
  const void* w;         // [N, K], with a gate [2N, K]: gate, then up
  const float* ws;       // e4m3: scales of rows
  const uint8_t* we;     // MXFP4: exponents [rows, K/32]
  const void* x;         // bf16 or fp32; with wait (*)
  const u16* h;          // NORM2: the stream; null: what the last one left
  const float* g;        // weights of the norm; NORM2: of the first,
  const float* g2;       //   of the second
  const u16* add;        // bias or residual; own: y of an earlier product
  void* y;
  u16* hout;             // NORM2: the stream behind it, or null
  int N, K, kind, x_f32, wait, glu, y_f32, own;
  float softcap;         // of the outputs, or 0
  // Routed experts.  slot 1 .. CH_TOP: the product of one that was chosen, W
  // and ws of expert e wstep bytes and sstep floats on; scaled: its result by
  // its weight.  route, with slot 1: the router [experts, K] in bf16, dotted
  // with the normed x; `top` are chosen.  same: x is what the last product
  // had.  add2: y, in fp32, of the product before this one.
  int slot;
  const u16* route;
  const float* add2;
  long wstep, sstep;
  int scaled, same, experts, top;
  float* tops;           // the largest output of each wave's, CH_TOPS of them
};
// and how it is shared out
struct ChStep {
  ChStage s;
  int rpb, kwl, cols, groups, ngate, ng, keep, pad;
};
struct ChArgs {
  ChStep st[CH_MAX];
  int n, act, total, slots, xbytes, hbytes, rbytes, limit;
  float eps;
  uint32_t* claims;      // CH_BLOCKS words that held ones, or null
};

DEVINL int ch_s(int v) { return __builtin_amdgcn_readfirstlane(v); }
template <class T> DEVINL T* ch_p(T* p) {
  const ch_u8 u = (ch_u8)p;
  return (T*)((ch_u8)(uint32_t)ch_s((int)u) |
              (ch_u8)(uint32_t)ch_s((int)(u >> 32)) << 32);
}
// Counters in LDS, by hand: beside loads into LDS the compiler waits for all
// of these first.
DEVINL int ch_get(ch_lp p) {
  uint32_t v;
  asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)"
               : "=v"(v) : "v"(p) : "memory");
  return ch_s((int)v);
}
DEVINL void ch_set(ch_lp p, uint32_t v) {
  asm volatile("ds_write_b32 %0, %1" :: "v"(p), "v"(v) : "memory");
}
DEVINL void ch_done(ch_lp p, int lane) {   // one more wave, its LDS behind it
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  if (lane == 0)
    asm volatile("ds_add_u32 %0, %1" :: "v"(p), "v"(1u) : "memory");
}
// until n have; whether the block goes on
template <int NAP> DEVINL bool ch_wait(ch_lp p, int n) {
  int v;
  while ((v = ch_get(p)) < n) __builtin_amdgcn_s_sleep(NAP);
  return v < CH_QUIT;
}
template <int N> DEVINL void ch_arrived() {
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory");
}

DEVINL ch_u8 ch_word(const void* p) {
  return __hip_atomic_load((const ch_u8*)p, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
}
// 16 bytes of x past the L2 (sc1, as that load has it; each value in them is
// looked at by itself, so they need not be of one moment)
DEVINL u4v_ ch_fresh(__amdgpu_buffer_rsrc_t r, int at) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, 16);
}
template <bool F32> DEVINL bool ch_there(u4v_ v) {
  bool all = true;
#pragma unroll
  for (int k = 0; k < 4; k++)
    all = all && (F32 ? v[k] != ~0u
                      : v[k] < 0xffff0000u && (v[k] & 0xffffu) != 0xffffu);
  return all;
}
DEVINL float ch_value(const void* y, int f32, int n, bool* there) {
  if (f32) {
    const uint32_t v = __hip_atomic_load((const uint32_t*)y + n,
                                         __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
    *there = v != ~0u;
    return __uint_as_float(v);
  }
  const u16 v = __hip_atomic_load((const u16*)y + n, __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT);
  *there = v != 0xffff;
  return b2f(v);
}
DEVINL void ch_put(void* y, int f32, int n, float v) {
  // a NaN is never all ones (f2b makes its own)
  if (f32)
    __hip_atomic_store((uint32_t*)y + n,
                       v != v ? 0x7fc00000u : __float_as_uint(v),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else
    __hip_atomic_store((u16*)y + n, f2b(v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
DEVINL f4v ch_quad(uint32_t a, uint32_t b) {    // four bf16
  return f4v{__uint_as_float(a << 16), __uint_as_float(a & 0xffff0000u),
             __uint_as_float(b << 16), __uint_as_float(b & 0xffff0000u)};
}
DEVINL f4v ch_quad(ch_u8 v) { return ch_quad((uint32_t)v, (uint32_t)(v >> 32)); }
DEVINL ch_u8 ch_pack(f4v v) {
  return (ch_u8)(f2b(v[0]) | (uint32_t)f2b(v[1]) << 16) |
         (ch_u8)(f2b(v[2]) | (uint32_t)f2b(v[3]) << 16) << 32;
}
// the same for x in LDS, by the unit's own conversion
DEVINL ch_u8 ch_pack_x(f4v v) {
  union { __bf16 b[4]; ch_u8 u; } r;
#pragma unroll
  for (int k = 0; k < 4; k++) r.b[k] = (__bf16)v[k];
  return r.u;
}
DEVINL float ch_squares(f4v a, f4v b) {
  return a[0] * a[0] + a[1] * a[1] + a[2] * a[2] + a[3] * a[3] +
         (b[0] * b[0] + b[1] * b[1] + b[2] * b[2] + b[3] * b[3]);
}

// Adds to R rows' sums a 16-byte piece of each times x: bf16 as it is (xb),
// else fp32.  Row by row the same bits whatever R is.
template <int WT, int R>
DEVINL void ch_dot(const u4v_* w, u4v_ xb, const f4v* x, const uint32_t* e,
                   bool in, float* acc) {
  float p[R], o[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    p[r] = acc[r];
    o[r] = 0.f;
  }
#pragma unroll
  for (int d = 0; d < 4; d++)
#pragma unroll
    for (int r = 0; r < R; r++) {
      const uint32_t v = w[r][d];
      if constexpr (WT == GV_BF16) {
        union { uint32_t u; ch_b2 b; } s = {v}, t = {xb[d]};
        p[r] = __builtin_amdgcn_fdot2_f32_bf16(s.b, t.b, p[r], false);
      } else if constexpr (WT == GV_FP8) {
        const f2v l = __builtin_amdgcn_cvt_pk_f32_fp8(v, false);
        const f2v h = __builtin_amdgcn_cvt_pk_f32_fp8(v, true);
        p[r] += l[0] * x[d][0];
        o[r] += l[1] * x[d][1];
        p[r] += h[0] * x[d][2];
        o[r] += h[1] * x[d][3];
      } else {
        const float s = __uint_as_float(e[r] << 23);
        const f2v t[4] = {__builtin_amdgcn_cvt_scalef32_pk_f32_fp4(v, s, 0),
                          __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(v, s, 1),
                          __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(v, s, 2),
                          __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(v, s, 3)};
#pragma unroll
        for (int i = 0; i < 4; i++) {
          p[r] += t[i][0] * x[d * 2 + i / 2][i % 2 * 2];
          o[r] += t[i][1] * x[d * 2 + i / 2][i % 2 * 2 + 1];
        }
      }
    }
#pragma unroll
  for (int r = 0; r < R; r++) {
    if constexpr (WT != GV_BF16) p[r] += o[r];
    acc[r] = in ? p[r] : acc[r];           // nothing behind the row's end
  }
}

// An output from its sums, on either way
template <int WT>
DEVINL float ch_finish(const ChStage& s, int act, float v, float up, float rn,
                       float s1, float s2, float add, float scale = 1.f) {
  const float cap = s.softcap;
  v *= rn;
  if constexpr (WT == GV_FP8) v *= s1;
  v *= scale;
  if (s.glu) {
    up *= rn;
    if constexpr (WT == GV_FP8) up *= s2;
    v = gate_act(v, act) * up;
  }
  if (cap > 0.f) v = cap * tanhf(v / cap);
  return v + add;
}

// Rows of product t that are quarter q of block b's, by one wave: every 16 rows
// four of them, in the order of sums of the waves that multiply, so the same
// bits.  r1 and rn: the factors of its norms.  hs: the last product's stream,
// where it stands in LDS alone.  look: only what is not there yet.
template <int WT>
DEVINL void ch_unit(CH_LDS_OF(ChStep)* st, int t, int b, int q, int lane,
                    int act, float r1, float rn, CH_LDS_OF(int)* eid,
                    CH_LDS_OF(float)* ew, CH_LDS_OF(char)* hs, bool look) {
  constexpr int E = gv_e<WT>(), Q = E / 4;
  ChStep p;
  uint32_t words[sizeof(p) / 4];
  for (int i = 0; i < (int)sizeof(p) / 4; i++)
    words[i] = ch_s(((CH_LDS_OF(uint32_t)*)(st + t))[i]);
  __builtin_memcpy(&p, words, sizeof(p));
  const ChStage& s = p.s;
  const int K = s.K, N = s.N, rpb = p.rpb, kwl = p.kwl;
  const int P = K / E, kind = s.kind;
  const int n0 = b * rpb, nn = min(rpb, N - n0);
  const bool glu = s.glu, f32 = s.x_f32;
  // whoever is at a product behind the router's has its choice
  const int ex = s.slot ? ch_s(eid[s.slot - 1]) : 0;
  const float scale = s.scaled ? ew[s.slot - 1] : 1.f;
  const char* const W = (const char*)s.w + ex * s.wstep;
  const float* const ws = WT == GV_FP8 ? s.ws + ex * s.sstep : nullptr;
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      (void*)s.x, 0, K * (f32 ? 4 : 2), 0x00027000);
  // quads 2i and 2i + 1 of x, by its norm but for the factor behind the product
  auto pair = [&](int i, f4v* v, bool stream) {
    if (f32) {
      union { u4v_ u; f4v f; } a = {ch_fresh(xr, i * 32)},
                               c = {ch_fresh(xr, i * 32 + 16)};
      v[0] = a.f;
      v[1] = c.f;
      return;
    }
    if (kind == CH_NORM2 && !s.h) {        // behind its first norm
      const u4v_ h = *(CH_LDS_OF(u4v_)*)(hs + i * 16);
      v[0] = ch_quad(h[0], h[1]);
      v[1] = ch_quad(h[2], h[3]);
    } else {
      const u4v_ a = ch_fresh(xr, i * 16);
      v[0] = ch_quad(a[0], a[1]);
      v[1] = ch_quad(a[2], a[3]);
      if (kind == CH_NORM2) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
          const f4v h = ch_quad(*(const ch_u8*)(s.h + i * 8 + j * 4));
          const f4v g = *(const f4v*)(s.g + i * 8 + j * 4);
#pragma unroll
          for (int k = 0; k < 4; k++)
            v[j][k] = b2f(f2b(v[j][k] * r1 * g[k] + h[k]));
        }
      }
    }
    if (kind == CH_RAW || stream) return;
    const float* const g = kind == CH_NORM2 ? s.g2 : s.g;
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const f4v m = *(const f4v*)(g + i * 8 + j * 4);
#pragma unroll
      for (int k = 0; k < 4; k++) v[j][k] *= m[k];
    }
  };
  if (b == 0 && s.hout)
    for (int i = q * 64 + lane; i < K / 8; i += 256) {
      f4v v[2];
      pair(i, v, true);
      *(ch_u8*)(s.hout + i * 8) = ch_pack(v[0]);
      *(ch_u8*)(s.hout + i * 8 + 4) = ch_pack(v[1]);
    }
  float most = -INFINITY;
  for (int r0 = q * 4; r0 < nn; r0 += 4 * CH_NS) {
    const int n = n0 + r0 + lane;
    const bool mine = lane < 4 && r0 + lane < nn;
    if (look) {
      bool there = true;
      if (mine) ch_value(s.y, s.y_f32, n, &there);
      if (__all(there)) continue;
    }
    // U columns on their way at a time: a read past the L2 takes some 6 us while
    // weights stream (200 tokens of 1B bf16 beside another stream's prompts 446
    // ms, a column at a time 472; e4m3 alike)
    constexpr int U = WT == GV_BF16 ? 4 : WT == GV_FP8 ? 1 : 2;
    float v = 0.f, up = 0.f;
    for (int side = 0; side <= glu; side++) {
      float sum = 0.f;
      for (int kw = 0; kw < 1 << kwl; kw++) {
        float acc[4] = {};
        for (int cc = 0; cc < p.cols; cc += U) {
          f4v x[U][Q];
          u4v_ w[U][4];
          uint32_t e[U][4] = {};
#pragma unroll
          for (int j = 0; j < U; j++) {
            const int at = min((((cc + j) << kwl) + kw) * 64 + lane, P - 1);
#pragma unroll
            for (int r = 0; r < 4; r++) {
              const size_t row = n0 + min(r0 + r, nn - 1) + (side ? N : 0);
              w[j][r] = __builtin_nontemporal_load(
                  (const u4v_*)(W + row * P * 16) + at);
              if constexpr (WT == GV_FP4) e[j][r] = s.we[row * P + at];
            }
#pragma unroll
            for (int i = 0; i < Q; i += 2)
              pair(at * (Q / 2) + i / 2, x[j] + i, false);
          }
#pragma unroll
          for (int j = 0; j < U; j++) {    // nothing behind the row's end
            u4v_ xb = {};
            if constexpr (WT == GV_BF16) {
              union { ch_u8 u[2]; u4v_ v; } o = {
                  {ch_pack_x(x[j][0]), ch_pack_x(x[j][1])}};
              xb = o.v;
            }
            ch_dot<WT, 4>(w[j], xb, x[j], e[j],
                          (((cc + j) << kwl) + kw) * 64 + lane < P, acc);
          }
        }
        sum += gv_rows<4>(acc, lane);
      }
      (side ? up : v) = sum;
    }
    if (!mine) continue;
    float add = 0.f, s1 = 1.f, s2 = 1.f;
    bool yes;                              // own: bf16, add2: fp32
    if (s.add) add = s.own ? ch_value(s.add, 0, n, &yes) : b2f(s.add[n]);
    if (s.add2) add += ch_value(s.add2, 1, n, &yes);
    if (WT == GV_FP8) {
      s1 = ws[n];
      if (glu) s2 = ws[N + n];
    }
    const float o = ch_finish<WT>(s, act, v, up, rn, s1, s2, add, scale);
    ch_put(s.y, s.y_f32, n, o);
    most = fmaxf(most, o);
  }
  if (s.tops) {
    most = wave_reduce_max(most);
    if (lane == 0) s.tops[b * CH_NS + q] = most;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// A block that has not started, for good, or -1; while fewer than half have, -1
// but for `any`: then another launch of the kind may have most CUs, and it is
// better that one of the two goes on.  Ends: each turn that fails has seen a bit
// of a word go.
DEVINL int ch_adopt(uint32_t* claims, int lane, bool any, int* seen) {
  for (;;) {
    uint32_t w[4], free = 0;
    int cared = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      w[k] = __hip_atomic_load(claims + lane * 4 + k, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
      if ((w[k] & CH_GIVEN) && ((w[k] & CH_STARTED) || !(w[k] & CH_ABSENT)))
        free |= 1u << k;
      cared += __builtin_popcountll(__ballot((w[k] & (CH_STARTED | CH_GIVEN)) !=
                                             (CH_STARTED | CH_GIVEN)));
    }
    const ch_u8 some = __ballot(free != 0);
    const bool more = cared > *seen;       // blocks still come
    *seen = cared;
    if (!some || (!any && (more || cared < CH_BLOCKS / 2))) return -1;
    // every block from another place on
    const int l0 = blockIdx.x >> 2, k0 = blockIdx.x & 3;
    const int l = (__builtin_ctzll(some >> l0 | some << (-l0 & 63)) + l0) & 63;
    const uint32_t f = __builtin_amdgcn_readlane(free, l);
    const int k = (__builtin_ctz((f >> k0 | f << (4 - k0)) & 15) + k0) & 3;
    bool got = false;
    if (lane == l) {
      uint32_t old = k == 0 ? w[0] : k == 1 ? w[1] : k == 2 ? w[2] : w[3];
      got = __hip_atomic_compare_exchange_strong(
          claims + lane * 4 + k, &old, old & ~CH_GIVEN, __ATOMIC_RELAXED,
          __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (__ballot(got)) return l * 4 + k;
  }
}

// a product as a block's loaders and multipliers see it
struct ChCur {
  const char* w;         // first row of the block
  const char* we;
  int N, P, C, rpb, nn, kwl, cols, groups, ngate, ng;
};
template <bool MOE = false>
DEVINL ChCur ch_take(const ChStep* st, int i, int wt, const int* eid = nullptr) {
  const ChStep* q = st + i;
  ChCur c;
  const int K = ch_s(q->s.K), E = 8 << wt, rpb = ch_s(q->rpb);
  c.N = ch_s(q->s.N);
  c.P = K / E;
  c.C = (c.P + 63) / 64;
  c.rpb = rpb;
  // a block without rows of its own sees the last one again
  const int n0 = min((int)blockIdx.x * rpb, c.N - 1);
  c.nn = min(rpb, c.N - n0);
  c.w = ch_p((const char*)q->s.w) + (size_t)n0 * c.P * 16;
  if (MOE && ch_s(q->s.slot))
    c.w += (size_t)ch_s(eid[ch_s(q->s.slot) - 1]) * q->s.wstep;
  c.we = ch_p((const char*)q->s.we) + (size_t)n0 * (K / 32);
  c.kwl = ch_s(q->kwl);
  c.cols = ch_s(q->cols);
  c.groups = ch_s(q->groups);
  c.ngate = ch_s(q->ngate);
  c.ng = ch_s(q->ng);
  return c;
}
// the g-th four rows of a wave: the first, and whether they are up rows
DEVINL int ch_rows(const ChCur& c, int g, int wave, bool* up) {
  const int G = min(g * (CH_NC >> c.kwl) + (wave >> c.kwl), c.ng - 1);
  *up = G >= c.ngate;
  return (G - (*up ? c.ngate : 0)) * 4;
}

template <int WT, bool MOE>
__global__ void __launch_bounds__(64 * (CH_NC + CH_NL + CH_NS))
k_chain(ChArgs a) {
  constexpr int E = gv_e<WT>(), Q = E / 4;
  constexpr int SLOT = WT == GV_FP4 ? 4096 + 256 : 4096;
  constexpr int LD = WT == GV_FP4 ? 5 : 4; // loads of a slot
  __shared__ ChStep st[CH_MAX];
  __shared__ float ssq[4][CH_NS], own[CH_NT];
  __shared__ uint32_t full[CH_NC], freed[CH_NC], xcnt, scnt, sub;
  // it stays; products whose norms are there; blocks taken over, whether all
  __shared__ uint32_t stays, ncnt, nothers, closed;
  __shared__ float norms[CH_MAX][2];         // factors of each product's
  __shared__ uint8_t others[CH_BLOCKS];
  // routed experts: the router's sums, the choice, what add2 is
  __shared__ float rsum[MOE ? CH_NS : 1][CH_EXPERTS], ew[CH_TOP];
  __shared__ float own2[MOE ? CH_NT : 1];
  __shared__ int eid[CH_TOP];
  __shared__ uint32_t dots, routed;
  // x | the stream | sums [row][wave] | rings
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = ch_s(tid >> 6);
  char* const xs = lds;
  char* const hs = xs + a.xbytes;
  float* const red = (float*)(hs + a.hbytes);
  char* const ring = hs + a.hbytes + a.rbytes;

  if (tid < CH_NC) full[tid] = freed[tid] = 0;
  if (tid == 0) xcnt = scnt = sub = stays = ncnt = nothers = closed = dots = routed = 0;
  {
    typedef const __attribute__((address_space(4))) uint32_t* kp;
    const kp from = (kp)__builtin_amdgcn_kernarg_segment_ptr();
    for (int i = tid; i < (int)sizeof(st) / 4; i += blockDim.x)
      ((uint32_t*)st)[i] = from[i];
  }
  __syncthreads();

  if (wave < CH_NC) {                      // ---- multiply
    const ch_lp fullp = (ch_lp)&full[wave], freep = (ch_lp)&freed[wave];
    int at = 0, have = 0, u = 0;           // slot, slots told, rounds
    // looked at behind the first product (a read past the L2 ahead of x, by
    // the waves that bring it, held each launch up by 2 us)
    uint32_t word = ~0u;
    if (a.claims && tid == 0)
      word = __hip_atomic_fetch_and(a.claims + blockIdx.x, ~CH_STARTED,
                                    __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    auto multiply = [&](const ChCur& c) {
      const int kw = wave & ((1 << c.kwl) - 1);
      for (int g = 0; g < c.groups; g++) {
        float acc[4] = {};
        for (int cc = 0; cc < c.cols; cc++) {
          while (have <= u) {
            have = ch_get(fullp);
            if (have <= u) __builtin_amdgcn_s_sleep(1);
          }
          const int col = (cc << c.kwl) + kw;
          const char* x0 = xs + min(col, c.C - 1) *
                                (WT == GV_BF16 ? 1024 : 256 * E) + lane * 16;
          const char* sl = ring + (wave * a.slots + at) * SLOT;
          if (++at == a.slots) at = 0;
          u4v_ w[4], xb = {};
          f4v x[Q];
          uint32_t e[4] = {};
          if constexpr (WT == GV_BF16) {
            xb = *(const u4v_*)x0;
          } else {
#pragma unroll
            for (int k = 0; k < Q; k++) x[k] = *(const f4v*)(x0 + k * 1024);
          }
#pragma unroll
          for (int r = 0; r < 4; r++) {
            w[r] = *(const u4v_*)(sl + r * 1024 + lane * 16);
            if constexpr (WT == GV_FP4)
              e[r] = *(const uint8_t*)(sl + 4096 + r * 64 + lane);
          }
          ch_set(freep, ++u);              // LDS keeps a wave's order
          ch_dot<WT, 4>(w, xb, x, e, col * 64 + lane < c.P, acc);
        }
        const float s = gv_rows<4>(acc, lane);
        bool up;
        const int r0 = ch_rows(c, g, wave, &up);
        if (lane < 4 && r0 + lane < c.rpb)
          red[((up ? c.rpb : 0) + r0 + lane) * CH_NC + kw] = s;
      }
      ch_done((ch_lp)&scnt, lane);
    };
    // A wave that has waited for long goes on below: what it does for others
    // has registers of its own there (in one loop with the products it cost
    // each launch 2 to 3 us).
    int i = 0;
    for (; i < a.n; i++) {
      const ChCur c = ch_take(st, i, WT);
      // The block's rows are another's: multipliers and loaders end, and the
      // others go through what is left without waiting or writing.  All
      // counters say so, what the former look at behind what the latter do.
      if (i == 1 && wave == 0) {
        if (~ch_s((int)word) & (CH_GIVEN | CH_ABSENT)) {
          if (lane < a.n) {                // what waits and writes besides
            st[lane].s.wait = 0;
            st[lane].s.hout = nullptr;
            st[lane].s.tops = nullptr;
          }
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          ch_set((ch_lp)&scnt, CH_QUIT);
          ch_set((ch_lp)&sub, CH_QUIT);
          ch_set((ch_lp)&dots, CH_QUIT);
          ch_set((ch_lp)&routed, CH_QUIT);
          ch_set((ch_lp)&xcnt, CH_QUIT);
          return;
        }
        ch_set((ch_lp)&stays, 1);
      }
      int v, polls = 0;
      while ((v = ch_get((ch_lp)&xcnt)) < CH_NS * (i + 1)) {
        if (++polls >= a.limit && ch_get((ch_lp)&stays)) break;
        __builtin_amdgcn_s_sleep(1);
      }
      if (v >= CH_QUIT) return;
      if (__builtin_expect(v < CH_NS * (i + 1), 0)) break;
      if (i == a.n - 1 && wave == 0) ch_set((ch_lp)&closed, 1);
      multiply(c);
    }
    if (__builtin_expect(i == a.n, 1)) {
      ch_wait<1>((ch_lp)&closed, 1);
      if (__builtin_expect(!ch_get((ch_lp)&nothers), 1)) return;
    }
    // blocks taken over, of which `kept` are as far as this one; looks in vain;
    // the next of all blocks, where their turn has come
    int kept = 0, looks = 0, all = CH_BLOCKS, seen = 0;
    for (; i <= a.n; i++) {
      // Until x is there (behind the last product: to the end of those taken
      // over) a quarter of another block's rows, products from t0 on.
      for (int k = 0, polls = a.limit, had = ch_get((ch_lp)&nothers);;) {
        int b, t0 = 0;
        const bool look = all < CH_BLOCKS;
        if (k < had) {
          b = ch_s(((CH_VOL(uint8_t)*)others)[k]);
          if (k < kept) t0 = i - 1;
          k++;
        } else if (look) {
          b = (int)(blockIdx.x + all++ * 101) & (CH_BLOCKS - 1);
        } else if (i < a.n) {
          const int v = ch_get((ch_lp)&xcnt);
          if (v >= CH_QUIT) return;
          if (v >= CH_NS * (i + 1)) break;
          __builtin_amdgcn_s_sleep(1);
          if (++polls < a.limit) continue;
          // someone's rows are not there
          polls = a.limit / 4 * 3;
          had = ch_get((ch_lp)&nothers);
          if (k < had) continue;
          b = wave == 0 && a.claims
                  ? ch_adopt(a.claims, lane, looks >= CH_MINOR, &seen) : -1;
          if (b >= 0) {
            if (lane == 0) ((CH_VOL(uint8_t)*)others)[k] = b;
            ch_set((ch_lp)&nothers, ++had);   // LDS keeps a wave's order
            polls = a.limit;
          } else if (++looks > (a.limit == 0 ? 0 : a.claims ? CH_PATIENCE : 8)) {
            all = 0;
          }
          continue;
        } else {
          // wave 0 has taken over its last one
          ch_wait<1>((ch_lp)&closed, 1);
          had = ch_get((ch_lp)&nothers);
          if (k < had) continue;
          break;
        }
        ch_wait<1>((ch_lp)&ncnt, i);
        for (int t = t0; t < i; t++)
          ch_unit<WT>((CH_LDS_OF(ChStep)*)st, t, b, wave, lane, a.act,
                      ((CH_VOL(float)*)norms[t])[1],
                      ((CH_VOL(float)*)norms[t])[0], (CH_LDS_OF(int)*)eid,
                      (CH_LDS_OF(float)*)ew, (CH_LDS_OF(char)*)hs, look);
        kept = max(kept, k);
      }
      if (i == a.n) break;
      if (i == a.n - 1 && wave == 0) ch_set((ch_lp)&closed, 1);
      multiply(ch_take(st, i, WT));
    }
  } else if (wave < CH_NC + CH_NL) {       // ---- load
    const int wv = wave - CH_NC;
    const ch_lp fullp = (ch_lp)&full[wv], freep = (ch_lp)&freed[wv];
    int ps = 0, pg = 0, pc = 0, at = 0, freedv = 0;
    ChCur c = ch_take(st, 0, WT);
    // Slots that have arrived are told as the next one is asked for: one in
    // flight behind the newest.
    // x of the first product ahead of weights that are soon through: us a launch
    // at once, after 6 and 12 x 64 cycles, MXFP4 1B 20.0, 18.6, 18.4, 8B 32.4,
    // 32.1, 32.4, e4m3 1B 20.9, 20.5, 20.2, 8B 46.4, 46.3, 46.7, bf16 1B 25.7,
    // 26.1, 26.3.
    if constexpr (WT != GV_BF16) __builtin_amdgcn_s_sleep(6);
    for (int u = 0; u < a.total; u++) {
      if (u - freedv >= a.slots) {
        freedv = ch_get(freep);
        if (u - freedv >= a.slots) {       // none free: wait for the newest
          ch_arrived<0>();
          ch_set(fullp, u);
          for (int n = 1; u - (freedv = ch_get(freep)) >= a.slots; n++) {
            if (!(n & 15) && ch_get((ch_lp)&xcnt) >= CH_QUIT) {
              ch_set(fullp, CH_QUIT);      // who still multiplies, for nothing
              return;
            }
            __builtin_amdgcn_s_sleep(1);
          }
        }
      }
      bool up;
      const int r0 = ch_rows(c, pg, wv, &up);
      const int col =
          min((pc << c.kwl) + (wv & ((1 << c.kwl) - 1)), c.C - 1);
      const int piece = min(col * 64 + lane, c.P - 1);
      char* const sl = ring + (wv * a.slots + at) * SLOT;
      const char* w = c.w + (up ? (size_t)c.N * c.P * 16 : 0);
#pragma unroll
      for (int r = 0; r < 4; r++)
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) uint32_t*)(
                w + (size_t)min(r0 + r, c.nn - 1) * c.P * 16 +
                (size_t)piece * 16),
            (__attribute__((address_space(3))) uint32_t*)(sl + r * 1024), 16,
            0, 2);
      if constexpr (WT == GV_FP4) {        // four bytes a lane
        const int row = min(r0 + (lane >> 4), c.nn - 1);
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) uint32_t*)(
                c.we + (up ? (size_t)c.N * c.P : 0) + (size_t)row * c.P +
                min(col * 64 + (lane & 15) * 4, c.P - 4)),
            (__attribute__((address_space(3))) uint32_t*)(sl + 4096), 4, 0, 2);
      }
      if (u > 0) {
        ch_arrived<LD>();
        ch_set(fullp, u);
      }
      if (++at == a.slots) at = 0;
      if (++pc < c.cols) continue;
      pc = 0;
      if (++pg < c.groups) continue;
      pg = 0;
      if (++ps >= a.n) continue;
      if constexpr (MOE)
        if (ch_s(st[ps].s.slot)) {
          if (!ch_get((ch_lp)&routed)) {
            ch_arrived<0>();
            ch_set(fullp, u + 1);          // all that the router waits for
          }
          if (!ch_wait<1>((ch_lp)&routed, 1)) {
            ch_arrived<0>();               // none on its way when a block ends
            ch_set(fullp, CH_QUIT);
            return;
          }
        }
      c = ch_take<MOE>(st, ps, WT, eid);
    }
    ch_arrived<0>();
    ch_set(fullp, a.total);
  } else {                                 // ---- bring x, finish outputs
    __builtin_amdgcn_s_setprio(3);         // what all others wait for
    const int t = tid - 64 * (CH_NC + CH_NL), sw = wave - CH_NC - CH_NL;
    int sums = 0;                          // over all of x, so far
    auto add_up = [&](float v) {           // one more: this wave's share
      v = wave_reduce_sum(v);
      if (lane == 0) ssq[sums & 3][sw] = v;
      sums++;
      ch_done((ch_lp)&sub, lane);
    };
    auto factor = [&](int K) {             // of the last one
      ch_wait<0>((ch_lp)&sub, CH_NS * sums);   // (or others have the rows)
      float v = 0.f;
#pragma unroll
      for (int k = 0; k < CH_NS; k++)
        v += ((CH_VOL(float)*)ssq[(sums - 1) & 3])[k];
      return rsqrtf(v / (float)K + a.eps);
    };
    float rn = 1.f, r1 = 1.f;
    for (int i = 0; i < a.n; i++) {
      const ChStage& s = st[i].s;
      const int K = ch_s(s.K), skind = ch_s(s.kind);
      const u16* const route = MOE ? ch_p(s.route) : nullptr;
      const int slot = MOE ? ch_s(s.slot) : 0;
      const bool add2 = MOE && ch_p(s.add2);
      [[maybe_unused]] float scale = 1.f;

      const int rpb = ch_s(st[i].rpb), n0 = blockIdx.x * rpb;
      const int nn = max(0, min(rpb, ch_s(s.N) - n0));
      const bool wait = ch_s(s.wait), glu = ch_s(s.glu);
      const char* const src = (const char*)ch_p(s.x);
      const float *const g = ch_p(s.g), *const g2 = ch_p(s.g2);
      const u16* const hsrc = ch_p(s.h);
      const u16* const addp = ch_p(s.add);
      u16* const hout = ch_p(s.hout);
      const bool fromown = ch_s(s.own);
      const int keep = ch_s(st[i].keep);
      const int kw = 1 << ch_s(st[i].kwl);
      const float* wsp = ch_p(s.ws) + n0;
      const int N = ch_s(s.N), yf32 = ch_s(s.y_f32);
      void* const y = ch_p(s.y);
      // what an output needs besides its sums
      float add = 0.f, s1 = 1.f, s2 = 1.f;
      auto rest = [&](int r) {
        if (addp) add = fromown ? own[r] : b2f(addp[n0 + r]);
        if (MOE && add2) add += own2[r];
        if constexpr (WT == GV_FP8) {
          s1 = wsp[r];
          if (glu) s2 = wsp[N + r];
        }
      };
      // an expert's are known only behind its router
      if (t < nn && !(MOE && route)) {
        if constexpr (MOE) {
          if (slot && WT == GV_FP8) wsp += (size_t)ch_s(eid[slot - 1]) * s.sstep;
          if (s.scaled) scale = ew[slot - 1];
        }
        rest(t);
      }

      // G pieces of 16 bytes a thread at a time; norms take all of x in one
      auto bring = [&](auto gn, auto f32, auto norms, auto routes) {
        constexpr int G = decltype(gn)::value;
        constexpr bool F32 = decltype(f32)::value;
        constexpr bool NORMS = decltype(norms)::value;
        constexpr bool ROUTES = decltype(routes)::value;   // by NORM alone
        const int kind = ROUTES ? CH_NORM : skind;
        constexpr int V = F32 ? 1 : 2;     // quads of a piece
        const int np = K / (4 * V);
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            (void*)src, 0, np * 16, 0x00027000);
        for (int b0 = 0; b0 < np; b0 += G * CH_NT) {
          auto piece = [&](int j) { return min(b0 + j * CH_NT + t, np - 1); };
          auto real = [&](int j) { return b0 + j * CH_NT + t < np; };
          f4v ga[G][V], gb[G][V];
          ch_u8 hv[G][V];
          if (NORMS && kind != CH_RAW)     // asked for ahead of x
#pragma unroll
            for (int j = 0; j < G; j++)
#pragma unroll
              for (int k = 0; k < V; k++) {
                const int q = piece(j) * V + k;
                ga[j][k] = *(const f4v*)(g + q * 4);
                if (kind == CH_NORM2) {
                  gb[j][k] = *(const f4v*)(g2 + q * 4);
                  hv[j][k] = hsrc ? *(const ch_u8*)(hsrc + q * 4)
                                  : *(const ch_u8*)(hs + q * 8);
                }
              }
          [[maybe_unused]] ch_u8 wg[ROUTES ? CH_EXPERTS : 1][G][V];
          if constexpr (ROUTES)
#pragma unroll
            for (int e = 0; e < CH_EXPERTS; e++)
#pragma unroll
              for (int j = 0; j < G; j++)
#pragma unroll
                for (int k = 0; k < V; k++)
                  wg[e][j][k] = *(const ch_u8*)(
                      route + (size_t)min(e, ch_s(s.experts) - 1) * K +
                      (piece(j) * V + k) * 4);
          u4v_ v[G];
          uint32_t todo = wait ? (1u << G) - 1 : 0;
          if (!wait)
#pragma unroll
            for (int j = 0; j < G; j++) v[j] = ((const u4v_*)src)[piece(j)];
          // what the other blocks are still at is not there at once
          if (wait && b0 == 0) __builtin_amdgcn_s_sleep(12);
          while (todo) {
            asm volatile("" ::: "memory");  // read again each time
#pragma unroll
            for (int j = 0; j < G; j++)
              if (todo >> j & 1) v[j] = ch_fresh(rs, piece(j) * 16);
#pragma unroll
            for (int j = 0; j < G; j++)
              if (todo >> j & 1 && __all(ch_there<F32>(v[j])))
                todo &= ~(1u << j);
          }
          f4v x[G][V];
#pragma unroll
          for (int j = 0; j < G; j++) {
            if constexpr (F32) {
              union { u4v_ u; f4v f; } r = {v[j]};
              x[j][0] = r.f;
            } else {
              x[j][0] = ch_quad(v[j][0], v[j][1]);
              x[j][V - 1] = ch_quad(v[j][2], v[j][3]);
            }
          }
          auto squares = [&]() {
            float ss = 0.f;
#pragma unroll
            for (int j = 0; j < G; j++)
              ss += real(j) ? ch_squares(x[j][0], x[j][V - 1]) : 0.f;
            return ss;
          };
          float ss = 0.f;
          if constexpr (NORMS) {
            if (kind == CH_NORM2) {
              add_up(squares());
              r1 = factor(K);
#pragma unroll
              for (int j = 0; j < G; j++)
#pragma unroll
                for (int k = 0; k < V; k++) {
                  const f4v h = ch_quad(hv[j][k]);
#pragma unroll
                  for (int e = 0; e < 4; e++)
                    x[j][k][e] = x[j][k][e] * r1 * ga[j][k][e] + h[e];
                  const ch_u8 o = ch_pack(x[j][k]);
                  x[j][k] = ch_quad(o);
                  const int q = piece(j) * V + k;
                  if (real(j)) {
                    *(ch_u8*)(hs + q * 8) = o;
                    if (hout && blockIdx.x == 0) *(ch_u8*)(hout + q * 4) = o;
                  }
                  ga[j][k] = gb[j][k];
                }
            }
            if (kind != CH_RAW) ss = squares();
          }
#pragma unroll
          for (int j = 0; j < G; j++)
#pragma unroll
            for (int k = 0; k < V; k++) {
              if (NORMS && kind != CH_RAW)
#pragma unroll
                for (int e = 0; e < 4; e++) x[j][k][e] *= ga[j][k][e];
              if (!real(j)) continue;
              const int q = piece(j) * V + k;
              if constexpr (WT == GV_BF16)
                *(ch_u8*)(xs + q * 8) = ch_pack_x(x[j][k]);
              else                         // a lane's quads a KB apart
                *(f4v*)(xs + q / (Q * 64) * (256 * E) + q % Q * 1024 +
                        q / Q % 64 * 16) = x[j][k];
            }
          if constexpr (ROUTES) {
            float d[CH_EXPERTS];
#pragma unroll
            for (int e = 0; e < CH_EXPERTS; e++) {
              d[e] = 0.f;
#pragma unroll
              for (int j = 0; j < G; j++)
#pragma unroll
                for (int k = 0; k < V; k++) {
                  const f4v w = ch_quad(wg[e][j][k]);
                  if (real(j))
                    d[e] += x[j][k][0] * w[0] + x[j][k][1] * w[1] +
                            (x[j][k][2] * w[2] + x[j][k][3] * w[3]);
                }
            }
            const float r = gv_rows<CH_EXPERTS>(d, lane);
            if (lane < CH_EXPERTS) rsum[sw][lane] = r;
            ch_done((ch_lp)&dots, lane);
          }
          if (b0 + G * CH_NT >= np) {
            ch_done((ch_lp)&xcnt, lane);
            if (NORMS && kind != CH_RAW) add_up(ss);
          }
        }
      };
      using yes = std::true_type;
      using no = std::false_type;
      const std::integral_constant<int, 1> one;
      const std::integral_constant<int, 2> two;
      const std::integral_constant<int, 4> four;
      const std::integral_constant<int, 7> seven;
      const std::integral_constant<bool, MOE> moe;
      if (MOE && ch_s(s.same)) ch_done((ch_lp)&xcnt, lane);
      else if (MOE && route) K <= 8 * CH_NT ? bring(one, no(), yes(), moe)
                                            : bring(two, no(), yes(), moe);
      else if (ch_s(s.x_f32)) bring(seven, yes(), no(), no());
      else if (K > CH_NORM_K) bring(four, no(), no(), no());
      else K <= 8 * CH_NT ? bring(one, no(), yes(), no())
                          : bring(two, no(), yes(), no());

      if (!(MOE && ch_s(s.same))) rn = skind == CH_RAW ? 1.f : factor(K);
      if (sw == 0) {
        if (lane == 0) {
          ((CH_VOL(float)*)norms[i])[0] = rn;
          ((CH_VOL(float)*)norms[i])[1] = r1;
        }
        ch_set((ch_lp)&ncnt, i + 1);       // LDS keeps a wave's order
      }
      if constexpr (MOE) if (route) {
        // Every wave by itself, to the same: probabilities of all experts,
        // the largest of them (the first of equals), by their sum.
        ch_wait<0>((ch_lp)&dots, CH_NS);
        const int ne = ch_s(s.experts), top = ch_s(s.top);
        const int e = lane & (CH_EXPERTS - 1);
        auto most = [&](float v) {         // over eight lanes
          v = fmaxf(v, gv_from<1>(v));
          v = fmaxf(v, gv_from<2>(v));
          return fmaxf(v, gv_from<7>(v));
        };
        float z = 0.f;
#pragma unroll
        for (int k = 0; k < CH_NS; k++) z += ((CH_VOL(float)*)rsum[k])[e];
        z = e < ne ? z * rn : -INFINITY;
        float p = __expf(z - most(z)), sum = 0.f, pv[CH_TOP];
        if (!(p == p)) p = 0.f;            // an index is one of an expert
        p = e < ne ? p : -2.f;
#pragma unroll
        for (int j = 0; j < CH_TOP; j++) {
          pv[j] = most(p);
          const int best = min(
              __builtin_ctz((uint32_t)__ballot(p == pv[j]) & 0xff | 256), ne - 1);
          if (j < top) sum += pv[j];
          if (e == best) p = -1.f;
          ((CH_VOL(int)*)eid)[j] = j < top ? best : 0;
        }
#pragma unroll
        for (int j = 0; j < CH_TOP; j++) ((CH_VOL(float)*)ew)[j] = pv[j] / sum;
        ch_done((ch_lp)&routed, lane);
        if (t < nn) {
          if (WT == GV_FP8) wsp += (size_t)ch_s(eid[slot - 1]) * s.sstep;
          rest(t);
        }
      }
      // nothing to finish where the block's rows are another's
      const int mine = ch_wait<0>((ch_lp)&scnt, CH_NC * (i + 1)) ? nn : 0;
      float* const tops = ch_p(((CH_VOL(ChStep)*)st)[i].s.tops);
      float most = -INFINITY;
      for (int r = t; r < mine; r += CH_NT) {
        if (r != t) rest(r);
        const f4v p = *(const f4v*)&red[r * CH_NC];
        const f4v o = *(const f4v*)&red[((glu ? rpb : 0) + r) * CH_NC];
        float v = 0.f, up = 0.f;
#pragma unroll
        for (int k = 0; k < CH_NC; k++)
          if (k < kw) {
            v += p[k];
            up += o[k];
          }
        v = ch_finish<WT>(s, a.act, v, up, rn, s1, s2, add, scale);
        if (keep == 1) own[r] = b2f(f2b(v));
        if (MOE && keep == 2) own2[r] = v;
        ch_put(y, yf32, n0 + r, v);
        most = fmaxf(most, v);
      }
      if (tops) {                          // not a NaN
        most = wave_reduce_max(most);
        if (lane == 0) tops[blockIdx.x * CH_NS + sw] = most;
      }
    }
  }
}

// How a step's rows of K weights are shared out: the split of K over the
// waves that multiply with the fewest rounds.
static ChStep ch_share(const ChStage& s, int wt) {
  ChStep q = {};
  q.s = s;
  const int C = (s.K / (8 << wt) + 63) / 64;
  q.rpb = (s.N + CH_BLOCKS - 1) / CH_BLOCKS;
  q.ngate = (q.rpb + 3) / 4;
  q.ng = s.glu ? 2 * q.ngate : q.ngate;
  int best = 1 << 30;
  for (int l = 0; 1 << l <= CH_NC; l++) {
    const int cols = (C + (1 << l) - 1) >> l, nw = CH_NC >> l;
    const int groups = (q.ng + nw - 1) / nw;
    if (cols * groups >= best) continue;
    best = cols * groups;
    q.kwl = l;
    q.cols = cols;
    q.groups = groups;
  }
  return q;
}

static int ch_plan(ChArgs* a, const ChStage* s, int n, int wt) {
  const int E = 8 << wt, slot = wt == GV_FP4 ? 4096 + 256 : 4096;
  int x = 0, h = 0, rows = 0;
  a->n = n;
  a->total = 0;
  for (int i = 0; i < n; i++) {
    if (s[i].N < 1 || s[i].K < E || s[i].K % E || s[i].K % 8 ||
        (wt == GV_FP4 && s[i].K % 128) ||
        (s[i].kind != CH_RAW && (s[i].K > CH_NORM_K || s[i].x_f32)))
      return 0;
    a->st[i] = ch_share(s[i], wt);
    const int C = (s[i].K / E + 63) / 64;
    const int xb = C * 64 * E * (wt == GV_BF16 ? 2 : 4);
    const int r = a->st[i].rpb * (s[i].glu ? 2 : 1);
    x = xb > x ? xb : x;
    rows = r > rows ? r : rows;
    if (s[i].kind == CH_NORM2 && s[i].K * 2 > h) h = s[i].K * 2;
    a->total += a->st[i].cols * a->st[i].groups;
  }
  a->xbytes = x;
  a->hbytes = (h + 15) / 16 * 16;
  a->rbytes = rows * CH_NC * 4;
  const long left = (long)CH_LDS - x - a->hbytes - a->rbytes;
  const int slots = left < 0 ? 0 : (int)(left / (CH_NC * slot));
  a->slots = slots < CH_SLOTS ? slots : CH_SLOTS;
  return a->slots;
}

// Slots of a ring that these products leave room for.  With fewer than two they
// are not taken, with two they should not be: us, four launches -> here, 4096
// wide, as many in the middle as leave 4, 3 and 2 slots:
//   bf16  36864 168 -> 157, 45056 198 -> 196, 52224 223 -> 250
//   e4m3  19456 61.7 -> 58.1, 23552 69.1 -> 68.6, 27648 77.7 -> 85.7
//   MXFP4 17408 46.3 -> 37.2, 21504 49.9 -> 42.9, 25600 54.0 -> 57.3
extern "C" int chain_slots(const ChStage* s, int n, int wt) {
  ChArgs a = {};
  if (!s || n < 1 || n > CH_MAX || wt < GV_BF16 || wt > GV_FP4) return 0;
  return ch_plan(&a, s, n, wt);
}

template <int WT, bool MOE>
static hipError_t ch_launch(const ChArgs& a, size_t bytes, hipStream_t s) {
  static const hipError_t raised = hipFuncSetAttribute(
      (const void*)&k_chain<WT, MOE>,
      hipFuncAttributeMaxDynamicSharedMemorySize, CH_LDS);
  (void)raised;
  hipLaunchKernelGGL((k_chain<WT, MOE>), dim3(CH_BLOCKS),
                     dim3(64 * (CH_NC + CH_NL + CH_NS)), bytes, s, a);
  return hipGetLastError();
}

// wt as of launch_gemv; limit: how long a wave waits, in steps of some 1.6 us,
// ahead of looking for blocks that have not started; claims: CH_BLOCKS words of
// ones, or null.
extern "C" hipError_t launch_chain(const ChStage* s, int n, int wt, int act,
                                   float eps, int limit, void* claims,
                                   hipStream_t stream) {
  ChArgs a = {};
  if (!s || n < 1 || n > CH_MAX || wt < GV_BF16 || wt > GV_FP4 || limit < 0 ||
      (size_t)claims % 16 || ch_plan(&a, s, n, wt) < 2)
    return hipErrorInvalidValue;
  int left = -1;                           // who left the stream in LDS
  int chosen = 0;                          // experts that a router has chosen
  for (int i = 0; i < n; i++) {
    if (s[i].route) {
      if (chosen || i == 0 || s[i].slot != 1 || s[i].kind != CH_NORM ||
          s[i].experts < 1 || s[i].experts > CH_EXPERTS || s[i].top < 1 ||
          s[i].top > CH_TOP || s[i].top > s[i].experts)
        return hipErrorInvalidValue;
      chosen = s[i].top;
    }
    // a block that ends leaves no stream behind, not even a wrong one
    if (claims && s[i].hout && i < 2) return hipErrorInvalidValue;
    if (!s[i].w || !s[i].x || !s[i].y || (wt == GV_FP8 && !s[i].ws) ||
        (wt == GV_FP4 && !s[i].we) || s[i].kind < CH_RAW ||
        s[i].kind > CH_NORM2 || (s[i].kind != CH_RAW && !s[i].g) ||
        (s[i].kind == CH_NORM2 &&
         (!s[i].g2 || (!s[i].h && (left < 0 || s[left].K != s[i].K)))) ||
        (s[i].slot && (wt == GV_FP4 || s[i].slot < 0 || !chosen ||
                       s[i].slot > chosen || s[i].kind == CH_NORM2)) ||
        (!s[i].slot && s[i].scaled) ||
        // the last product's x, and its norm
        (s[i].tops && (!s[i].y_f32 || i != n - 1)) ||
        (s[i].same && (i == 0 || s[i].x != s[i - 1].x || s[i].K != s[i - 1].K ||
                       s[i].kind != s[i - 1].kind || s[i].g != s[i - 1].g)) ||
        (s[i].add2 && (i < 2 || s[i].add2 != s[i - 1].y || !s[i - 1].y_f32 ||
                       s[i].N != s[i - 1].N || a.st[0].rpb > CH_NT ||
                       a.st[i].rpb > CH_NT || s[i - 1].glu)) ||
        // only the first product's outputs are kept, for as many rows
        (s[i].own && (i == 0 || s[i].add != s[0].y || s[0].glu || s[0].y_f32 ||
                      s[i].N != s[0].N || a.st[0].rpb > CH_NT)) ||
        // who takes over rows reads a stream from memory, or the last one's
        (s[i].kind == CH_NORM2 && !s[i].h && i != n - 1))
      return hipErrorInvalidValue;
    if (s[i].kind == CH_NORM2) left = i;
    if (s[i].own) a.st[0].keep = 1;
    if (s[i].add2) a.st[i - 1].keep = 2;
  }
  a.act = act;
  a.eps = eps;
  a.limit = (limit < 1 << 20 ? limit : 1 << 20) * 16;  // looks at LDS
  a.claims = (uint32_t*)claims;
  const size_t bytes = (size_t)a.xbytes + a.hbytes + a.rbytes +
                       (size_t)a.slots * CH_NC * (wt == GV_FP4 ? 4352 : 4096);
  switch (wt) {
    case GV_BF16:
      return chosen ? ch_launch<GV_BF16, true>(a, bytes, stream)
                    : ch_launch<GV_BF16, false>(a, bytes, stream);
    case GV_FP8:
      return chosen ? ch_launch<GV_FP8, true>(a, bytes, stream)
                    : ch_launch<GV_FP8, false>(a, bytes, stream);
    case GV_FP4: return ch_launch<GV_FP4, false>(a, bytes, stream);
  }
  return hipErrorInvalidValue;
}
