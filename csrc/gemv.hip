// gemv.hip — linears of one row: y[N] = W[N,K] stage(x)[K] (+ res), the
// products of a decode step.
//
// Bound by streaming W once, and for the small ones by the time until the
// stream runs.  So the first rows of W are asked for before x is staged, and
// x goes no further than registers: KW waves share out K, each lane keeps
// its pieces of x (fp32) for all the rows that it sees, and the other waves
// of a block (NW of them for each piece) take other rows.  Nothing is read
// from LDS per weight: widening and a product an element are all the work.
// Sums over the lanes are folded R rows at a time, sums over the waves meet
// in LDS once, behind a block's last row.
//
// Staged from LDS as fp32 (as before) e4m3 weights had 4 bytes of LDS read a
// weight, and every block waited for x, its norm and the first weights in
// turn.  us and TB/s, before -> here:
//   bf16   2048x8192, gate before it  11.2 -> 8.8 (the gate is taken by the
//          product before: 16384x2048 14.5 -> 14.4 with it), 3072x2048 5.7
//          -> 5.5, 128256x2048 85 -> 83.5 (6.3 TB/s)
//   e4m3   4096x14336, gate before it 17.6 -> 13.9, 28672x4096 23.7 -> 22.2,
//          128256x4096 87 -> 86 (6.1 TB/s)
//   MXFP4  3584x18944, gate before it 20.8 -> 13.8, 37888x3584 24.7 -> 19.0,
//          152064x3584 82.7 -> 53 (5.5 TB/s)
// Of the small ones 2 us are the launch, 1 the first loads, 0.7 to 2 the work
// on x and on the last rows; MXFP4 is bound by widening (13 us of 37888x3584
// without its loads).
#include "common.h"
#include "gemv.h"

typedef float gv_f4 __attribute__((ext_vector_type(4), aligned(4)));
typedef __bf16 gv_b2 __attribute__((ext_vector_type(2)));
typedef uint32_t gv_u2 __attribute__((ext_vector_type(2), aligned(4)));

struct GvArgs {
  const void* w;         // [N, K]; with a gate [2N, K]: gate, then up
  const float* ws;       // e4m3: scale of a row
  const uint8_t* we;     // MXFP4: exponents [rows, K/32]
  const void* x;         // bf16 (fp32: x_f32); STAGE_NORM_EMBED: the table
  const u16* x2;         // up half / residual stream / token
  const float* g;
  const float* g2;
  void* y;
  const u16* res;
  u16* hout;             // the residual stream that a stage writes back
  const int* eidx;       // experts: W, ws of eidx[i]
  const float* oscale;   // and the weight of its result
  long wstride, sstride;
  int N, K, stage, act, glu, x_f32, out_f32, kw, nw, rpb, ne;
  int kwl, nwl, kwel;    // log2 of kw, nw, kw / ne
  float eps, softcap, escale;
  u4v_* ones;            // filled with ones, words of 16 bytes
  long nones;
};

// LDS only: weights stay in flight across it
DEVINL void gv_meet() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// J loads of 1 KB (64 lanes x 16 bytes) a wave and row; R rows in flight
// while R others are multiplied.  T: x as it is (GV_RAW), staged by all
// threads of the block, 2048 elements at a time (T times), or by each group of
// waves that covers K by itself (GV_OWN: rows too long for T).
enum { GV_RAW = 0, GV_OWN = -1 };
template <int WT, int J, int R, int T>
__global__ void __launch_bounds__(512) k_gemv(GvArgs a) {
  constexpr int E = gv_e<WT>();
  constexpr bool RAW = T == GV_RAW, ALL = T > 0;
  __shared__ float ssq[2][8];
  // [kw][rows of the block], then x (or a stretch for each wave to turn)
  extern __shared__ __attribute__((aligned(16))) float red[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // a.kw is a power of two where more than one wave shares a piece of K
  const int kw = a.nw > 1 ? wave & (a.kw - 1) : wave;
  const int nw = a.nw > 1 ? wave >> a.kwl : 0;
  const int n0 = blockIdx.x * a.rpb, nn = min(a.rpb, a.N - n0);
  const int nr = a.glu ? 2 * nn : nn;      // rows of W
  // experts apart (rows of y) or added up (waves of each)
  const int kwe = 1 << a.kwel;
  const int ex = gridDim.y > 1 ? blockIdx.y : kw >> a.kwel;
  const int C = a.K / E;                   // 16-byte pieces of a row
  const size_t rowb = (size_t)a.K * 16 / E;
  const int stage = RAW ? STAGE_RAW : a.stage, rs = a.glu ? 2 * a.rpb : a.rpb;

  // what an output needs besides its sum: the first of a thread ahead of all
  float add = 0.f, s1 = 1.f, s2 = 1.f;
  auto rest = [&](int i) {
    const int n = n0 + i;
    if (a.res) add = b2f(a.res[n]);
    if (WT == GV_FP8 && !a.eidx) {
      s1 = a.ws[n];
      if (a.glu) s2 = a.ws[a.N + n];
    }
  };
  if (tid < nn) rest(tid);

  const int e0 = a.eidx ? a.eidx[ex] : 0;
  const char* W = (const char*)a.w + (size_t)e0 * a.wstride * 16 / E;
  int pc[J];                               // this lane's pieces of a row
  bool in[J];
  const int per = kwe * 64 * J;            // pieces of a pass over K
  constexpr int RP = R > 4 ? 8 : R > 2 ? 4 : R;
  float acc[RP] = {};
  u4v_ wa[R][J], wb[R][J];
  uint32_t xa[R][J], xb[R][J];             // MXFP4: exponents
  const int ng = ((nr + R - 1) / R + a.nw - 1) >> a.nwl;
  auto row_of = [&](int q, int r) {
    const int i = min((q * a.nw + nw) * R + r, nr - 1);
    return i < nn ? n0 + i : a.N + n0 + i - nn;
  };
  auto load = [&](u4v_ (&w)[R][J], uint32_t (&x)[R][J], int q) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int row = row_of(q, r);
      const char* p = W + (size_t)row * rowb;
#pragma unroll
      for (int j = 0; j < J; j++) {
        w[r][j] = __builtin_nontemporal_load(
            (const u4v_*)(p + (size_t)pc[j] * 16));
        if constexpr (WT == GV_FP4)
          x[r][j] = a.we[(size_t)row * (a.K / 32) + pc[j]];
      }
    }
  };

  for (int c0 = 0; c0 < C; c0 += per) {
#pragma unroll
    for (int j = 0; j < J; j++) {
      const int c = c0 + (j * kwe + (kw & (kwe - 1))) * 64 + lane;
      in[j] = c < C;
      pc[j] = in[j] ? c : C - 1;
    }
    constexpr int Q = E / 4;
    f4v* const turn = (f4v*)(red + ((a.kw * rs + 3) & ~3));
    const u16* xs = (const u16*)a.x;
    if (stage == STAGE_NORM_EMBED)
      xs += (size_t)(*(const int*)a.x2) * a.K;
    if (a.ne > 1 && gridDim.y == 1) xs += (size_t)ex * a.K * (a.x_f32 ? 2 : 1);
    auto clip = [&](int e) { return min(e, a.K - 4); };
    auto bf = [](gv_u2 u, int k) {
      return __uint_as_float(k & 1 ? u[k >> 1] & 0xffff0000u : u[k >> 1] << 16);
    };
    // What a stage does to NV pieces of four, at(i) the first element of the
    // i-th: v from x, hr from x2, gg and g1 from the last and the first norm's
    // g.  sums of n of the block's waves from w0 on; keeps: hout is written.
    auto staged = [&](auto& v, auto& hr, auto& gg, auto& g1, auto at, int w0,
                      int n, bool keeps) {
      constexpr int NV = sizeof(v) / sizeof(v[0]);
      // 1 / root mean square over all of x
      auto norm = [&](float* sq) {
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < NV; i++) {
          float t = 0.f;
#pragma unroll
          for (int k = 0; k < 4; k++) t += v[i][k] * v[i][k];
          ss += at(i) < a.K ? t : 0.f;
        }
        ss = gv_sum(ss);
        if (lane == 0) sq[wave] = ss;
        gv_meet();
        float t = 0.f;
        for (int k = 0; k < n; k++) t += sq[w0 + k];
        return rsqrtf(t / (float)a.K + a.eps);
      };
      auto round = [](float f) { return WT == GV_BF16 ? b2f(f2b(f)) : f; };
      if (stage == STAGE_GLU) {
#pragma unroll
        for (int i = 0; i < NV; i++)
#pragma unroll
          for (int k = 0; k < 4; k++)
            v[i][k] = round(gate_act(v[i][k], a.act) * bf(hr[i], k));
        return;
      }
      if (stage != STAGE_NORM) {           // the residual stream is bf16
        const float rn = stage == STAGE_NORM2 ? norm(ssq[1]) : a.escale;
#pragma unroll
        for (int i = 0; i < NV; i++) {
          const int e = at(i);
          u16 o[4];
#pragma unroll
          for (int k = 0; k < 4; k++) {
            float f = v[i][k] * rn;
            if (stage == STAGE_NORM2) f = f * g1(i, k) + bf(hr[i], k);
            o[k] = f2b(f);
            v[i][k] = b2f(o[k]);
          }
          if (keeps && e < a.K) *(gv_u2*)(a.hout + e) = *(gv_u2*)o;
        }
      }
      const float rn = norm(ssq[0]);
#pragma unroll
      for (int i = 0; i < NV; i++)
#pragma unroll
        for (int k = 0; k < 4; k++) v[i][k] = round(v[i][k] * rn * gg[i][k]);
    };
    // x, ahead of W: it comes from L2 and loads return in order.
    if constexpr (ALL) {
      auto at = [&](int i) { return (i * 512 + tid) * 4; };
      gv_f4 v[T], gg[T], ga[T];
      gv_u2 xr[T], hr[T];
#pragma unroll
      for (int i = 0; i < T; i++) xr[i] = *(const gv_u2*)(xs + clip(at(i)));
      if (stage == STAGE_GLU || stage == STAGE_NORM2)
#pragma unroll
        for (int i = 0; i < T; i++)
          hr[i] = *(const gv_u2*)(a.x2 + clip(at(i)));
      if (stage != STAGE_GLU) {
        const float* g = stage == STAGE_NORM2 ? a.g2 : a.g;
#pragma unroll
        for (int i = 0; i < T; i++) gg[i] = *(const gv_f4*)(g + clip(at(i)));
        if (stage == STAGE_NORM2)
#pragma unroll
          for (int i = 0; i < T; i++)
            ga[i] = *(const gv_f4*)(a.g + clip(at(i)));
      }
      load(wa, xa, 0);
#pragma unroll
      for (int i = 0; i < T; i++)
#pragma unroll
        for (int k = 0; k < 4; k++) v[i][k] = bf(xr[i], k);
      auto g1 = [&](int i, int k) { return ga[i][k]; };
      staged(v, hr, gg, g1, at, 0, 8, blockIdx.x == 0);
#pragma unroll
      for (int i = 0; i < T; i++) {
        const int n = i * 512 + tid;
        if (n * 4 < a.K) turn[n ^ (n / Q & (Q - 1))] = v[i];
      }
      gv_meet();
    }
    // Here lane l has elements 4l.. of every 256 of the wave's stretch: whole
    // lines.
    constexpr int NV = ALL ? 1 : J * Q;
    gv_f4 v[NV];
    auto at = [&](int i) {
      return ((c0 + (i / Q * kwe + (kw & (kwe - 1))) * 64) * Q + i % Q * 64 +
              lane) * 4;
    };
    auto each = [&](auto f) {
#pragma unroll
      for (int i = 0; i < NV; i++) f(i);
    };
    if (RAW && a.x_f32) {
      each([&](int i) {
        v[i] = *(const gv_f4*)((const float*)xs + clip(at(i)));
      });
      load(wa, xa, 0);
    } else if constexpr (!ALL) {
      gv_f4 gg[NV];
      gv_u2 xr[NV], hr[NV];
      each([&](int i) { xr[i] = *(const gv_u2*)(xs + clip(at(i))); });
      if constexpr (!RAW) {
        if (stage == STAGE_GLU || stage == STAGE_NORM2)
          each([&](int i) { hr[i] = *(const gv_u2*)(a.x2 + clip(at(i))); });
        if (stage != STAGE_GLU) {
          const float* g = stage == STAGE_NORM2 ? a.g2 : a.g;
          each([&](int i) { gg[i] = *(const gv_f4*)(g + clip(at(i))); });
        }
      }
      load(wa, xa, 0);
      each([&](int i) {
#pragma unroll
        for (int k = 0; k < 4; k++) v[i][k] = bf(xr[i], k);
      });
      if constexpr (!RAW) {
        auto g1 = [&](int i, int k) { return a.g[clip(at(i)) + k]; };
        staged(v, hr, gg, g1, at, nw << a.kwl, a.kw,
               blockIdx.x == 0 && nw == 0);
      }
    }
    // each lane's E elements in a row, by way of LDS
    float xv[J][E];
    gv_b2 xb2[J][4];                       // bf16 weights: x as it is
#pragma unroll
    for (int j = 0; j < J; j++) {
      f4v* to = turn + wave * (64 * Q);
      if constexpr (ALL) {
        to = turn + (j * kwe + (kw & (kwe - 1))) * (64 * Q);
      } else {
#pragma unroll
        for (int i = 0; i < Q; i++) {
          const int n = i * 64 + lane;
          to[n ^ (n / Q & (Q - 1))] = v[j * Q + i];
        }
      }
#pragma unroll
      for (int i = 0; i < Q; i++) {
        const f4v t = to[lane * Q + (i ^ (lane & (Q - 1)))];
#pragma unroll
        for (int k = 0; k < 4; k++) {
          if constexpr (WT == GV_BF16) xb2[j][i * 2 + k / 2][k & 1] = (__bf16)t[k];
          else xv[j][i * 4 + k] = t[k];
        }
      }
    }

    auto mul = [&](u4v_ (&w)[R][J], uint32_t (&ee)[R][J], int q) {
#pragma unroll
      for (int r = 0; r < R; r++) {
        acc[r] = 0.f;
#pragma unroll
        for (int j = 0; j < J; j++) {
          float p = 0.f, o = 0.f;
#pragma unroll
          for (int d = 0; d < 4; d++) {
            const uint32_t v = w[r][j][d];
            if constexpr (WT == GV_BF16) {
              // two products, exact, in one
              union { uint32_t u; gv_b2 b; } t = {v};
              float& q = d & 1 ? o : p;
              q = __builtin_amdgcn_fdot2_f32_bf16(t.b, xb2[j][d], q, false);
            } else if constexpr (WT == GV_FP8) {
              const f2v l = __builtin_amdgcn_cvt_pk_f32_fp8(v, false);
              const f2v h = __builtin_amdgcn_cvt_pk_f32_fp8(v, true);
              p += l[0] * xv[j][d * 4];
              o += l[1] * xv[j][d * 4 + 1];
              p += h[0] * xv[j][d * 4 + 2];
              o += h[1] * xv[j][d * 4 + 3];
            } else {
              const float s = __uint_as_float(ee[r][j] << 23);
              const f2v t[4] = {
                  __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(v, s, 0),
                  __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(v, s, 1),
                  __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(v, s, 2),
                  __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(v, s, 3)};
#pragma unroll
              for (int i = 0; i < 4; i++) {
                p += t[i][0] * xv[j][d * 8 + i * 2];
                o += t[i][1] * xv[j][d * 8 + i * 2 + 1];
              }
            }
          }
          acc[r] += in[j] ? p + o : 0.f;   // nothing behind the row's end
        }
      }
      const float s = gv_rows<RP>(acc, lane);
      const int i = (q * a.nw + nw) * R + lane;
      if (lane < R && i < nr) {
        float* t = red + kw * rs + i;
        *t = c0 ? *t + s : s;
      }
    };
    if (ng == 1) {
      mul(wa, xa, 0);
    } else {
      load(wb, xb, 1);
      for (int q = 0;; q += 2) {
        mul(wa, xa, q);
        if (q + 2 >= ng) {
          mul(wb, xb, q + 1);
          break;
        }
        load(wa, xa, q + 2);
        mul(wb, xb, q + 1);
        if (q + 3 >= ng) {
          mul(wa, xa, q + 2);
          break;
        }
        load(wb, xb, q + 3);
      }
    }
  }

  gv_meet();
  for (int i = tid; i < nn; i += blockDim.x) {
    const int n = n0 + i;
    if (i != tid) rest(i);
    float v = 0.f, up = 0.f;
    for (int k = 0; k < a.kw; k++) {
      const int e = gridDim.y > 1 ? blockIdx.y : k >> a.kwel;
      float s = a.oscale ? a.oscale[e] : 1.f, t = 1.f;
      if (WT == GV_FP8 && a.eidx) {
        const float* p = a.ws + (size_t)a.eidx[e] * a.sstride + n;
        s *= p[0];
        if (a.glu) t = p[a.N];
      }
      v += s * red[k * rs + i];
      if (a.glu) up += t * red[k * rs + nn + i];
    }
    v *= s1;
    if (a.glu) v = gate_act(v, a.act) * (up * s2);
    if (a.softcap > 0.f) v = a.softcap * tanhf(v / a.softcap);
    v += add;
    const size_t at = (size_t)blockIdx.y * a.N + n;
    if (a.out_f32) ((float*)a.y)[at] = v;
    else ((u16*)a.y)[at] = f2b(v);
  }
  for (long i = (long)blockIdx.x * blockDim.x + tid; i < a.nones;
       i += (long)gridDim.x * blockDim.x)
    a.ones[i] = u4v_{~0u, ~0u, ~0u, ~0u};
}

#define GV_ROOM (80 * 1024)                // LDS for the sums of a block

template <int WT, int J, int R, int T>
static hipError_t gv_launch(const GvArgs& a, dim3 grid, hipStream_t s) {
  static const hipError_t raised = hipFuncSetAttribute(
      (const void*)&k_gemv<WT, J, R, T>,
      hipFuncAttributeMaxDynamicSharedMemorySize, 159 * 1024);
  (void)raised;
  const int waves = T > 0 ? (1 << a.kwel) * J : a.kw * a.nw;
  hipLaunchKernelGGL((k_gemv<WT, J, R, T>), grid, dim3(64 * a.kw * a.nw),
                     ((size_t)a.kw * (a.glu ? 2 : 1) * a.rpb + 3 +
                      waves * 64 * gv_e<WT>()) * 4, s, a);
  return hipGetLastError();
}

// How x is staged: by all threads of a block, each element once, up to 8192 of
// them (every model's rows).  By each group of waves that covers K for itself
// two norms took longer than the 256 threads that staged into LDS before; us,
// one norm and two, that -> by groups -> here:
//   64x512 e4m3         3.6, 4.2 -> 4.3, 6.4 -> 3.6, 4.0
//   2048x16384 e4m3     8.3, 9.4 -> 7.8, 13.0 -> 6.8, 7.2
//   2304x4096 bf16      5.9, 7.6 -> 6.0, 8.5 -> 5.4, 6.3
//   3584x4608 MXFP4     7.0, 8.5 -> 7.0, 12.0 -> 5.9, 6.7
//   8192x10240 e4m3     16.9, 18.1 -> 14.6, 19.9 -> 14.2, 15.5
// (weights of the small ones from L2).
template <int WT, int J, int R>
static hipError_t gv_stage(const GvArgs& a, dim3 grid, hipStream_t s) {
  if (a.stage == STAGE_RAW) return gv_launch<WT, J, R, GV_RAW>(a, grid, s);
  // up to 8192 elements are two loads at most, one of MXFP4
  if constexpr (J <= (WT == GV_FP4 ? 1 : 2)) {
    if (a.K <= 2048)
      return gv_launch<WT, J, R, WT == GV_BF16 && J == 2 ? 2 : 1>(a, grid, s);
    if constexpr (WT == GV_FP4 || J == 2) {
      if (a.K <= 4096) return gv_launch<WT, J, R, 2>(a, grid, s);
      if constexpr (WT != GV_FP4 || R <= 6)
        if (a.K <= 8192) return gv_launch<WT, J, R, 4>(a, grid, s);
    }
  }
  if constexpr (J > (WT == GV_BF16 ? 2 : WT == GV_FP8 ? 1 : 0))
    return gv_launch<WT, J, R, GV_OWN>(a, grid, s);
  return hipErrorInvalidValue;
}

template <int WT, int J>
static hipError_t gv_go(const GvArgs& a, dim3 grid, int rows, hipStream_t s) {
  constexpr int RM = 8 / J > 1 ? 8 / J : 1;
  // rows in flight: the wave's, in equal turns of up to 8 KB
  // (six of MXFP4 beside 8192 staged elements: registers)
  const bool wide = WT == GV_FP4 && J == 1 && a.stage != STAGE_RAW &&
                    a.K > 4096 && a.K <= 8192;
  const int most = wide ? 6 : RM;
  const int turns = (rows + most - 1) / most, r = (rows + turns - 1) / turns;
#define GV_ROWS(RV)                                                          \
  if constexpr (RV <= RM)                                                    \
    if (r <= RV) return gv_stage<WT, J, RV>(a, grid, s);
  GV_ROWS(1)
  GV_ROWS(2)
  GV_ROWS(3)
  GV_ROWS(4)
  GV_ROWS(6)
  GV_ROWS(8)
#undef GV_ROWS
  return hipErrorInvalidValue;
}

template <int WT>
static hipError_t gv_run(GvArgs a, int maxblocks, hipStream_t s) {
  constexpr int E = gv_e<WT>(), JM = WT == GV_BF16 ? 8 : WT == GV_FP8 ? 5 : 3;
  const bool apart = a.ne > 1 && a.glu;    // a block an expert
  const int add = apart ? 1 : a.ne;        // experts that a block adds up
  const int loads = (a.K / E + 63) / 64;   // KB of a row
  // Waves of K: one a KB of a row of MXFP4 (two take the registers of x
  // that rows need); e4m3 two KB a wave (4096x4096 6.2 us, one 6.9); bf16 two
  // from four waves on (4096x4096 8.5 us, eight of one 9.0; 3072x2048 5.5,
  // two waves of two 5.8).
  int kwe = 1;
  while (kwe * 2 * add <= 8 &&
         (WT == GV_FP4 || (WT == GV_BF16 && kwe < 4) ? kwe : kwe * 2) < loads)
    kwe *= 2;
  int j = (loads + kwe - 1) / kwe;
  if (j > JM) {
    if (a.stage != STAGE_RAW && a.stage != STAGE_GLU)
      return hipErrorInvalidValue;
    const int passes = (j + JM - 1) / JM;  // over K
    j = (j + passes - 1) / passes;
  }
  a.kw = kwe * add;
  a.nw = a.kw & (a.kw - 1) ? 1 : 8 / a.kw;
  a.kwl = __builtin_ctz(a.kw);
  a.nwl = __builtin_ctz(a.nw);
  a.kwel = __builtin_ctz(kwe);
  const int P = a.glu ? 2 : 1, ny = apart ? a.ne : 1;
  if (apart) a.ne = 1;
  // A block a CU: with two, x is staged twice over and rows of a wave are
  // few (16384x2048 14.4 us, 512 blocks 16.5).
  int nb = 256 / ny;
  if (maxblocks > 0 && nb > maxblocks) nb = maxblocks;
  if (nb < 1) nb = 1;
  const int most = GV_ROOM / (a.kw * P * 4);
  if (nb < (a.N + most - 1) / most) nb = (a.N + most - 1) / most;
  a.rpb = (a.N + nb - 1) / nb;
  const dim3 grid((a.N + a.rpb - 1) / a.rpb, ny);
  const int rows = (a.rpb * P + a.nw - 1) / a.nw;
  switch (j) {
    case 1: return gv_go<WT, 1>(a, grid, rows, s);
    case 2: return gv_go<WT, 2>(a, grid, rows, s);
    case 3: return gv_go<WT, 3>(a, grid, rows, s);
  }
  if constexpr (JM >= 5) {
    if (j == 4) return gv_go<WT, 4>(a, grid, rows, s);
    if (j == 5) return gv_go<WT, 5>(a, grid, rows, s);
  }
  if constexpr (JM >= 8) {
    if (j <= 6) return gv_go<WT, 6>(a, grid, rows, s);
    return gv_go<WT, 8>(a, grid, rows, s);
  }
  return hipErrorInvalidValue;
}

// wt: 0 bf16, 1 e4m3 with ws, 2 MXFP4 with we.  glu: W holds 2N rows, gate
// then up, and y = act(gate) * up.  eidx: ne experts' W; their results stand
// in y one after the other with glu, else they are added up, x [ne, K].
// ones: bytes that are filled with ones besides (what a later launch leaves
// there is not there yet; a launch for that alone takes 2 us).
extern "C" hipError_t launch_gemv(
    const void* W, const void* ws, const void* we, const void* x,
    const void* x2, const void* g, const void* g2, void* y, const void* res,
    int wt, int N, int K, int stage, int act, int glu, int x_f32, int out_f32,
    float eps, float softcap, float escale, int maxblocks, const void* eidx,
    int ne, long wstride, long sstride, const void* oscale, void* ones,
    long ones_bytes, hipStream_t stream) {
  const bool keeps = stage == STAGE_NORM2 || stage == STAGE_NORM_EMBED;
  if (N < 1 || K < 1 || K % (wt == GV_BF16 ? 8 : wt == GV_FP8 ? 16 : 32) ||
      stage < 0 || stage > STAGE_NORM_EMBED || ne < 1 || ne > 8 ||
      (ne > 1 && (!eidx || (!glu && stage != STAGE_RAW) || keeps)) ||
      (x_f32 && stage != STAGE_RAW) || (keeps && !res) ||
      (wt == GV_FP8 && !ws) || (wt == GV_FP4 && (!we || eidx)) ||
      (ones ? ones_bytes < 16 || ones_bytes % 16 || ne > 1 : ones_bytes != 0))
    return hipErrorInvalidValue;
  GvArgs a = {W, (const float*)ws, (const uint8_t*)we, x, (const u16*)x2,
              (const float*)g, (const float*)g2, y,
              keeps ? nullptr : (const u16*)res, (u16*)res, (const int*)eidx,
              (const float*)oscale, wstride, sstride, N, K, stage, act, glu,
              x_f32, out_f32, 0, 0, 0, ne, 0, 0, 0, eps, softcap, escale,
              (u4v_*)ones, ones_bytes / 16};
  switch (wt) {
    case GV_BF16: return gv_run<GV_BF16>(a, maxblocks, stream);
    case GV_FP8: return gv_run<GV_FP8>(a, maxblocks, stream);
    case GV_FP4: return gv_run<GV_FP4>(a, maxblocks, stream);
  }
  return hipErrorInvalidValue;
}
