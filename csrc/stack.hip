// stack.hip — the launches of a prompt's rows through all layers.
//
// A chunk of a prompt is 7 to 13 launches a layer.  One by one through the
// bindings each cost the host 9 to 10 us, as much as the kernels of a short
// prompt run (37 rows through 16 layers: 1280 us of launching for 1345 us of
// kernels), so here a chunk is one call: 364 us of launching, and the first
// kernel runs when the host has asked for it and not 35 us later (those 37
// rows 1463 -> 1382 us, five rows through three layers 425 -> 388).  What is
// launched is what the engine launches for a step of several sequences or
// over several ranks, which need the host between layers.
#include "common.h"

struct StackLin {          // as it is multiplied: bf16, e4m3 or MXFP4
  const void *w, *s, *e;   // scales of rows; exponents
};

struct StackLayer {
  const void *g_in, *g_post, *g_preffn, *g_postffn, *bqkv, *wg;
  StackLin qkv, o, gu, down;               // gu, down: of all experts
  void *kc, *vc, *kS, *vS;                 // of all sequences
  long window;
};

struct StackPlan {
  const StackLayer* layers;
  const void *embed, *cos, *sin;
  void *h, *xn, *t1, *qkv, *att, *gate, *acc, *row_cnt, *tile_cnt, *xq,
      *sx, *len, *moe_idx, *moe_w, *moe_order, *pairs, *aq, *sa;
  long acc_floats, order_room;
  int nlayers, H, I, nh, kvh, hd, S, wt, kv8, gemma, act, E, topk, nrow_cnt,
      ntile_cnt, mfma, rows, pools;        // rows that fit, sequences
  float eps, scale, softcap, escale;
};

extern "C" {
hipError_t launch_gemv(
    const void* W, const void* ws, const void* we, const void* x,
    const void* x2, const void* g, const void* g2, void* y, const void* res,
    int wt, int N, int K, int stage, int act, int glu, int x_f32, int out_f32,
    float eps, float softcap, float escale, int maxblocks, const void* eidx,
    int ne, long wstride, long sstride, const void* oscale, void* ones,
    long ones_bytes, hipStream_t);
hipError_t launch_rmsnorm(const void* x, const void* g, const void* res,
                          void* y, const void* g2, void* y2, void* q2,
                          void* s2, int M, int H, float eps, hipStream_t);
hipError_t launch_rope_cache(void* q, const void* kin, const void* vin,
                             void* kc, void* vc, void* kS, void* vS, int kv8,
                             const void* cost, const void* sint,
                             const void* pos_ptr, const void* rows, int M,
                             int nh, int kvh, int hd, int S, int ldq,
                             int ldkv, hipStream_t);
hipError_t launch_attn(const void* q, const void* kc, const void* vc,
                       void* out, const void* len_ptr, const void* kS,
                       const void* vS, int kv8, int M, int nh, int kvh,
                       int hd, int ldq, int S, float scale, float softcap,
                       int window, hipStream_t);
hipError_t launch_attn_prefill_mfma(
    const void* q, const void* kc, const void* vc, void* out,
    const void* len_ptr, const void* tiles, const void* kS, const void* vS,
    void* part, long part_floats, int kv8, int M, int nh, int kvh, int hd,
    int ldq, int S, int keys, int most, int ntiles, float scale,
    float softcap, int window, hipStream_t);
float gemm_prompt_time(int fp4, int M, int N, int K, int act, long part_floats,
                       int ncnt);
hipError_t launch_gemm_prompt(
    const void* x, const void* w, const void* sx, const void* sw,
    const void* res, const void* bias, void* y, void* part, void* cnt,
    long part_floats, int ncnt, int M, int N, int K, int act, hipStream_t);
hipError_t launch_row_gemm(
    const void* x, const void* sx, const void* w, const void* ws,
    const void* we, const void* g, const void* bias, const void* res, void* y,
    void* part, void* cnt, long part_floats, int ncnt, int wt, int M, int N,
    int K, int ldx, int ldr, int ldy, int act, int out_f32, int n16,
    float eps, float softcap, hipStream_t);
hipError_t launch_quant_fp8(const void* X, void* Q, void* S, int f32, int M,
                            int K, hipStream_t);
hipError_t launch_gemm_fp4w(
    const void* x, const void* w, const void* we, const void* res,
    const void* bias, void* y, void* part, void* cnt, long part_floats,
    int ncnt, int M, int N, int K, int act, hipStream_t);
hipError_t launch_moe_route(const void* h, const void* g, const void* wg,
                            int M, int H, int E, int topk, float eps,
                            void* idx, void* wout, void* dense, hipStream_t);
hipError_t launch_expert_sort(const void* idx, void* sorted, int pairs, int E,
                              long room, hipStream_t);
hipError_t launch_expert_gemm(const void* x, const void* w, const void* sx,
                              const void* sw, void* y, const void* sorted,
                              int pairs, int E, int top, int gather, int N,
                              int K, int act, hipStream_t);
hipError_t launch_expert_sum(const void* y, const void* w, const void* idx,
                             void* h, int M, int top, int H, hipStream_t);
}

#define ST_FEW 16          // rows that row_gemm takes
#define ST_NORM_K 4096     // the longest row that it norms
#define ST(call)                                                             \
  do {                                                                       \
    const hipError_t err = (call);                                           \
    if (err != hipSuccess) return err;                                       \
  } while (0)

namespace {

enum { ST_BF16 = 0, ST_FP8 = 1, ST_FP4 = 2 };

// y [M, N] = x [M, K] W^T, N outputs (with act: of 2N rows, gate then up);
// g: of few rows, their norm on the way
hipError_t st_linear(const StackPlan& p, const StackLin& w, const void* x,
                     void* y, int M, int N, int K, const void* g,
                     const void* res, const void* bias, int act,
                     hipStream_t s) {
  if (M > ST_FEW) {
    if (p.wt == ST_FP4)
      return launch_gemm_fp4w(x, w.w, w.e, res, bias, y, p.acc, p.tile_cnt,
                              p.acc_floats, p.ntile_cnt, M, N, K, act, s);
    const void* sx = nullptr;
    if (p.wt == ST_FP8) {
      ST(launch_quant_fp8(x, p.xq, p.sx, 0, M, K, s));
      x = p.xq;
      sx = p.sx;
    }
    return launch_gemm_prompt(x, w.w, sx, w.s, res, bias, y, p.acc,
                              p.tile_cnt, p.acc_floats, p.ntile_cnt, M, N, K,
                              act, s);
  }
  if (p.wt == ST_FP8 && M == 1) {          // not rounded to e4m3
    if (g) {
      ST(launch_rmsnorm(x, g, nullptr, p.xn, nullptr, nullptr, nullptr,
                        nullptr, 1, K, p.eps, s));
      x = p.xn;
    }
    if (bias && res) return hipErrorInvalidValue;
    return launch_gemv(w.w, w.s, nullptr, x, nullptr, nullptr, nullptr, y,
                       bias ? bias : res, ST_FP8, N, K, 0, act > 0 ? act : 0,
                       act >= 0, 0, 0, 1e-5f, 0.f, 1.f, 0, nullptr, 1, 0, 0,
                       nullptr, nullptr, 0, s);
  }
  if (g && K > ST_NORM_K) {
    ST(launch_rmsnorm(x, g, nullptr, p.xn, nullptr, nullptr, nullptr, nullptr,
                      M, K, p.eps, s));
    x = p.xn;
    g = nullptr;
  }
  const void* sx = nullptr;
  if (p.wt == ST_FP8 && !g) {
    ST(launch_quant_fp8(x, p.xq, p.sx, 0, M, K, s));
    x = p.xq;
    sx = p.sx;
  }
  // a prompt's rows are bf16 on their way to e4m3
  return launch_row_gemm(x, sx, w.w, w.s, w.e, g, bias, res, y, p.acc,
                         p.row_cnt, p.acc_floats, p.nrow_cnt, p.wt, M, N, K,
                         K, res ? N : 0, N, act, 0, p.wt == ST_FP8, p.eps,
                         0.f, s);
}

// routed experts over the rows' own choices, into h
hipError_t st_experts(const StackPlan& p, const StackLayer& l, int M,
                      hipStream_t s) {
  const int pairs = M * p.topk;
  ST(launch_moe_route(p.h, l.g_post, l.wg, M, p.H, p.E, p.topk, p.eps,
                      p.moe_idx, p.moe_w, nullptr, s));
  ST(launch_expert_sort(p.moe_idx, p.moe_order, pairs, p.E, p.order_room, s));
  const bool f8 = p.wt == ST_FP8;
  if (f8) ST(launch_quant_fp8(p.xn, p.xq, p.sx, 0, M, p.H, s));
  ST(launch_expert_gemm(f8 ? p.xq : p.xn, l.gu.w, f8 ? p.sx : nullptr, l.gu.s,
                        p.gate, p.moe_order, pairs, p.E, p.topk, 1, p.I, p.H,
                        p.act, s));
  if (f8) ST(launch_quant_fp8(p.gate, p.aq, p.sa, 0, pairs, p.I, s));
  ST(launch_expert_gemm(f8 ? p.aq : p.gate, l.down.w, f8 ? p.sa : nullptr,
                        l.down.s, p.pairs, p.moe_order, pairs, p.E, p.topk, 0,
                        p.H, p.I, -1, s));
  return launch_expert_sum(p.pairs, p.moe_w, p.moe_idx, p.h, M, p.topk, p.H,
                           s);
}

}  // namespace

// Rows [0, M) of h through layers [first, last).  The last row sees `keys`
// keys; the rows follow *len in cache `pool`, or, with ntiles, are several
// sequences' (rows, tiles, most: of the cache and attention launches).
extern "C" hipError_t stack_forward(const StackPlan* plan, int M, int keys,
                                    int pool, int first, int last,
                                    const void* rows, const void* tiles,
                                    int ntiles, int most, hipStream_t s) {
  const StackPlan& p = *plan;
  // a chunk of one sequence ends inside its cache, one of several brings the
  // positions and pools of its rows
  if (M < 1 || M > p.rows || keys > p.S || first < 0 || last > p.nlayers ||
      (ntiles ? ntiles < 0 || !p.mfma || !rows || !tiles || most < 1 || most > M
              : M > p.S || pool < 0 || pool >= p.pools))
    return hipErrorInvalidValue;
  const bool few = M <= ST_FEW;
  const int nq = p.nh * p.hd, nkv = p.kvh * p.hd, nqkv = nq + 2 * nkv;
  u16 *q = (u16*)p.qkv, *k = q + nq, *v = k + nkv;
  auto norm = [&](const void* g) {         // xn = norm(h) g
    return launch_rmsnorm(p.h, g, nullptr, p.xn, nullptr, nullptr, nullptr,
                          nullptr, M, p.H, p.eps, s);
  };
  // h += x W^T, Gemma's through its norm and, with g, on to the next one
  auto into_h = [&](const StackLin& w, const void* x, int K, const void* post,
                    const void* g) {
    if (!p.gemma)
      return st_linear(p, w, x, p.h, M, p.H, K, nullptr, p.h, nullptr, -1, s);
    ST(st_linear(p, w, x, p.t1, M, p.H, K, nullptr, nullptr, nullptr, -1, s));
    return launch_rmsnorm(p.t1, post, p.h, p.h, g, g ? p.xn : nullptr,
                          nullptr, nullptr, M, p.H, p.eps, s);
  };
  for (int i = first; i < last; i++) {
    const StackLayer& l = p.layers[i];
    if (!few && (!p.gemma || i == 0)) ST(norm(l.g_in));
    ST(st_linear(p, l.qkv, few ? p.h : p.xn, p.qkv, M, nqkv, p.H,
                 few ? l.g_in : nullptr, nullptr, l.bqkv, -1, s));
    const size_t key = ntiles ? 0 : (size_t)pool * p.kvh * p.S;
    char* kc = (char*)l.kc + key * p.hd * (p.kv8 ? 1 : 2);
    char* vc = (char*)l.vc + key * p.hd * (p.kv8 ? 1 : 2);
    float* kS = p.kv8 ? (float*)l.kS + key : nullptr;
    float* vS = p.kv8 ? (float*)l.vS + key : nullptr;
    ST(launch_rope_cache(q, k, v, kc, vc, kS, vS, p.kv8, p.cos, p.sin, p.len,
                         ntiles ? rows : nullptr, M, p.nh, p.kvh, p.hd, p.S,
                         nqkv, nqkv, s));
    if (p.mfma)
      ST(launch_attn_prefill_mfma(
          q, kc, vc, p.att, p.len, ntiles ? tiles : nullptr, kS, vS, p.acc,
          p.acc_floats, p.kv8, M, p.nh, p.kvh, p.hd, nqkv, p.S,
          keys > M || ntiles ? keys : M, ntiles ? most : 0, ntiles, p.scale,
          p.softcap, (int)l.window, s));
    else
      ST(launch_attn(q, kc, vc, p.att, p.len, kS, vS, p.kv8, M, p.nh, p.kvh,
                     p.hd, nqkv, p.S, p.scale, p.softcap, (int)l.window, s));
    const void* g_mlp = p.gemma ? l.g_preffn : l.g_post;
    ST(into_h(l.o, p.att, nq, l.g_post, few ? nullptr : g_mlp));
    if (p.E) {
      ST(norm(g_mlp));
      ST(st_experts(p, l, M, s));
      continue;
    }
    if (!few && !p.gemma) ST(norm(g_mlp));
    ST(st_linear(p, l.gu, few ? p.h : p.xn, p.gate, M, p.I, p.H,
                 few ? g_mlp : nullptr, nullptr, nullptr, p.act, s));
    ST(into_h(l.down, p.gate, p.I, l.g_postffn,
              few || i + 1 == p.nlayers ? nullptr : p.layers[i + 1].g_in));
  }
  return hipSuccess;
}

// Rows of a chunk of a prompt of n, at most `most`: those, or fewer whole tiles
// of 128 where as many chunks take less so by the numbers that choose the
// products' tiles.  2048 rows of 2304 outputs are 288 tiles, one round of 256
// CUs and a rest; 1792 are 252.  ms, chunks of 2048 -> as here, four layers 2304
// wide: 2100 rows 2.29 -> 2.11, 3000 3.04 -> 2.80, 5003 5.02 -> 4.49.  Where 2048
// rows are whole rounds they stay: two layers 4096 wide, 5003 rows 4.47, in
// chunks of 1792 4.78.  A chunk more costs what it saves (2048 rows 2304 wide
// 1.91, as 1792 and 256 2.08).  A rest of 64 rows and fewer goes by other
// kernels than the numbers are of, and attention is in them by 3% alone: over
// 24 lengths up to 8000 rows of six widths none took longer (0.995 to 1.12 times
// as fast).  Beside e4m3 rows sums in another order are other
// values, and routed experts' rows are where the router sends them: these stay.
extern "C" int stack_chunk_rows(const StackPlan* plan, int n, int most) {
  const StackPlan& p = *plan;
  if (p.wt == ST_FP8 || p.E || most < 1 || n <= most) return most;
  const int nq = p.nh * p.hd, nqkv = nq + 2 * p.kvh * p.hd;
  auto product = [&](int M, int N, int K, int act) {
    return gemm_prompt_time(p.wt == ST_FP4, M, N, K, act, p.acc_floats,
                            p.ntile_cnt);
  };
  auto layer = [&](int M) {
    return M == 0 ? 0.f
                  : product(M, nqkv, p.H, -1) + product(M, p.H, nq, -1) +
                        product(M, p.I, p.H, p.act) + product(M, p.H, p.I, -1);
  };
  auto all = [&](int rows) {
    return (float)(n / rows) * layer(rows) + layer(n % rows);
  };
  // the numbers are 1 to 3% off, and attention would rather have large chunks
  float least = 0.97f * all(most);
  int best = most;
  const int chunks = (n + most - 1) / most, alike = (n + chunks - 1) / chunks;
  for (int rows = (most - 1) / 128 * 128; rows >= alike; rows -= 128) {
    const float t = all(rows);
    if (t >= least) continue;
    least = t;
    best = rows;
  }
  return best;
}

// h = rows of the embedding of up to ST_IDS tokens that come with the launch
// (a copy of them ahead of it takes 16 us); *len = pos0.
#define ST_IDS 128
struct StackIds { int v[ST_IDS]; };

__global__ void __launch_bounds__(256)
k_embed_list(const u16* __restrict__ embed, StackIds ids,
             const int* __restrict__ list, u16* __restrict__ out,
             int* __restrict__ len, int pos0, int H, float scale) {
  const int m = blockIdx.x, id = list ? list[m] : ids.v[m];
  if (m == 0 && threadIdx.x == 0) *len = pos0;
  const u16* src = embed + (size_t)id * H;
  u16* dst = out + (size_t)m * H;
  for (int i = threadIdx.x * 8; i < H; i += 2048) {
    const s8v v = *(const s8v*)(src + i);
    u16 o[8];
#pragma unroll
    for (int j = 0; j < 8; j++) o[j] = f2b(b2f(((const u16*)&v)[j]) * scale);
    *(s8v*)(dst + i) = *(s8v*)o;
  }
}

// ids: the tokens on the host, M <= 128, or list: on the device.  pos0 is a
// position of the cache; where several sequences share the rows it is not used.
extern "C" hipError_t stack_embed(const StackPlan* plan, const int* ids,
                                  const void* list, int M, int pos0,
                                  hipStream_t s) {
  const StackPlan& p = *plan;
  StackIds v = {};
  if (M < 1 || M > p.rows || pos0 < 0 || pos0 >= p.S || !ids == !list ||
      (ids && M > ST_IDS))
    return hipErrorInvalidValue;
  for (int i = 0; ids && i < M; i++) v.v[i] = ids[i];
  hipLaunchKernelGGL(k_embed_list, dim3(M), dim3(256), 0, s,
                     (const u16*)p.embed, v, (const int*)list, (u16*)p.h,
                     (int*)p.len, pos0, p.H, p.escale);
  return hipGetLastError();
}
