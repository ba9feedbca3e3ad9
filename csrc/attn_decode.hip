// attn_decode.hip — one new token of each sequence against the KV pool:
// RoPE of q and k, the pool write, online softmax, fp32 throughout.
//
// A block takes up to four query heads of one kv head (K and V are read once
// for them) over a range of the history.  How many ranges there are is
// decided on the device from the sequence's length (a captured step keeps
// its grid; blocks without a range leave), so that a short history has no
// merge at all.  The last block to arrive merges.
//
// k_attn_dec (head dims 64, 128, 256) keeps fp32 on the bf16 matrix cores: a
// query, and later a probability, is the sum of three bf16 numbers (8 bits of
// its mantissa each), and the three stand as columns of their own beside K
// and V, which are bf16 already: four heads fill 12 of 16 columns, products
// are exact, sums fp32.  The three columns of a result are added at the end.
// On the VALU the same took 2600 cycles for 16 keys of 4 heads of 128, and
// that bounded it.
//
// A wave takes 32 keys at a time by itself: K in operand order straight from
// the pool, V through its own stretch of LDS, turned by ds_read_b64_tr_b16
// (see attn_prefill.hip).  Loads are hidden by the eight waves of a block, not
// by a pipeline in one: a wave rarely has a second tile, since a block's range
// is a tile for each wave.  64 keys in four waves took 1.7 us more at 90 keys
// and as long at 6000.  Of 256 dims, where eight waves are a CU's whole LDS,
// short histories come in ranges of four tiles.
//
// What is left at a short history is one trip for the position, one for the
// loads it allows, the score -> probability -> value chain and the launch:
// 4.3 us at no history, 128 dims.  us, blocks a head apart and two fixed
// ranges (as before) -> here:
//   32/8 heads of 64, 90 keys 7.6 -> 4.6; 4000 keys 22.2 -> 10.0
//   32/8 of 128, 6040 e4m3 keys 39.2 -> 13.5; 160 keys 9.8 -> 6.4
//   16/8 of 256, 16 sequences of 620 keys, softcap 52.3 -> 25.4 (two ranges);
//     by eight waves a block for four 23.5 -> 20.0 (3.1 TB/s), 16 of 1500 keys
//     46.6 -> 40.7, one of 2000 13.5 -> 12.2, 8/4 heads, 220 keys 11.7 -> 10.1
//   64/8 of 128, 4 sequences of 2000 keys 97 -> 23
//   16/4 of 128, 32000 keys 131 -> 38 (1.7 TB/s: few blocks, long ranges)
//
// k_attn_dec_any serves the other head dims on the VALU.
#include "common.h"

typedef short ad_s4 __attribute__((ext_vector_type(4)));
typedef __bf16 ad_b8 __attribute__((ext_vector_type(8)));
typedef __bf16 ad_b2 __attribute__((ext_vector_type(2)));

struct AdArgs {
  const u16* qkv;        // [batch, (nh + 2 kvh) * hd]
  void* kc;              // [batch, kvh, S, hd]
  void* vc;
  u16* out;              // [batch, nh * hd]
  const int* len;        // [batch] positions of the new tokens
  const float* cost;     // [S, hd/2]
  const float* sint;
  float* kS;             // [batch, kvh, S] scales of an e4m3 pool
  float* vS;
  float* part;           // [batch, nh, split, hd + 2]: maximum, sum, values
  int* cnt;
  int nh, kvh, S, hg;    // hg: blocks of a kv head
  float scale, softcap;
  int window;
};

#define AD_NW 8
#define AD_UN 4
#define AD_LOG2E 1.4426950408889634f

// v op its value at lane ^ W; for W = 4 the four lanes around must agree
template <int W, class F> DEVINL float ad_pair(float v, F op) {
  const uint32_t u = __float_as_uint(v);
  if constexpr (W == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
  } else if constexpr (W == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
  } else {
    // quad_perm, row_half_mirror, row_ror:8
    constexpr int C = W == 1 ? 0xB1 : W == 2 ? 0x4E : W == 4 ? 0x141 : 0x128;
    return op(v, __uint_as_float(__builtin_amdgcn_update_dpp(0, u, C, 0xf,
                                                             0xf, true)));
  }
}
template <int LO, int HI, class F> DEVINL float ad_fold(float v, F op) {
  if constexpr (LO < HI) return ad_fold<LO * 2, HI>(ad_pair<LO>(v, op), op);
  else return v;
}

#define AD_MAX_SPLIT 64

// The last of a head group's `eff` blocks to arrive adds the parts.  Every
// load goes out before any is waited for: one trip, whatever eff.
template <int HD, int GB>
DEVINL void ad_merge(const AdArgs& a, const float* part, u16* out, int ng,
                     int eff, int* last_flag) {
  __shared__ float wt[GB][AD_MAX_SPLIT], sum[GB];
  const int tid = threadIdx.x;
  const size_t rowp = (size_t)gridDim.y * (HD + 2);
  if (!last_block(a.cnt + blockIdx.z * gridDim.x + blockIdx.x, eff,
                  last_flag))
    return;
  // a wave a head: the weights of its parts and their sum
  for (int g = tid >> 6; g < ng; g += blockDim.x >> 6) {
    const int c = tid & 63;
    float m = -INFINITY, l = 0.f;
    if (c < eff) {
      m = part_get(part + g * rowp + c * (HD + 2));
      l = part_get(part + g * rowp + c * (HD + 2) + 1);
    }
    float mt = m;
#pragma unroll
    for (int w = 1; w < 64; w <<= 1) mt = fmaxf(mt, __shfl_xor(mt, w));
    const float al = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mt);
    l = wave_reduce_sum(l * al);
    wt[g][c] = al;
    if (c == 0) sum[g] = l;
  }
  constexpr int Q = 16;                        // parts asked for at a time
  for (int e0 = 0; e0 < ng * HD; e0 += blockDim.x) {
    const int e = min(e0 + tid, ng * HD - 1), g = e / HD, d = e % HD;
    const float* pp = part + g * rowp + 2 + d;
    float v = 0.f;
    for (int c0 = 0; c0 < eff; c0 += Q) {
      float x[Q];
#pragma unroll
      for (int i = 0; i < Q; i++)
        x[i] = part_get(pp + (size_t)min(c0 + i, eff - 1) * (HD + 2));
      if (e0 == 0 && c0 == 0) __syncthreads();
#pragma unroll
      for (int i = 0; i < Q; i++)
        if (c0 + i < eff) v += x[i] * wt[g][c0 + i];
    }
    if (e0 + tid < ng * HD) out[e] = f2b(v / sum[g]);
  }
}

template <int HD, int GB, bool KV8>
__global__ void __launch_bounds__(64 * AD_NW) k_attn_dec_any(AdArgs a) {
  constexpr int LP = HD / 8, PP = 64 / LP, HD2 = HD / 2;
  constexpr int STEP = AD_NW * AD_UN * PP;   // keys of a block at a time
  __shared__ float accs[AD_NW][GB][HD];
  __shared__ float ml[AD_NW][GB][2];
  __shared__ int last_flag;
  const auto add = [](float x, float y) { return x + y; };
  const auto max2 = [](float x, float y) { return fmaxf(x, y); };

  const int b = blockIdx.z, chunk = blockIdx.y;
  const int kvhead = blockIdx.x / a.hg, grp = a.nh / a.kvh;
  const int g0 = blockIdx.x % a.hg * GB, ng = min(GB, grp - g0);
  const int h0 = kvhead * grp + g0;
  const int pos = a.len[b];
  const int start = a.window > 0 ? max(0, pos + 1 - a.window) : 0;
  const int hist = pos - start;
  // ranges of at least two steps each
  const int eff = min(max(1, (hist + 2 * STEP - 1) / (2 * STEP)),
                      (int)gridDim.y);
  if (chunk >= eff) return;
  const int clen = (hist + eff - 1) / eff;
  const int c0 = start + chunk * clen, c1 = min(c0 + clen, pos);
  const bool last_chunk = chunk == eff - 1;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int p = lane / LP, d0 = (lane % LP) * 8;
  const size_t pool = ((size_t)b * a.kvh + kvhead) * a.S;
  const u16* K0 = (const u16*)a.kc + pool * HD + d0;
  const u16* V0 = (const u16*)a.vc + pool * HD + d0;
  const uint8_t* K8 = (const uint8_t*)a.kc + pool * HD + d0;
  const uint8_t* V8 = (const uint8_t*)a.vc + pool * HD + d0;
  const float* kS = KV8 ? a.kS + pool : nullptr;
  const float* vS = KV8 ? a.vS + pool : nullptr;

  // ---- q and the new k, v: raw, then rotated ----
  const u16* row = a.qkv + (size_t)b * (a.nh + 2 * a.kvh) * HD;
  const bool lo = d0 < HD2;
  const int dp = lo ? d0 + HD2 : d0 - HD2, ci = lo ? d0 : d0 - HD2;
  s8v qa[GB], qb[GB];
#pragma unroll
  for (int g = 0; g < GB; g++) {
    const u16* q = row + (size_t)(h0 + min(g, ng - 1)) * HD;
    qa[g] = *(const s8v*)(q + d0);
    qb[g] = *(const s8v*)(q + dp);
  }
  const u16* kh = row + (size_t)(a.nh + kvhead) * HD;
  const s8v ka = *(const s8v*)(kh + d0), kb = *(const s8v*)(kh + dp);
  const s8v va = *(const s8v*)(kh + (size_t)a.kvh * HD + d0);
  float cs[8], sn[8];
  {
    const float* cp = a.cost + (size_t)pos * HD2 + ci;
    const float* sp = a.sint + (size_t)pos * HD2 + ci;
    *(f4v*)cs = *(const f4v*)cp;
    *(f4v*)(cs + 4) = *(const f4v*)(cp + 4);
    *(f4v*)sn = *(const f4v*)sp;
    *(f4v*)(sn + 4) = *(const f4v*)(sp + 4);
  }

  // ---- keys of a step: AD_UN loads of PP keys a wave ----
  struct Keys {
    s8v k[AD_UN], v[AD_UN];
    unsigned long long k8[AD_UN], v8[AD_UN];
    float ks[AD_UN], vs[AD_UN];
  };
  auto load = [&](Keys& x, int t0) {
#pragma unroll
    for (int u = 0; u < AD_UN; u++) {
      const int t = min(t0 + (wave * AD_UN + u) * PP + p, c1 - 1);
      if constexpr (KV8) {
        x.k8[u] = *(const unsigned long long*)(K8 + (size_t)t * HD);
        x.v8[u] = *(const unsigned long long*)(V8 + (size_t)t * HD);
        x.ks[u] = kS[t];
        x.vs[u] = vS[t];
      } else {
        x.k[u] = *(const s8v*)(K0 + (size_t)t * HD);
        x.v[u] = *(const s8v*)(V0 + (size_t)t * HD);
      }
    }
  };
  Keys cur, nxt;
  if (c0 < c1) load(cur, c0);

  float qf[GB][8], kn[8], vn[8];
  {
    const float sgn = lo ? -1.f : 1.f;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const float s = sgn * sn[j];
#pragma unroll
      for (int g = 0; g < GB; g++)
        qf[g][j] = b2f(((u16*)&qa[g])[j]) * cs[j] + b2f(((u16*)&qb[g])[j]) * s;
      kn[j] = b2f(((u16*)&ka)[j]) * cs[j] + b2f(((u16*)&kb)[j]) * s;
      vn[j] = b2f(((u16*)&va)[j]);
    }
  }
  if (last_chunk && g0 == 0 && wave == 0 && p == 0) {
    const size_t at = (pool + pos) * HD + d0;
    if constexpr (KV8) {
      float km = 0.f, vm = 0.f;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        km = fmaxf(km, fabsf(kn[j]));
        vm = fmaxf(vm, fabsf(vn[j]));
      }
      for (int w = 1; w < LP; w <<= 1) {
        km = fmaxf(km, __shfl_xor(km, w));
        vm = fmaxf(vm, __shfl_xor(vm, w));
      }
      const float k_s = fmaxf(km, 1e-8f) / 448.0f;
      const float v_s = fmaxf(vm, 1e-8f) / 448.0f;
      *(unsigned long long*)((uint8_t*)a.kc + at) = f32x8_to_fp8(kn, 1.f / k_s);
      *(unsigned long long*)((uint8_t*)a.vc + at) = f32x8_to_fp8(vn, 1.f / v_s);
      if (lane == 0) {
        a.kS[pool + pos] = k_s;
        a.vS[pool + pos] = v_s;
      }
    } else {
      u16 ko[8], vo[8];
#pragma unroll
      for (int j = 0; j < 8; j++) { ko[j] = f2b(kn[j]); vo[j] = f2b(vn[j]); }
      *(s8v*)((u16*)a.kc + at) = *(s8v*)ko;
      *(s8v*)((u16*)a.vc + at) = *(s8v*)vo;
    }
  }

  // scores in units of log2; the maximum is the wave's, so that its keys'
  // sums add up without weights
  const float c1s = a.softcap > 0.f ? a.scale / a.softcap : a.scale * AD_LOG2E;
  auto capped = [&](float s) {
    s *= c1s;
    if (a.softcap > 0.f) {
      const float e = __builtin_amdgcn_exp2f(s * (2.f * AD_LOG2E));
      s = a.softcap * AD_LOG2E * (1.f - 2.f * __builtin_amdgcn_rcpf(e + 1.f));
    }
    return s;
  };
  float m[GB], l[GB], acc[GB][8];
#pragma unroll
  for (int g = 0; g < GB; g++) {
    m[g] = -INFINITY;
    l[g] = 0.f;
#pragma unroll
    for (int j = 0; j < 8; j++) acc[g][j] = 0.f;
  }
  auto wide = [&](const s8v& v, unsigned long long v8, float* f) {
    if constexpr (KV8) {
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const uint32_t w = (uint32_t)(v8 >> (32 * h));
        const f2v x = __builtin_amdgcn_cvt_pk_f32_fp8(w, false);
        const f2v y = __builtin_amdgcn_cvt_pk_f32_fp8(w, true);
        f[h * 4] = x[0]; f[h * 4 + 1] = x[1];
        f[h * 4 + 2] = y[0]; f[h * 4 + 3] = y[1];
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; j++) f[j] = b2f(((u16*)&v)[j]);
    }
  };
  for (int t0 = c0; t0 < c1; t0 += STEP) {
    if (t0 + STEP < c1) load(nxt, t0 + STEP);
    const int tw = t0 + wave * AD_UN * PP;
    if (tw < c1) {
      float s[GB][AD_UN];
#pragma unroll
      for (int u = 0; u < AD_UN; u++) {
        float kf[8];
        wide(cur.k[u], cur.k8[u], kf);
        const bool in = tw + u * PP + p < c1;
#pragma unroll
        for (int g = 0; g < GB; g++) {
          float d = 0.f;
#pragma unroll
          for (int j = 0; j < 8; j++) d += qf[g][j] * kf[j];
          d = ad_fold<1, LP>(d, add);
          s[g][u] = in ? capped(KV8 ? d * cur.ks[u] : d) : -INFINITY;
        }
      }
#pragma unroll
      for (int g = 0; g < GB; g++) {
        float mx = s[g][0];
#pragma unroll
        for (int u = 1; u < AD_UN; u++) mx = fmaxf(mx, s[g][u]);
        mx = fmaxf(m[g], ad_fold<LP, 64>(mx, max2));
        const float mu = mx == -INFINITY ? 0.f : mx;
        const float al = __builtin_amdgcn_exp2f(m[g] - mu);
        m[g] = mx;
        l[g] *= al;
#pragma unroll
        for (int j = 0; j < 8; j++) acc[g][j] *= al;
#pragma unroll
        for (int u = 0; u < AD_UN; u++) {
          s[g][u] = __builtin_amdgcn_exp2f(s[g][u] - mu);
          l[g] += s[g][u];
          if (KV8) s[g][u] *= cur.vs[u];
        }
      }
#pragma unroll
      for (int u = 0; u < AD_UN; u++) {
        float vf[8];
        wide(cur.v[u], cur.v8[u], vf);
#pragma unroll
        for (int g = 0; g < GB; g++)
#pragma unroll
          for (int j = 0; j < 8; j++) acc[g][j] += s[g][u] * vf[j];
      }
    }
    cur = nxt;
  }

  // the new token, by the lanes of one key
  if (last_chunk && wave == 0) {
#pragma unroll
    for (int g = 0; g < GB; g++) {
      float d = 0.f;
#pragma unroll
      for (int j = 0; j < 8; j++) d += qf[g][j] * kn[j];
      const float s = capped(ad_fold<1, LP>(d, add));
      const float mx = fmaxf(m[g], s);
      const float al = __builtin_amdgcn_exp2f(m[g] - mx);
      const float pv = p == 0 ? __builtin_amdgcn_exp2f(s - mx) : 0.f;
      m[g] = mx;
      l[g] = l[g] * al + pv;
#pragma unroll
      for (int j = 0; j < 8; j++) acc[g][j] = acc[g][j] * al + pv * vn[j];
    }
  }

  // sums over the keys of the wave, then over the waves
#pragma unroll
  for (int g = 0; g < GB; g++) {
    l[g] = ad_fold<LP, 64>(l[g], add);
#pragma unroll
    for (int j = 0; j < 8; j++) {
      if constexpr (LP < 8) {       // lanes of a quad hold different dims
        for (int w = LP; w < 64; w <<= 1)
          acc[g][j] += __shfl_xor(acc[g][j], w);
      } else {
        acc[g][j] = ad_fold<LP, 64>(acc[g][j], add);
      }
    }
    if (p == 0) {
#pragma unroll
      for (int j = 0; j < 8; j++) accs[wave][g][d0 + j] = acc[g][j];
    }
    if (lane == 0) {
      ml[wave][g][0] = m[g];
      ml[wave][g][1] = l[g];
    }
  }
  __syncthreads();
  u16* out = a.out + ((size_t)b * a.nh + h0) * HD;
  const size_t rowp = (size_t)gridDim.y * (HD + 2);     // parts of a head
  float* part = a.part + ((size_t)b * a.nh + h0) * rowp;
  for (int e = tid; e < ng * HD; e += 64 * AD_NW) {
    const int g = e / HD, d = e % HD;
    float mt = -INFINITY, lt = 0.f, v = 0.f;
#pragma unroll
    for (int w = 0; w < AD_NW; w++) mt = fmaxf(mt, ml[w][g][0]);
#pragma unroll
    for (int w = 0; w < AD_NW; w++) {
      const float mw = ml[w][g][0];
      const float al = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - mt);
      lt += ml[w][g][1] * al;
      v += accs[w][g][d] * al;
    }
    if (eff == 1) {
      out[e] = f2b(v / lt);
    } else {
      float* pp = part + g * rowp + chunk * (HD + 2);
      part_put(pp + 2 + d, v);
      if (d == 0) {
        part_put(pp, mt);
        part_put(pp + 1, lt);
      }
    }
  }
  if (eff == 1) return;

  ad_merge<HD, GB>(a, part, out, ng, eff, &last_flag);
}

// eight e4m3 numbers as bf16, exact (by way of fp32 and f2b, as keys went
// before, 6040 of 32/8 heads of 128 took 1.4 us longer)
DEVINL s8v ad_widen(unsigned long long v) {
  union { ad_b2 p[4]; s8v s; } w;
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const uint32_t u = (uint32_t)(v >> (32 * i));
    w.p[i * 2] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(u, 1.0f, false);
    w.p[i * 2 + 1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(u, 1.0f, true);
  }
  return w.s;
}

// value * (1, 2^-8, 2^-16, 0): part `part` of its split into bf16 numbers
DEVINL float ad_part(float v, int part) {
  const float r1 = v - (float)(__bf16)v;
  const float r2 = r1 - (float)(__bf16)r1;
  return part == 0 ? v : part == 1 ? r1 : part == 2 ? r2 : 0.f;
}

template <int HD, bool KV8>
__global__ void __launch_bounds__(64 * 8)
k_attn_dec(AdArgs a) {
  constexpr int NW = 8, NS = 2, TK = 16 * NS;  // keys of a tile
  constexpr int KC = HD / 32, DT = HD / 16, HD2 = HD / 2, RB = HD * 2;
  constexpr int VT = TK * RB;                // bytes of a wave's V tile
  __shared__ __attribute__((aligned(16))) char Vs[NW][VT];
  __shared__ float ml[NW][4][2];
  // rotated; the new value
  __shared__ __attribute__((aligned(16))) float qs[4][HD], kn[HD], vn[HD];
  __shared__ __attribute__((aligned(16))) u16 qp[12][HD + 8];  // split
  __shared__ int last_flag;
  const auto add = [](float x, float y) { return x + y; };
  const auto max2 = [](float x, float y) { return fmaxf(x, y); };

  const int b = blockIdx.z, chunk = blockIdx.y;
  const int kvhead = blockIdx.x / a.hg, grp = a.nh / a.kvh;
  const int g0 = blockIdx.x % a.hg * 4, ng = min(4, grp - g0);
  const int h0 = kvhead * grp + g0;
  const int pos = a.len[b];
  const int start = a.window > 0 ? max(0, pos + 1 - a.window) : 0;
  const int hist = pos - start;
  // A tile for every wave of a block, more where the grid ends; one range as
  // long as two rounds will do (345 keys of 128, 6 sequences: 8.9 us, two
  // ranges and their merge 10.0; of 256 dims one round: 300 keys 12.1, three
  // ranges 9.9).  Of 256 dims up to 2048 keys are in ranges of four tiles (700
  // keys, 4 sequences 13.9, so 11.4; 2000 keys 14.4, 12.2; 5000 15.6 both).
  constexpr int ONE = HD == 256 ? NW : 2 * NW;
  const int tiles = (hist + TK - 1) / TK;
  const int most = HD == 256 && tiles <= 64 ? 4 : NW;
  const int eff = tiles <= ONE ? 1 : min((tiles + most - 1) / most,
                                         (int)gridDim.y);
  if (chunk >= eff) return;
  const int per = (tiles + eff - 1) / eff;
  const int c0 = start + chunk * per * TK, c1 = min(c0 + per * TK, pos);
  const bool last_chunk = chunk == eff - 1;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, gq = lane >> 4;  // operand row / column, k group
  const int part = lr >> 2;
  const size_t pool = ((size_t)b * a.kvh + kvhead) * a.S;
  const size_t esz = KV8 ? 1 : 2;
  const char* Kg = (const char*)a.kc + pool * HD * esz;
  const char* Vg = (const char*)a.vc + pool * HD * esz;

  // K of a tile: key 16n + lr, dims 32c + 8gq; issued before all else
  s8v kf[NS][KC];
  unsigned long long k8[NS][KC];
  u4v_ v8[KV8 ? VT / 2048 : 1];
  float ks[NS][4], vs[NS][4];
  auto load = [&](int t0) {
#pragma unroll
    for (int n = 0; n < NS; n++) {
      const size_t t = min(t0 + n * 16 + lr, c1 - 1);
#pragma unroll
      for (int c = 0; c < KC; c++) {
        const char* p = Kg + (t * HD + c * 32 + gq * 8) * esz;
        if constexpr (KV8) k8[n][c] = *(const unsigned long long*)p;
        else kf[n][c] = *(const s8v*)p;
      }
      if constexpr (KV8) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int tr = min(t0 + n * 16 + gq * 4 + r, c1 - 1);
          ks[n][r] = a.kS[pool + tr];
          vs[n][r] = a.vS[pool + tr];
        }
      }
    }
    // V into LDS, rows of 16-byte slots swizzled by 64-byte chunks
    constexpr int SL = HD / 8;
    if constexpr (KV8) {
#pragma unroll
      for (int i = 0; i < VT / 2048; i++) {
        const int e = i * 64 + lane, r = e / (SL / 2), s2 = e % (SL / 2);
        v8[i] = *(const u4v_*)(Vg + (size_t)min(t0 + r, c1 - 1) * HD + s2 * 16);
      }
    } else {
#pragma unroll
      for (int i = 0; i < VT / 1024; i++) {
        const int e = i * 64 + lane, r = e / SL;
        const int x = HD == 64 ? (r >> 1) & 1 : r & 3;
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) uint32_t*)(
                Vg + (size_t)min(t0 + r, c1 - 1) * RB +
                ((e % SL) ^ (x << 2)) * 16),
            (__attribute__((address_space(3))) uint32_t*)(
                &Vs[wave][i * 1024]), 16, 0, 0);
      }
    }
  };
  int t0 = c0 + wave * TK;
  if (t0 < c1) load(t0);

  // q of the heads and the new k, rotated; q split for the matrix cores
  const u16* row = a.qkv + (size_t)b * (a.nh + 2 * a.kvh) * HD;
  const u16* kh = row + (size_t)(a.nh + kvhead) * HD;
  const u16* vh = kh + (size_t)a.kvh * HD;
  for (int e = tid; e < (ng + 2) * HD2; e += 64 * NW) {
    const int h = e / HD2, i = e % HD2;
    if (h > ng) {
      vn[i] = b2f(vh[i]);
      vn[i + HD2] = b2f(vh[i + HD2]);
      continue;
    }
    const u16* x = h < ng ? row + (size_t)(h0 + h) * HD : kh;
    const float c = a.cost[(size_t)pos * HD2 + i];
    const float s = a.sint[(size_t)pos * HD2 + i];
    const float x1 = b2f(x[i]), x2 = b2f(x[i + HD2]);
    const float y1 = x1 * c - x2 * s, y2 = x2 * c + x1 * s;
    float* o = h < ng ? qs[h] : kn;
    o[i] = y1;
    o[i + HD2] = y2;
    if (h < ng)
#pragma unroll
      for (int q = 0; q < 3; q++) {
        qp[q * 4 + h][i] = f2b(ad_part(y1, q));
        qp[q * 4 + h][i + HD2] = f2b(ad_part(y2, q));
      }
  }
  union Op { s8v s; __bf16 e[8]; ad_b8 v; };
  Op qf[KC];
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
  for (int c = 0; c < KC; c++)
    qf[c].s = part < 3 ? *(const s8v*)&qp[lr][c * 32 + gq * 8] : s8v{};

  // the pool takes the new key and value: by the last wave, 8 dims a lane
  if (last_chunk && g0 == 0 && wave == NW - 1 && lane < HD / 8) {
    const float* k = kn + lane * 8;
    const float* v = vn + lane * 8;
    const size_t at = (pool + pos) * HD + lane * 8;
    if constexpr (KV8) {
      float km = 0.f, vm = 0.f;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        km = fmaxf(km, fabsf(k[j]));
        vm = fmaxf(vm, fabsf(v[j]));
      }
#pragma unroll
      for (int w = 1; w < HD / 8; w <<= 1) {
        km = fmaxf(km, __shfl_xor(km, w));
        vm = fmaxf(vm, __shfl_xor(vm, w));
      }
      const float k_s = fmaxf(km, 1e-8f) / 448.0f;
      const float v_s = fmaxf(vm, 1e-8f) / 448.0f;
      *(unsigned long long*)((uint8_t*)a.kc + at) = f32x8_to_fp8(k, 1.f / k_s);
      *(unsigned long long*)((uint8_t*)a.vc + at) = f32x8_to_fp8(v, 1.f / v_s);
      if (lane == 0) {
        a.kS[pool + pos] = k_s;
        a.vS[pool + pos] = v_s;
      }
    } else {
      u16 o[8], w[8];
#pragma unroll
      for (int j = 0; j < 8; j++) { o[j] = f2b(k[j]); w[j] = f2b(v[j]); }
      *(s8v*)((u16*)a.kc + at) = *(s8v*)o;
      *(s8v*)((u16*)a.vc + at) = *(s8v*)w;
    }
  }

  // scores in units of log2
  const float c1s = a.softcap > 0.f ? a.scale / a.softcap : a.scale * AD_LOG2E;
  auto capped = [&](float s) {
    s *= c1s;
    if (a.softcap > 0.f) {
      const float e = __builtin_amdgcn_exp2f(s * (2.f * AD_LOG2E));
      s = a.softcap * AD_LOG2E * (1.f - 2.f * __builtin_amdgcn_rcpf(e + 1.f));
    }
    return s;
  };
  float m = -INFINITY, l = 0.f;    // of head lr & 3, alike in its lanes
  f4v o[DT];
#pragma unroll
  for (int d = 0; d < DT; d++) o[d] = {0.f, 0.f, 0.f, 0.f};

  // V^T operand: dim 16d + lr, keys 32q + 4gq + 0..3 and 16 more, as the
  // scores lie in their lanes
  const int vrow = gq * 4 + (lr >> 2);
  const int vx = HD == 64 ? (vrow >> 1) & 1 : vrow & 3;
  for (; t0 < c1; t0 += NW * TK) {
    if constexpr (KV8) {
      constexpr int SL = HD / 8;
#pragma unroll
      for (int i = 0; i < VT / 2048; i++) {
        const int e = i * 64 + lane, r = e / (SL / 2), s2 = e % (SL / 2);
        const int x = HD == 64 ? (r >> 1) & 1 : r & 3;
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const s8v w = ad_widen((unsigned long long)v8[i][h * 2] |
                                 (unsigned long long)v8[i][h * 2 + 1] << 32);
          *(s8v*)(&Vs[wave][r * RB + ((s2 * 2 + h) ^ (x << 2)) * 16]) = w;
        }
      }
    }
    float p[NS][4], mx = m;
#pragma unroll
    for (int n = 0; n < NS; n++) {
      f4v s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < KC; c++) {
        Op k;
        if constexpr (KV8) k.s = ad_widen(k8[n][c]);
        else k.s = kf[n][c];
        s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k.v, qf[c].v, s, 0, 0, 0);
      }
      // key 16n + 4gq + r: the three parts of its score are 4 and 8 lanes on
#pragma unroll
      for (int r = 0; r < 4; r++) {
        float v = s[r];
        v += __uint_as_float(__builtin_amdgcn_update_dpp(
            0, __float_as_uint(v), 0x128, 0xf, 0xf, true));
        v += __uint_as_float(__builtin_amdgcn_update_dpp(
            0, __float_as_uint(v), 0x124, 0xf, 0xf, true));
        if constexpr (KV8) v *= ks[n][r];
        v = t0 + n * 16 + gq * 4 + r < c1 ? capped(v) : -INFINITY;
        p[n][r] = v;
        mx = fmaxf(mx, v);
      }
    }
    mx = ad_fold<16, 64>(mx, max2);
    const float mu = mx == -INFINITY ? 0.f : mx;
    const float al = __builtin_amdgcn_exp2f(m - mu);
    m = mx;
    l *= al;
#pragma unroll
    for (int d = 0; d < DT; d++)
#pragma unroll
      for (int r = 0; r < 4; r++) o[d][r] *= al;
    Op pf[NS / 2];
#pragma unroll
    for (int n = 0; n < NS; n++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        float v = __builtin_amdgcn_exp2f(p[n][r] - mu);
        l += v;
        if constexpr (KV8) v *= vs[n][r];
        pf[n / 2].e[n % 2 * 4 + r] = (__bf16)ad_part(v, part);
      }
#pragma unroll
    for (int q = 0; q < NS / 2; q++)
#pragma unroll
      for (int d = 0; d < DT; d++) {
        union { ad_s4 h[2]; ad_b8 v; } vf;
        const int slot = d * 2 + ((lr & 3) >> 1);
#pragma unroll
        for (int h = 0; h < 2; h++)
          vf.h[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) ad_s4*)(
                  &Vs[wave][(q * 32 + h * 16 + vrow) * RB +
                            (slot ^ (vx << 2)) * 16 + (lr & 1) * 8]));
        o[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf.v, pf[q].v, o[d], 0,
                                                       0, 0);
      }
    if (t0 + NW * TK < c1) load(t0 + NW * TK);
  }
  l = ad_fold<16, 64>(l, add);

  // o element r of d: dim 16d + 4gq + r of head lr & 3, in three lanes
#pragma unroll
  for (int d = 0; d < DT; d++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      float v = o[d][r];
      v += __uint_as_float(__builtin_amdgcn_update_dpp(
          0, __float_as_uint(v), 0x128, 0xf, 0xf, true));
      v += __uint_as_float(__builtin_amdgcn_update_dpp(
          0, __float_as_uint(v), 0x124, 0xf, 0xf, true));
      o[d][r] = v;
    }
  if (last_chunk && wave == 0) {             // the new token
    const int h = min(lr & 3, ng - 1);
    float fresh = 0.f;             // 16 lanes share a head's dims
#pragma unroll
    for (int d = 0; d < HD; d += 16) {
      const int i = d + part * 4 + gq;
      fresh += qs[h][i] * kn[i];
    }
    fresh += __uint_as_float(__builtin_amdgcn_update_dpp(
        0, __float_as_uint(fresh), 0x128, 0xf, 0xf, true));
    fresh += __uint_as_float(__builtin_amdgcn_update_dpp(
        0, __float_as_uint(fresh), 0x124, 0xf, 0xf, true));
    const float s = capped(ad_fold<16, 64>(fresh, add)), mx = fmaxf(m, s);
    const float mu = mx == -INFINITY ? 0.f : mx;
    const float al = __builtin_amdgcn_exp2f(m - mu);
    const float pv = __builtin_amdgcn_exp2f(s - mu);
    m = mx;
    l = l * al + pv;
#pragma unroll
    for (int d = 0; d < DT; d++) {
      const f4v x = *(const f4v*)&vn[d * 16 + gq * 4];
#pragma unroll
      for (int r = 0; r < 4; r++) o[d][r] = o[d][r] * al + pv * x[r];
    }
  }
  if (lr < 4) {                    // over the wave's V tile
#pragma unroll
    for (int d = 0; d < DT; d++)
      *(f4v*)&Vs[wave][(lr * HD + d * 16 + gq * 4) * 4] = o[d];
    if (gq == 0) {
      ml[wave][lr][0] = m;
      ml[wave][lr][1] = l;
    }
  }
  __syncthreads();
  u16* out = a.out + ((size_t)b * a.nh + h0) * HD;
  const size_t rowp = (size_t)gridDim.y * (HD + 2);     // parts of a head
  float* parts = a.part + ((size_t)b * a.nh + h0) * rowp;
  for (int e = tid; e < ng * HD; e += 64 * NW) {
    const int h = e / HD, d = e % HD;
    float mt = -INFINITY, lt = 0.f, v = 0.f;
#pragma unroll
    for (int w = 0; w < NW; w++) mt = fmaxf(mt, ml[w][h][0]);
#pragma unroll
    for (int w = 0; w < NW; w++) {
      const float mw = ml[w][h][0];
      const float al = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - mt);
      lt += ml[w][h][1] * al;
      v += *(const float*)&Vs[w][(h * HD + d) * 4] * al;
    }
    if (eff == 1) {
      out[e] = f2b(v / lt);
    } else {
      float* pp = parts + h * rowp + chunk * (HD + 2);
      part_put(pp + 2 + d, v);
      if (d == 0) {
        part_put(pp, mt);
        part_put(pp + 1, lt);
      }
    }
  }
  if (eff == 1) return;
  ad_merge<HD, 4>(a, parts, out, ng, eff, &last_flag);
}

template <int HD>
static hipError_t ad_mfma(AdArgs a, int kv8, int split, int batch,
                          hipStream_t s) {
  a.hg = (a.nh / a.kvh + 3) / 4;
  const dim3 grid(a.kvh * a.hg, split, batch);
  if (kv8)
    hipLaunchKernelGGL((k_attn_dec<HD, true>), grid, dim3(512), 0, s, a);
  else
    hipLaunchKernelGGL((k_attn_dec<HD, false>), grid, dim3(512), 0, s, a);
  return hipGetLastError();
}

template <int HD, int GB>
static hipError_t ad_go(const AdArgs& a, int kv8, int split, int batch,
                        hipStream_t s) {
  const dim3 grid(a.kvh * a.hg, split, batch);
  if (kv8)
    hipLaunchKernelGGL((k_attn_dec_any<HD, GB, true>), grid, dim3(64 * AD_NW), 0,
                       s, a);
  else
    hipLaunchKernelGGL((k_attn_dec_any<HD, GB, false>), grid, dim3(64 * AD_NW), 0,
                       s, a);
  return hipGetLastError();
}

template <int HD>
static hipError_t ad_run(AdArgs a, int kv8, int split, int batch,
                         hipStream_t s) {
  const int grp = a.nh / a.kvh;
  if (grp == 1) { a.hg = 1; return ad_go<HD, 1>(a, kv8, split, batch, s); }
  if (grp == 2) { a.hg = 1; return ad_go<HD, 2>(a, kv8, split, batch, s); }
  a.hg = (grp + 3) / 4;
  return ad_go<HD, 4>(a, kv8, split, batch, s);
}

// scratch: batch * nh * split * (hd + 2) floats; cnt: batch * nh ints, zero,
// left zero
extern "C" hipError_t launch_attn_dec(const void* qkv, void* kc, void* vc,
                                      void* out, const void* len_ptr,
                                      const void* cost, const void* sint,
                                      void* kS, void* vS, int kv8,
                                      void* scratch, void* cnt, int split,
                                      int batch, int nh, int kvh, int hd,
                                      int S, float scale, float softcap,
                                      int window, hipStream_t stream) {
  if (split < 1 || batch < 1 || kvh < 1 || nh % kvh)
    return hipErrorInvalidValue;
  split = split < AD_MAX_SPLIT ? split : AD_MAX_SPLIT;
  AdArgs a = {(const u16*)qkv, kc, vc, (u16*)out, (const int*)len_ptr,
              (const float*)cost, (const float*)sint, (float*)kS, (float*)vS,
              (float*)scratch, (int*)cnt, nh, kvh, S, 1, scale, softcap,
              window};
  switch (hd) {
    case 16: return ad_run<16>(a, kv8, split, batch, stream);
    case 32: return ad_run<32>(a, kv8, split, batch, stream);
    case 64: return ad_mfma<64>(a, kv8, split, batch, stream);
    case 128: return ad_mfma<128>(a, kv8, split, batch, stream);
    case 256: return ad_mfma<256>(a, kv8, split, batch, stream);
    case 512: return ad_run<512>(a, kv8, split, batch, stream);
  }
  return hipErrorInvalidValue;
}
