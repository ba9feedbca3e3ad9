// rglru.hip — gated linear recurrence behind a short causal convolution.
//
//   u_t = conv of the last `taps` inputs x (per channel, with bias)
//   r, i = sigmoid(block-diagonal maps of u_t)
//   log a = r * nl[c]           (nl = -C softplus(lam), from the host)
//   S_t = a S_{t-1} + sqrt(1 - a^2) i u_t,   out = S_t * gelu_tanh(y_t)
//
// Everything here is fp32.  With bf16 weights the gate products run on bf16
// MFMA with u cut into three bf16 pieces, which hold all its bits, so the
// products are exact and the sums fp32.
//
// State, one slot per sequence: S [slot, C], and a ring of the last `taps`
// inputs [slot, taps, C], the input of position p at p % taps, so a step
// writes an entry that no block of it reads.  Positions before 0 read as
// zero whatever the slot held.
//
// A run of tokens: chunks of 64 scan their own tokens with the channel's
// state as 0 (the run's first chunk: the stored state) and keep, per token,
// the state so far and the product of the decays; a second kernel folds
// the chunks before each one in.
#include "gemm_tile.h"
#include "hybrid.h"

#define CH 64      // chunk length
#define LS 68      // LDS row stride of a 64-wide fp32 tile (16-byte aligned)

struct RglruArgs {
  const float* P;             // fp32 projections [rows, ldp], biases added
  const float *cw, *cb;       // [taps, C], [C]
  const void* gates;          // [blocks, 2 (r, i), KP, KP], T, zero-padded
  const float *rb, *ib, *nl;  // [C]
  float *S, *ring;            // [slots, C], [slots, taps, C]
  float *A, *h;               // [rows, C]: decay products, local states
  void* out;                  // [rows, ldo]
  const int *slot, *pos;      // per row
  const int *seg_row0, *seg_len, *seg_slot, *seg_pos0;
  const int *chunk_row0, *chunk_len, *chunk_seg;
  int ldp, oy, ox, C, nb, bw, KP, taps, ldo, rows, nchunk;
};

DEVINL float gelu_tanh_f(float z) {
  // 0.5 (1 + tanh(w)) = sigmoid(2w)
  return z * fast_sigmoid(1.5957691216057308f * (z + 0.044715f * z * z * z));
}

// 1 - e^-x for x >= 0, without the cancellation near 0
DEVINL float one_minus_exp(float x, float e) {
  if (x > 0.5f) return 1.f - e;
  float s = 1.f - x * (1.f / 8.f);
#pragma unroll
  for (int k = 7; k >= 2; k--) s = 1.f - x * (1.f / (float)k) * s;
  return x * s;
}

// decay and input weight of one channel from the gate sums, their biases and
// its rate
DEVINL void recur(float rb, float ib, float nl, float r, float i, float u,
                  float& dec, float& add) {
  const float la = fast_sigmoid(r + rb) * nl;
  dec = fast_exp(la);
  add = __builtin_amdgcn_sqrtf(one_minus_exp(-2.f * la, dec * dec)) *
        fast_sigmoid(i + ib) * u;
}

// C += A B^T of 16 rows of fp32 `u` (LDS, this lane's row) and 16 rows of
// gate weights, over 64 bytes of the weights' rows; g is the lane group
template <typename T> struct GateMma;
template <> struct GateMma<float> {
  f4v a;
  DEVINL void load(const float* u, int g) { a = ld16(u + g * 4); }
  DEVINL f4v mma(f4v w, f4v c) const { return GemmMma<float>::mma(a, w, c); }
};
template <> struct GateMma<u16> {
  f4v p[3];
  DEVINL void load(const float* u, int g) {
    union { f4v f; u16 h[8]; } o[3];
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const f4v v = ld16(u + g * 8 + h * 4);
#pragma unroll
      for (int j = 0; j < 4; j++) {
        union { float f; uint32_t i; } x, q;
        x.f = v[j];
#pragma unroll
        for (int k = 0; k < 3; k++) {      // truncated, so the rest is exact
          q.i = x.i & 0xffff0000u;
          o[k].h[h * 4 + j] = (u16)(q.i >> 16);
          x.f -= q.f;
        }
      }
    }
#pragma unroll
    for (int k = 0; k < 3; k++) p[k] = o[k].f;
  }
  DEVINL f4v mma(f4v w, f4v c) const {
#pragma unroll
    for (int k = 2; k >= 0; k--) c = GemmMma<u16>::mma(p[k], w, c);
    return c;
  }
};

// ---- one token per row ------------------------------------------------
// a block: 16 channels of one part; 16 lanes per channel share its two dot
// products over the part's convolved inputs.  What bounds it is the way of all
// that it reads, so nothing waits for something else: taps, states and what
// the epilogue takes are asked for ahead of the convolution (us, 16 parts of
// 128, 4 taps: 4 rows 4.2 -> 3.3, 16 rows 6.3 -> 5.2, 64 rows 16.8 -> 13.1; tap
// after tap, behind a division of its own each, and the state at the end).
#define STEP_TAPS 4
template <typename T>
__global__ void __launch_bounds__(256) k_rglru_step(RglruArgs a) {
  constexpr int V = El<T>::V;
  extern __shared__ __attribute__((aligned(16))) float us[];   // [KP]
  const int r = blockIdx.y, nsl = (a.bw + 15) / 16;
  const int b = blockIdx.x / nsl, n0 = (blockIdx.x - b * nsl) * 16;
  const int tid = threadIdx.x, l = tid & 15, n = n0 + (tid >> 4);
  const size_t slot = a.slot[r];
  const int pos = a.pos[r];
  const float* x = a.P + (size_t)r * a.ldp + a.ox + b * a.bw;
  float* ring = a.ring + slot * a.taps * a.C + b * a.bw;
  const int nc = min(n, a.bw - 1);
  const T* wr = (const T*)a.gates + ((size_t)(2 * b) * a.KP + nc) * a.KP;
  const T* wi = wr + (size_t)a.KP * a.KP;
  f4v pr = ld16(wr + (l * V < a.KP ? l * V : 0));     // on their way early
  f4v pi = ld16(wi + (l * V < a.KP ? l * V : 0));
  const int cn = b * a.bw + nc, place = pos % a.taps;
  float* const S = a.S + slot * a.C + cn;
  const float s0 = *S, xn = x[nc], yn = a.P[(size_t)r * a.ldp + a.oy + cn];
  const float rb = a.rb[cn], ib = a.ib[cn], nl = a.nl[cn];
  for (int j = tid; j < a.KP; j += 256) {
    float u = 0.f;
    if (j < a.bw) {
      const int c = b * a.bw + j;
      const float wx = a.cw[(a.taps - 1) * a.C + c], xj = x[j];
      u = a.cb[c];
      // STEP_TAPS of them on the way at a time; those ahead of the first
      // position are read, in some place of the ring, and left out
      for (int t0 = 1; t0 < a.taps; t0 += STEP_TAPS) {
        float w[STEP_TAPS], v[STEP_TAPS];
#pragma unroll
        for (int i = 0; i < STEP_TAPS; i++) {
          const int t = min(t0 + i, a.taps - 1), at = place + t;
          w[i] = a.cw[(t - 1) * a.C + c];
          v[i] = ring[(at < a.taps ? at : at - a.taps) * a.C + j];
        }
#pragma unroll
        for (int i = 0; i < STEP_TAPS; i++)
          if (t0 + i < a.taps && pos - a.taps + t0 + i >= 0)
            u = fmaf(w[i], v[i], u);
      }
      u = fmaf(wx, xj, u);
    }
    us[j] = u;
  }
  __syncthreads();
  float sr = 0.f, si = 0.f;
  for (int k = l * V; k < a.KP; k += 16 * V) {
    union { f4v f; T t[V]; } vr, vi;
    vr.f = k == l * V ? pr : ld16(wr + k);
    vi.f = k == l * V ? pi : ld16(wi + k);
#pragma unroll
    for (int j = 0; j < V; j++) {
      sr = fmaf(El<T>::ld(vr.t[j]), us[k + j], sr);
      si = fmaf(El<T>::ld(vi.t[j]), us[k + j], si);
    }
  }
#pragma unroll
  for (int m = 1; m < 16; m <<= 1) {
    sr += __shfl_xor(sr, m);
    si += __shfl_xor(si, m);
  }
  if (l == 0 && n < a.bw) {
    const int c = b * a.bw + n;
    float dec, add;
    recur(rb, ib, nl, sr, si, us[n], dec, add);
    const float s = pos == 0 ? add : dec * s0 + add;
    *S = s;
    ring[place * a.C + n] = xn;
    ((T*)a.out)[(size_t)r * a.ldo + c] = El<T>::st(s * gelu_tanh_f(yn));
  }
}

// ---- runs of tokens -----------------------------------------------------
// input of channel c at position p of a run (its first row0 holds pos0);
// p >= pos0 - taps + 1
DEVINL float run_input(const RglruArgs& a, const float* x, const float* ring,
                       int pos0, int p, int c) {
  if (p >= pos0) return x[(size_t)(p - pos0) * a.ldp + c];
  return p >= 0 ? ring[(p % a.taps) * a.C + c] : 0.f;
}

// convolution, gates and the scan inside a chunk, 64 channels of one part:
// wave w holds tokens 16w .. 16w+15
template <typename T>
__global__ void __launch_bounds__(256) k_rglru_local(RglruArgs a) {
  // inputs u, then the weighted inputs; decays
  __shared__ __attribute__((aligned(16))) float us[CH * LS], ds[CH * LS];
  __shared__ float endA[4][64], endH[4][64];
  constexpr int KC = 64 / sizeof(T);         // weights in 64 bytes
  const int nsl = (a.bw + 63) / 64, c = blockIdx.y;
  const int b = blockIdx.x / nsl, n0 = (blockIdx.x - b * nsl) * 64;
  const int tid = threadIdx.x, wave = wave_index(), lane = tid & 63;
  const int lr = lane & 15, g = lane >> 4;
  const int sg = a.chunk_seg[c], crow = a.chunk_row0[c], len = a.chunk_len[c];
  const int row0 = a.seg_row0[sg], pos0 = a.seg_pos0[sg];
  const size_t slot = a.seg_slot[sg];
  const float* x = a.P + (size_t)row0 * a.ldp + a.ox + b * a.bw;
  const float* ring = a.ring + slot * a.taps * a.C + b * a.bw;
  const int at = pos0 + crow - row0;                // position of token 0
  f4v ar[4], ai[4];
#pragma unroll
  for (int j = 0; j < 4; j++) ar[j] = ai[j] = f4v{0.f, 0.f, 0.f, 0.f};
  // the slab of this block's own channels comes last and stays in us
  const int nk = a.KP / 64;
  for (int s = 1; s <= nk; s++) {
    const int k0 = (n0 / 64 + s) % nk * 64, j = k0 + lane, cj = b * a.bw + j;
    float u[16];
    const bool live = j < a.bw;
#pragma unroll
    for (int t = 0; t < 16; t++) u[t] = live ? a.cb[cj] : 0.f;
    if (live) {
      const int p0 = at + wave * 16;
      if (a.taps <= 4) {
        float w[4], xv[19];
#pragma unroll
        for (int q = 0; q < 4; q++)
          w[q] = q < a.taps ? a.cw[(a.taps - 1 - q) * a.C + cj] : 0.f;
#pragma unroll
        for (int t = 0; t < 19; t++) xv[t] = 0.f;
        if (p0 - 3 >= pos0 && p0 + 15 < at + len) {      // all in the run
          const float* xp = x + (size_t)(p0 - 3 - pos0) * a.ldp + j;
#pragma unroll
          for (int t = 0; t < 19; t++) xv[t] = xp[(size_t)t * a.ldp];
        } else {
#pragma unroll
          for (int t = 0; t < 19; t++) {
            const int p = p0 + t - 3;
            if (p - at < len && p >= pos0 - a.taps + 1)
              xv[t] = run_input(a, x, ring, pos0, p, j);
          }
        }
#pragma unroll
        for (int t = 0; t < 16; t++)
#pragma unroll
          for (int q = 3; q >= 0; q--) u[t] = fmaf(w[q], xv[t + 3 - q], u[t]);
      } else {
        for (int q = a.taps - 1; q >= 0; q--) {
          const float w = a.cw[(a.taps - 1 - q) * a.C + cj];
#pragma unroll
          for (int t = 0; t < 16; t++)
            if (p0 + t - at < len)
              u[t] = fmaf(w, run_input(a, x, ring, pos0, p0 + t - q, j), u[t]);
        }
      }
    }
    const T* gr = (const T*)a.gates +
                  ((size_t)(2 * b) * a.KP + n0 + lr) * a.KP + k0 + g * (KC / 4);
    const T* gi = gr + (size_t)a.KP * a.KP;
    // the tokens of a wave are its own: no barrier until the chunk's scan
    wave_sync();
#pragma unroll
    for (int t = 0; t < 16; t++) us[(wave * 16 + t) * LS + lane] = u[t];
    wave_sync();
#pragma unroll
    for (int k = 0; k < 64; k += KC) {
      f4v wr[4], wi[4];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        wr[q] = ld16(gr + (size_t)q * 16 * a.KP + k);
        wi[q] = ld16(gi + (size_t)q * 16 * a.KP + k);
      }
      GateMma<T> m;
      m.load(us + (wave * 16 + lr) * LS + k, g);
#pragma unroll
      for (int q = 0; q < 4; q++) {
        ar[q] = m.mma(wr[q], ar[q]);
        ai[q] = m.mma(wi[q], ai[q]);
      }
    }
  }
  // decays and weighted inputs of the wave's tokens
  wave_sync();
#pragma unroll
  for (int q = 0; q < 4; q++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int t = wave * 16 + g * 4 + r, n = q * 16 + lr;
      float dec = 1.f, add = 0.f;
      if (t < len && n0 + n < a.bw) {
        const int c = b * a.bw + n0 + n;
        recur(a.rb[c], a.ib[c], a.nl[c], ar[q][r], ai[q][r], us[t * LS + n],
              dec, add);
      }
      ds[t * LS + n] = dec;
      us[t * LS + n] = add;
    }
  wave_sync();
  float pa = 1.f, ph = 0.f, da[16], ha[16];
#pragma unroll
  for (int t = 0; t < 16; t++) {
    const int o = (wave * 16 + t) * LS + lane;
    pa *= ds[o];
    ph = fmaf(ds[o], ph, us[o]);
    da[t] = pa;
    ha[t] = ph;
  }
  endA[wave][lane] = pa;
  endH[wave][lane] = ph;
  __syncthreads();
  if (n0 + lane >= a.bw) return;
  const int ch = b * a.bw + n0 + lane;
  float ca = 1.f, chs = crow == row0 && pos0 > 0 ? a.S[slot * a.C + ch] : 0.f;
  for (int w = 0; w < wave; w++) {
    chs = fmaf(endA[w][lane], chs, endH[w][lane]);
    ca *= endA[w][lane];
  }
#pragma unroll
  for (int t = 0; t < 16; t++) {
    const int tt = wave * 16 + t;
    if (tt < len) {
      a.A[(size_t)(crow + tt) * a.C + ch] = da[t] * ca;
      a.h[(size_t)(crow + tt) * a.C + ch] = fmaf(da[t], chs, ha[t]);
    }
  }
}

// fold in the chunks before, gate, and leave the run's last state and inputs
template <typename T>
__global__ void __launch_bounds__(256) k_rglru_finish(RglruArgs a) {
  const int lane = threadIdx.x & 63, wave = wave_index();
  const int ch = blockIdx.x * 64 + lane, c = blockIdx.y;
  if (ch >= a.C) return;
  const int sg = a.chunk_seg[c], crow = a.chunk_row0[c], len = a.chunk_len[c];
  const int row0 = a.seg_row0[sg], slen = a.seg_len[sg];
  const int first = c - (crow - row0) / CH;
  float carry = 0.f;                   // the first chunk's states are whole
#pragma unroll 8
  for (int k = first; k < c; k++) {
    const size_t e = (size_t)(a.chunk_row0[k] + CH - 1) * a.C + ch;
    carry = fmaf(a.A[e], carry, a.h[e]);
  }
  float s = 0.f;
#pragma unroll 4
  for (int t = wave; t < len; t += 4) {
    const size_t r = crow + t;
    s = fmaf(a.A[r * a.C + ch], carry, a.h[r * a.C + ch]);
    ((T*)a.out)[r * a.ldo + ch] =
        El<T>::st(s * gelu_tanh_f(a.P[r * a.ldp + a.oy + ch]));
  }
  if (crow + len != row0 + slen) return;
  const size_t slot = a.seg_slot[sg];
  if (wave == (len - 1) % 4) a.S[slot * a.C + ch] = s;
  for (int q = wave; q < min(a.taps, slen); q += 4) {
    const int t = slen - 1 - q, p = a.seg_pos0[sg] + t;
    a.ring[(slot * a.taps + p % a.taps) * a.C + ch] =
        a.P[(size_t)(row0 + t) * a.ldp + a.ox + ch];
  }
}

// ---- launchers ------------------------------------------------------------
static bool bad_shape(const RglruArgs& a) {
  return a.rows < 1 || a.nb < 1 || a.bw < 1 || a.C != a.nb * a.bw ||
         a.KP % 64 || a.KP < a.bw || a.taps < 1 || a.ldo < a.C;
}

extern "C" hipError_t launch_rglru_step(int f32, const RglruArgs* a,
                                        hipStream_t s) {
  if (bad_shape(*a)) return hipErrorInvalidValue;
  dim3 grid(a->nb * ((a->bw + 15) / 16), a->rows);
  const size_t lds = (size_t)a->KP * sizeof(float);
  if (lds > 150 * 1024) return hipErrorInvalidValue;
  if (f32) {
    RAISE_LDS(k_rglru_step<float>);
    hipLaunchKernelGGL(k_rglru_step<float>, grid, dim3(256), lds, s, *a);
  } else {
    RAISE_LDS(k_rglru_step<u16>);
    hipLaunchKernelGGL(k_rglru_step<u16>, grid, dim3(256), lds, s, *a);
  }
  return hipGetLastError();
}

extern "C" hipError_t launch_rglru_run(int f32, const RglruArgs* a,
                                       hipStream_t s) {
  if (bad_shape(*a) || a->nchunk < 1) return hipErrorInvalidValue;
  dim3 local(a->nb * ((a->bw + 63) / 64), a->nchunk);
  dim3 fin((a->C + 63) / 64, a->nchunk);
  if (f32) {
    hipLaunchKernelGGL(k_rglru_local<float>, local, dim3(256), 0, s, *a);
    hipLaunchKernelGGL(k_rglru_finish<float>, fin, dim3(256), 0, s, *a);
  } else {
    hipLaunchKernelGGL(k_rglru_local<u16>, local, dim3(256), 0, s, *a);
    hipLaunchKernelGGL(k_rglru_finish<u16>, fin, dim3(256), 0, s, *a);
  }
  return hipGetLastError();
}
