// gemv.h — products of one row: kinds of weights, sums over lanes, and what a
// product does to its input on the way:
//   RAW         x
//   NORM        rmsnorm(x) * g            (g fp32, Gemma's +1 folded in)
//   GLU         act(x) * x2               (act 0: SiLU, 1: tanh-GELU)
//   NORM2       h' = x2 + rmsnorm(x) * g, kept by one block; then
//               rmsnorm(h') * g2          (Gemma's two norms around a branch)
//   NORM_EMBED  row *x2 of the table x times escale, kept by one block; then
//               rmsnorm * g
#pragma once
#include "common.h"

#define STAGE_RAW 0
#define STAGE_NORM 1
#define STAGE_GLU 2
#define STAGE_NORM2 3
#define STAGE_NORM_EMBED 4

enum { GV_BF16 = 0, GV_FP8 = 1, GV_FP4 = 2 };

template <int WT> constexpr int gv_e() {   // weights of 16 bytes
  return WT == GV_BF16 ? 8 : WT == GV_FP8 ? 16 : 32;
}

// the value of lane ^ W (W 7: mirrored in eight, W 8 and 12: turned in 16)
template <int W> DEVINL float gv_from(float v) {
  constexpr int C = W == 1 ? 0xB1 : W == 2 ? 0x4E : W == 7 ? 0x141
                    : W == 8 ? 0x128 : 0x124;
  return __uint_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_uint(v), C, 0xf, 0xf, true));
}
DEVINL float gv_halves(float v) {          // sums of 16 lanes -> of 64
  uint32_t u = __float_as_uint(v);
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  u = __float_as_uint(v);
  const auto s = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}
DEVINL float gv_sum(float v) {
  v += gv_from<1>(v);
  v += gv_from<2>(v);
  v += gv_from<8>(v);
  v += gv_from<12>(v);
  return gv_halves(v);
}
// sums of R rows (to the next power of two) over the lanes: row l in lane l
template <int R> DEVINL float gv_rows(float* v, int lane) {
  if constexpr (R == 8) {                  // pairs of lanes that add up to 7
    const bool up = lane & 4;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const float keep = up ? v[r + 4] : v[r], give = up ? v[r] : v[r + 4];
      v[r] = keep + gv_from<7>(give);
    }
  }
  if constexpr (R >= 4) {
    const bool up = lane & 2;
#pragma unroll
    for (int r = 0; r < 2; r++) {
      const float keep = up ? v[r + 2] : v[r], give = up ? v[r] : v[r + 2];
      v[r] = keep + gv_from<2>(give);
    }
  }
  float s;
  if constexpr (R >= 2) {
    const bool up = lane & 1;
    const float keep = up ? v[1] : v[0], give = up ? v[0] : v[1];
    s = keep + gv_from<1>(give);
  } else {
    s = v[0] + gv_from<1>(v[0]);
  }
  if constexpr (R < 4) s += gv_from<2>(s);
  s += gv_from<8>(s);
  if constexpr (R < 8) s += gv_from<12>(s);
  return gv_halves(s);
}
