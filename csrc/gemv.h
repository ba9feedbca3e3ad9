// gemv.h — what a product of one row does to its input on the way:
//   RAW         x
//   NORM        rmsnorm(x) * g            (g fp32, Gemma's +1 folded in)
//   GLU         act(x) * x2               (act 0: SiLU, 1: tanh-GELU)
//   NORM2       h' = x2 + rmsnorm(x) * g, kept by one block; then
//               rmsnorm(h') * g2          (Gemma's two norms around a branch)
//   NORM_EMBED  row *x2 of the table x times escale, kept by one block; then
//               rmsnorm * g
#pragma once
#define STAGE_RAW 0
#define STAGE_NORM 1
#define STAGE_GLU 2
#define STAGE_NORM2 3
#define STAGE_NORM_EMBED 4
