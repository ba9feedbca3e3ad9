// attn_prefill.h — arguments of the prompt attention kernels.
#pragma once
#include "common.h"

struct ApArgs {
  const u16* q;          // [M, ldq], heads of head_dim values, rotated
  const void* kc;        // [kvh, S, head_dim] bf16, or e4m3 with kS / vS
  const void* vc;
  u16* out;              // [M, nh * head_dim]
  const int* len_ptr;    // position of row 0
  // Rows of several sequences, kc .. vS the pools of all: of each block's
  // tile its number in the sequence, the sequence's first row, rows,
  // position of the first and pool.
  const int* tiles;
  const float* kS;       // [kvh, S]
  const float* vS;
  float* part;           // split keys: [split, kvh, rows, head_dim + 4]
  int M, nh, kvh, ldq, S, fold, by_row;
  float scale, softcap;
  int window;
};
