// common.h — shared types/helpers for the CDNA4 kernel sources.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

typedef unsigned short u16;
typedef short s8v __attribute__((ext_vector_type(8)));    // 16 B of bf16
typedef float f4v __attribute__((ext_vector_type(4)));
typedef uint32_t u4v_ __attribute__((ext_vector_type(4)));  // 16 B raw

#define DEVINL __device__ __forceinline__

DEVINL float b2f(u16 u) {
  union { float f; uint32_t i; } c;
  c.i = ((uint32_t)u) << 16;
  return c.f;
}

DEVINL u16 f2b(float f) {
  union { float f; uint32_t i; } c;
  c.f = f;
  uint32_t u = c.i;
  if ((u & 0x7fffffffu) > 0x7f800000u) return (u16)0x7fc0;  // NaN
  u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even
  return (u16)(u >> 16);
}

// Sum over a wave, alike in all lanes.  Lanes 1, 2, 4 and 8 away are operands
// of the add itself (where four lanes agree, the mirror image in eight is the
// lane four away), rows of 16 and halves are swapped in registers: 40 cycles,
// by ds_bpermute 400.
template <int C> DEVINL float dpp_from(float v) {
  return __uint_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_uint(v), C, 0xf, 0xf, true));
}
DEVINL float wave_reduce_sum(float v) {
  v += dpp_from<0xB1>(v);
  v += dpp_from<0x4E>(v);
  v += dpp_from<0x141>(v);
  v += dpp_from<0x128>(v);
  uint32_t u = __float_as_uint(v);
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  u = __float_as_uint(v);
  const auto s = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}
DEVINL float wave_reduce_max(float v) {
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) v = fmaxf(v, __shfl_xor(v, m));
  return v;
}

// act 0: SiLU, 1: tanh-GELU
DEVINL float gate_act(float x, int act) {
  if (act == 0) return x / (1.f + __expf(-x));
  const float c = 0.7978845608028654f * (x + 0.044715f * x * x * x);
  return 0.5f * x * (1.f + tanhf(c));
}

typedef float f2v __attribute__((ext_vector_type(2)));

// 8 floats (pre-scaled by rs) -> 8 packed e4m3 bytes
DEVINL unsigned long long f32x8_to_fp8(const float* f, float rs) {
  uint32_t lo = 0, hi = 0;
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(f[0] * rs, f[1] * rs, lo, false);
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(f[2] * rs, f[3] * rs, lo, true);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(f[4] * rs, f[5] * rs, hi, false);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(f[6] * rs, f[7] * rs, hi, true);
  return (unsigned long long)lo | ((unsigned long long)hi << 32);
}

// What a block leaves for the last of several blocks to add up.  They may run
// on dies with an L2 of their own: a release at device scope writes a die's
// L2 back and an acquire empties the reader's, which cost a product of 256
// blocks 3 us and one of 384 eleven (37x2048x2048 in two parts of K: 10.9 us
// with them, 8.0 without; 37x3072x2048 in two: 21.2 and 10.9).  So the parts
// themselves go past the L2 (relaxed atomics of device scope are coherent by
// themselves), and a wait puts them ahead of the block's arrival.
DEVINL void part_put(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
DEVINL float part_get(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Four of them, the last two `far` floats behind the first: lanes side by side
// leave whole lines (16 bytes a lane in two halves of their own left half lines
// twice: 1999x2048x8192 in two parts of K by 128x256 81 us, so 72; 300 rows in
// three 36.6, 33.9; 700x3584x14336 in three 103, 95).
union PartSums { f4v v; unsigned long long u[2]; };
DEVINL void part_put4(float* p, int far, f4v v) {     // 8-byte aligned
  const PartSums s = {v};
#pragma unroll
  for (int i = 0; i < 2; i++)
    __hip_atomic_store((unsigned long long*)(p + i * far), s.u[i],
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
DEVINL f4v part_get4(const float* p, int far) {
  PartSums s;
#pragma unroll
  for (int i = 0; i < 2; i++)
    s.u[i] = __hip_atomic_load((const unsigned long long*)(p + i * far),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return s.v;
}
// True in the last of n blocks at cnt, which is left zero; all threads.
DEVINL bool last_block(int* cnt, int n, int* flag) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    const int t = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
    if (t == n - 1)
      __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *flag = t == n - 1;
  }
  __syncthreads();
  return *flag;
}
