// mid_gemm.h — products of some rows (mid_gemm.hip) for the launchers that
// hand theirs on.
#pragma once
#include <hip/hip_runtime.h>

// Whether it is faster than row_gemm, up to 16 rows without a gate.
bool mid_takes(bool f8, int M, int N, int K);

// How long it takes, to be compared with gemm_prompt's tiles: without end for
// more rows than it takes, nothing where it is faster than any.
float mid_time(bool f8, int M, int N, int K, bool glu, long part_floats,
               int ncnt);

extern "C" hipError_t launch_mid_gemm(
    const void* x, const void* w, const void* sx, const void* sw,
    const void* res, const void* bias, void* y, void* part, void* cnt,
    long part_floats, int ncnt, int M, int N, int K, int ldx, int ldr,
    int ldy, int act, int out_f32, float softcap, hipStream_t stream);
