// mid_gemm.h — products of some rows (mid_gemm.hip) for the launchers that
// hand theirs on.
#pragma once
#include <hip/hip_runtime.h>

// Whether it is the faster one: gate, and M at most 16 beside row_gemm, more
// beside gemm_prompt.
bool mid_takes(bool f8, int M, int N, int K, bool glu);

extern "C" hipError_t launch_mid_gemm(
    const void* x, const void* w, const void* sx, const void* sw,
    const void* res, const void* bias, void* y, void* part, void* cnt,
    long part_floats, int ncnt, int M, int N, int K, int ldx, int ldr,
    int ldy, int act, int out_f32, float softcap, hipStream_t stream);
