// gemm_tile.h — the MFMA main loop that the dense, per-head and grouped
// GEMM kernels share: C[BM,BN] += A[BM,K] * B[BN,K]^T.
//
// T = u16 (bf16, v_mfma_f32_16x16x32_bf16) or float (true fp32,
// v_mfma_f32_16x16x4_f32).  A K-slab is 128 bytes a row for both types
// (64 bf16 or 32 floats), so the staging, the swizzle and the fragment
// addresses are the same; a 16-byte fragment feeds one bf16 MFMA or four
// fp32 ones (the order of k inside a slab is free as long as A and B
// agree on it).
//
// 4 waves (2x2), each a (BM/2)x(BN/2) sub-tile of 16x16 fragments.  Two to
// four LDS buffers (up to 72 KB, for two blocks a CU) filled by
// global_load_lds (16 B/lane), one barrier per slab that waits for the next
// slab and leaves the DMA behind it in flight: drained at each barrier a slab
// cost the one to two microseconds that a trip takes.  An array a buffer and
// a loop unrolled over them let the compiler see that a DMA into one does not
// touch what is read from another; it would wait for all of it before the
// reads otherwise.  1664x2048 outputs of K 2048 and 8192, 128x64 tiles: 70 us
// on average, now 51.
// Without DEEP two buffers, drained at each barrier, and the schedule is the
// compiler's: for 128x128, which has no room for a third, for fp32, which is
// bound by its products (2048x6144x1024: 202 us, in flight 273), and where
// more than two blocks would share a CU, which they do with two buffers only
// (513x8192x2048 in 640 blocks of 128x64: 30.7 us, in flight 33.5).
// LDS rows are XOR-swizzled (slot ^= row & 7); the DMA writes lane-linear, so
// the swizzle sits in the per-lane source address and in the fragment reads.
//
// `arow` / `brow` map a tile row (clamped by the caller to something
// readable) to its first element, which is how row gathers and
// per-expert weight bases come in.  K must be a multiple of 64.
#pragma once
#include "common.h"

typedef short gt_bf8 __attribute__((ext_vector_type(8)));

template <typename T> struct GemmMma;

template <> struct GemmMma<u16> {
  static constexpr int BK = 64;
  DEVINL static f4v mma(f4v a, f4v b, f4v c) {
    union { f4v f; gt_bf8 h; } ua, ub;
    ua.f = a; ub.f = b;
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(ua.h, ub.h, c, 0, 0, 0);
  }
};

template <> struct GemmMma<float> {
  static constexpr int BK = 32;
  DEVINL static f4v mma(f4v a, f4v b, f4v c) {
#pragma unroll
    for (int j = 0; j < 4; j++)
      c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], c, 0, 0, 0);
    return c;
  }
};

// Barrier after the wave's LDS reads and all but its last N DMA loads; the
// builtin tells the compiler which of them are over.
template <int N> DEVINL void gemm_meet() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | (N >> 4 << 14) | 7 << 4);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <int BM, int BN, typename T, bool DEEP = true, class ARow, class BRow>
DEVINL void gemm_mainloop(f4v (&acc)[BM / 32][BN / 32], ARow arow, BRow brow,
                          int k_lo, int nt) {
  constexpr int FM = BM / 32, FN = BN / 32;
  constexpr int BK = GemmMma<T>::BK;
  constexpr int VE = 16 / sizeof(T);   // elements of a 16-byte slot
  constexpr int ROOM = 73728 / ((BM + BN) * 128);       // buffers
  constexpr bool DRAIN = !DEEP || ROOM < 3;
  constexpr int NS = DRAIN ? 2 : ROOM > 4 ? 4 : ROOM;
  constexpr int PS = FM + FN;                // DMA of a wave and slab
#define GEMM_BUF(i)                                                          \
  __shared__ __attribute__((aligned(16))) char A##i[NS > i ? BM * 128 : 16], \
      B##i[NS > i ? BN * 128 : 16];
  GEMM_BUF(0) GEMM_BUF(1) GEMM_BUF(2) GEMM_BUF(3)
#undef GEMM_BUF
  char* const A[4] = {A0, A1, A2, A3};
  char* const B[4] = {B0, B1, B2, B3};
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int wrow = wave >> 1, wcol = wave & 1;
  const int g_r = lane >> 3, g_s = lane & 7;

#pragma unroll
  for (int i = 0; i < FM; i++)
#pragma unroll
    for (int j = 0; j < FN; j++) acc[i][j] = {0.f, 0.f, 0.f, 0.f};

  const T* pa[FM];
  const T* pb[FN];
#pragma unroll
  for (int i = 0; i < FM; i++) {
    int r = wave * (BM / 4) + i * 8 + g_r;
    pa[i] = arow(r) + k_lo + (g_s ^ (r & 7)) * VE;
  }
#pragma unroll
  for (int i = 0; i < FN; i++) {
    int r = wave * (BN / 4) + i * 8 + g_r;
    pb[i] = brow(r) + k_lo + (g_s ^ (r & 7)) * VE;
  }
  auto stage = [&](char* As, char* Bs, int kt) {
#pragma unroll
    for (int i = 0; i < FM; i++)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) uint32_t*)(
              pa[i] + (size_t)kt * BK),
          (__attribute__((address_space(3))) uint32_t*)(
              As + (wave * (BM / 4) + i * 8) * 128),
          16, 0, 0);
#pragma unroll
    for (int i = 0; i < FN; i++)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) uint32_t*)(
              pb[i] + (size_t)kt * BK),
          (__attribute__((address_space(3))) uint32_t*)(
              Bs + (wave * (BN / 4) + i * 8) * 128),
          16, 0, 0);
  };

  const int fr = lane & 15, fk = lane >> 4;
  if (nt < 1) return;
  if constexpr (DRAIN) {
    stage(A0, B0, 0);
    __syncthreads();
    for (int t = 0; t < nt; t++) {
      const char *As = t & 1 ? A1 : A0, *Bs = t & 1 ? B1 : B0;
      if (t + 1 < nt) stage(t & 1 ? A0 : A1, t & 1 ? B0 : B1, t + 1);
#pragma unroll
      for (int h = 0; h < 2; h++) {
        f4v a[FM], b[FN];
#pragma unroll
        for (int i = 0; i < FM; i++) {
          const int ra = wrow * (BM / 2) + i * 16 + fr;
          a[i] = *(const f4v*)(As + ra * 128 + ((h * 4 + fk) ^ (ra & 7)) * 16);
        }
#pragma unroll
        for (int j = 0; j < FN; j++) {
          const int rb = wcol * (BN / 2) + j * 16 + fr;
          b[j] = *(const f4v*)(Bs + rb * 128 + ((h * 4 + fk) ^ (rb & 7)) * 16);
        }
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
          for (int j = 0; j < FN; j++)
            acc[i][j] = GemmMma<T>::mma(a[i], b[j], acc[i][j]);
      }
      __syncthreads();               // the DMA is over, the reads are done
    }
    return;
  }
  // Half a slab of fragments ahead: the hand-over stands between two halves'
  // products, when the second half is in registers already.
  f4v a[2][FM], b[2][FN];
  auto fetch = [&](int h, const char* As, const char* Bs) {
#pragma unroll
    for (int i = 0; i < FM; i++) {
      int ra = wrow * (BM / 2) + i * 16 + fr;
      a[h][i] = *(const f4v*)(As + ra * 128 + ((h * 4 + fk) ^ (ra & 7)) * 16);
    }
#pragma unroll
    for (int j = 0; j < FN; j++) {
      int rb = wcol * (BN / 2) + j * 16 + fr;
      b[h][j] = *(const f4v*)(Bs + rb * 128 + ((h * 4 + fk) ^ (rb & 7)) * 16);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto mma = [&](int h) {
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
      for (int j = 0; j < FN; j++)
        acc[i][j] = GemmMma<T>::mma(a[h][i], b[h][j], acc[i][j]);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto slab = [&](char* As, char* Bs, const char* An, const char* Bn, int t,
                  bool steady) {
    fetch(1, As, Bs);
    mma(0);
    if (steady) {
      gemm_meet<PS * (NS - 2)>();
      stage(As, Bs, t + NS);
      fetch(0, An, Bn);
    } else if (t + 1 < nt) {
      gemm_meet<0>();
      if (t + NS < nt) stage(As, Bs, t + NS);
      fetch(0, An, Bn);
    }
    mma(1);
  };
#pragma unroll
  for (int u = 0; u < NS; u++)
    if (u < nt) stage(A[u], B[u], u);
  if (nt >= NS) gemm_meet<PS * (NS - 1)>();
  else gemm_meet<0>();
  fetch(0, A[0], B[0]);
  int t = 0;
  for (; t + 2 * NS <= nt; t += NS) {        // free of conditions
#pragma unroll
    for (int u = 0; u < NS; u++)
      slab(A[u], B[u], A[(u + 1) % NS], B[(u + 1) % NS], t + u, true);
  }
  for (; t < nt; t += NS) {
#pragma unroll
    for (int u = 0; u < NS; u++)
      if (t + u < nt)
        slab(A[u], B[u], A[(u + 1) % NS], B[(u + 1) % NS], t + u, false);
  }
}

// C layout: element (row, col) of fragment (i, j), register r
//   row = wrow*BM/2 + i*16 + (lane>>4)*4 + r, col = wcol*BN/2 + j*16 + lane%16
template <int BM> DEVINL int gemm_row0(int i) {
  return ((threadIdx.x >> 6) >> 1) * (BM / 2) + i * 16 +
         ((threadIdx.x & 63) >> 4) * 4;
}
template <int BN> DEVINL int gemm_col(int j) {
  return ((threadIdx.x >> 6) & 1) * (BN / 2) + j * 16 + (threadIdx.x & 15);
}
