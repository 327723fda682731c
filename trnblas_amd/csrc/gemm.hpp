// What gemm.hip and sgemm.hip share: the argument block of a GEMM / SYRK
// launch and the accumulation chain length.
#pragma once

#include "common.hpp"

namespace trnblas {

struct GemmArgs {
  int M, N, K;
  float alpha, beta;
  const void* A;
  int64_t lda, sA;
  const void* B;
  int64_t ldb, sB;
  const void* C;
  int64_t ldc, sC;
  void* D;
  int64_t ldd, sD;
  int batch;
  int tiles_m, tiles_n;  // tile grid of one batch entry
  int ntiles;            // tiles of the launch (all batch entries, or the SYRK triangle)
  int nk;                // k-tiles per tile
  int uplo;              // SYRK: 0 = lower triangle of C referenced, 1 = upper
  const int32_t* tri;    // SYRK: triangle flags of C (device), or null; see syrk_upper
  int vec4;              // SYRK: C and D take 4-element vector accesses (aligned, ld % 4 == 0)
  int vec2;              // sgemm_pipe_kernel: C and D take 2-element accesses (aligned, ld even)
  int sk_groups;         // stream-K workgroups (0 = data-parallel)
  int dp_tiles;          // under stream-K: leading tiles computed whole
  float* ws;             // stream-K partial tiles [sk_groups][2][BM * BN]
  int span;              // k-tiles per MFMA accumulation chain (chain_length / k-tile)
  int splits;            // sgemm.hip: k ranges per tile, partial tiles in ws (1 = whole tiles)
};

// Accumulation: the MFMA accumulator of a tile restarts from zero every
// chain_length(K) k values and each finished chain is added into a separate
// fp32 sum with a VALU add (fold_span). One chain over all of K rounds the
// running sum at every step: a sum of 8192 same-sign products (a SYRK
// diagonal) came out 5.3e-6 off. With chains of L values folded into the sum
// the error is that of one L-long chain (averaged over the K / L chains)
// plus that of K / L folds. Measured on the MI355X, largest componentwise
// error over the whole output with U(0, 1) operands, L = 64 / 128 / 256:
// SYRK 1030 x 260 (one chain dominates) 3.5e-7 / 5.7e-7 / 1.05e-6; SYRK
// 4096 x 8192 (the folds dominate) 7.8e-7 / 6.2e-7 / 4.5e-7; C2a (N(0, 1))
// 6.1e-7 / 4.2e-7 / 3.6e-7, at 1.094 / 1.057 / 1.046 ms. Hence L grows with
// K. 16-bit operands keep L >= 128 (two of their 64-wide k-tiles: the DMA
// kernel folds after an even number of k-tiles).
static inline int chain_length(int64_t K, int elem_bytes) {
  const int L = K <= 1024 ? 64 : K <= 4096 ? 128 : K < 16384 ? 256 : K < 65536 ? 512 : 1024;
  return elem_bytes == 2 && L < 128 ? 128 : L;
}

// fp32 GEMM on operands of any alignment (sgemm.hip): true, with *rc the
// launch's status, when one of its kernels serves these arguments better
// than gemm.hip's (`aligned`: the operands are ready for LDS DMA).
bool sgemm_launch(const GemmArgs& g, bool akc, bool bkc, bool aligned, size_t ws_bytes,
                  hipStream_t s, int* rc);

}  // namespace trnblas
