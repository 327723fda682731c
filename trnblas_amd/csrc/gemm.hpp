// What the GEMM / SYRK sources share: the argument block of a launch, the
// accumulation chain length, the SYRK tile order and triangle rule, and the
// epilogue of the 32 x 32 kernels.
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
  const char** plan;     // trnblas_hip_gemm_plan: receives the kernel's name, nothing is launched
};

// True when only the kernel's name is asked for.
static inline bool planned(const GemmArgs& g, const char* kernel) {
  if (g.plan) *g.plan = kernel;
  return g.plan != nullptr;
}

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

// Lower-triangle tile t -> (tm, tn), tm >= tn, of a triangle T tiles on a
// side, in groups of 8 tile rows: group G (rows 8G .. 8G + R - 1, R = 8 but
// for the last) lists its whole columns tn < 8G (R tiles each, top to
// bottom), then its own R-row triangle column by column; groups start at
// tile 32 G^2 + 4 G. Consecutive tiles (one XCD's share of a round) then
// cover an 8-row, 8-column block of operand panels (13-20 distinct panels per
// 64 tiles of a 32-tile side, against ~35 for a row-major walk).
__device__ __forceinline__ void tri_tile(int t, int T, int& tm, int& tn) {
  int G = (int)((sqrtf(16.0f + 128.0f * (float)t) - 4.0f) * (1.0f / 64.0f));
  while (G > 0 && 32 * G * G + 4 * G > t) --G;
  while ((G + 1) * 8 < T && 32 * (G + 1) * (G + 1) + 4 * (G + 1) <= t) ++G;
  int u = t - (32 * G * G + 4 * G);
  const int R = min(8, T - 8 * G);
  if (u < 8 * G * R) {
    tm = 8 * G + u % R;
    tn = u / R;
    return;
  }
  u -= 8 * G * R;
  int c = 0;
  while (u >= R - c) {
    u -= R - c;
    ++c;
  }
  tm = 8 * G + c + u;
  tn = 8 * G + c;
}

// SYRK: whether the upper triangle of C is the one referenced: g.uplo, or,
// with triangle flags (flags[0]: the strict upper triangle holds a nonzero,
// flags[1]: the strict lower one), the other triangle when only that one
// holds off-diagonal entries (the rule of trnblas/level3.py:305-329, decided
// on the device so the host need not wait for the flags before the launch).
__device__ __forceinline__ int syrk_upper(const GemmArgs& g) {
  int up = g.uplo;
  if (g.tri != nullptr) {
    const int has_up = g.tri[0], has_lo = g.tri[1];
    if (up ? (has_lo && !has_up) : (has_up && !has_lo)) up ^= 1;
  }
  return up;
}

// The end of a 32 x 32 tile (corner (m0, n0)) whose raw sums the workgroup's
// waves left in part[wave]: the sums added in wave order, alpha / beta, and
// the store, by the first 256 threads, four columns each. SYRK: only elements
// on or below the diagonal, each written to both triangles.
template <typename T, bool SYRK, int WAVES>
__device__ __forceinline__ void direct_out(const GemmArgs& g, const float (&part)[WAVES][32 * 32],
                                           int bat, int m0, int n0) {
  typedef T vec4 __attribute__((ext_vector_type(4), aligned(sizeof(T))));
  const int tid = threadIdx.x;
  if (tid >= 256) return;
  const int m = m0 + (tid >> 3), n = n0 + 4 * (tid & 7);
  f32x4 v = *reinterpret_cast<const f32x4*>(&part[0][4 * tid]);
#pragma unroll
  for (int s = 1; s < WAVES; ++s) v += *reinterpret_cast<const f32x4*>(&part[s][4 * tid]);
  const int last = SYRK ? m + 1 : g.N;  // columns of this row
  if (m >= g.M || n >= last) return;
  const T* C = static_cast<const T*>(g.C) + (g.C ? bat * g.sC : 0);
  T* D = static_cast<T*>(g.D) + bat * g.sD;
  const bool up = SYRK && g.beta != 0.0f && syrk_upper(g);
  float c[4];
#pragma unroll
  for (int u = 0; u < 4; ++u)
    c[u] = g.beta != 0.0f && n + u < last
               ? (float)C[up ? (int64_t)(n + u) * g.ldc + m : (int64_t)m * g.ldc + n + u]
               : 0.0f;
  T o[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    v[u] *= g.alpha;
    if (g.beta != 0.0f) v[u] = __builtin_fmaf(g.beta, c[u], v[u]);
    o[u] = (T)v[u];
  }
  if (n + 4 <= last) {
    *reinterpret_cast<vec4*>(D + (int64_t)m * g.ldd + n) = vec4{o[0], o[1], o[2], o[3]};
  } else {
#pragma unroll
    for (int u = 0; u < 3; ++u)
      if (n + u < last) D[(int64_t)m * g.ldd + n + u] = o[u];
  }
  if constexpr (SYRK) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (n + u < last) D[(int64_t)(n + u) * g.ldd + m] = o[u];
  }
}

// fp32 GEMM on operands of any alignment (sgemm.hip): true, with *rc the
// launch's status, when one of its kernels serves these arguments better
// than gemm.hip's (`aligned`: the operands are ready for LDS DMA).
bool sgemm_launch(const GemmArgs& g, bool akc, bool bkc, bool aligned, size_t ws_bytes,
                  hipStream_t s, int* rc);

// fp32 SYRK on sgemm.hip's 32 x 32 kernel, likewise (kc: A is K-contiguous).
bool ssyrk_launch(const GemmArgs& g, bool kc, bool aligned, hipStream_t s, int* rc);

// 16-bit GEMM and SYRK of any alignment on hgemm.hip's 32 x 32 kernel, likewise.
template <typename T, bool SYRK>
bool hgemm_launch(const GemmArgs& g, bool akc, bool bkc, bool aligned, hipStream_t s, int* rc);

}  // namespace trnblas
