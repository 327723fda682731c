// Native drivers of the metric stage: the blocked Cholesky inverse factor
// (metric_inv_half, trnblas/level3.py:365-380) and the blocked triangular
// solve (trsm, level3.py:332-362; the reference's blocked solve is
// `_nki_trsm_left`, trnblas/nki/dispatch.py:1740-1799). Each is one C-ABI
// call that issues its whole launch sequence from C++: the 128-wide
// diagonal-block kernels (metric.hip) and the GEMMs around them (dgemm.hip,
// and gemm.hip for fp32 trsm). Issued from Python, each launch's host cost
// (~50 us through ctypes) exceeded its GPU time, and the GPU waited.
//
// metric_inv_half: right-looking blocked Cholesky in steps of 256 columns
// (two 128-wide diagonal blocks) with look-ahead. After a step's two panels
// only the next step's columns are updated on the caller's stream, so that
// they are factored while a second stream (per device, default priority)
// applies the rest of the trailing update (lower triangle only, rank 256)
// with the other CUs; the caller's stream waits for it before it next writes
// there. Y = L^-1 is built beside the factorisation on a third stream: the
// rows B of a step are Y[B, :k0] = -Y_BB T_B with T_B = L[B, :k0] Y[:k0, :k0],
// which is formed before B is factored, so that only the short product
// follows the last diagonal block. Then X = Y^T. A hand-over between streams
// costs some 10 us beside the 35 us that the caller's stream works per 128
// columns: with one per 128 columns, the rows' long products after their
// diagonal block, and W and Y cleared by passes of their own, naux 384 /
// 1024 / 2304 / 4096 took 185 / 545 / 1117 / 2500 us against 157 / 404 / 926 /
// 2244.
#include <mutex>

#include "common.hpp"

namespace trnblas {

constexpr int kNB = 128;

constexpr int kStep = 2 * kNB;  // columns of a step of metric_inv_half

// dst[i * dr + j * dc] = alpha * src[i * sr + j * sc], rows x cols (rows by
// blockIdx.y and columns by blockIdx.x, grid-strided both ways)
template <typename TS, typename TD>
__global__ __launch_bounds__(256) void copy2d_kernel(int64_t rows, int64_t cols, const TS* src,
                                                     int64_t sr, int64_t sc, TD* dst,
                                                     int64_t dr, int64_t dc, double alpha) {
  for (int64_t i = blockIdx.y; i < rows; i += gridDim.y)
    for (int64_t j = blockIdx.x * 256ll + threadIdx.x; j < cols; j += (int64_t)gridDim.x * 256)
      dst[i * dr + j * dc] = (TD)(alpha * (double)src[i * sr + j * sc]);
}

static dim3 grid2d(int64_t rows, int64_t cols) {
  const int64_t gx = (cols + 255) / 256, gy = rows;
  return dim3((unsigned)(gx < 64 ? (gx > 0 ? gx : 1) : 64), (unsigned)(gy < 4096 ? (gy > 0 ? gy : 1) : 4096));
}

// X[j][i] = f Y[i][j] for j <= i < n and zeros for j > i, through a 64 x 64 LDS
// tile (both sides coalesced; only Y's lower tiles are read); f: metric_init_kernel's
__global__ __launch_bounds__(256) void transpose_kernel(int n, const double* Y, int64_t ldy,
                                                        const double* factor, double* X,
                                                        int64_t ldx) {
  __shared__ double t[64][65];
  const double f = *factor;
  const int i0 = blockIdx.y * 64, j0 = blockIdx.x * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  if (i0 >= j0) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int i = i0 + ty + 4 * r, j = j0 + tx;
      t[ty + 4 * r][tx] = i < n && j <= i ? f * Y[(int64_t)i * ldy + j] : 0.0;
    }
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int j = j0 + ty + 4 * r, i = i0 + tx;
    if (i < n && j < n) X[(int64_t)j * ldx + i] = i0 >= j0 ? t[tx][ty + 4 * r] : 0.0;
  }
}

// W's lower 128 x 128 blocks = J's, zeros past n; zeros in Y's last diagonal
// block when it is partial (its padding takes part in the products); info =
// 0. A metric whose first diagonal element is below 2^-960 is factored as 2^120
// times itself (the diagonal kernel divides by the pivots, and 1 / d overflows
// below 2^-1024), and *factor brings X back. Grid: (blocks of a row, block rows, 8 slices of 16 rows).
__global__ __launch_bounds__(256) void metric_init_kernel(int64_t n, int64_t npad, const double* J,
                                                          int64_t ldj, double* W, double* Y,
                                                          double* factor, int32_t* info) {
  const int64_t bi = blockIdx.y, bj = blockIdx.x;
  if (bj > bi) return;
  const bool small = J[0] < 0x1p-960;
  if (bi == 0 && blockIdx.z == 0 && threadIdx.x == 0) {
    *factor = small ? 0x1p60 : 1.0;
    *info = 0;
  }
  const bool tail = bi == bj && (bi + 1) * 128 > n;
  const double f = small ? 0x1p120 : 1.0;
  const int64_t j = bj * 128 + (threadIdx.x & 127);
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const int64_t i = bi * 128 + blockIdx.z * 16 + (threadIdx.x >> 7) + 2 * u;
    W[i * npad + j] = i < n && j < n ? f * J[i * ldj + j] : 0.0;
    if (tail) Y[i * npad + j] = 0.0;
  }
}

static int grid_for(int64_t elems) {
  const int64_t g = (elems + 255) / 256;
  return (int)(g < 4096 ? (g > 0 ? g : 1) : 4096);
}

// Per device: the side stream of the look-ahead and the two events that
// hand work between the streams (re-recorded every step; a wait uses the
// record that precedes it), and the mutex that keeps calls on one device
// from interleaving their use.
struct SideStream {
  std::mutex mu;
  hipStream_t side = nullptr, inv = nullptr;
  hipEvent_t ready = nullptr, done = nullptr, inverted = nullptr;
};

static SideStream* side_stream(int& rc) {
  static SideStream devs[64];
  int dev = 0;
  rc = TRNBLAS_OK;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
    set_error("metric_inv_half: no current device");
    rc = TRNBLAS_E_LAUNCH;
    return nullptr;
  }
  return &devs[dev];
}

static int side_init(SideStream* ss) {
  if (ss->side) return TRNBLAS_OK;
  if (hipStreamCreateWithFlags(&ss->side, hipStreamNonBlocking) != hipSuccess ||
      hipStreamCreateWithFlags(&ss->inv, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreateWithFlags(&ss->ready, hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&ss->done, hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&ss->inverted, hipEventDisableTiming) != hipSuccess) {
    set_error("metric_inv_half: cannot create the side stream / events");
    return TRNBLAS_E_LAUNCH;
  }
  return TRNBLAS_OK;
}

static void metric_layout(int64_t n, int64_t& npad, size_t off[6]) {
  npad = (n + kNB - 1) / kNB * kNB;
  const size_t sq = (size_t)npad * npad * 8;
  auto up = [](size_t v) { return (v + 255) & ~(size_t)255; };
  off[0] = 0;                                // W: J, updated in place
  off[1] = up(off[0] + sq);                  // L: panels of the factor
  off[2] = up(off[1] + sq);                  // Y: L^-1 (diagonal blocks from the kernel)
  off[3] = up(off[2] + sq);                  // T: a step's rows L[B, :k0] Y[:k0, :k0]
  off[4] = up(off[3] + (size_t)kStep * npad * 8);  // S: L_10 Y_00 of a step's blocks 0, 1
  off[5] = up(off[4] + (size_t)kNB * kNB * 8);     // the factor of X
}

#define TRY(x)                        \
  do {                                \
    const int rc_ = (x);              \
    if (rc_ != TRNBLAS_OK) return rc_; \
  } while (0)

}  // namespace trnblas

using namespace trnblas;

extern "C" size_t trnblas_hip_metric_inv_half_workspace(int64_t n) {
  if (n <= 0) return 0;
  int64_t npad;
  size_t off[6];
  metric_layout(n, npad, off);
  return off[5] + sizeof(double);
}

extern "C" int trnblas_hip_metric_inv_half(int64_t n, const double* J, int64_t ldj, double* X,
                                           int64_t ldx, int32_t* info, void* workspace,
                                           size_t workspace_bytes, void* stream) {
  clear_error();
  TRNBLAS_CHECK_ARG(n >= 0 && n < (1ll << 20), "metric_inv_half: bad n %lld", (long long)n);
  if (n == 0) return TRNBLAS_OK;
  TRNBLAS_CHECK_ARG(J && X && info && workspace, "metric_inv_half: NULL pointer");
  TRNBLAS_CHECK_ARG(ldj >= n && ldx >= n, "metric_inv_half: leading dimension below n");
  TRNBLAS_CHECK_ARG(workspace_bytes >= trnblas_hip_metric_inv_half_workspace(n),
                    "metric_inv_half: workspace %zu bytes, %zu needed", workspace_bytes,
                    trnblas_hip_metric_inv_half_workspace(n));
  TRNBLAS_CHECK_ARG((reinterpret_cast<uintptr_t>(workspace) & 255) == 0,
                    "metric_inv_half: workspace must be 256-byte aligned");
  hipStream_t main = (hipStream_t)stream;
  int64_t npad;
  size_t off[6];
  metric_layout(n, npad, off);
  char* ws = static_cast<char*>(workspace);
  double* W = reinterpret_cast<double*>(ws + off[0]);
  double* L = reinterpret_cast<double*>(ws + off[1]);
  double* Y = reinterpret_cast<double*>(ws + off[2]);
  double* T = reinterpret_cast<double*>(ws + off[3]);
  double* S = reinterpret_cast<double*>(ws + off[4]);
  double* factor = reinterpret_cast<double*>(ws + off[5]);
  int rc = TRNBLAS_OK;
  SideStream* ss = side_stream(rc);
  if (!ss) return rc;
  std::lock_guard<std::mutex> lock(ss->mu);
  TRY(side_init(ss));
  auto wait = [](hipStream_t s, hipEvent_t e) {
    return hipStreamWaitEvent(s, e, 0) == hipSuccess ? TRNBLAS_OK : TRNBLAS_E_LAUNCH;
  };
  auto record = [](hipEvent_t e, hipStream_t s) {
    return hipEventRecord(e, s) == hipSuccess ? TRNBLAS_OK : TRNBLAS_E_LAUNCH;
  };

  const unsigned nblk = (unsigned)(npad / kNB);
  hipLaunchKernelGGL(metric_init_kernel, dim3(nblk, nblk, 8), dim3(256), 0, main, n, npad, J, ldj, W,
                     Y, factor, info);
  TRY(check_launch("metric_inv_half(init)"));
  // D = alpha A op(B) + beta D over blocks of W, L, Y (ld npad)
  auto mm = [&](bool bt, int64_t M, int64_t N, int64_t K, double alpha, const double* A,
                const double* B, int64_t ldb, double beta, double* D, int64_t ldd, int lower, int tri,
                hipStream_t s) {
    return trnblas_hip_dgemm(0, bt, M, N, K, alpha, A, npad, 0, B, ldb, 0, beta, D, ldd, 0, D, ldd,
                             0, 1, lower, tri, s);
  };
  auto chol = [&](int64_t k) {  // L_bb into W (lower triangle), L_bb^-1 = Y_bb into Y
    return chol_block(n - k < kNB ? n - k : kNB, W + k * npad + k, npad, Y + k * npad + k, npad, info,
                      k, false, main);
  };

  // up to two steps there is no trailing update, and the hand-overs to the
  // inverse stream cost what it would overlap
  hipStream_t inv = npad <= 2 * kStep ? main : ss->inv;
  bool rest = false;  // the side stream has a trailing update pending
  for (int64_t k0 = 0; k0 < npad; k0 += kStep) {
    const int64_t k1 = k0 + kNB;
    const int64_t k2 = k1 < npad ? k1 + kNB : k1;  // the step's columns k0 .. k2
    const int64_t k3 = k2 + kStep < npad ? k2 + kStep : npad;  // the next step's end
    double* Y00 = Y + k0 * npad + k0;
    double* Y11 = Y + k1 * npad + k1;
    TRY(chol(k0));
    if (k2 > k1) {
      const int64_t rows = npad - k1;
      double* P = L + k1 * npad + k0;  // the panel of block 0: W[k1:, k0:k1] Y00^T
      TRY(mm(true, rows, kNB, kNB, 1.0, W + k1 * npad + k0, Y00, npad, 0.0, P, npad, 0, 0, main));
      TRY(mm(true, rows, kNB, kNB, -1.0, P, P, npad, 1.0, W + k1 * npad + k1, npad, 0, 0, main));
      TRY(chol(k1));
      if (k2 < npad)
        TRY(mm(true, npad - k2, kNB, kNB, 1.0, W + k2 * npad + k1, Y11, npad, 0.0,
               L + k2 * npad + k1, npad, 0, 0, main));
    }
    if (k2 < npad) {  // the next step's columns
      if (rest) TRY(wait(main, ss->done));
      rest = false;
      const double* R = L + k2 * npad + k0;
      TRY(mm(true, npad - k2, k3 - k2, k2 - k0, -1.0, R, R, npad, 1.0, W + k2 * npad + k2, npad, 0, 0,
             main));
    }
    // one event for both: the side stream's trailing update and the
    // inverse stream's rows
    if (inv != main) TRY(record(ss->ready, main));
    if (k3 < npad) {
      const double* R = L + k3 * npad + k0;
      TRY(wait(ss->side, ss->ready));
      TRY(mm(true, npad - k3, npad - k3, k2 - k0, -1.0, R, R, npad, 1.0, W + k3 * npad + k3, npad, 1,
             0, ss->side));
      TRY(record(ss->done, ss->side));
      rest = true;
    }
    if (inv != main) TRY(wait(inv, ss->ready));
    if (k2 > k1) {  // Y_10 = -Y_11 (L_10 Y_00)
      TRY(mm(false, kNB, kNB, kNB, 1.0, L + k1 * npad + k0, Y00, npad, 0.0, S, kNB, 0,
             TRNBLAS_TRI_B_LOWER, inv));
      TRY(mm(false, kNB, kNB, kNB, -1.0, Y11, S, kNB, 0.0, Y + k1 * npad + k0, npad, 0,
             TRNBLAS_TRI_A_LOWER, inv));
    }
    if (k0 > 0)  // Y[B, :k0] = -Y_BB T
      TRY(mm(false, k2 - k0, k0, k2 - k0, -1.0, Y00, T, npad, 0.0, Y + k0 * npad, npad, 0,
             TRNBLAS_TRI_A_LOWER, inv));
    if (k2 < npad)  // T = L[B', :k2] Y[:k2, :k2] of the next rows B'
      TRY(mm(false, k3 - k2, k2, k2, 1.0, L + k2 * npad, Y, npad, 0.0, T, npad, 0,
             TRNBLAS_TRI_B_LOWER, inv));
  }
  if (inv != main) {
    TRY(record(ss->inverted, inv));
    TRY(wait(main, ss->inverted));
  }
  const unsigned tb = (unsigned)((n + 63) / 64);
  hipLaunchKernelGGL(transpose_kernel, dim3(tb, tb), dim3(256), 0, main, (int)n, Y, npad,
                     factor, X, ldx);
  return check_launch("metric_inv_half(transpose)");
}

// ── trsm ─────────────────────────────────────────────────────────────────────

static void trsm_layout(int dtype, int64_t n, int64_t nrhs, int64_t& nblk, int64_t& npad,
                        int64_t& mp, size_t off[5]) {
  const size_t es = dtype == TRNBLAS_F64 ? 8 : 4;
  nblk = (n + kNB - 1) / kNB;
  npad = nblk * kNB;
  mp = nrhs + (nrhs & 1);
  auto up = [](size_t v) { return (v + 255) & ~(size_t)255; };
  off[0] = 0;                                            // Dinv
  off[1] = up(off[0] + (size_t)nblk * kNB * kNB * es);   // T, padded copy
  off[2] = up(off[1] + (size_t)npad * npad * es);        // R, the running right-hand side
  off[3] = up(off[2] + (size_t)npad * mp * es);          // X, padded
  off[4] = up(off[3] + (size_t)npad * mp * es);          // fp32 GEMM workspace
}

extern "C" size_t trnblas_hip_gemm_workspace(void);

extern "C" size_t trnblas_hip_trsm_workspace(int dtype, int64_t n, int64_t nrhs) {
  if (n <= 0 || nrhs <= 0 || (dtype != TRNBLAS_F32 && dtype != TRNBLAS_F64)) return 0;
  int64_t nblk, npad, mp;
  size_t off[5];
  trsm_layout(dtype, n, nrhs, nblk, npad, mp, off);
  return off[4] + (dtype == TRNBLAS_F32 ? trnblas_hip_gemm_workspace() : 0);
}

namespace trnblas {

struct TrsmCtx {
  int dtype, upper;
  int64_t npad, mp;
  char *Dinv, *T, *R, *X, *gws;
  size_t gws_bytes;
  hipStream_t s;
  size_t es;
  // element pointers
  char* at(char* base, int64_t i, int64_t j, int64_t ld) const {
    return base + (size_t)(i * ld + j) * es;
  }
  // D = alpha A B + beta C (C may be D), row-major operands of this solve
  int mm(int64_t M, int64_t N, int64_t K, double alpha, const char* A, int64_t lda,
         const char* B, int64_t ldb, double beta, char* D, int64_t ldd, int tri) const {
    if (dtype == TRNBLAS_F64)
      return trnblas_hip_dgemm(0, 0, M, N, K, alpha, reinterpret_cast<const double*>(A), lda, 0,
                               reinterpret_cast<const double*>(B), ldb, 0, beta,
                               reinterpret_cast<const double*>(D), ldd, 0,
                               reinterpret_cast<double*>(D), ldd, 0, 1, 0, tri, s);
    return trnblas_hip_gemm(TRNBLAS_F32, 0, 0, M, N, K, alpha, A, lda, 0, B, ldb, 0, beta, D, ldd, 0,
                            D, ldd, 0, 1, gws, gws_bytes, s);
  }
  // blocks [b0, b1): X rows from R rows (R is consumed)
  int solve(int64_t b0, int64_t b1) const {
    if (b1 - b0 == 1) {
      const int64_t r = b0 * kNB;
      return mm(kNB, mp, kNB, 1.0, Dinv + (size_t)b0 * kNB * kNB * es, kNB, at(R, r, 0, mp), mp, 0.0,
                at(X, r, 0, mp), mp, upper ? TRNBLAS_TRI_A_UPPER : TRNBLAS_TRI_A_LOWER);
    }
    const int64_t bm = (b0 + b1) / 2, lo = b0 * kNB, mid = bm * kNB, hi = b1 * kNB;
    if (!upper) {  // forward: the first half, then the rest of R
      TRY(solve(b0, bm));
      TRY(mm(hi - mid, mp, mid - lo, -1.0, at(T, mid, lo, npad), npad, at(X, lo, 0, mp), mp, 1.0,
             at(R, mid, 0, mp), mp, 0));
      return solve(bm, b1);
    }
    TRY(solve(bm, b1));  // backward: the second half first
    TRY(mm(mid - lo, mp, hi - mid, -1.0, at(T, lo, mid, npad), npad, at(X, mid, 0, mp), mp, 1.0,
           at(R, lo, 0, mp), mp, 0));
    return solve(b0, bm);
  }
};

template <typename E>
static int trsm_copies(int64_t n, int64_t nrhs, double alpha, const void* T, int64_t tr, int64_t tc,
                       const void* B, int64_t br, int64_t bc, const TrsmCtx& c) {
  hipLaunchKernelGGL((copy2d_kernel<E, E>), grid2d(n, n), dim3(256), 0, c.s, n, n,
                     static_cast<const E*>(T), tr, tc, reinterpret_cast<E*>(c.T), c.npad,
                     (int64_t)1, 1.0);
  TRY(check_launch("trsm(copy T)"));
  hipLaunchKernelGGL((copy2d_kernel<E, E>), grid2d(n, nrhs), dim3(256), 0, c.s, n, nrhs,
                     static_cast<const E*>(B), br, bc, reinterpret_cast<E*>(c.R), c.mp, (int64_t)1,
                     alpha);
  return check_launch("trsm(copy B)");
}

template <typename E>
__global__ __launch_bounds__(256) void fill_t_kernel(E* p, int64_t n) {
  for (int64_t x = blockIdx.x * 256ll + threadIdx.x; x < n; x += (int64_t)gridDim.x * 256) p[x] = E(0);
}

}  // namespace trnblas

extern "C" int trnblas_hip_trsm(int dtype, int64_t n, int64_t nrhs, int upper, int unit,
                                double alpha, const void* T, int64_t ldt_r, int64_t ldt_c,
                                const void* B, int64_t ldb_r, int64_t ldb_c, void* X,
                                int64_t ldx_r, int64_t ldx_c, void* workspace,
                                size_t workspace_bytes, void* stream) {
  clear_error();
  TRNBLAS_CHECK_ARG(dtype == TRNBLAS_F32 || dtype == TRNBLAS_F64, "trsm: dtype %d not supported",
                    dtype);
  TRNBLAS_CHECK_ARG(n >= 0 && nrhs >= 0 && n < (1ll << 20) && nrhs < (1ll << 30),
                    "trsm: bad sizes");
  if (n == 0 || nrhs == 0) return TRNBLAS_OK;
  TRNBLAS_CHECK_ARG(T && B && X && workspace, "trsm: NULL pointer");
  TRNBLAS_CHECK_ARG(ldt_r > 0 && ldt_c > 0 && ldb_r > 0 && ldb_c > 0 && ldx_r > 0 && ldx_c > 0,
                    "trsm: strides must be positive");
  const size_t need = trnblas_hip_trsm_workspace(dtype, n, nrhs);
  TRNBLAS_CHECK_ARG(workspace_bytes >= need, "trsm: workspace %zu bytes, %zu needed",
                    workspace_bytes, need);
  TRNBLAS_CHECK_ARG((reinterpret_cast<uintptr_t>(workspace) & 255) == 0,
                    "trsm: workspace must be 256-byte aligned");
  TrsmCtx c{};
  int64_t nblk;
  size_t off[5];
  trsm_layout(dtype, n, nrhs, nblk, c.npad, c.mp, off);
  char* ws = static_cast<char*>(workspace);
  c.dtype = dtype;
  c.upper = upper != 0;
  c.es = dtype == TRNBLAS_F64 ? 8 : 4;
  c.Dinv = ws + off[0];
  c.T = ws + off[1];
  c.R = ws + off[2];
  c.X = ws + off[3];
  c.gws = ws + off[4];
  c.gws_bytes = workspace_bytes - off[4];
  c.s = (hipStream_t)stream;
  // zero T, R (their padding takes part in the products) and X
  const int64_t zero_elems = (int64_t)((off[4] - off[1]) / c.es);
  if (dtype == TRNBLAS_F64)
    hipLaunchKernelGGL(fill_t_kernel<double>, dim3(grid_for(zero_elems)), dim3(256), 0, c.s,
                       reinterpret_cast<double*>(c.T), zero_elems);
  else
    hipLaunchKernelGGL(fill_t_kernel<float>, dim3(grid_for(zero_elems)), dim3(256), 0, c.s,
                       reinterpret_cast<float*>(c.T), zero_elems);
  TRY(check_launch("trsm(fill)"));
  if (dtype == TRNBLAS_F64)
    TRY(trsm_copies<double>(n, nrhs, alpha, T, ldt_r, ldt_c, B, ldb_r, ldb_c, c));
  else
    TRY(trsm_copies<float>(n, nrhs, alpha, T, ldt_r, ldt_c, B, ldb_r, ldb_c, c));
  TRY(trnblas_hip_tri_inv_blocks(dtype, n, upper, unit, T, ldt_r, ldt_c, c.Dinv, stream));
  TRY(c.solve(0, nblk));
  if (dtype == TRNBLAS_F64)
    hipLaunchKernelGGL((copy2d_kernel<double, double>), grid2d(n, nrhs), dim3(256), 0, c.s, n, nrhs,
                       reinterpret_cast<const double*>(c.X), c.mp, (int64_t)1,
                       static_cast<double*>(X), ldx_r, ldx_c, 1.0);
  else
    hipLaunchKernelGGL((copy2d_kernel<float, float>), grid2d(n, nrhs), dim3(256), 0, c.s, n, nrhs,
                       reinterpret_cast<const float*>(c.X), c.mp, (int64_t)1,
                       static_cast<float*>(X), ldx_r, ldx_c, 1.0);
  return check_launch("trsm(copy X)");
}
