// 128-wide diagonal blocks of the metric stage, fp64, for gfx950.
//
// metric_inv_half (trnblas/level3.py:365-380; the reference's device route is
// torch.linalg.cholesky + a blocked trsm, trnblas/nki/dispatch.py:1854-1881)
// returns X = L^-T for J = L L^T, and trsm (level3.py:332-362, the blocked
// solve of dispatch.py:1740-1799) solves with a triangular matrix. On the
// device both are blocked by 128: the panels, trailing updates and block
// products are fp64 GEMMs (dgemm.hip); these kernels do what a GEMM cannot,
// on one 128 x 128 diagonal block per workgroup:
//  * chol128_kernel: the Cholesky factor L of an updated SPD block and L^-1
//    (the panel solve then is a GEMM with L^-1, and L^-1 seeds the block
//    inverse of the whole factor);
//  * trinv128_kernel: the inverse of each 128 x 128 diagonal block of a
//    triangular matrix (trsm's diagonal solves become GEMMs).
//
// Inside a workgroup (8 waves) the block is a grid of 8 x 8 sub-blocks of
// 16 x 16 in LDS, lower sub-blocks only, each column-major with column pitch
// 17 doubles. With that pitch the three access patterns of the 16x16x4 f64
// MFMA are cheap: an A fragment (lane l: X[l % 16][4 q + l / 16]) reads 16
// consecutive doubles per 16-lane group, a B fragment (X[4 q + l / 16][l % 16])
// and the accumulator layout (lane l, register e: row 4 e + l / 16, column
// l % 16) fall on distinct banks.
//
// Cholesky: a serial chain of 128 columns, so everything else runs beside
// it. Per 16-wide block column p (two barriers):
//  A. the sub-blocks below the diagonal one become L_ip = A_ip (L_pp^-1)^T,
//     one wave each (MFMA);
//  B. wave 0 updates sub-block (p + 1, p + 1) with L_{p+1,p} and factors and
//     inverts it (chol16: no memory access on its column chain); the other
//     waves meanwhile apply the rest of the trailing update and form block
//     row p of the inverse, Y_pj = -Y_pp sum_k L_pk Y_kj.
// L and Y go to memory from the registers they are formed in. 25.4 us a
// block under the tracer (45.4 us with the diagonal sub-block's columns exchanged through LDS,
// its factorisation and the trailing update one after the other, and the
// inverse by recursive doubling after all of them).
// trinv128: the 8 diagonal sub-blocks inverted at once (inv16), then
// recursive doubling over halves of 16, 32 and 64,
// Y21 = -Y22 (L21 Y11), in place over L21, through an LDS scratch for the
// intermediate product.
#include <type_traits>

#include "common.hpp"

namespace trnblas {

typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int kCholNB = 128;
constexpr int kSP = 17;          // column pitch of a sub-block (doubles)
constexpr int kSB = 16 * kSP;    // doubles per sub-block
constexpr int kNS = 8;           // sub-blocks per side
constexpr int kNLow = kNS * (kNS + 1) / 2;  // lower sub-blocks
constexpr int kThreads = 512;    // 8 waves

__device__ __forceinline__ int sidx(int i, int j) { return i * (i + 1) / 2 + j; }  // i >= j

// 1 / sqrt(d) for d > 0: the hardware estimate (v_rsq_f64) refined by two
// Newton-Raphson steps y <- y (3 - d y^2) / 2; NaN for d <= 0.
__device__ __forceinline__ double rsqrt_nr(double d) {
  double y = __builtin_amdgcn_rsq(d);
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const double h = 0.5 * d * y;
    y = fma(-h, y, 1.5) * y;
  }
  return d > 0.0 ? y : __builtin_nan("");
}

// 1 / d: the hardware estimate (v_rcp_f64) refined by two Newton-Raphson
// steps y <- y + y (1 - d y).
__device__ __forceinline__ double rcp_nr(double d) {
  double y = __builtin_amdgcn_rcp(d);
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const double e = fma(-d, y, 1.0);
    y = fma(y, e, y);
  }
  return y;
}

__device__ __forceinline__ double readlane_f64(double v, int l) {
  const long long b = __builtin_bit_cast(long long, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)b, l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), l);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// MFMA operand and accumulator access of one sub-block (slice q = 0..3).
__device__ __forceinline__ double frag_a(const double* s, int lane, int q) {
  return s[(4 * q + (lane >> 4)) * kSP + (lane & 15)];  // X[l % 16][4 q + l / 16]
}
__device__ __forceinline__ double frag_b(const double* s, int lane, int q) {
  return s[(lane & 15) * kSP + 4 * q + (lane >> 4)];  // X[4 q + l / 16][l % 16]
}
__device__ __forceinline__ f64x4 load_acc(const double* s, int lane) {
  const double* p = s + (lane & 15) * kSP + (lane >> 4);
  return f64x4{p[0], p[4], p[8], p[12]};
}
__device__ __forceinline__ void store_acc(double* s, int lane, const f64x4& v) {
  double* p = s + (lane & 15) * kSP + (lane >> 4);
#pragma unroll
  for (int e = 0; e < 4; ++e) p[4 * e] = v[e];
}
// acc += sgn X Y^T (BT) or sgn X Y
template <bool BT>
__device__ __forceinline__ void mma16(f64x4& acc, const double* X, const double* Y, double sgn,
                                      int lane) {
  double a[4], b[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    a[q] = sgn * frag_a(X, lane, q);
    b[q] = BT ? frag_a(Y, lane, q) : frag_b(Y, lane, q);
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[q], b[q], acc, 0, 0, 0);
}

template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (N > 0) {
    static_for<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

// v from lane SRC of the lane's 16-lane row (DPP row_newbcast: every lane has
// a source, so the destination's old value does not matter).
template <int SRC>
__device__ __forceinline__ double row_bcast(double v) {
  const long long b = __builtin_bit_cast(long long, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)b, 0x150 + SRC, 0xf, 0xf, true);
  const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)(b >> 32), 0x150 + SRC, 0xf, 0xf, true);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// One wave on a 16 x 16 diagonal sub-block `blk` (lower part read, SPD):
// blk becomes L^-1 (blk = L L^T); in register e of lane (h = l / 16,
// r = l % 16), l receives L[r][4 e + h] and y L^-1[4 e + h][r]. Returns 0, or
// column + 1 of the first pivot that is not positive and finite among the
// leading nb columns.
//
// Elimination without square roots, U D U^T, four columns at a time: every
// 16-lane row h of the wave holds the four columns of row r (p) and
// eliminates them by itself, the pivots and multipliers' rows coming from
// other lanes of the row by DPP, with no memory access. The steps act on a
// 4-column identity as well (column h of it on row h: w), and then one MFMA
// applies them to the rest of the matrix (S -= M P^T, rank 4) and one to the
// inverse (E = W E_4 + the rows of E outside the four). S is kept whole, so
// that by its symmetry an accumulator register t (row 4 t + h, column r) is
// column 4 t + h of row r, the next four columns. Then L = U D^1/2 and L^-1 =
// D^-1/2 E, the 16 inverse roots at once. A lone wave issues an instruction
// every 7 cycles or so, which bounds this: column by column on the whole block
// the elimination took 7400 cycles, this way about 4100. ex: 64 doubles of LDS.
__device__ __forceinline__ int chol16(double* blk, double* ex, int lane, int nb, f64x4& l, f64x4& y) {
  // (an opaque copy of the lane index: otherwise the per-column lane masks
  // are computed once, outside the caller's loop, and spill)
  asm volatile("" : "+v"(lane));
  const int r = lane & 15, h = lane >> 4;
  f64x4 S, E;
  double p[4], u[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) p[e] = blk[min(r, e) * kSP + max(r, e)];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int s = 4 * e + h;
    S[e] = blk[min(r, s) * kSP + max(r, s)];
    E[e] = s == r ? 1.0 : 0.0;
  }
  double mine = 1.0;  // lanes h = r % 4: the pivot of column r
  static_for<4>([&](auto tI) {
    constexpr int t = decltype(tI)::value;
    double mh = 0.0, uh = 0.0;        // multiplier and value of column 4 t + h
    double w = r == 4 * t + h ? 1.0 : 0.0;  // W[r][h]
    static_for<4>([&](auto kI) {
      constexpr int k = decltype(kI)::value, c = 4 * t + k;
      const double d = row_bcast<c>(p[k]);
      // 1 / d: the hardware estimate x and one step x (1 + e + e^2), e = 1 - d x
      double rd = __builtin_amdgcn_rcp(d);
      const double er = fma(-d, rd, 1.0);
      rd = fma(rd, fma(er, er, er), rd);
      const double m = r > c ? p[k] * rd : 0.0;
      static_for<3 - k>([&](auto sI) {
        constexpr int s = k + 1 + decltype(sI)::value;
        p[s] = fma(-m, row_bcast<4 * t + s>(p[k]), p[s]);
      });
      w = fma(-m, row_bcast<c>(w), w);
      mh = h == k ? m : mh;
      uh = h == k ? p[k] : uh;
    });
    u[t] = uh;
    mine = r == 4 * t + h ? uh : mine;
    if constexpr (t < 3) {
      S = __builtin_amdgcn_mfma_f64_16x16x4f64(-mh, uh, S, 0, 0, 0);
      ex[lane] = S[t + 1];
    }
    const double e4 = E[t];
    E[t] = 0.0;
    E = __builtin_amdgcn_mfma_f64_16x16x4f64(w, e4, E, 0, 0, 0);
    if constexpr (t < 3) {
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int k = 0; k < 4; ++k) p[k] = ex[16 * k + r];
      __builtin_amdgcn_wave_barrier();
    }
  });
  // the lane that holds the pivot of column r
  const bool own = (r & 3) == h;
  const unsigned long long b = __ballot(own && !(mine > 0.0 && mine < __builtin_inf()) && r < nb);
  const unsigned cols = (unsigned)(b | b >> 16 | b >> 32 | b >> 48) & 0xffffu;
  if (own) ex[r] = rsqrt_nr(mine);
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int s = 4 * e + h;
    const double rs = ex[s];
    l[e] = u[e] * rs;
    y[e] = s >= r ? E[e] * rs : 0.0;
    blk[r * kSP + s] = y[e];
  }
  return cols ? (int)__builtin_ctz(cols) + 1 : 0;
}

// One wave on a 16 x 16 lower triangular sub-block `blk` (unit: its diagonal
// taken as ones), in place: blk becomes its inverse. Lane (h = l / 16,
// r = l % 16) holds columns 4 e + h of row r (e = 0..3) of the matrix and of
// E, the product of the elimination steps (the inverse is diag(1 / t_rr) E).
// Per column c every lane publishes its element of column 4 (c / 4) + h
// through LDS, of which the column-c ones are read back; row c of E comes
// from lane c of the lane's own 16-lane row (DPP). ex: 80 doubles of this
// wave's LDS.
__device__ __forceinline__ void inv16(double* blk, double* ex, int lane, bool unit) {
  double* colb = ex;        // colb[16 h + r]: lane (h, r)'s published value
  double* rinvb = ex + 64;  // 1 / t_cc
  // (an opaque copy of the lane index: otherwise the per-column lane masks
  // are computed once, outside the caller's loop, and spill)
  int ln = lane;
  asm volatile("" : "+v"(ln));
  const int r = ln & 15, h = ln >> 4;
  double a[4], E[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int s = 4 * e + h;
    a[e] = s <= r ? blk[s * kSP + r] : 0.0;
    if (unit && s == r) a[e] = 1.0;
    E[e] = s == r ? 1.0 : 0.0;
  }
  static_for<16>([&](auto cI) {
    constexpr int c = decltype(cI)::value, ch = c & 3, ce = c >> 2;
    const double d = readlane_f64(a[ce], c + 16 * ch);  // the pivot
    const double rinv = unit ? 1.0 : rcp_nr(d);
    colb[16 * h + r] = a[ce];
    rinvb[c] = rinv;
    double ev[4];  // E[c][4 e + h]
#pragma unroll
    for (int e = 0; e < 4; ++e) ev[e] = row_bcast<c>(E[e]);
    __builtin_amdgcn_wave_barrier();
    const double m = r > c ? colb[16 * ch + r] * rinv : 0.0;  // the multiplier of row r
#pragma unroll
    for (int e = 0; e < 4; ++e) E[e] = fma(-m, ev[e], E[e]);
    __builtin_amdgcn_wave_barrier();
  });
  const double rr = rinvb[r];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int s = 4 * e + h;
    blk[s * kSP + r] = s <= r ? E[e] * rr : 0.0;
  }
}

// acc += sgn sum_{t < n} X_t Y_t (n <= NMAX, wave-uniform) over sub-block
// pairs given by the offsets xo[t], yo[t] into G / Y buffers: every
// fragment is read before the first MFMA (offsets past n repeat a valid
// pair and their MFMAs are skipped), so the LDS reads overlap.
template <int NMAX>
__device__ __forceinline__ void mma16_sum(f64x4& acc, const double* X, const int (&xo)[NMAX],
                                          const double* Y, const int (&yo)[NMAX], int n, double sgn,
                                          int lane) {
  double a[NMAX][4], b[NMAX][4];
#pragma unroll
  for (int t = 0; t < NMAX; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      a[t][q] = sgn * frag_a(X + xo[t], lane, q);
      b[t][q] = frag_b(Y + yo[t], lane, q);
    }
#pragma unroll
  for (int t = 0; t < NMAX; ++t)
    if (t < n) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t][q], b[t][q], acc, 0, 0, 0);
    }
}

// The block inverse Y = L^-1 in place over the lower sub-block grid G, whose
// off-diagonal sub-blocks hold L and diagonal ones their inverses: for
// halves of h = 1, 2, 4 sub-blocks and each column j of a half, T = L21 Y11
// (column j) into scr, then Y21 = -Y22 T (column j) over L21. A round
// handles one column of every pair: 4 sub-blocks of T, so scr holds 4
// (later rounds read only columns of L21 that earlier rounds left).
__device__ __forceinline__ void block_inverse(double* G, double* scr, int wave, int lane) {
  static_for<3>([&](auto lI) {
    constexpr int h = 1 << decltype(lI)::value;
    for (int j = 0; j < h; ++j) {
      if (wave < 4) {  // item = (pair pi, row i of the half)
        const int pi = wave / h, i = wave % h, b0 = 2 * h * pi;
        int xo[h], yo[h];
#pragma unroll
        for (int t = 0; t < h; ++t) {  // k = j + t < h
          const int k = min(j + t, h - 1);
          xo[t] = sidx(b0 + h + i, b0 + k) * kSB;
          yo[t] = sidx(b0 + k, b0 + j) * kSB;
        }
        f64x4 acc = {0.0, 0.0, 0.0, 0.0};
        mma16_sum<h>(acc, G, xo, G, yo, h - j, 1.0, lane);
        store_acc(scr + wave * kSB, lane, acc);
      }
      __syncthreads();
      if (wave < 4) {
        const int pi = wave / h, i = wave % h, b0 = 2 * h * pi;
        int xo[h], yo[h];
#pragma unroll
        for (int t = 0; t < h; ++t) {  // k = t <= i
          const int k = min(t, i);
          xo[t] = sidx(b0 + h + i, b0 + h + k) * kSB;
          yo[t] = (pi * h + k) * kSB;
        }
        f64x4 acc = {0.0, 0.0, 0.0, 0.0};
        mma16_sum<h>(acc, G, xo, scr, yo, i + 1, -1.0, lane);
        store_acc(G + sidx(b0 + h + i, b0 + j) * kSB, lane, acc);
      }
      __syncthreads();
    }
  });
}

// The lower triangle of a 128 x 128 block (element (i, k) at
// X[i * ri + k * ci], the identity past nb) into the sub-block grid. Thread
// t takes column k = t % 128 of rows t / 128 + 4 u (u = 0..31), so its
// addresses step by a constant and the sub-block of each u is known at
// compile time; all 32 loads issue before the first LDS store.
template <typename TT>
__device__ __forceinline__ void load_lower(double* G, const TT* X, int64_t ri, int64_t ci, int nb,
                                           int tid) {
  constexpr int PER = kCholNB * kCholNB / kThreads;  // 32
  const int k = tid & 127, i0 = tid >> 7;
  const TT* p = X + i0 * ri + k * ci;
  double v[PER];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int i = i0 + 4 * u;
    v[u] = (k <= i && i < nb) ? (double)p[(int64_t)(4 * u) * ri] : (i == k ? 1.0 : 0.0);
  }
  double* g = G + (k >> 4) * kSB + (k & 15) * kSP + i0;
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int i = i0 + 4 * u;
    if (k <= i) g[sidx(u >> 2, 0) * kSB + 4 * (u & 3)] = v[u];
  }
}

// The lower triangle of the grid out to Z[i * zr + k * zc] for i, k < nb,
// zeros above the diagonal, in the thread mapping of load_lower.
template <typename TT>
__device__ __forceinline__ void store_lower(const double* G, TT* Z, int64_t zr, int64_t zc, int nb,
                                            int tid) {
  constexpr int PER = kCholNB * kCholNB / kThreads;
  asm volatile("" : "+v"(tid));  // (its masks and addresses computed here, not at kernel entry)
  const int k = tid & 127, i0 = tid >> 7;
  const double* g = G + (k >> 4) * kSB + (k & 15) * kSP + i0;
  double v[PER];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int i = i0 + 4 * u;
    v[u] = k <= i ? g[sidx(u >> 2, 0) * kSB + 4 * (u & 3)] : 0.0;
  }
  TT* z = Z + (int64_t)i0 * zr + (int64_t)k * zc;
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int i = i0 + 4 * u;
    if (i < nb && k < nb) z[(int64_t)(4 * u) * zr] = (TT)v[u];
  }
}

// LDS: the sub-block grid and a 16 x 16 scratch per wave, 96 KB, so the
// workgroup shares a CU with a GEMM workgroup (64 KB) of a concurrent
// stream instead of waiting for a whole free CU. chol16 divides by its
// pivots, and 1 / d overflows below 2^-1024: with SCALE, a block with a diagonal
// element below 2^-960 is factored as 2^120 times itself (a pivot that the
// updates leave of a larger one is at least its rounding, 2^-53 of it; 1 us
// more a block: the metric driver scales the whole matrix instead). The
// sub-blocks of Li above its diagonal ones are cleared: the triangular products
// that read it take them as zeros.
template <bool SCALE>
__global__ __launch_bounds__(kThreads) void chol128_kernel(int nb, double* A, int64_t lda,
                                                           double* Li, int64_t ldl, int32_t* info,
                                                           int offset) {
  constexpr int NW = kThreads / 64;
  __shared__ double G[kNLow * kSB];
  __shared__ double scr[NW][kSB];  // T of the inverse's block row; chol16's exchange
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  bool small = false;
  if constexpr (SCALE) {
#pragma unroll
    for (int x = lane; x < kCholNB; x += 64) small |= x < nb && A[(int64_t)x * (lda + 1)] < 0x1p-960;
    small = __any(small);
  }
  // sub-block (i, k) of an accumulator to Z, rows and columns below nb; f: of a
  // scaled block
  auto put = [&](double* Z, int64_t ld, int i, int k, f64x4 v, double f) __attribute__((always_inline)) {
    if (small) v *= f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = 16 * i + 4 * e + lg, col = 16 * k + li;
      if (row < nb && col < nb) Z[(int64_t)row * ld + col] = v[e];
    }
  };
  // sub-block (i, k) of A, the identity past nb
  auto get = [&](int i, int k) __attribute__((always_inline)) {
    f64x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = 16 * i + 4 * e + lg, col = 16 * k + li;
      v[e] = row == col ? 1.0 : 0.0;
      if (row < nb && col <= row) v[e] = A[(int64_t)row * lda + col];
    }
    if (small) v *= 0x1p120;
    return v;
  };
  int bad = 0;  // wave 0: the first pivot that is not positive, 1-based
  // wave 0: chol16's l and y of step p; the others: the panel sub-block and
  // the inverse's (with its partial sum t)
  f64x4 l = {0.0, 0.0, 0.0, 0.0}, y = l, t = l;
  if (wave == 0) {
    store_acc(G, lane, get(0, 0));
    __builtin_amdgcn_wave_barrier();
    bad = chol16(G, scr[0], lane, nb, l, y);
  } else {  // the other 35 sub-blocks meanwhile, five per wave
    f64x4 v[5];
#pragma unroll
    for (int x = 0; x < 5; ++x) {
      const int q = wave + 7 * x;
      int i = 0;
      while ((i + 1) * (i + 2) / 2 <= q) ++i;
      v[x] = get(i, q - i * (i + 1) / 2);
    }
#pragma unroll
    for (int x = 0; x < 5; ++x) store_acc(G + (wave + 7 * x) * kSB, lane, v[x]);
    for (int x = tid - 64; x < kCholNB * kCholNB; x += kThreads - 64) {
      const int i = x >> 7, k = x & 127;
      if ((k >> 4) > (i >> 4) && i < nb && k < nb) Li[(int64_t)i * ldl + k] = 0.0;
    }
  }
  __syncthreads();
  for (int p = 0; p < kNS; ++p) {
    const double* D = G + sidx(p, p) * kSB;  // L_pp^-1
    // A. the panel (wave 0 has no row of it: it stores L_pp and its inverse)
    const int pi = p + NW - wave;
    if (wave == 0) {
      if (small) {
        l *= 0x1p-60;
        y *= 0x1p60;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 16 * p + li, s = 16 * p + 4 * e + lg;
        if (r < nb && s < nb) {
          Li[(int64_t)s * ldl + r] = y[e];
          if (s <= r) A[(int64_t)r * lda + s] = l[e];
        }
      }
    } else if (pi < kNS) {
      l = f64x4{0.0, 0.0, 0.0, 0.0};
      mma16<true>(l, G + sidx(pi, p) * kSB, D, 1.0, lane);
      store_acc(G + sidx(pi, p) * kSB, lane, l);
    }
    __syncthreads();
    // B. wave 0 the next diagonal sub-block; the others block row p of the
    // inverse (column j on wave j + 1), the part of row p + 1 that is known,
    // and the rest of the trailing update
    const bool last = p + 1 == kNS;
    if (wave == 0 && !last) {
      double* N = G + sidx(p + 1, p + 1) * kSB;
      const double* X = G + sidx(p + 1, p) * kSB;
      f64x4 acc = load_acc(N, lane);
      mma16<true>(acc, X, X, -1.0, lane);
      store_acc(N, lane, acc);
      __builtin_amdgcn_wave_barrier();
      const int b = chol16(N, scr[0], lane, nb - 16 * (p + 1), l, y);
      if (bad == 0 && b != 0) bad = 16 * (p + 1) + b;
    } else {
      if (pi < kNS) put(A, lda, pi, p, l, 0x1p-60);
      const int j = wave - 1;
      if (wave != 0 && j < p) {
        // t holds sum_{k < p - 1} L_pk Y_kj from the step before
        mma16<false>(t, G + sidx(p, p - 1) * kSB, G + sidx(p - 1, j) * kSB, 1.0, lane);
        store_acc(scr[wave], lane, t);
        __builtin_amdgcn_wave_barrier();
        y = f64x4{0.0, 0.0, 0.0, 0.0};
        mma16<false>(y, D, scr[wave], -1.0, lane);
        put(Li, ldl, p, j, y, 0x1p60);
        t = f64x4{0.0, 0.0, 0.0, 0.0};
        if (!last)
          for (int k = j; k < p; ++k)
            mma16<false>(t, G + sidx(p + 1, k) * kSB, G + sidx(k, j) * kSB, 1.0, lane);
      }
      const int nt = kNS - 1 - p, items = nt * (nt + 1) / 2;
      for (int it = NW - wave; it < items; it += NW - 1) {  // item 0 is wave 0's
        int ri = 0;
        while ((ri + 1) * (ri + 2) / 2 <= it) ++ri;
        const int i = p + 1 + ri, k = p + 1 + (it - ri * (ri + 1) / 2);
        f64x4 acc = load_acc(G + sidx(i, k) * kSB, lane);
        mma16<true>(acc, G + sidx(i, p) * kSB, G + sidx(k, p) * kSB, -1.0, lane);
        store_acc(G + sidx(i, k) * kSB, lane, acc);
      }
    }
    __syncthreads();
    // Y_pj over L_pj, which every wave has now read
    if (!last && wave >= 1 && wave - 1 < p) store_acc(G + sidx(p, wave - 1) * kSB, lane, y);
  }
  if (tid == 0 && bad != 0 && info[0] == 0) info[0] = offset + bad;
}

// Inverse of diagonal block b of the n x n triangular matrix T: element
// (i, k) of the lower matrix inverted is T[k0 + i][k0 + k] (lower) or
// T[k0 + k][k0 + i] (upper: T^T is inverted and the result transposed back),
// read through the strides (sr, sc) in T's element type. Dinv[b] (128 x 128
// row-major) receives the inverse, the identity past the matrix.
template <typename TT>
__global__ __launch_bounds__(kThreads) void trinv128_kernel(int n, int upper, int unit,
                                                            const TT* T, int64_t sr, int64_t sc,
                                                            TT* Dinv) {
  __shared__ double G[kNLow * kSB];
  __shared__ double scr[4 * kSB];
  __shared__ double ex[kThreads / 64][80];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.x, k0 = b * kCholNB, nb = min(kCholNB, n - k0);
  const int64_t ri = upper ? sc : sr, ci = upper ? sr : sc;  // strides of the lower view
  load_lower(G, T + (int64_t)k0 * (sr + sc), ri, ci, nb, tid);
  __syncthreads();
  // the 8 diagonal sub-blocks' inverses, one wave each, in place
  inv16(G + sidx(wave, wave) * kSB, ex[wave], lane, unit != 0);
  __syncthreads();
  block_inverse(G, scr, wave, lane);
  // lower: out[i][k] = Y[i][k]; upper: out[k][i] = Y[i][k]
  TT* out = Dinv + (int64_t)b * kCholNB * kCholNB;
  store_lower(G, out, upper ? (int64_t)1 : (int64_t)kCholNB, upper ? (int64_t)kCholNB : (int64_t)1,
              kCholNB, tid);
}

}  // namespace trnblas

using namespace trnblas;

int trnblas::chol_block(int64_t nb, double* A, int64_t lda, double* Linv, int64_t ldl,
                        int32_t* info, int64_t offset, bool any_scale, hipStream_t stream) {
  TRNBLAS_CHECK_ARG(nb >= 0 && nb <= kCholNB, "chol_block: nb %lld not in [0, %d]", (long long)nb,
                    kCholNB);
  if (nb == 0) return TRNBLAS_OK;
  TRNBLAS_CHECK_ARG(A && Linv && info, "chol_block: NULL pointer");
  TRNBLAS_CHECK_ARG(lda >= nb && ldl >= nb, "chol_block: leading dimension below nb");
  TRNBLAS_CHECK_ARG(offset >= 0 && offset < (1ll << 30), "chol_block: bad offset");
  auto kern = any_scale ? chol128_kernel<true> : chol128_kernel<false>;
  hipLaunchKernelGGL(kern, dim3(1), dim3(kThreads), 0, stream, (int)nb, A, lda, Linv, ldl, info,
                     (int)offset);
  return check_launch("chol_block");
}

extern "C" int trnblas_hip_chol_block(int64_t nb, double* A, int64_t lda, double* Linv,
                                      int64_t ldl, int32_t* info, int64_t offset, void* stream) {
  clear_error();
  return chol_block(nb, A, lda, Linv, ldl, info, offset, true, (hipStream_t)stream);
}

extern "C" int trnblas_hip_tri_inv_blocks(int dtype, int64_t n, int upper, int unit, const void* T,
                                          int64_t ldt_r, int64_t ldt_c, void* Dinv, void* stream) {
  clear_error();
  TRNBLAS_CHECK_ARG(dtype == TRNBLAS_F32 || dtype == TRNBLAS_F64,
                    "tri_inv_blocks: dtype %d not supported (f32, f64)", dtype);
  TRNBLAS_CHECK_ARG(n >= 0 && n < (1ll << 30), "tri_inv_blocks: bad n %lld", (long long)n);
  if (n == 0) return TRNBLAS_OK;
  TRNBLAS_CHECK_ARG(T && Dinv, "tri_inv_blocks: NULL pointer");
  TRNBLAS_CHECK_ARG(ldt_r > 0 && ldt_c > 0 && (ldt_r >= n || ldt_c >= n || n == 1),
                    "tri_inv_blocks: bad strides");
  const int nblk = (int)((n + kCholNB - 1) / kCholNB);
  if (dtype == TRNBLAS_F64)
    hipLaunchKernelGGL(trinv128_kernel<double>, dim3(nblk), dim3(kThreads), 0, (hipStream_t)stream,
                       (int)n, upper, unit, static_cast<const double*>(T), ldt_r, ldt_c,
                       static_cast<double*>(Dinv));
  else
    hipLaunchKernelGGL(trinv128_kernel<float>, dim3(nblk), dim3(kThreads), 0, (hipStream_t)stream,
                       (int)n, upper, unit, static_cast<const float*>(T), ldt_r, ldt_c,
                       static_cast<float*>(Dinv));
  return check_launch("tri_inv_blocks");
}
