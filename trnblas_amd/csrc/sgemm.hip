// fp32 GEMM for the sizes and alignments that gemm.hip's LDS-DMA kernels do
// not serve: operands that are not 16-byte ready (odd orbital counts), too
// few 128 x 128 tiles to fill the chip, and few rows against very many
// columns. D = alpha op(A) op(B) + beta C on v_mfma_f32_16x16x4_f32, the
// semantics and the chains of gemm.hip (MFMA chains of chain_length(K)
// values folded into a separate fp32 sum).
//
// Every operand access is a buffer load of 4 consecutive floats at 4-byte
// alignment (buffer_load_dwordx4 needs no more), so odd leading dimensions
// and bases cost nothing but split cache lines. A group is loaded as one
// only when all four values are inside the matrix; groups cut by its edge
// take single loads, in the last k-tile. Nothing outside the operands is read.
//
// MFMA 16x16x4 f32: lane l holds k = l / 16 of A (row l % 16) and of B
// (column l % 16); D row 4 (l / 16) + r in register r, column l % 16. In
// every kernel lane group g = l / 16 takes k = 4 g + q of a 16-wide k chunk
// for MFMA q (0..3), the same for both operands, so that
//  * of an operand stored K-contiguous a lane needs the four consecutive
//    values 4 g .. 4 g + 3 of its row (one 16-byte access for four MFMAs);
//    its block i is rows 16 i .. 16 i + 15;
//  * of one stored M / N-contiguous it needs F consecutive values of row
//    4 g + q (F: the wave's blocks), and block i is rows F r + i.
#include <algorithm>
#include <cmath>

#include "gemm.hpp"

namespace trnblas {

constexpr uint32_t kSOob = 0x80000000u;  // offsets >= this read as zero, with no access

__device__ __forceinline__ __amdgpu_buffer_rsrc_t srsrc(const float* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), (short)0, 0x7ffffff0,
                                           0x00020000);
}
__device__ __forceinline__ f32x4 load4f(__amdgpu_buffer_rsrc_t rs, uint32_t off) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
}
// The leading nv (0..4) of 4 consecutive floats, zeros after them.
__device__ __forceinline__ f32x4 load_part(__amdgpu_buffer_rsrc_t rs, uint32_t off, int nv) {
  i32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rs, nv >= 4 ? off : kSOob, 0, 0);
#pragma unroll
  for (int e = 0; e < 3; ++e)
    v[e] |= (int)__builtin_amdgcn_raw_buffer_load_b32(rs, nv > e && nv < 4 ? off + 4 * e : kSOob, 0, 0);
  return __builtin_bit_cast(f32x4, v);
}

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef f32x4 __attribute__((aligned(4))) f32x4u;
typedef f32x2 __attribute__((aligned(4))) f32x2u;

// One operand panel of W rows (m or n) x 32 k, moved by 256 threads through
// registers into LDS: [row][k] with pitch 36 (KC) or [k][row] with pitch
// W + 8. Both pitches put the 16 lanes of a fragment read on distinct banks
// and lane groups g, g + 1 on different halves of them.
template <bool KC, int W>
struct Panel {
  static constexpr int BK = 32;
  static constexpr int NG = W * BK / 4;           // 4-float groups
  static constexpr int NV = (NG + 255) / 256;     // per thread
  static constexpr int GR = KC ? BK / 4 : W / 4;  // groups per stored row
  static constexpr int PITCH = KC ? BK + 4 : W + 8;
  static constexpr int SIZE = KC ? W * PITCH : BK * PITCH;
  const float* X;     // the panel's corner at k = 0
  int64_t step;       // floats from one k-tile to the next
  int ld, rows, K;    // leading dimension; m / n left from the corner; k
  int nwhole;         // leading k-tiles without a group cut by an edge
  uint32_t off[NV];   // byte offset of each group, kSOob outside the rows
  f32x4 v[NV];

  __device__ __forceinline__ void init(const float* base, int64_t ld_, int row0, int nrows, int K_,
                                       int tid) {
    ld = (int)ld_;
    rows = nrows - row0;
    K = K_;
    X = base + (KC ? row0 * ld_ : (int64_t)row0);
    step = KC ? (int64_t)BK : BK * ld_;
    // An M / N-contiguous group cut by the matrix's edge is loaded as one as
    // long as it ends inside the operand (on the next row's values, which only
    // reach outputs outside D): all but the last rows of k, 3 floats from its
    // end. A K-contiguous one must read zeros past K.
    const bool cut = !KC && rows < W && (rows & 3) != 0;
    nwhole = (cut ? max(K - (ld > 2 ? 1 : ld > 1 ? 2 : 3), 0) : K) / BK;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int idx = tid + 256 * i, r = idx / GR, c = 4 * (idx % GR);
      off[i] = idx < NG && (KC ? r < rows : c < rows) ? 4u * ((uint32_t)r * (uint32_t)ld + (uint32_t)c)
                                                      : kSOob;
    }
  }
  __device__ __forceinline__ void load(int kt, int tid) {
    const __amdgpu_buffer_rsrc_t rs = srsrc(X + kt * step);
    if (kt < nwhole) {
#pragma unroll
      for (int i = 0; i < NV; ++i) v[i] = load4f(rs, off[i]);
    } else {
      const int kl = K - kt * BK;
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int idx = tid + 256 * i, r = idx / GR, c = 4 * (idx % GR);
        v[i] = load_part(rs, off[i], off[i] == kSOob ? 0 : KC ? kl - c : r < kl ? rows - c : 0);
      }
    }
  }
  __device__ __forceinline__ void store(float* lds, int tid) const {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int idx = tid + 256 * i, r = idx / GR, c = 4 * (idx % GR);
      if (NG % 256 == 0 || idx < NG) *reinterpret_cast<f32x4*>(lds + r * PITCH + c) = v[i];
    }
  }
};

// F values a[i][q] (block i, MFMA q) of the 16-wide k chunk at kk, for the
// wave's rows w0 .. w0 + 16 F - 1.
template <bool KC, int W, int F>
__device__ __forceinline__ void frags(const float* p, int w0, int kk, int li, int g,
                                      float (&a)[F][4]) {
  constexpr int P = Panel<KC, W>::PITCH;
  if constexpr (KC) {
#pragma unroll
    for (int i = 0; i < F; ++i) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(p + (w0 + 16 * i + li) * P + kk + 4 * g);
#pragma unroll
      for (int q = 0; q < 4; ++q) a[i][q] = x[q];
    }
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float* r = p + (kk + 4 * g + q) * P + w0 + F * li;
      if constexpr (F == 4) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(r);
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i][q] = x[i];
      } else if constexpr (F == 2) {
        const f32x2 x = *reinterpret_cast<const f32x2*>(r);
        a[0][q] = x[0];
        a[1][q] = x[1];
      } else {
#pragma unroll
        for (int i = 0; i < F; ++i) a[i][q] = r[i];
      }
    }
  }
}

// row / column of block b, index x (0..15) of a wave's F blocks
template <bool KC, int F>
__device__ __forceinline__ int blk_row(int b, int x) {
  return KC ? 16 * b + x : F * x + b;
}

// D = alpha acc + beta C for the FM x FN blocks of a wave whose corner is
// (m0, n0) of the matrix. C's values are all read before the first store of
// a block row: D may be C. BNC (B N-contiguous): a lane's FN columns are
// consecutive.
template <bool AKC, bool BKC, int FM, int FN>
__device__ __forceinline__ void store_wave(const GemmArgs& g, int bat, int m0, int n0, int lane,
                                           const f32x4 (&acc)[FM][FN]) {
  const float* C = static_cast<const float*>(g.C) + (g.C ? bat * g.sC : 0);
  float* D = static_cast<float*>(g.D) + bat * g.sD;
  const int li = lane & 15, lg = lane >> 4;
  const float alpha = g.alpha, beta = g.beta;
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    float c[4][FN];
    if (beta != 0.0f) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + blk_row<AKC, FM>(i, 4 * lg + r);
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const int n = n0 + blk_row<BKC, FN>(j, li);
          c[r][j] = 0.0f;
          if (m < g.M && n < g.N) c[r][j] = C[(int64_t)m * g.ldc + n];
        }
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = m0 + blk_row<AKC, FM>(i, 4 * lg + r);
      float v[FN];
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        v[j] = alpha * acc[i][j][r];
        if (beta != 0.0f) v[j] = __builtin_fmaf(beta, c[r][j], v[j]);
      }
      if (m >= g.M) continue;
      float* d = D + (int64_t)m * g.ldd;
      const int nc = n0 + FN * li;
      if constexpr (!BKC && (FN == 4 || FN == 2)) {
        if (nc + FN <= g.N) {
          if constexpr (FN == 4)
            *reinterpret_cast<f32x4u*>(d + nc) = f32x4{v[0], v[1], v[2], v[3]};
          else
            *reinterpret_cast<f32x2u*>(d + nc) = f32x2{v[0], v[1]};
          continue;
        }
      }
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int n = n0 + blk_row<BKC, FN>(j, li);
        if (n < g.N) d[n] = v[j];
      }
    }
  }
}

// BM x BN tiles, 4 waves (WGM of them along M), k-tiles of 32 through
// registers into two LDS stages: the loads of k-tile t + 1 are in flight
// behind the MFMAs of k-tile t, one barrier per k-tile, and the workgroups
// that share a CU (64 x 64: four) fill each other's gaps. Under a split
// (g.splits > 1) workgroup (tile, s) takes the k-tiles [s nk / splits,
// (s + 1) nk / splits) and leaves its raw sums in ws; sgemm_sum_kernel adds
// them in order.
template <int BM, int BN, int WGM, bool AKC, bool BKC>
__global__ __launch_bounds__(256, 2) void sgemm_tile_kernel(GemmArgs g) {
  using PA = Panel<AKC, BM>;
  using PB = Panel<BKC, BN>;
  constexpr int BK = 32, WGN = 4 / WGM, WM = BM / WGM, WN = BN / WGN, FM = WM / 16, FN = WN / 16;
  __shared__ __attribute__((aligned(16))) float lds[2][PA::SIZE + PB::SIZE];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm0 = (wave / WGN) * WM, wn0 = (wave % WGN) * WN;
  const int w = xcd_remap(blockIdx.x, gridDim.x);
  const int t = w / g.splits, sp = w - t * g.splits;
  const int per = g.tiles_m * g.tiles_n;
  const int bat = t / per;
  int tm, tn;
  grouped_tile(t - bat * per, g.tiles_m, g.tiles_n, 8, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int kb0 = (int)((int64_t)sp * g.nk / g.splits);
  const int kb1 = (int)((int64_t)(sp + 1) * g.nk / g.splits);

  PA pa;
  PB pb;
  pa.init(static_cast<const float*>(g.A) + bat * g.sA, g.lda, m0, g.M, g.K, tid);
  pb.init(static_cast<const float*>(g.B) + bat * g.sB, g.ldb, n0, g.N, g.K, tid);
  f32x4 acc[FM][FN], sum[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = sum[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  if (kb1 > kb0) {
    pa.load(kb0, tid);
    pb.load(kb0, tid);
    pa.store(lds[0], tid);
    pb.store(lds[0] + PA::SIZE, tid);
  }
  __syncthreads();
  int chain = g.span;
  for (int kt = kb0; kt < kb1; ++kt) {
    const float* cur = lds[(kt - kb0) & 1];
    float* oth = lds[(kt - kb0 + 1) & 1];
    if (kt + 1 < kb1) {
      pa.load(kt + 1, tid);
      pb.load(kt + 1, tid);
    }
    float fa[2][FM][4], fb[2][FN][4];
    frags<AKC, BM, FM>(cur, wm0, 0, li, lg, fa[0]);
    frags<BKC, BN, FN>(cur + PA::SIZE, wn0, 0, li, lg, fb[0]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < BK / 16; ++c) {
      if (c + 1 < BK / 16) {  // the next chunk's reads go out before this one's MFMAs
        frags<AKC, BM, FM>(cur, wm0, 16 * (c + 1), li, lg, fa[(c + 1) & 1]);
        frags<BKC, BN, FN>(cur + PA::SIZE, wn0, 16 * (c + 1), li, lg, fb[(c + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[c & 1][i][q], fb[c & 1][j][q],
                                                             acc[i][j], 0, 0, 0);
    }
    if (--chain == 0) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          sum[i][j] += acc[i][j];
          acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
      chain = g.span;
    }
    if (kt + 1 < kb1) {
      pa.store(oth, tid);
      pb.store(oth + PA::SIZE, tid);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) sum[i][j] += acc[i][j];
  if (g.splits == 1) {
    store_wave<AKC, BKC, FM, FN>(g, bat, m0 + wm0, n0 + wn0, lane, sum);
    return;
  }
  float* P = g.ws + (int64_t)w * (BM * BN);
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float* p = P + (wm0 + blk_row<AKC, FM>(i, 4 * lg + r)) * BN + wn0;
#pragma unroll
      for (int j = 0; j < FN; ++j) p[blk_row<BKC, FN>(j, li)] = sum[i][j][r];
    }
}

// The split tiles' sums (ws, in split order) and the epilogue: one thread
// per 4 consecutive columns of a tile row, grid (tiles, BM BN / 1024).
template <int BM, int BN>
__global__ __launch_bounds__(256) void sgemm_sum_kernel(GemmArgs g) {
  const int t = blockIdx.x, per = g.tiles_m * g.tiles_n, bat = t / per;
  int tm, tn;
  grouped_tile(t - bat * per, g.tiles_m, g.tiles_n, 8, tm, tn);
  const int e = (blockIdx.y * 256 + threadIdx.x) * 4;
  const int m = tm * BM + e / BN, n = tn * BN + e % BN;
  if (m >= g.M || n >= g.N) return;
  const float* P = g.ws + (int64_t)t * g.splits * (BM * BN) + e;
  f32x4 v = *reinterpret_cast<const f32x4*>(P);
  int s = 1;
  for (; s + 4 <= g.splits; s += 4) {
    f32x4 x[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      x[u] = *reinterpret_cast<const f32x4*>(P + (int64_t)(s + u) * (BM * BN));
#pragma unroll
    for (int u = 0; u < 4; ++u) v += x[u];
  }
  for (; s < g.splits; ++s) v += *reinterpret_cast<const f32x4*>(P + (int64_t)s * (BM * BN));
  const float* C = static_cast<const float*>(g.C) + (g.C ? bat * g.sC : 0) + (int64_t)m * g.ldc + n;
  float* D = static_cast<float*>(g.D) + bat * g.sD + (int64_t)m * g.ldd + n;
  float c[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) c[u] = g.beta != 0.0f && n + u < g.N ? C[u] : 0.0f;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    float x = g.alpha * v[u];
    if (g.beta != 0.0f) x = __builtin_fmaf(g.beta, c[u], x);
    if (n + u < g.N) D[u] = x;
  }
}

// 32 x 32 tiles for small products: one workgroup per tile, its waves split
// K between them (16-wide chunks, chunk c to wave c % WAVES), each reading
// its fragments straight from memory into registers two chunks ahead (no
// LDS, no barrier in the loop), and the partial tiles are summed through LDS
// in wave order. The loop is short: a one-workgroup launch of the 128 x 128
// kernel spends most of its time fetching instructions.
template <int WAVES, bool AKC, bool BKC, bool SYRK>
__global__ __launch_bounds__(64 * WAVES) void sgemm_direct_kernel(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) float part[WAVES][32 * 32];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int t = xcd_remap(blockIdx.x, gridDim.x);
  const int per = SYRK ? g.ntiles : g.tiles_m * g.tiles_n;
  const int bat = t / per;
  int tm, tn;
  if (SYRK)
    tri_tile(t, g.tiles_m, tm, tn);
  else
    grouped_tile(t - bat * per, g.tiles_m, g.tiles_n, 8, tm, tn);
  const int m0 = tm * 32, n0 = tn * 32, K = g.K;
  const uint32_t lda = (uint32_t)g.lda, ldb = (uint32_t)g.ldb;
  const float* A = static_cast<const float*>(g.A) + bat * g.sA + (AKC ? (int64_t)m0 * lda : m0);
  const float* B = static_cast<const float*>(g.B) + bat * g.sB + (BKC ? (int64_t)n0 * ldb : n0);
  const int nch = (K + 15) / 16;

  // f[i][q]: block i, MFMA q of the 16-wide chunk at k0 (kl = K - k0 left)
  auto fetch = [&](const float* X, uint32_t ld, bool kc, int rows, int k0, float (&f)[2][4])
                   __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rs = srsrc(kc ? X + k0 : X + (int64_t)k0 * ld);
    const int kl = K - k0;
    if (kc) {
      const bool whole = kl >= 16;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r = 16 * i + li;
        const uint32_t off = 4u * ((uint32_t)r * ld + 4u * lg);
        f32x4 x;
        if (whole)
          x = load4f(rs, r < rows ? off : kSOob);
        else
          x = load_part(rs, off, r < rows ? kl - 4 * lg : 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) f[i][q] = x[q];
      }
    } else {
      const bool whole = rows >= 32 || (rows & 1) == 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int k = 4 * lg + q;
        const uint32_t off = 4u * ((uint32_t)k * ld + 2u * li);
        if (whole) {
          const f32x2 x = __builtin_bit_cast(
              f32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, k < kl && 2 * li < rows ? off : kSOob, 0, 0));
          f[0][q] = x[0];
          f[1][q] = x[1];
        } else {
#pragma unroll
          for (int e = 0; e < 2; ++e)
            f[e][q] = __builtin_bit_cast(
                float, __builtin_amdgcn_raw_buffer_load_b32(
                           rs, k < kl && 2 * li + e < rows ? off + 4 * e : kSOob, 0, 0));
        }
      }
    }
  };
  f32x4 acc[2][2], sum[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = sum[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float fa[2][2][4], fb[2][2][4];
  auto get = [&](int c, int s) __attribute__((always_inline)) {
    fetch(A, lda, AKC, g.M - m0, 16 * c, fa[s]);
    fetch(B, ldb, BKC, g.N - n0, 16 * c, fb[s]);
  };
  int chain = g.span;  // 16-wide chunks per MFMA chain (even)
  auto mm = [&](int s) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[s][i][q], fb[s][j][q], acc[i][j], 0, 0, 0);
  };
  int c = wave;
  if (c < nch) get(c, 0);
  if (c + WAVES < nch) get(c + WAVES, 1);
  for (; c < nch; c += 2 * WAVES) {
    mm(0);
    if (c + 2 * WAVES < nch) get(c + 2 * WAVES, 0);
    if (c + WAVES < nch) {
      mm(1);
      if (c + 3 * WAVES < nch) get(c + 3 * WAVES, 1);
    }
    chain -= 2;
    if (chain == 0) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          sum[i][j] += acc[i][j];
          acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
      chain = g.span;
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        part[wave][blk_row<AKC, 2>(i, 4 * lg + r) * 32 + blk_row<BKC, 2>(j, li)] =
            sum[i][j][r] + acc[i][j][r];
  __syncthreads();
  direct_out<float, SYRK, WAVES>(g, part, bat, m0, n0);
}

template <int BM, int BN, int WGM, bool AKC, bool BKC>
static int run_tile(GemmArgs g, int splits, hipStream_t s) {
  g.tiles_m = (g.M + BM - 1) / BM;
  g.tiles_n = (g.N + BN - 1) / BN;
  g.ntiles = g.tiles_m * g.tiles_n * g.batch;
  g.nk = (g.K + 31) / 32;
  g.span = chain_length(g.K, 4) / 32;
  g.splits = splits;
  if (g.plan) {
    static thread_local char name[48];
    snprintf(name, sizeof name, "sgemm_tile_kernel<%d, %d> in %d", BM, BN, splits);
    *g.plan = name;
    return TRNBLAS_OK;
  }
  hipLaunchKernelGGL((sgemm_tile_kernel<BM, BN, WGM, AKC, BKC>), dim3(g.ntiles * g.splits), dim3(256), 0,
                     s, g);
  int rc = check_launch("trnblas_hip_gemm");
  if constexpr (BM == 64 && BN == 64) {  // the split tile
    if (rc || splits == 1) return rc;
    hipLaunchKernelGGL((sgemm_sum_kernel<BM, BN>), dim3(g.ntiles, BM * BN / 1024), dim3(256), 0, s, g);
    rc = check_launch("trnblas_hip_gemm(sum)");
  }
  return rc;
}

template <int WAVES, bool AKC, bool BKC, bool SYRK = false>
static int run_direct(GemmArgs g, hipStream_t s) {
  g.tiles_m = (g.M + 31) / 32;
  g.tiles_n = (g.N + 31) / 32;
  g.ntiles = SYRK ? g.tiles_m * (g.tiles_m + 1) / 2 : g.tiles_m * g.tiles_n * g.batch;
  g.span = chain_length(g.K, 4) / 16;
  if (planned(g, "sgemm_direct_kernel")) return TRNBLAS_OK;
  hipLaunchKernelGGL((sgemm_direct_kernel<WAVES, AKC, BKC, SYRK>), dim3(g.ntiles), dim3(64 * WAVES), 0,
                     s, g);
  return check_launch(SYRK ? "trnblas_hip_syrk" : "trnblas_hip_gemm");
}

// Which kernel: the least of these estimates (microseconds), each fitted to
// the measured times of its kernel (rms 4-10 %) over 9058 random shapes, the
// layouts mixed (M, N, K from 16 to 8192, batches to 256): a fixed cost, then
// the longer of one workgroup's chain (`chunk` per k step) and the CU's share
// of the MFMAs (`work` per k step and resident round), and the epilogue's
// share. The choice is within 2 % of the best kernel on average (1.2x at the
// 99th percentile). Against gemm.hip's kernels (packed where those need it)
// 2.6x faster over M, N, K log-uniform in 16..4096, e.g. (us) 96^3 3.9 /
// 13.1, 512^3 7.1 / 15.6, 1024^3 29 / 34, 1535^3 79 / 100, 16 x (112 x 384 x
// 384) 11.2 / 33.2, 48 x 442368 x 384 A^T B 190 / 409.
struct Est {
  double fixed, chunk, work, tail;
};
// tiles of one round, in CUs
static double rounds_of(double q) { return q <= 1.0 ? 1.0 : q > 6.0 ? q + 0.35 : std::ceil(q); }

static double est_tile(const Est& e, double tiles, double nk) {
  const double q = tiles / device_cus();
  return e.fixed + std::max(nk * e.chunk, rounds_of(q) * nk * e.work) + e.tail * std::max(q, 1.0);
}

static double tiles_of(const GemmArgs& g, int bm, int bn) {
  return (double)((g.M + bm - 1) / bm) * (double)((g.N + bn - 1) / bn) * (double)g.batch;
}

// gemm_dma_kernel (aligned operands): whole rounds of two 128 x 128 tiles per
// CU, or balanced by narrow tiles (half the work where N <= 64) / stream-K
// (choose_sk, narrow_tiles_pay), of which a tile takes up to 63 pieces. Fitted
// to 330 products' times (rms 7 %) and set against this file's (whose 64 x 64
// tiles are estimated 10 % high at 1 ms and more) where the two cross.
static double est_dma(const GemmArgs& g) {
  const double cus = device_cus(), t = tiles_of(g, 128, 128), nk = (g.K + 31) / 32;
  const double whole = std::floor(t / (2.0 * cus)), left = t - whole * 2.0 * cus;
  const double rounds = std::ceil(t / (2.0 * cus)), eff = t / (rounds * 2.0 * cus);
  if (t <= cus)
    return nk < 16 ? 7.1 + 2.25 * nk
                   : 18.0 + std::max(2.18 * 0.5 * tiles_of(g, 128, 64) / cus * nk, 0.65 * nk / 63.0);
  // (after whole rounds stream-K needs 4 k-tiles or 1 / 63 of K a workgroup)
  if (nk >= 16 && eff < 0.9 && rounds <= 8 &&
      (whole == 0.0 || left * nk / (2.0 * cus) >= std::max(4.0, std::ceil(nk / 63.0))))
    return 30.0 + (2.14 * nk + 3.0) * t / cus;
  const double last = left == 0.0 ? 0.0 : left <= cus && nk >= 16 ? 1.1 : 2.0;  // tiles per CU
  return 4.1 + 2.1 * (2.0 * whole + last) * nk + 3.75 * t / cus;
}

// The time of sgemm_direct_kernel for q 32 x 32 tiles per CU of `chunks`
// 16-wide chunks (w: the CU's MFMA time per chunk).
static double est_direct(int waves, double q, double chunks, double w) {
  return waves == 4 ? 3.3 + std::max(0.54 * std::ceil(chunks / 4), w * chunks) + 0.59 * q
                    : 3.25 + std::max(0.80 * std::ceil(chunks / 8), w * chunks) + 0.95 * q;
}

enum Kind { kDirect4, kDirect8, kT32x64, kT64x64, kT48x128, kT64x128 };

template <bool AKC, bool BKC>
static int run(Kind kind, int splits, const GemmArgs& g, hipStream_t s) {
  switch (kind) {
    case kDirect4:
      return run_direct<4, AKC, BKC>(g, s);
    case kDirect8:
      return run_direct<8, AKC, BKC>(g, s);
    case kT32x64:
      return run_tile<32, 64, 2, AKC, BKC>(g, 1, s);
    case kT64x64:
      return run_tile<64, 64, 2, AKC, BKC>(g, splits, s);
    case kT48x128:
      return run_tile<48, 128, 1, AKC, BKC>(g, 1, s);
    default:
      return run_tile<64, 128, 2, AKC, BKC>(g, 1, s);
  }
}

struct Choice {
  Kind kind;
  int splits;
  double us;
};

static Choice choose(const GemmArgs& g, size_t ws_bytes) {
  const double nk = (g.K + 31) / 32, chunks = (g.K + 15) / 16;
  Choice best{kT64x128, 1, est_tile({4.2, 0.0, 1.21, 1.53}, tiles_of(g, 64, 128), nk)};
  auto take = [&](Kind k, double t, int sp) {
    if (t < best.us) best = Choice{k, sp, t};
  };
  take(kT48x128, est_tile({4.9, 1.09, 0.954, 1.06}, tiles_of(g, 48, 128), nk), 1);
  take(kT32x64, est_tile({3.7, 0.486, 0.322, 0.67}, tiles_of(g, 32, 64), nk), 1);
  const double t64 = tiles_of(g, 64, 64), q32 = tiles_of(g, 32, 32) / device_cus();
  take(kT64x64, est_tile({4.0, 0.737, 0.591, 1.1}, t64, nk), 1);
  // split along K (at least 8 k-tiles each): the sum kernel's launch, the
  // partial tiles' bytes and its serial reads of one tile's. Fitted (rms 6 %) over 216
  // products of few tiles, K 2000 to 1200000, up to 512 splits: 63 x 63 x 1000001
  // 138 us (16 splits 2120)
  for (int sp = 2; sp <= 512 && 8 * sp <= nk; sp *= 2)
    if (t64 * sp <= 4.0 * device_cus() && t64 * sp * (64 * 64 * 4) <= (double)ws_bytes)
      take(kT64x64,
           est_tile({5.8, 0.741, 0.591, 0.0}, t64 * sp, std::ceil(nk / sp)) + t64 * sp * 0.0048 + sp * 0.073,
           sp);
  // (whole-K workgroups: past the fitted K their panels fall out of the caches
  // together, 10 x (549 x 174 x 41161) 2104 us against 1135 estimated)
  if (chunks <= 512.0) {
    // (past 128 chunks the last round costs as much as a full one)
    const double w = chunks > 128.0 ? 0.095 * rounds_of(q32) : 0.104 * q32;
    take(kDirect4, est_direct(4, q32, chunks, w), 1);
    take(kDirect8, est_direct(8, q32, chunks, 1.02 * w), 1);
  }
  return best;
}

bool sgemm_launch(const GemmArgs& g, bool akc, bool bkc, bool aligned, size_t ws_bytes,
                  hipStream_t s, int* rc) {
  const Choice c = choose(g, g.ws ? ws_bytes : 0);
  if (aligned && est_dma(g) <= c.us) return false;
  if (akc)
    *rc = bkc ? run<true, true>(c.kind, c.splits, g, s) : run<true, false>(c.kind, c.splits, g, s);
  else
    *rc = bkc ? run<false, true>(c.kind, c.splits, g, s) : run<false, false>(c.kind, c.splits, g, s);
  return true;
}

// Packing (M + N) K elements moves them twice (at about 4 TB/s) in one or two
// launches, and the packed product takes gemm_dma_kernel. The copy's share falls
// with M and N, so that near-cubes pay from 3500 up, skinny products never, and
// those whose K no kernel here splits well early. Us packed / in place: 1535^3
// 98 / 77, 3071^3 491 / 485, 4095^3 1091 / 1118, 6143^3 3520 / 3740, 1258 x 1258
// x 19063 600 / 751, 9722 x 19004 x 205 870 / 928, 17517 x 702 x 11415 2758 /
// 2540. Short K, whose time is the store of D, is estimated 3 % high in place.
// Over 285 unaligned products of 2^30 to 2^38 multiply-adds the choice is 0.3 %
// off the better one on average, at most 10 %.
extern "C" int trnblas_hip_gemm_pack_pays(int64_t M, int64_t N, int64_t K, int64_t batch,
                                          int64_t elements) {
  if (M < 1 || N < 1 || K < 1 || batch < 1 || M >= (1ll << 31) || N >= (1ll << 31) ||
      K >= (1ll << 31) - 4 || batch >= (1ll << 31))
    return 0;
  GemmArgs g{};
  g.M = (int)M;
  g.N = (int)N;
  g.K = (int)K;
  g.batch = (int)batch;
  const double in_place = choose(g, trnblas_hip_gemm_workspace()).us;
  const double packed = est_dma(g) + 6.0 + 8.0 * (double)elements / 4e6;
  return in_place > (K < 1024 ? 1.03 : 1.0) * packed;
}

// SYRK of few 128 x 128 tiles: gemm.hip's kernels spend it on instruction
// fetch and idle CUs, and unaligned operands ran at half the rate. Limits: a
// wave's serial chain (K to 3072 aligned, 4096 not: past them stream-K over
// more CUs is faster) and, aligned, q chunks <= 300, past which the LDS-DMA
// kernel's fewer L2 bytes count. Over 300 random SYRKs (n to 5000, k to 12000, those
// past the limits among them) 1.75x faster aligned and 2.5x unaligned on average,
// one 4 % slower. GPU time (us), n x k, before / after: 125 x 160 17.3 / 4.9, 241
// x 357 (unaligned) 50.8 / 6.6, 1072 x 116 (A^T A) 17.5 / 7.8, 506 x 2606
// (unaligned) 35.2 / 21.9.
bool ssyrk_launch(const GemmArgs& g, bool kc, bool aligned, hipStream_t s, int* rc) {
  const double t = (g.M + 31) / 32, chunks = (g.K + 15) / 16;
  const double q = 0.5 * t * (t + 1.0) / device_cus();
  if (aligned ? q > 12.0 || q * chunks > 300.0 || chunks > 192.0 : q > 20.0 || chunks > 256.0) return false;
  if (est_direct(4, q, chunks, 0.104 * q) <= est_direct(8, q, chunks, 0.106 * q))
    *rc = kc ? run_direct<4, true, true, true>(g, s) : run_direct<4, false, false, true>(g, s);
  else
    *rc = kc ? run_direct<8, true, true, true>(g, s) : run_direct<8, false, false, true>(g, s);
  return true;
}

}  // namespace trnblas
