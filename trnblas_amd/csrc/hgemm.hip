// 16-bit GEMM and SYRK for the sizes and alignments that gemm.hip's LDS-DMA
// kernels do not serve: small products, and operands that are not 16-byte
// ready (odd orbital counts). D = alpha op(A) op(B) + beta C on
// v_mfma_f32_16x16x32_{bf16,f16} with the semantics and the chains of gemm.hip
// (MFMA chains of chain_length(K) values folded into a separate fp32 sum).
//
// MFMA 16x16x32: lane l holds 8 k values of A (row l % 16) and of B (column
// l % 16); D row 4 (l / 16) + r in register r, column l % 16. Lane group
// g = l / 16 takes k = 8 g .. 8 g + 7 of a 32-wide chunk of both operands:
//  * of an operand stored K-contiguous, 8 consecutive values of its row
//    (from five 4-byte words); block i is rows 16 i .. 16 i + 15;
//  * of one stored M / N-contiguous, the pair at 2 (l % 16) of 8 rows of k
//    (4-byte loads); block i is rows 2 r + i.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "gemm.hpp"

namespace trnblas {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 __attribute__((aligned(4))) u32x4w;
typedef uint32_t __attribute__((aligned(2))) u32h;

template <typename T>
__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (std::is_same_v<T, __bf16>)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// One operand of a 32 x 32 tile: rows m or n, of which `rows` are inside the
// matrix. Rows past the edge repeat the last one (their outputs are not
// stored); k values past K are zeroed in both operands, in the last chunk
// only. Loads touch only the 4-byte words that hold values of the operand.
// ODD: K-contiguous rows that start inside a word are read as the five words
// around 8 values (a 16-byte load two bytes past a word takes about twice as
// long: 30^2 x 6683 SYRK 62 us).
template <bool KC, bool ODD>
struct Direct16 {
  static constexpr bool WORDS = KC && ODD;
  static constexpr int NW = WORDS ? 10 : 8;
  const char* X;        // the tile's corner at k = 0 (WORDS: the word that holds it)
  uint32_t ld, off[2];  // bytes
  uint32_t sh[2];       // WORDS: bits of block i's first word before its first value
  uint32_t lo;          // M / N-contiguous: byte selector of block 0 in two pairs
  bool pairs;
  __device__ __forceinline__ void init(const void* base, int64_t ld_, int row0, int rows, int li, int lg) {
    X = static_cast<const char*>(base) + 2 * (KC ? row0 * ld_ : (int64_t)row0);
    ld = 2u * (uint32_t)ld_;
    sh[0] = sh[1] = 0;
    if constexpr (KC) {
      const uint32_t d = WORDS ? (uint32_t)(uintptr_t)X & 2u : 0u;
      X -= d;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        off[i] = (uint32_t)min(16 * i + li, rows - 1) * ld + 16u * lg + d;
        if constexpr (WORDS) {
          sh[i] = 8u * (off[i] & 2u);
          off[i] &= ~3u;
        }
      }
    } else {
      // the last of an odd number of rows is the high half of the pair before
      pairs = rows > 1;
      off[0] = 2u * (uint32_t)max(min(2 * li, rows - 2), 0);
      lo = pairs && 2 * li == rows - 1 ? 0x07060302u : 0x05040100u;
    }
  }
  // the raw words of the whole chunk at k0
  __device__ __forceinline__ void load(int k0, int lg, uint32_t (&w)[NW]) const {
    if constexpr (KC) {
      const char* p = X + 2 * (int64_t)k0;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const u32x4 x = *reinterpret_cast<const u32x4w*>(p + off[i]);
#pragma unroll
        for (int e = 0; e < 4; ++e) w[NW / 2 * i + e] = x[e];
        if constexpr (WORDS)
          w[5 * i + 4] = *reinterpret_cast<const uint32_t*>(p + (off[i] + (sh[i] ? 16u : 12u)));
      }
    } else {
      const char* p = X + (int64_t)k0 * ld;
      const uint32_t o = off[0] + 8u * lg * ld;
      if (pairs) {
#pragma unroll
        for (int e = 0; e < 8; ++e) w[e] = *reinterpret_cast<const u32h*>(p + (o + e * ld));
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) w[e] = *reinterpret_cast<const uint16_t*>(p + (o + e * ld));
      }
    }
  }
  // of the last chunk, with 0 < kl < 32 values of k
  __device__ __forceinline__ void load_tail(int k0, int kl, int lg, uint32_t (&w)[NW]) const {
    if constexpr (KC) {
      const char* p = X + 2 * (int64_t)k0;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t o = off[i] - 16u * lg + (sh[i] >> 3);  // k = 0 of the chunk
#pragma unroll
        for (int e = 0; e < NW / 2; ++e) {
          uint32_t h[2];
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const int k = 8 * lg + 2 * e + u - (int)(sh[i] >> 4);
            h[u] = *reinterpret_cast<const uint16_t*>(p + (o + 2u * (uint32_t)max(min(k, kl - 1), 0)));
            if (k < 0 || k >= kl) h[u] = 0;
          }
          w[NW / 2 * i + e] = h[0] | h[1] << 16;
        }
      }
    } else {
      const char* p = X + (int64_t)k0 * ld + off[0];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int k = 8 * lg + e;
        const char* q = p + (uint32_t)min(k, kl - 1) * ld;
        w[e] = pairs ? *reinterpret_cast<const u32h*>(q) : *reinterpret_cast<const uint16_t*>(q);
        if (k >= kl) w[e] = 0;
      }
    }
  }
  // the fragments of blocks 0 and 1
  __device__ __forceinline__ void frags(const uint32_t (&w)[NW], u32x4 (&f)[2]) const {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (WORDS) {
#pragma unroll
        for (int i = 0; i < 2; ++i) f[i][e] = __builtin_amdgcn_alignbit(w[5 * i + e + 1], w[5 * i + e], sh[i]);
      } else if constexpr (KC) {
        f[0][e] = w[e];
        f[1][e] = w[4 + e];
      } else {
        f[0][e] = __builtin_amdgcn_perm(w[2 * e + 1], w[2 * e], lo);
        f[1][e] = __builtin_amdgcn_perm(w[2 * e + 1], w[2 * e], 0x07060302u);
      }
    }
  }
};

// 32 x 32 tiles: one workgroup per tile, its waves split K between them
// (32-wide chunks, chunk c to wave c % WAVES), each reading its fragments
// straight from memory two chunks ahead (no LDS, no barrier in the loop);
// the partial tiles are summed through LDS in wave order. A last chunk that K
// cuts goes before the loop, behind the first loads, so that the loop stays
// short (a workgroup runs it once, and fetching its code counts).
template <typename T, int WAVES, bool AKC, bool BKC, bool ODD, bool SYRK>
__global__ __launch_bounds__(64 * WAVES, 4) void hgemm_direct_kernel(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) float part[WAVES][32 * 32];
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int t = xcd_remap(blockIdx.x, gridDim.x);
  const int per = SYRK ? g.ntiles : g.tiles_m * g.tiles_n;
  const int bat = t / per;
  int tm, tn;
  if (SYRK)
    tri_tile(t, g.tiles_m, tm, tn);
  else
    grouped_tile(t - bat * per, g.tiles_m, g.tiles_n, 8, tm, tn);
  const int m0 = tm * 32, n0 = tn * 32;
  Direct16<AKC, ODD> A;
  Direct16<BKC, ODD> B;
  A.init(static_cast<const T*>(g.A) + bat * g.sA, g.lda, m0, g.M - m0, li, lg);
  B.init(static_cast<const T*>(g.B) + bat * g.sB, g.ldb, n0, g.N - n0, li, lg);
  const int nch = g.K / 32;
  f32x4 acc[2][2], sum[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = sum[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  uint32_t wa[2][Direct16<AKC, ODD>::NW], wb[2][Direct16<BKC, ODD>::NW];
  auto get = [&](int c, int s) __attribute__((always_inline)) {
    A.load(32 * c, lg, wa[s]);
    B.load(32 * c, lg, wb[s]);
  };
  auto mm = [&](const auto& xa, const auto& xb) __attribute__((always_inline)) {
    u32x4 fa[2], fb[2];
    A.frags(xa, fa);
    B.frags(xb, fb);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = mfma16<T>(fa[i], fb[j], acc[i][j]);
  };
  int chain = g.span;  // 32-wide chunks per MFMA chain (even)
  int c = wave;
  if (c < nch) get(c, 0);
  if (c + WAVES < nch) get(c + WAVES, 1);
  if (wave == nch % WAVES && (g.K & 31)) {
    uint32_t ta[Direct16<AKC, ODD>::NW], tb[Direct16<BKC, ODD>::NW];
    A.load_tail(32 * nch, g.K & 31, lg, ta);
    B.load_tail(32 * nch, g.K & 31, lg, tb);
    mm(ta, tb);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        sum[i][j] = acc[i][j];
        acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      }
  }
  for (; c < nch; c += 2 * WAVES) {
    mm(wa[0], wb[0]);
    if (c + 2 * WAVES < nch) get(c + 2 * WAVES, 0);
    if (c + WAVES < nch) {
      mm(wa[1], wb[1]);
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
      for (int r = 0; r < 4; ++r) {
        const int m = AKC ? 16 * i + 4 * lg + r : 2 * (4 * lg + r) + i;
        const int n = BKC ? 16 * j + li : 2 * li + j;
        part[wave][m * 32 + n] = sum[i][j][r] + acc[i][j][r];
      }
  __syncthreads();
  direct_out<T, SYRK, WAVES>(g, part, bat, m0, n0);
}

template <typename T, bool AKC, bool BKC, bool ODD, bool SYRK>
static int run_direct(int waves, GemmArgs g, hipStream_t s) {
  g.tiles_m = (g.M + 31) / 32;
  g.tiles_n = (g.N + 31) / 32;
  g.ntiles = SYRK ? g.tiles_m * (g.tiles_m + 1) / 2 : g.tiles_m * g.tiles_n * g.batch;
  g.span = chain_length(g.K, 2) / 32;
  if (planned(g, "hgemm_direct_kernel")) return TRNBLAS_OK;
  if (waves == 4)
    hipLaunchKernelGGL((hgemm_direct_kernel<T, 4, AKC, BKC, ODD, SYRK>), dim3(g.ntiles), dim3(256), 0, s, g);
  else
    hipLaunchKernelGGL((hgemm_direct_kernel<T, 8, AKC, BKC, ODD, SYRK>), dim3(g.ntiles), dim3(512), 0, s, g);
  return check_launch(SYRK ? "trnblas_hip_syrk" : "trnblas_hip_gemm");
}

// Where it serves (q: 32 x 32 tiles per CU, ch: 32-wide chunks of K): products
// of up to a few tiles per CU, whose time is launch, latency and, on the
// 128 x 128 kernels, instruction fetch and idle CUs. Aligned operands: q <= 6
// (SYRK 8) and q ch <= 200 (150 past 96 chunks: 1200 x 256 x 4792, 178, 30.3 us
// here, 23.8 on narrow tiles); above, the LDS-DMA kernels read each operand less
// often from L2. Unaligned ones up to q = 12 (SYRK 20): gemm_kernel runs
// them at half this kernel's rate, but for K of a few values, where the store
// of D counts and larger tiles store longer rows. The limits of ch are where
// one workgroup's serial chain takes as long as stream-K over the chip: 64 x
// 64 x 65536 (4 workgroups) 130 us here and 27 there, SYRK 56 x 181568 609 and
// 47. Both operands K-contiguous read 32 rows at once, words of odd rows five
// at a time, so these limits are lower (aligned 80 x 4416 SYRK 17.8 us here, 12.6
// there; unaligned 58 x 7427 37.8 and 27.4).
// Over 1500 random products (bf16, M and N 8 .. 3000, K 32 .. 20000, batches
// to 64, the layouts mixed), those past the rule among them, against gemm.hip's
// kernels (packed where those need it): GEMM 1.65x aligned and 2.5x unaligned
// faster on average, SYRK 1.65x and 2.3x, one 7 % and one 6 % slower. GPU time (us)
// before / after: 64 x 267 x 892 (A^T B) 19.9 / 5.3, 33 x (518 x 106 x 197) 28.6 /
// 13.4, aligned 913 x 224 x 408 (A B^T) 11.3 / 5.6. Four waves or eight: the smaller of two fitted times
// (rms 15 %; within 0.5 % of the better one on average).
template <typename T, bool SYRK>
bool hgemm_launch(const GemmArgs& g, bool akc, bool bkc, bool aligned, hipStream_t s, int* rc) {
  const double tm = (g.M + 31) / 32, tn = (g.N + 31) / 32, ch = (g.K + 31) / 32;
  const double q = (SYRK ? 0.5 * tm * (tm + 1.0) : tm * tn * g.batch) / device_cus();
  auto odd = [](const void* p, int64_t ld, int64_t st) {
    return (((uintptr_t)p >> 1 | ld | st) & 1) != 0;
  };
  const bool words = (akc && odd(g.A, g.lda, g.sA)) || (bkc && odd(g.B, g.ldb, g.sB));
  const bool kk = akc && bkc;
  if (aligned ? q > (kk ? 5.0 : SYRK ? 8.0 : 6.0) || ch > (kk ? 96.0 : 192.0) ||
                    q * ch > (kk ? 120.0 : ch > 96.0 ? 150.0 : 200.0)
              : q > (SYRK ? 20.0 : 12.0) || ch > (words ? (kk ? 128.0 : 256.0) : SYRK ? 256.0 : 384.0))
    return false;
  const double t4 = 3.3 + std::max(0.31 * std::ceil(ch / 4), 0.096 * q * ch) + 0.45 * q;
  const double t8 = 3.0 + std::max(0.58 * std::ceil(ch / 8), 0.092 * q * ch) + 0.88 * q;
  const int waves = t4 <= t8 ? 4 : 8;
  if constexpr (SYRK) {
    *rc = !akc    ? run_direct<T, false, false, false, true>(waves, g, s)
          : words ? run_direct<T, true, true, true, true>(waves, g, s)
                  : run_direct<T, true, true, false, true>(waves, g, s);
  } else if (!akc && !bkc) {
    *rc = run_direct<T, false, false, false, false>(waves, g, s);
  } else if (akc && bkc) {
    *rc = words ? run_direct<T, true, true, true, false>(waves, g, s)
                : run_direct<T, true, true, false, false>(waves, g, s);
  } else if (akc) {
    *rc = words ? run_direct<T, true, false, true, false>(waves, g, s)
                : run_direct<T, true, false, false, false>(waves, g, s);
  } else {
    *rc = words ? run_direct<T, false, true, true, false>(waves, g, s)
                : run_direct<T, false, true, false, false>(waves, g, s);
  }
  return true;
}

template bool hgemm_launch<__bf16, false>(const GemmArgs&, bool, bool, bool, hipStream_t, int*);
template bool hgemm_launch<__bf16, true>(const GemmArgs&, bool, bool, bool, hipStream_t, int*);
template bool hgemm_launch<_Float16, false>(const GemmArgs&, bool, bool, bool, hipStream_t, int*);
template bool hgemm_launch<_Float16, true>(const GemmArgs&, bool, bool, bool, hipStream_t, int*);

}  // namespace trnblas
