// Batched dense GEMM on the CDNA matrix cores:  C_b = alpha A_b B_b + beta C_b
// (row major, one pointer per batch entry).
//
// Block tile BM x BN with 256 threads = 4 waves in a 2 x 2 arrangement; each
// wave owns a (BM/2) x (BN/2) sub-tile made of 16 x 16 MFMA tiles
// (v_mfma_f64_16x16x4f64 for double, v_mfma_f32_16x16x4f32 for float).  The products
// are bound by the matrix cores; a loop of nothing but these instructions reaches
// 70 TF/s (FP64) and 130 (FP32) here.  With two LDS buffers and one barrier per chunk
// (GemmTile) 64 products of 768 run at 62 TF/s in FP64 and 122 in FP32, 7 of 4096 at
// 66 and 139; with one buffer, two barriers and loads of single elements they ran at
// 48 and 99, 59 and 125.
//
// MFMA 16x16x4 operand layout (one wave, lane l):
//   A fragment: A[l % 16][l / 16]   (16 x 4)
//   B fragment: B[l / 16][l % 16]   (4 x 16)
//   D: 4 values per lane, v = 0..3:
//      f32: D[4 (l / 16) + v][l % 16]
//      f64: D[(l / 16) + 4 v][l % 16]   (rows interleaved)
// (both measured on gfx950 with row-sum / column-sum inputs).
#pragma once

#include <cstdint>
#include <type_traits>

#include "tf_common.h"

namespace tf {

typedef double tf_double4 __attribute__((ext_vector_type(4)));
typedef float tf_float4 __attribute__((ext_vector_type(4)));

template <typename T>
struct Mfma;
template <>
struct Mfma<double> {
  typedef tf_double4 acc_t;
  static __device__ __forceinline__ int row(int lk, int v) { return lk + 4 * v; }
  static __device__ __forceinline__ acc_t mma(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mfma<float> {
  typedef tf_float4 acc_t;
  static __device__ __forceinline__ int row(int lk, int v) { return 4 * lk + v; }
  static __device__ __forceinline__ acc_t mma(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};

// FP32 operands as sums of BF16 terms for v_mfma_f32_16x16x16bf16_1k (lane l):
//   a[i] = A[l % 16][4 (l / 16) + i], b[i] = B[4 (l / 16) + i][l % 16],
//   D[4 (l / 16) + v][l % 16] (the f32 layout), measured on gfx950.
// x = hi + lo with hi = bf16(x), lo = bf16(x - hi) (round to nearest even): the
// three-term product hi*hi + hi*lo + lo*hi drops lo*lo and the rounding of lo,
// about 2^-16 relative per product.
typedef short tf_bf16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ unsigned short tf_bf16_rne(float f) {
  unsigned u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ __forceinline__ void tf_split4(const float v[4], tf_bf16x4& hi, tf_bf16x4& lo) {
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const unsigned short h = tf_bf16_rne(v[c]);
    hi[c] = (short)h;
    lo[c] = (short)tf_bf16_rne(v[c] - __uint_as_float((unsigned)h << 16));
  }
}

// One BM x BN tile of A B (added to acc with add) on 256 threads (4 waves, 2 x 2; each wave TM x TN MFMA
// tiles).  K is consumed in chunks of BK through two LDS buffers: while a chunk is
// multiplied the next one is stored from registers into the other buffer and the one
// after that is loaded, so a chunk costs one barrier and its loads have a whole
// chunk's MFMAs to arrive.  A is kept row-major in LDS (rows of BK + W elements), B
// k-major (rows of BN + W): 16-byte stores, few bank conflicts on the fragment reads
// (a pitch without any takes 5 KB more and a block less per CU: 45 for 57 TF/s).
// FAST: 16-byte loads from pointers that only advance with k; rows and columns past
// the edge are read from the last ones (never stored).  Needs 16-byte aligned operands
// and rows, K a multiple of BK and N of W (gemm_fast).  Otherwise every element is
// loaded by itself, zero past the edges.
// SPLIT 0: the type's own MFMA; SPLIT 1 or 3 (float only): BF16 terms of the FP32
// operands, one (hi*hi) or three products, FP32 accumulation.
template <typename T, int BM, int BN, int BK, bool FAST, int SPLIT = 0>
struct GemmTile {
  static constexpr int TM = BM / 32, TN = BN / 32;       // 16 x 16 tiles per wave
  static constexpr int W = 16 / (int)sizeof(T);
  static constexpr int PA = BK + W, PB = BN + W;         // LDS row pitches
  static constexpr int NA = BM * BK / 256, NB = BK * BN / 256;  // elements per thread and chunk
  typedef typename Mfma<T>::acc_t acc_t;
  typedef T V __attribute__((ext_vector_type(W)));
  typedef typename Global<const T>::type GT;
  typedef typename Global<const V>::type GV;
  struct Lds {
    T a[2][BM * PA];
    T b[2][BK * PB];
  };

  // row of value v of tile (i, j) and its column, relative to the block's tile
  static __device__ __forceinline__ int row(int i, int v) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    return (wave >> 1) * (BM / 2) + i * 16 + Mfma<T>::row(lane >> 4, v);
  }
  static __device__ __forceinline__ int col(int j) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    return (wave & 1) * (BN / 2) + j * 16 + (lane & 15);
  }

  static __device__ __forceinline__ void run(int M, int N, int K, GT* __restrict__ A, int lda,
                                             GT* __restrict__ B, int ldb, int m0, int n0, Lds& sh,
                                             acc_t (&acc)[TM][TN], bool add = false) {
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm0 = (wave >> 1) * (BM / 2), wn0 = (wave & 1) * (BN / 2);
    const int lr = lane & 15, lk = lane >> 4;
    if (add) {
      __syncthreads();  // an earlier product of the block has left the buffers
    } else {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = acc_t{0, 0, 0, 0};
    }
    V va[FAST ? NA / W : 1], vb[FAST ? NB / W : 1];
    T ra[FAST ? 1 : NA], rb[FAST ? 1 : NB];
    GT* pa[FAST ? NA / W : 1];
    GT* pb[FAST ? NB / W : 1];
    if constexpr (FAST) {
#pragma unroll
      for (int q = 0; q < NA / W; ++q) {
        const int e = t + q * 256, r = m0 + e / (BK / W);
        pa[q] = A + (long)(r < M ? r : M - 1) * lda + (e % (BK / W)) * W;
      }
#pragma unroll
      for (int q = 0; q < NB / W; ++q) {
        const int e = t + q * 256, c = n0 + (e % (BN / W)) * W;
        pb[q] = B + (long)(e / (BN / W)) * ldb + (c < N ? c : N - W);
      }
    }
    auto load = [&](int k0) {
      if constexpr (FAST) {
#pragma unroll
        for (int q = 0; q < NA / W; ++q) va[q] = *(GV*)(pa[q] + k0);
#pragma unroll
        for (int q = 0; q < NB / W; ++q) vb[q] = *(GV*)(pb[q] + (long)k0 * ldb);
      } else {
#pragma unroll
        for (int q = 0; q < NA; ++q) {
          const int e = t + q * 256, r = e / BK, c = e % BK;
          ra[q] = (m0 + r < M && k0 + c < K) ? A[(long)(m0 + r) * lda + k0 + c] : (T)0;
        }
#pragma unroll
        for (int q = 0; q < NB; ++q) {
          const int e = t + q * 256, r = e / BN, c = e % BN;
          rb[q] = (k0 + r < K && n0 + c < N) ? B[(long)(k0 + r) * ldb + n0 + c] : (T)0;
        }
      }
    };
    auto store = [&](int s) {
      if constexpr (FAST) {
#pragma unroll
        for (int q = 0; q < NA / W; ++q) {
          const int e = t + q * 256;
          *(V*)(sh.a[s] + e / (BK / W) * PA + (e % (BK / W)) * W) = va[q];
        }
#pragma unroll
        for (int q = 0; q < NB / W; ++q) {
          const int e = t + q * 256;
          *(V*)(sh.b[s] + e / (BN / W) * PB + (e % (BN / W)) * W) = vb[q];
        }
      } else {
#pragma unroll
        for (int q = 0; q < NA; ++q) {
          const int e = t + q * 256;
          sh.a[s][e / BK * PA + e % BK] = ra[q];
        }
#pragma unroll
        for (int q = 0; q < NB; ++q) {
          const int e = t + q * 256;
          sh.b[s][e / BN * PB + e % BN] = rb[q];
        }
      }
    };
    load(0);
    store(0);
    if (BK < K) load(BK);
    int s = 0;
    for (int k0 = 0; k0 < K; k0 += BK, s ^= 1) {
      __syncthreads();  // buffer s is stored, the other one consumed
      if (k0 + BK < K) {
        store(s ^ 1);
        if (k0 + 2 * BK < K) load(k0 + 2 * BK);
      }
      const T* __restrict__ As = sh.a[s];
      const T* __restrict__ Bs = sh.b[s];
      if constexpr (SPLIT == 0) {
#pragma unroll
        for (int ks = 0; ks < BK; ks += 4) {
          T a[TM], b[TN];
#pragma unroll
          for (int i = 0; i < TM; ++i) a[i] = As[(wm0 + i * 16 + lr) * PA + ks + lk];
#pragma unroll
          for (int j = 0; j < TN; ++j) b[j] = Bs[(ks + lk) * PB + wn0 + j * 16 + lr];
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = Mfma<T>::mma(a[i], b[j], acc[i][j]);
        }
      } else {
        static_assert(sizeof(T) == 4 && BK % 16 == 0, "BF16 terms need FP32 operands and 16-wide k chunks");
#pragma unroll
        for (int ks = 0; ks < BK; ks += 16) {
          tf_bf16x4 ah[TM], al[TM], bh[TN], bl[TN];
#pragma unroll
          for (int i = 0; i < TM; ++i) {
            float v[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) v[c] = As[(wm0 + i * 16 + lr) * PA + ks + 4 * lk + c];
            tf_split4(v, ah[i], al[i]);
          }
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            float v[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) v[c] = Bs[(ks + 4 * lk + c) * PB + wn0 + j * 16 + lr];
            tf_split4(v, bh[j], bl[j]);
          }
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
              if constexpr (SPLIT == 3) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(al[i], bh[j], acc[i][j], 0, 0, 0);
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ah[i], bl[j], acc[i][j], 0, 0, 0);
              }
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ah[i], bh[j], acc[i][j], 0, 0, 0);
            }
        }
      }
    }
  }
};

// Whether the products of a batch may use the FAST loads.  The operands are blocks of
// hipMalloc'ed arrays at multiples of their row lengths, so rows of whole 16-byte
// units make every operand aligned.
template <typename T>
inline bool gemm_fast(int N, int K, int lda, int ldb, int BK = 16) {
  constexpr int W = 16 / (int)sizeof(T);
  return lda % W == 0 && ldb % W == 0 && N % W == 0 && K % BK == 0 && K > 0;
}

// C_b = alpha (A_b B_b [+ A2_b B2_b]) + beta C_b (ADD: beta is not zero).  A2 may be a
// null list; with one, null operands of either pair leave that product out.  The old values of C are
// read before the product is formed: read after it they stand alone at the end of
// every tile (the rank-64 update of 128 matrices of 768 took 1.7 times as long).
template <typename T, int BM, int BN, int MINW, bool FAST, bool ADD, int SPLIT = 0, int BK = 16>
__global__ __launch_bounds__(256, MINW) void k_gemm_mfma(int M, int N, int K, T* const* __restrict__ Ap,
                                                         int lda, T* const* __restrict__ Bp, int ldb,
                                                         T* const* __restrict__ Cp, int ldc, double alpha,
                                                         double beta, T* const* __restrict__ A2p,
                                                         T* const* __restrict__ B2p) {
  typedef GemmTile<T, BM, BN, BK, FAST, SPLIT> Tile;
  __shared__ __align__(16) typename Tile::Lds sh;
  typename Global<T>::type* __restrict__ C = global_ptr(Cp[blockIdx.z]);
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  T prev[ADD ? Tile::TM : 1][Tile::TN][4];
  if constexpr (ADD) {
#pragma unroll
    for (int i = 0; i < Tile::TM; ++i)
#pragma unroll
      for (int j = 0; j < Tile::TN; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int gm = m0 + Tile::row(i, v), gn = n0 + Tile::col(j);
          prev[i][j][v] = C[(long)(gm < M ? gm : M - 1) * ldc + (gn < N ? gn : N - 1)];
        }
  }
  typename Tile::acc_t acc[Tile::TM][Tile::TN];
  const T *A = Ap[blockIdx.z], *A2 = A2p ? A2p[blockIdx.z] : nullptr;
  if (A || !A2p) Tile::run(M, N, K, global_ptr(A), lda, global_ptr((const T*)Bp[blockIdx.z]), ldb, m0, n0, sh, acc);
  if (A2) Tile::run(M, N, K, global_ptr(A2), lda, global_ptr((const T*)B2p[blockIdx.z]), ldb, m0, n0, sh, acc, A != nullptr);
#pragma unroll
  for (int i = 0; i < Tile::TM; ++i)
#pragma unroll
    for (int j = 0; j < Tile::TN; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int gm = m0 + Tile::row(i, v), gn = n0 + Tile::col(j);
        if (gm < M && gn < N) {
          double r = alpha * (double)acc[i][j][v];
          if constexpr (ADD) r += beta * (double)prev[i][j][v];
          C[(long)gm * ldc + gn] = (T)r;
        }
      }
}

}  // namespace tf

// ---- launch + tile autotuner ------------------------------------------------
//
// The first call with a given (type, M, N, K, batch) times every candidate tile on
// scratch operands of that shape (every batch entry aliases one scratch matrix, so the
// scratch stays at one A, B and C), and the fastest is cached for the life of the
// process.  With tuning off a fixed rule is used.
namespace tf {

enum GemmTileId : int { GEMM_128x128 = 0, GEMM_64x64 = 1, GEMM_32x32 = 2, GEMM_TILES = 3 };

template <typename T, int BM, int BN, int MINW, int SPLIT, int BK = 16>
inline void gemm_launch_tile(int M, int N, int K, T* const* A, int lda, T* const* B, int ldb, T* const* C, int ldc,
                             double alpha, double beta, int batch, hipStream_t st, T* const* A2, T* const* B2) {
  const dim3 grid((N + BN - 1) / BN, (M + BM - 1) / BM, batch);
  auto go = [&](auto fast, auto add) {
    hipLaunchKernelGGL((k_gemm_mfma<T, BM, BN, MINW, decltype(fast)::value, decltype(add)::value, SPLIT, BK>), grid,
                       dim3(256), 0, st, M, N, K, A, lda, B, ldb, C, ldc, alpha, beta, A2, B2);
  };
  const bool f = gemm_fast<T>(N, K, lda, ldb, BK), a = beta != 0.0;
  if (f && a) go(std::true_type(), std::true_type());
  else if (f) go(std::true_type(), std::false_type());
  else if (a) go(std::false_type(), std::true_type());
  else go(std::false_type(), std::false_type());
}

template <typename T, int SPLIT = 0>
inline void gemm_launch(int tile, int M, int N, int K, T* const* A, int lda, T* const* B, int ldb, T* const* C,
                        int ldc, double alpha, double beta, int batch, hipStream_t st, T* const* A2 = nullptr,
                        T* const* B2 = nullptr) {
  switch (tile) {
    case GEMM_128x128:
      gemm_launch_tile<T, 128, 128, 2, SPLIT>(M, N, K, A, lda, B, ldb, C, ldc, alpha, beta, batch, st, A2, B2);
      break;
    case GEMM_32x32:
      gemm_launch_tile<T, 32, 32, 4, SPLIT, 32>(M, N, K, A, lda, B, ldb, C, ldc, alpha, beta, batch, st, A2, B2);
      break;
    default:
      gemm_launch_tile<T, 64, 64, 4, SPLIT>(M, N, K, A, lda, B, ldb, C, ldc, alpha, beta, batch, st, A2, B2);
  }
}

int gemm_tuned_tile(int single, int M, int N, int K, int batch, hipStream_t st);

// C_b = alpha (A_b B_b [+ A2_b B2_b]) + beta C_b for b < batch (device pointer lists).
// split (float only): 1 or 3 BF16 terms per operand (hi*hi; hi*hi + hi*lo + lo*hi), with
// the tile that the tuner picked for the FP32 kernel of the same shape.
template <typename T>
inline void gemm_batched(int M, int N, int K, T* const* A, int lda, T* const* B, int ldb, T* const* C, int ldc,
                         double alpha, double beta, int batch, hipStream_t st, T* const* A2 = nullptr,
                         T* const* B2 = nullptr, int split = 0) {
  if (batch <= 0 || M <= 0 || N <= 0) return;
  const int tile = gemm_tuned_tile(sizeof(T) == 4, M, N, K, batch, st);
  if constexpr (sizeof(T) == 4) {
    if (split == 1) return gemm_launch<T, 1>(tile, M, N, K, A, lda, B, ldb, C, ldc, alpha, beta, batch, st, A2, B2);
    if (split == 3) return gemm_launch<T, 3>(tile, M, N, K, A, lda, B, ldb, C, ldc, alpha, beta, batch, st, A2, B2);
  }
  gemm_launch<T>(tile, M, N, K, A, lda, B, ldb, C, ldc, alpha, beta, batch, st, A2, B2);
}

}  // namespace tf
