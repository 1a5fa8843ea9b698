// Batched in-place inversion of dense m x m matrices by blocked Gauss-Jordan: panels of
// 128 columns, each inverted by one workgroup with implicit partial pivoting within its
// two halves (k_gj_block), then a rank-128 update of the whole matrix on the matrix
// cores (k_gj_rows, k_gj_update).  Shared by the line factorisations (bcr.hip,
// lineilu.hip).
#pragma once

#include <type_traits>

#include "gemm.h"
#include "tf_common.h"

namespace tf {
namespace gj {

constexpr int PB = 128;  // Gauss-Jordan panel width

template <typename T>
__device__ __forceinline__ T readlane_t(T v, int lane);
template <>
__device__ __forceinline__ double readlane_t<double>(double v, int lane) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
  return __hiloint2double(hi, lo);
}
template <>
__device__ __forceinline__ float readlane_t<float>(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// Largest value of v over the wave, in every lane's view (a scalar): six DPP steps
// (row shifts, then the row broadcasts), about 70 cycles where six ds_bpermute
// shuffles take about 500.
__device__ __forceinline__ unsigned wave_max(unsigned v) {
#define TF_DPP_MAX(ctrl, rows)                                                                       \
  {                                                                                                  \
    const unsigned o = (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, rows, 0xf, false);      \
    v = o > v ? o : v;                                                                               \
  }
  TF_DPP_MAX(0x111, 0xf)  // row_shr:1
  TF_DPP_MAX(0x112, 0xf)  // row_shr:2
  TF_DPP_MAX(0x114, 0xf)  // row_shr:4
  TF_DPP_MAX(0x118, 0xf)  // row_shr:8
  TF_DPP_MAX(0x142, 0xa)  // row_bcast:15
  TF_DPP_MAX(0x143, 0xc)  // row_bcast:31
#undef TF_DPP_MAX
  return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

// 1 / x to about one ulp from the hardware's estimate, for |x| well inside the
// exponent range: one Newton step (float), two (double).
template <typename T>
__device__ __forceinline__ T fast_rcp(T x);
template <>
__device__ __forceinline__ double fast_rcp<double>(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.0), r, r);
  return fma(fma(-x, r, 1.0), r, r);
}
template <>
__device__ __forceinline__ float fast_rcp<float>(float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  return fmaf(fmaf(-x, r, 1.0f), r, r);
}

// Magnitude bits of x as a float (the sign is masked by the caller), and the biased
// exponent of a scalar.
__device__ __forceinline__ unsigned mag_bits(double x) { return __float_as_uint((float)fabs(x)); }
__device__ __forceinline__ unsigned mag_bits(float x) { return __float_as_uint(x); }
__device__ __forceinline__ int exponent_of(double x) { return (__double2hiint(x) >> 20) & 0x7ff; }
__device__ __forceinline__ int exponent_of(float x) { return (__float_as_int(x) >> 23) & 0xff; }

// Gauss-Jordan inversion of a 64 x 64 matrix in place, by the 8 waves of a block:
// lane = row, wave w holds columns 8w .. 8w+7 (cur, nxt).  Implicit partial
// pivoting: step k takes the row p(k) of largest magnitude among those not used yet
// and replaces column k, which becomes a unit column, by column p(k) of the inverse.
// On return lane p(k) holds row k of the inverse (mystep = k there) and column slot k
// its column p(k) = piv_of[k].
//
// The 64 steps are a serial chain and its latency is the time of the routine: a step
// that crosses waves costs about 400 cycles for the barrier and the LDS round trip
// alone.  So the wave that owns them takes four columns at a time through their four
// steps in its registers and publishes the four columns G that result; for every
// other column v the four steps together are v <- (v with the pivot rows zeroed)
// + sum_j G_j v[p_j], applied after one barrier, by the next owner to its next four
// columns first, so that its chain runs beside the others' updates.  Within the chain
// the maximum is reduced by DPP while every lane forms the reciprocal of its own entry.
// Rows and columns from cols on are those of the identity: the turns end with the last of
// the others (a block of 111 rows 60.4 -> 55.6 us in FP64), and a row that no turn took
// is its own.
constexpr int NS = 4;  // columns per turn
template <typename T>
struct Turns {
  T G[2][NS][64];   // a turn's columns, by its parity
  int prow[2][NS];  // ... and pivot rows
  int piv_of[64];
  T wmax[8];
};

template <typename T>
__device__ __forceinline__ void invert64(T (&cur)[NS], T (&nxt)[NS], int& mystep, Turns<T>& sh, int cols,
                                         int* nperturb, double repl) {
  const int nturns = (cols + NS - 1) / NS;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  T mx = 0;
#pragma unroll
  for (int i = 0; i < NS; ++i) mx = fmax(mx, fmax(fabs(cur[i]), fabs(nxt[i])));
  for (int off = 32; off > 0; off >>= 1) mx = fmax(mx, __shfl_xor(mx, off, 64));
  if (lane == 0) sh.wmax[wave] = mx;
  if (wave == 0) sh.piv_of[lane] = lane;
  __syncthreads();
  T amax = 0;
  for (int w = 0; w < 8; ++w) amax = fmax(amax, sh.wmax[w]);
  if (amax == (T)0) amax = 1;
  const T tol = (sizeof(T) == 8 ? (T)1e-13 : (T)1e-6) * amax;
  // pivots of a smaller or larger exponent go the careful way (below tol, or too small or
  // large for the quick reciprocal; with tol itself that large only those just above it go
  // the quick one, and none do beside an infinite entry)
  const int elo = __builtin_amdgcn_readfirstlane(exponent_of(fmax(tol, (T)1e-30)) + 1);
  const int ehi = max(exponent_of((T)1e30), elo);
  mystep = 64;
  // pivot key: magnitude bits, then the lane (ties go to the lower one); used rows 0
  unsigned alive = 0x7fffffc0u, tag = 63u - (unsigned)lane;

  // the steps of turn s on its columns c; the quick way reports a pivot that needs the
  // careful one (a branch in every step would cost a quarter of the step)
  auto steps = [&](int s, T (&c)[NS], int (&pj)[NS], auto careful) {
    bool odd = false;
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      const T f = c[j];
      const T inv = fast_rcp<T>(f);
      const int p = 63 - (int)(wave_max((mag_bits(f) & alive) | tag) & 63u);
      const T piv = readlane_t<T>(f, p);
      T ip = readlane_t<T>(inv, p);
      if constexpr (!decltype(careful)::value) {
        odd |= (unsigned)(exponent_of(piv) - elo) > (unsigned)(ehi - elo);
      } else {
        // a (numerically) zero pivot becomes +-tol, or +-repl amax when the caller
        // asks for a regularising replacement (approximate factorisations)
        T d = piv;
        if (fabs(piv) < tol) {
          const T rep = repl > 0.0 ? (T)repl * amax : tol;
          d = piv < (T)0 ? -rep : rep;
          if (lane == 0) atomicAdd(nperturb, 1);
        }
        ip = (T)1 / d;
      }
      const bool here = lane == p;
      const T g = here ? -ip : f * ip;
      T vp[NS];
#pragma unroll
      for (int i = 0; i < NS; ++i)
        if (i != j) vp[i] = readlane_t<T>(c[i], p);
      if (here) {
        alive = 0;
        tag = 0;
        mystep = s * NS + j;
#pragma unroll
        for (int i = 0; i < NS; ++i)
          if (i != j) c[i] = 0;
      }
#pragma unroll
      for (int i = 0; i < NS; ++i)
        if (i != j) c[i] -= g * vp[i];
      c[j] = -g;  // the column of the inverse that takes column j's place
      pj[j] = p;
    }
    return odd;
  };
  auto turn = [&](int s, T (&c)[NS]) {
    int pj[NS];
    T c0[NS];
#pragma unroll
    for (int i = 0; i < NS; ++i) c0[i] = c[i];
    const unsigned alive0 = alive, tag0 = tag;
    const int mystep0 = mystep;
    if (__builtin_expect(steps(s, c, pj, std::false_type()), 0)) {
#pragma unroll
      for (int i = 0; i < NS; ++i) c[i] = c0[i];
      alive = alive0;
      tag = tag0;
      mystep = mystep0;
      (void)steps(s, c, pj, std::true_type());
    }
#pragma unroll
    for (int j = 0; j < NS; ++j) sh.G[s & 1][j][lane] = c[j];
    if (lane < NS) sh.prow[s & 1][lane] = lane < 2 ? (lane ? pj[1] : pj[0]) : (lane == 2 ? pj[2] : pj[3]);
  };

  if (wave == 0) turn(0, cur);
  // the halves swap every turn, so that the turn's columns are cur and the next turn's
  // nxt in the waves that own them
#pragma unroll 1
  for (int s = 0; s < nturns; ++s) {
    __syncthreads();
    T g[NS];
    int p[NS];
    bool in = false;
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      g[j] = sh.G[s & 1][j][lane];
      p[j] = __builtin_amdgcn_readfirstlane(sh.prow[s & 1][j]);
    }
#pragma unroll
    for (int j = 0; j < NS; ++j)
      if (lane == p[j]) {
        in = true;
        mystep = s * NS + j;
      }
    if (in) alive = tag = 0;
    auto apply = [&](T (&c)[NS]) {
      // all pivot-row entries first, each in scalar registers of its own (left alone the
      // compiler reads each into the same pair just before its use, 20 cycles apiece)
      T vp[NS][NS];
#pragma unroll
      for (int i = 0; i < NS; ++i)
#pragma unroll
        for (int j = 0; j < NS; ++j) vp[i][j] = readlane_t<T>(c[i], p[j]);
#pragma unroll
      for (int i = 0; i < NS; ++i)
#pragma unroll
        for (int j = 0; j < NS; ++j) asm volatile("" : "+s"(vp[i][j]));
#pragma unroll
      for (int i = 0; i < NS; ++i) c[i] = in ? (T)0 : c[i];
#pragma unroll
      for (int j = 0; j < NS; ++j)
#pragma unroll
        for (int i = 0; i < NS; ++i) c[i] += g[j] * vp[i][j];
    };
    apply(nxt);
    if (s + 1 < nturns && wave == (s + 1) * NS / 8) turn(s + 1, nxt);
    if (wave != s * NS / 8) apply(cur);
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      const T t = cur[i];
      cur[i] = nxt[i];
      nxt[i] = t;
    }
  }
  if (nturns & 1)
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      const T t = cur[i];
      cur[i] = nxt[i];
      nxt[i] = t;
    }
  if (mystep == 64) mystep = lane;
  if (wave == 0) sh.piv_of[mystep] = lane;
  __syncthreads();
}

// Inverse of the pb x pb diagonal panel block of X_b at k0 (pb <= 128, padded with the
// identity; Nb: of Nb_b, PB x PB, in its place), into P_b (PB x PB; in place when Pb is
// null and k0 = 0): one block of 8 waves per matrix.  The block
// is held in LDS as 2 x 2 blocks of 64 and inverted by two Gauss-Jordan steps of width
// 64 (invert64 each), their block products on the matrix cores.  The block of 128 takes
// 61 us in FP64 and 44 us in FP32, for one matrix or 128 (of it 2 x 21 and 2 x 16 us the
// invert64 chains, 14 and 8 the products, which one CU's matrix units bound); the earlier
// panels of 64, in registers with the identity beside them, LDS shuffles and the division
// on the chain, took 60 and 46 us each.
template <typename T>
struct BlockLds {
  static constexpr int LD = PB + 1;  // a column of 64 rows meets every bank
  T s[PB * LD];
  Turns<T> turns;
};

template <typename T>
__global__ __launch_bounds__(512) void k_gj_block(int m, int k0, int pb, T* const* __restrict__ Xp,
                                                  const T* __restrict__ Nb, T* __restrict__ Pb,
                                                  int* __restrict__ nperturb, double repl) {
  extern __shared__ __align__(16) char lds[];
  BlockLds<T>& sh = *(BlockLds<T>*)lds;
  constexpr int LD = BlockLds<T>::LD;
  typedef typename Mfma<T>::acc_t acc_t;
  typename Global<T>::type* X = global_ptr(Xp[blockIdx.x]);
  typename Global<T>::type* P = Pb ? global_ptr(Pb + (long)blockIdx.x * PB * PB) : X;
  const int pp = Pb ? PB : m;
  typename Global<const T>::type* A =
      Nb ? global_ptr(Nb + (long)blockIdx.x * PB * PB) : (typename Global<const T>::type*)X + (long)k0 * m + k0;
  const int pa = Nb ? PB : m;
  T* S = sh.s;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lr = lane & 15, lk = lane >> 4;
  const int nb = pb > 64 ? 2 : 1;
  // sixteen loads in flight a thread (one at a time, the loop took 6 us of the block's 65)
  for (int q = 0; q < nb; ++q) {
    T v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = q * 64 + (t >> 7) + 4 * i, c = t & 127;
      v[i] = A[(long)min(r, pb - 1) * pa + min(c, pb - 1)];
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = q * 64 + (t >> 7) + 4 * i, c = t & 127;
      if (c < nb * 64) S[r * LD + c] = (r < pb && c < pb) ? v[i] : (r == c ? (T)1 : (T)0);
    }
  }
  __syncthreads();
  // the 64 x 64 block at (o, o) <- its inverse
  auto invert = [&](int o) {
    T c[2][NS];
#pragma unroll
    for (int q = 0; q < 2 * NS; ++q) c[q / NS][q % NS] = S[(o + lane) * LD + o + wave * 8 + q];
    int mystep;
    invert64<T>(c[0], c[1], mystep, sh.turns, min(pb - o, 64), nperturb, repl);
#pragma unroll
    for (int q = 0; q < 2 * NS; ++q) S[(o + mystep) * LD + o + sh.turns.piv_of[wave * 8 + q]] = c[q / NS][q % NS];
    __syncthreads();
  };
  // acc[h] = rows 16 (wave / 2), columns 32 (wave % 2) + 16 h of S[ar.., ac..] S[br.., bc..]
  auto product = [&](int ar, int ac, int br, int bc, acc_t (&acc)[2]) {
    acc[0] = acc[1] = acc_t{0, 0, 0, 0};
    const T* A = S + (ar + (wave >> 1) * 16 + lr) * LD + ac + lk;
    const T* B = S + (br + lk) * LD + bc + (wave & 1) * 32 + lr;
#pragma unroll 4
    for (int k = 0; k < 64; k += 4) {
      const T a = A[k];
      acc[0] = Mfma<T>::mma(a, B[k * LD], acc[0]);
      acc[1] = Mfma<T>::mma(a, B[k * LD + 16], acc[1]);
    }
  };
  // S[r.., c..] <- beta S[r.., c..] + alpha acc
  auto put = [&](int r, int c, const acc_t (&acc)[2], T alpha, T beta) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        T* s = S + (r + (wave >> 1) * 16 + Mfma<T>::row(lk, v)) * LD + c + (wave & 1) * 32 + h * 16 + lr;
        *s = beta != (T)0 ? *s + alpha * acc[h][v] : alpha * acc[h][v];
      }
  };
  invert(0);
  if (nb == 2) {
    acc_t u[2], w[2];
    product(0, 0, 0, 64, u);  // T12 = P11 A12
    __syncthreads();
    put(0, 64, u, (T)1, (T)0);
    __syncthreads();
    product(64, 0, 0, 64, u);  // A22 - A21 T12, and A21 <- -A21 P11
    product(64, 0, 0, 0, w);
    __syncthreads();
    put(64, 64, u, (T)-1, (T)1);
    put(64, 0, w, (T)-1, (T)0);
    __syncthreads();
    invert(64);
    product(64, 64, 64, 0, u);  // T21 = P22 A21
    __syncthreads();
    put(64, 0, u, (T)1, (T)0);
    __syncthreads();
    product(0, 64, 64, 0, u);  // P11 - T12 T21, and A12 <- -T12 P22
    product(0, 64, 64, 64, w);
    __syncthreads();
    put(0, 0, u, (T)-1, (T)1);
    put(0, 64, w, (T)-1, (T)0);
    __syncthreads();
  }
  for (int q = 0; q < nb; ++q) {
    T v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = S[(q * 64 + (t >> 7) + 4 * i) * LD + (t & 127)];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = q * 64 + (t >> 7) + 4 * i, c = t & 127;
      if (r < pb && c < pb) P[(long)r * pp + c] = v[i];
    }
  }
}

// Panel K = [k0, k0 + pb): T_b = P_b X_b[K, :] with X_b[K, K] taken as the identity, and
// Kc_b = X_b[:, K] (the update overwrites both).  Grid: (column tiles, row tiles of T +
// one row of copies, batch).
template <typename T, bool FAST>
__global__ __launch_bounds__(256, 2) void k_gj_rows(int m, int k0, int pb, T* const* __restrict__ Xp,
                                                    const T* __restrict__ Pb, T* __restrict__ Tb,
                                                    T* __restrict__ Kb) {
  typedef GemmTile<T, 64, 64, 16, FAST> Tile;
  __shared__ __align__(16) typename Tile::Lds sh;
  typename Global<const T>::type* X = global_ptr((const T*)Xp[blockIdx.z]);
  typename Global<const T>::type* P = global_ptr(Pb + (long)blockIdx.z * PB * PB);
  const int n0 = blockIdx.x * 64;
  if (blockIdx.y == gridDim.y - 1) {
    typename Global<T>::type* Kc = global_ptr(Kb + (long)blockIdx.z * PB * m);
    for (int e = threadIdx.x; e < 64 * PB; e += 256) {
      const int r = n0 + (e >> 7), c = e & 127;
      if (r < m && c < pb) Kc[(long)r * PB + c] = X[(long)r * m + k0 + c];
    }
    return;
  }
  typename Global<T>::type* Tm = global_ptr(Tb + (long)blockIdx.z * PB * m);
  const int m0 = blockIdx.y * 64;
  if (n0 >= k0 && n0 < k0 + pb) {
    for (int e = threadIdx.x; e < 64 * 64; e += 256) {
      const int r = m0 + (e >> 6), c = n0 + (e & 63);
      if (r < pb && c < k0 + pb) Tm[(long)r * m + c] = P[r * PB + c - k0];
    }
    return;
  }
  typename Tile::acc_t acc[Tile::TM][Tile::TN];
  Tile::run(pb, m, pb, P, PB, X + (long)k0 * m, m, m0, n0, sh, acc);
#pragma unroll
  for (int i = 0; i < Tile::TM; ++i)
#pragma unroll
    for (int j = 0; j < Tile::TN; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = m0 + Tile::row(i, v), c = n0 + Tile::col(j);
        if (r < pb && c < m) Tm[(long)r * m + c] = acc[i][j][v];
      }
}

// X_b[K, :] = T_b; elsewhere X_b = (X_b with the columns K zeroed) - Kc_b T_b.  The old
// values are read before the product is formed.
template <typename T, bool FAST>
__global__ __launch_bounds__(256, 2) void k_gj_update(int m, int k0, int pb, T* const* __restrict__ Xp,
                                                      const T* __restrict__ Tb, const T* __restrict__ Kb) {
  typedef GemmTile<T, 64, 64, 16, FAST> Tile;
  __shared__ __align__(16) typename Tile::Lds sh;
  typename Global<T>::type* X = global_ptr(Xp[blockIdx.z]);
  typename Global<const T>::type* Tm = global_ptr(Tb + (long)blockIdx.z * PB * m);
  typename Global<const T>::type* Kc = global_ptr(Kb + (long)blockIdx.z * PB * m);
  const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
  if (m0 >= k0 && m0 < k0 + pb) {
    for (int e = threadIdx.x; e < 64 * 64; e += 256) {
      const int r = m0 + (e >> 6), c = n0 + (e & 63);
      if (r < k0 + pb && c < m) X[(long)r * m + c] = Tm[(long)(r - k0) * m + c];
    }
    return;
  }
  const bool fresh = n0 >= k0 && n0 < k0 + pb;
  T prev[Tile::TM][Tile::TN][4];
#pragma unroll
  for (int i = 0; i < Tile::TM; ++i)
#pragma unroll
    for (int j = 0; j < Tile::TN; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = m0 + Tile::row(i, v), c = n0 + Tile::col(j);
        prev[i][j][v] = X[(long)(r < m ? r : m - 1) * m + (c < m ? c : m - 1)];
      }
  typename Tile::acc_t acc[Tile::TM][Tile::TN];
  Tile::run(m, m, pb, Kc, PB, Tm, m, m0, n0, sh, acc);
#pragma unroll
  for (int i = 0; i < Tile::TM; ++i)
#pragma unroll
    for (int j = 0; j < Tile::TN; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = m0 + Tile::row(i, v), c = n0 + Tile::col(j);
        if (r < m && c < m) X[(long)r * m + c] = (fresh ? (T)0 : prev[i][j][v]) - acc[i][j][v];
      }
}

// The diagonal block at k1 as k_gj_update will leave it, into N_b (PB x PB), 64 x 64 a
// block.  Grid: (2, 2, batch).
template <typename T, bool FAST>
__global__ __launch_bounds__(256, 2) void k_gj_next(int m, int k1, int pb, T* const* __restrict__ Xp,
                                                    const T* __restrict__ Tb, const T* __restrict__ Kb,
                                                    T* __restrict__ Nb) {
  typedef GemmTile<T, 64, 64, 16, FAST> Tile;
  __shared__ __align__(16) typename Tile::Lds sh;
  typename Global<const T>::type* X = global_ptr((const T*)Xp[blockIdx.z]);
  typename Global<const T>::type* Tm = global_ptr(Tb + (long)blockIdx.z * PB * m);
  typename Global<const T>::type* Kc = global_ptr(Kb + (long)blockIdx.z * PB * m);
  typename Global<T>::type* N = global_ptr(Nb + (long)blockIdx.z * PB * PB);
  const int m0 = k1 + blockIdx.y * 64, n0 = k1 + blockIdx.x * 64;
  if (m0 >= m || n0 >= m) return;
  typename Tile::acc_t acc[Tile::TM][Tile::TN];
  Tile::run(m, m, pb, Kc, PB, Tm, m, m0, n0, sh, acc);
#pragma unroll
  for (int i = 0; i < Tile::TM; ++i)
#pragma unroll
    for (int j = 0; j < Tile::TN; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = m0 + Tile::row(i, v), c = n0 + Tile::col(j);
        if (r < m && c < m) N[(r - k1) * PB + c - k1] = X[(long)r * m + c] - acc[i][j][v];
      }
}

// A second stream for the update beside the next k_gj_block, and the events between the
// two (made on first use; default priority).
struct Side {
  hipStream_t st = nullptr;
  hipEvent_t go = nullptr, done = nullptr;
  int ready() {
    if (!st) TF_HIP(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
    if (!go) TF_HIP(hipEventCreateWithFlags(&go, hipEventDisableTiming));
    if (!done) TF_HIP(hipEventCreateWithFlags(&done, hipEventDisableTiming));
    return 0;
  }
  void release() {
    if (st) (void)hipStreamDestroy(st);
    for (hipEvent_t e : {go, done})
      if (e) (void)hipEventDestroy(e);
  }
};

// Scratch of an inversion, per matrix of the batch: P and N PB x PB, Kc m x PB, T PB x m.
// side, N: null for no look-ahead.
template <typename T>
struct Scratch {
  T *P, *Kc, *Tb;
  T* N = nullptr;
  Side* side = nullptr;
};
inline size_t scratch_P() { return (size_t)PB * PB; }
// Look-ahead: the diagonal block of the next panel is updated by itself (k_gj_next) and
// inverted while the rest of the update runs, on the side stream; the block goes first, on
// the caller's (behind the update it found no CU with room for its LDS until the update's
// end, and every inversion took 3 to 10% longer).  It pays from 36 MB of matrices, where
// the update hides more of the block's 60 us than the events cost, up to 64 of them (more
// blocks take too many CUs from the update).  One inversion without and with, ms: FP64 64 x
// 768 1.86 / 1.79, 16 x 768 0.79 / 0.67, 8 x 768 0.65 / 0.60, 10 x 1600 2.55 / 2.31, 1 x
// 1600 1.19 / 1.20, 1 x 4096 4.99 / 4.26, 128 x 768 3.22 / 3.25; FP32 32 x 768 0.69 / 0.62,
// 16 x 768 0.535 / 0.528, 1 x 4096 3.34 / 2.97.
inline bool look_ahead(int m, int batch, size_t es) {
  return (double)batch * m * m * es >= 3.6e7 && batch <= 64 && m > PB;
}
inline size_t scratch_K(int m) { return (size_t)PB * m; }

// X_b <- X_b^-1 for the matrices of a device pointer list.  Up to 128 rows: one launch;
// otherwise three per panel of 128 columns.  The
// update reads and writes the whole matrix once per panel, and HBM bounds it: with
// panels of 64 and separate copies and stores (five launches a panel) the 128 matrices
// of 768 took 540 us per 64 columns in FP64, now 280 (update 366 us, rows 115, block 70
// per 128 columns); one matrix of 768 takes 110 us per 128 columns (170).
template <typename T>
int invert(int m, T* const* Xp, int batch, const Scratch<T>& w, int* nperturb, double repl, hipStream_t st) {
  if (batch <= 0) return 0;
  const size_t lds = sizeof(BlockLds<T>);
  TF_HIP(hipFuncSetAttribute((const void*)k_gj_block<T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  const int nt = (m + 63) / 64;
  const bool ahead = w.side && w.N && look_ahead(m, batch, sizeof(T)) && !prof_on();
  if (ahead)
    if (int e = w.side->ready()) return e;
  for (int k0 = 0; k0 < m; k0 += PB) {
    const int pb = m - k0 < PB ? m - k0 : PB;
    TF_PROF_WORK(PROF_GJ_PANEL, 2.0 * pb * pb * pb * batch);
    TF_PROF_BEGIN(PROF_GJ_PANEL, st);
    if (m <= PB) {
      hipLaunchKernelGGL(k_gj_block<T>, dim3(batch), dim3(512), lds, st, m, 0, m, Xp, (const T*)nullptr, (T*)nullptr,
                         nperturb, repl);
      TF_PROF_END(PROF_GJ_PANEL, st);
      return 0;
    }
    if (!ahead || k0 == 0)
      hipLaunchKernelGGL(k_gj_block<T>, dim3(batch), dim3(512), lds, st, m, k0, pb, Xp, (const T*)nullptr, w.P,
                         nperturb, repl);
    TF_PROF_END(PROF_GJ_PANEL, st);
    TF_PROF_WORK(PROF_GEMM, 2.0 * pb * (double)m * (m + pb) * batch);
    TF_PROF_BEGIN(PROF_GEMM, st);
    const dim3 gr(nt, (pb + 63) / 64 + 1, batch), gu(nt, nt, batch);
    auto go = [&](auto f) -> int {
      constexpr bool F = decltype(f)::value;
      hipLaunchKernelGGL((k_gj_rows<T, F>), gr, dim3(256), 0, st, m, k0, pb, Xp, (const T*)w.P, w.Tb, w.Kc);
      const int k1 = k0 + pb;
      const bool next = ahead && k1 < m;
      if (next) {
        hipLaunchKernelGGL((k_gj_next<T, F>), dim3(2, 2, batch), dim3(256), 0, st, m, k1, pb, Xp, (const T*)w.Tb,
                           (const T*)w.Kc, w.N);
        TF_HIP(hipEventRecord(w.side->go, st));
        hipLaunchKernelGGL(k_gj_block<T>, dim3(batch), dim3(512), lds, st, m, k1, m - k1 < PB ? m - k1 : PB, Xp,
                           (const T*)w.N, w.P, nperturb, repl);
        TF_HIP(hipStreamWaitEvent(w.side->st, w.side->go, 0));
      }
      hipLaunchKernelGGL((k_gj_update<T, F>), gu, dim3(256), 0, next ? w.side->st : st, m, k0, pb, Xp,
                         (const T*)w.Tb, (const T*)w.Kc);
      if (next) {
        TF_HIP(hipEventRecord(w.side->done, w.side->st));
        TF_HIP(hipStreamWaitEvent(st, w.side->done, 0));
      }
      return 0;
    };
    if (int e = gemm_fast<T>(m, pb, PB, m) ? go(std::true_type()) : go(std::false_type())) return e;
    TF_PROF_END(PROF_GEMM, st);
  }
  return 0;
}

}  // namespace gj
}  // namespace tf
