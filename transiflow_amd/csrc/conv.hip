// Convolutions of the learned preconditioner on the cell grid (BF16 MFMA,
// FP32 accumulation): forward, backward-data, backward-weights, plus the
// elementwise pieces of training (MSE gradient, ReLU backward, Adam).
//
// Layouts.  Activations are cell-major [ncell][C] (the state vector layout:
// index c + C * cell, cell = i + nx (j + ny k)), BF16 stored as uint16.  A
// layer has taps = 3^dim neighbour offsets, tap = (dx+1) + 3 (dy+1) [+ 9 (dz+1)
// in 3D; dz = 0 in 2D], and zero padding outside the grid:
//
//   out[cell][co] = b[co] + sum_{tap, ci} W[tap][ci][co] in[cell + off(tap)][ci]
//
// which is a GEMM with K = taps * Cin (row k = tap * Cin + ci).  The MFMA
// copy of W is [Kpad][Npad] BF16 with K and Cout padded to multiples of 16.
//
// MFMA v_mfma_f32_16x16x16bf16_1k (one wave, lane l, measured on gfx950):
//   a[i] = A[l % 16][4 (l / 16) + i], b[i] = B[4 (l / 16) + i][l % 16],
//   D[4 (l / 16) + v][l % 16].
#include "tf_common.h"

#include <cstdint>
#include <type_traits>

namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((unsigned)h << 16); }
__device__ __forceinline__ uint16_t f2bf(float f) {  // round to nearest even
  unsigned u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)(u >> 16);  // inf / nan
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

struct Grid3 {
  int nx, ny, nz, dim;
};

// Cell c < ncell as coordinates.
__device__ __forceinline__ void coordinates(const Grid3& g, long ncell, long c, int& x, int& y, int& z) {
  if (ncell <= 0x7fffffffL) {
    const unsigned row = (unsigned)c / (unsigned)g.nx;
    x = (int)((unsigned)c - row * (unsigned)g.nx);
    z = (int)(row / (unsigned)g.ny);
    y = (int)(row - (unsigned)z * (unsigned)g.ny);
  } else {
    x = (int)(c % g.nx);
    y = (int)((c / g.nx) % g.ny);
    z = (int)(c / ((long)g.nx * g.ny));
  }
}

// Any number of input channels (the 2D networks' three).  One wave: 16 cells x all
// output tiles.  Block: 4 waves = 64 cells.  W (MFMA layout, BF16) and, per row k of it,
// the tap and the offset of its input from the cell's own are staged in LDS; a lane
// keeps one bit per tap that stays in the grid, so an A entry costs a bit test and a load.
constexpr int CONV_LDS = 28 * 1024;  // uint16 elements of W: K x N up to 864 x 32

struct TapRow {
  long off;
  int tap, pad;
};

__global__ __launch_bounds__(256) void k_conv_fwd(Grid3 g, long ncell, int cin, int cout, int kpad, int npad,
                                                  const uint16_t* __restrict__ in, const uint16_t* __restrict__ W,
                                                  const float* __restrict__ bias, int relu, float* __restrict__ out32,
                                                  uint16_t* __restrict__ out16) {
  extern __shared__ __align__(16) char conv_lds[];
  TapRow* rows = (TapRow*)conv_lds;                  // kpad
  uint16_t* Ws = (uint16_t*)(rows + kpad);           // kpad * npad
  const int taps = g.dim == 3 ? 27 : 9, K = taps * cin;
  for (int e = threadIdx.x; e < kpad * npad; e += 256) Ws[e] = W[e];
  for (int k = threadIdx.x; k < kpad; k += 256) {
    const int tap = k / cin, dx = tap % 3 - 1, dy = (tap / 3) % 3 - 1, dz = g.dim == 3 ? tap / 9 - 1 : 0;
    rows[k] = TapRow{((long)dx + (long)g.nx * (dy + (long)g.ny * dz)) * cin + (k - tap * cin), k < K ? tap : 31, 0};
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long cell0 = ((long)blockIdx.x * 4 + wave) * 16;
  const long cell = cell0 + (lane & 15);
  const int q = lane >> 4;
  unsigned inside = 0;  // bit per tap
  if (cell < ncell) {
    int x, y, z;
    coordinates(g, ncell, cell, x, y, z);
    for (int t = 0; t < taps; ++t) {
      const int X = x + t % 3 - 1, Y = y + (t / 3) % 3 - 1, Z = z + (g.dim == 3 ? t / 9 - 1 : 0);
      if ((unsigned)X < (unsigned)g.nx && (unsigned)Y < (unsigned)g.ny && (unsigned)Z < (unsigned)g.nz) inside |= 1u << t;
    }
  }
  const uint16_t* own = in + cell * cin;
  const int ntiles = npad / 16;
  f32x4 acc0 = {0, 0, 0, 0}, acc1 = {0, 0, 0, 0};
  for (int k0 = 0; k0 < kpad; k0 += 16) {
    bf16x4 a;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const TapRow row = rows[k0 + 4 * q + i];
      a[i] = (inside >> row.tap) & 1u ? (short)own[row.off] : (short)0;
    }
    bf16x4 b0, b1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      b0[i] = (short)Ws[(k0 + 4 * q + i) * npad + (lane & 15)];
      b1[i] = ntiles > 1 ? (short)Ws[(k0 + 4 * q + i) * npad + 16 + (lane & 15)] : (short)0;
    }
    acc0 = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b0, acc0, 0, 0, 0);
    if (ntiles > 1) acc1 = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b1, acc1, 0, 0, 0);
  }
  // D[4 q + v][lane % 16]: row = cell0 + 4 q + v, column = output channel
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    if (t >= ntiles) break;
    const int co = t * 16 + (lane & 15);
    if (co >= cout) continue;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const long c = cell0 + 4 * q + v;
      if (c >= ncell) continue;
      float s = (t == 0 ? acc0[v] : acc1[v]) + (bias ? bias[co] : 0.f);
      if (relu) s = s > 0.f ? s : 0.f;
      if (out32) out32[c * cout + co] = s;
      if (out16) out16[c * cout + co] = f2bf(s);
    }
  }
}

// W [kpad][npad] -> LDS transposed, [n] rows of kpad + WPAD entries: four k of two n per
// item, 8-byte stores.  The pad spreads the rows that a fragment read touches over the
// banks (kpad alone is a multiple of 32 dwords for 32 channels).
constexpr int WPAD = 8;

__device__ __forceinline__ void stage_weights(int kpad, int npad, const uint16_t* __restrict__ W,
                                              uint16_t* __restrict__ Ws) {
  const int kp = kpad + WPAD, half = npad / 2;
  for (int e = threadIdx.x; e < kpad / 4 * half; e += blockDim.x) {
    const int n = 2 * (e % half), k = 4 * (e / half);
    bf16x4 lo, hi;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned w = *reinterpret_cast<const unsigned*>(W + (k + i) * npad + n);
      lo[i] = (short)(w & 0xffffu);
      hi[i] = (short)(w >> 16);
    }
    *reinterpret_cast<bf16x4*>(Ws + n * kp + k) = lo;
    *reinterpret_cast<bf16x4*>(Ws + (n + 1) * kp + k) = hi;
  }
}

// Bias, ReLU and the stores of MT x NT tiles: D[4 q + v][r] is cell base + 16 m + 4 q + v,
// output channel 16 t + r.
template <int MT, int NT>
__device__ __forceinline__ void conv_store(const f32x4 (&acc)[MT][NT], long base, long ncell, int cout,
                                           const float* __restrict__ bias, int relu, float* __restrict__ out32,
                                           uint16_t* __restrict__ out16) {
  const int lane = threadIdx.x & 63, q = lane >> 4, r = lane & 15;
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int co = t * 16 + r;
      if (co >= cout) continue;
      const float bco = bias ? bias[co] : 0.f;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const long c = base + m * 16 + 4 * q + v;
        if (c >= ncell) continue;
        float sv = acc[m][t][v] + bco;
        if (relu) sv = sv > 0.f ? sv : 0.f;
        if (out32) out32[c * cout + co] = sv;
        if (out16) out16[c * cout + co] = f2bf(sv);
      }
    }
}

// The same layer when cin is a multiple of 4 (every layer of the 3D network and
// its data gradients): a lane's four K entries of one MFMA step are four
// consecutive channels of one tap, so the A fragment is one 8-byte load of the
// neighbour's activations; W is staged transposed ([n][k]) so the B fragment
// is one 8-byte LDS read.  Each wave computes MT tiles of 16 cells, reusing
// each B fragment MT times, and a block stages W once for 128 MT cells.
// The K order of the accumulation is that of k_conv_fwd.
// Bound by the latency of the neighbour loads: C32 (cin = 32) walks the taps with the
// next tap's loads in flight and finds a neighbour once per tap, and small grids take
// fewer tiles per wave, so that every CU has waves (conv_tiles).  32 -> 32 channels: 32^3 40 -> 15 us, 256^2
// 31 -> 14 us against one step's loads at a time, 4 waves a block and four tiles always.
template <int NT, int MT, bool C32>
__global__ __launch_bounds__(512) void k_conv_fwd_v(Grid3 g, long ncell, int cin, int cout, int kpad, int npad,
                                                    const uint16_t* __restrict__ in, const uint16_t* __restrict__ W,
                                                    const float* __restrict__ bias, int relu,
                                                    float* __restrict__ out32, uint16_t* __restrict__ out16) {
  extern __shared__ __align__(16) uint16_t Ws[];   // npad rows of kpad + WPAD
  stage_weights(kpad, npad, W, Ws);
  const int kp = kpad + WPAD;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int q = lane >> 4, r = lane & 15;
  const int taps = g.dim == 3 ? 27 : 9;
  const long base = ((long)blockIdx.x * 8 + wave) * (MT * 16);
  int xm[MT], ym[MT], zm[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const long cell = base + m * 16 + r;
    coordinates(g, ncell, cell < ncell ? cell : 0, xm[m], ym[m], zm[m]);
    if (cell >= ncell) zm[m] = -4;  // no neighbour of a cell past the end is in the grid
  }
  f32x4 acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[m][t] = f32x4{0, 0, 0, 0};
  // four channels from ci of the neighbour through a tap (zero outside the grid)
  auto piece = [&](int m, int tap, int ci, int channels) {
    const int X = xm[m] + tap % 3 - 1, Y = ym[m] + (tap / 3) % 3 - 1, Z = zm[m] + (g.dim == 3 ? tap / 9 - 1 : 0);
    bf16x4 a = {0, 0, 0, 0};
    if ((unsigned)X < (unsigned)g.nx && (unsigned)Y < (unsigned)g.ny && (unsigned)Z < (unsigned)g.nz)
      a = *reinterpret_cast<const bf16x4*>(in + ((long)X + (long)g.nx * (Y + (long)g.ny * Z)) * channels + ci);
    return a;
  };
  if constexpr (C32) {
    bf16x4 a[2][MT], nx[2][MT];
    auto load = [&](int tap, bf16x4 (&to)[2][MT]) {
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const int X = xm[m] + tap % 3 - 1, Y = ym[m] + (tap / 3) % 3 - 1, Z = zm[m] + (g.dim == 3 ? tap / 9 - 1 : 0);
        to[0][m] = to[1][m] = bf16x4{0, 0, 0, 0};
        if ((unsigned)X < (unsigned)g.nx && (unsigned)Y < (unsigned)g.ny && (unsigned)Z < (unsigned)g.nz) {
          const uint16_t* p = in + ((long)X + (long)g.nx * (Y + (long)g.ny * Z)) * 32 + 4 * q;
          to[0][m] = *reinterpret_cast<const bf16x4*>(p);
          to[1][m] = *reinterpret_cast<const bf16x4*>(p + 16);
        }
      }
    };
    load(0, nx);
    __syncthreads();
    for (int tap = 0; tap < taps; ++tap) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int m = 0; m < MT; ++m) a[h][m] = nx[h][m];
      if (tap + 1 < taps) load(tap + 1, nx);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        bf16x4 b[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t)
          b[t] = *reinterpret_cast<const bf16x4*>(&Ws[(t * 16 + r) * kp + tap * 32 + 16 * h + 4 * q]);
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int t = 0; t < NT; ++t)
            acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[h][m], b[t], acc[m][t], 0, 0, 0);
      }
    }
  } else {
    __syncthreads();
    const int K = taps * cin;
#pragma unroll 2
    for (int k0 = 0; k0 < kpad; k0 += 16) {
      const int k = k0 + 4 * q;  // this lane's four K entries: channels ci..ci+3 of one tap
      const int tap = k / cin;
      bf16x4 b[NT], a[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) a[m] = k < K ? piece(m, tap, k - tap * cin, cin) : bf16x4{0, 0, 0, 0};
#pragma unroll
      for (int t = 0; t < NT; ++t) b[t] = *reinterpret_cast<const bf16x4*>(&Ws[(t * 16 + r) * kp + k]);
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < NT; ++t)
          acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[m], b[t], acc[m][t], 0, 0, 0);
    }
  }
  conv_store<MT, NT>(acc, base, ncell, cout, bias, relu, out32, out16);
}

// Tiles of 16 cells per wave: one while that gives at most two blocks of 128 cells per
// CU, else four (a B fragment and a staging of W per four tiles).
inline int conv_tiles(long ncell) { return ncell <= 512L * 128 ? 1 : 4; }

// Partial weight and bias gradients, one block per chunk of cells:
//   partial[block][k][co] = sum over the block's cells of patch[cell][k] g[cell][co],
//   then 32 entries       sum over the block's cells of g32[cell][co] (the FP32 gradient;
//                         left unwritten when g32 is null)
// as MFMAs with M = k, N = co and the cells as the reduction dimension.  The
// block walks its cells WG_SUB at a time: the patch (all K values of WG_SUB
// cells, zero outside the grid) and the gradient are staged transposed in LDS
// ([k][cell], [co][cell]), so a lane's four reduction entries are one 8-byte
// LDS read for A and for B.  A staging item is VEC channels of one tap for four
// consecutive cells: four loads of VEC channels, VEC stores of four cells each.
// Wave w of the WG_WAVES owns the k-tiles w, w + WG_WAVES, ... for both n-tiles and
// keeps their accumulators in registers across the whole chunk, so a block writes its
// partial once.
// The staging bounds it (2-byte LDS stores of single cells took 331 us at 32^3 with 32
// channels in and out, in 32 blocks); chunks are sized for about 256 blocks:
// 20 us there, with the sum of the partials 26.
constexpr int WG_SUB = 32;
constexpr int WG_PITCH = WG_SUB + 4;  // LDS row pitch: 16 rows by 4 cells spread over the banks
constexpr int WG_WAVES = 8;
constexpr int WG_MAXT = 7;    // k-tiles per wave: 56 / 8
constexpr int WG_KMAX = 896;  // staged K rows

// cells per block (a multiple of WG_SUB) for about 256 blocks, at most 1024 (an empty
// grid, too, gets a block size to divide by)
inline long wgrad_chunk(long ncell) {
  const long c = ((ncell + 255) / 256 + WG_SUB - 1) / WG_SUB * WG_SUB;
  return c < WG_SUB ? WG_SUB : (c < 1024 ? c : 1024);
}
inline long wgrad_blocks(long ncell) { return (ncell + wgrad_chunk(ncell) - 1) / wgrad_chunk(ncell); }
inline size_t wgrad_lds(int kpad, int npad) { return sizeof(uint16_t) * (size_t)(kpad + npad) * WG_PITCH; }

template <int VEC>   // channels per staging load: 8 (16 bytes), 4 (8 bytes) or 1
__global__ __launch_bounds__(64 * WG_WAVES) void k_conv_wgrad(Grid3 g, long ncell, int chunk, int cin, int cout,
                                                              int kpad, int npad, const uint16_t* __restrict__ in,
                                                              const uint16_t* __restrict__ gout,
                                                              const float* __restrict__ g32,
                                                              float* __restrict__ partial) {
  extern __shared__ __align__(16) uint16_t lds[];
  uint16_t* pt = lds;                     // [kpad][WG_PITCH]
  uint16_t* gt = lds + kpad * WG_PITCH;   // [npad][WG_PITCH]
  constexpr int NT = 64 * WG_WAVES;
  const int taps = g.dim == 3 ? 27 : 9;
  const int K = taps * cin;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int q = lane >> 4, r = lane & 15;
  const int ktiles = kpad / 16, ntiles = npad / 16;
  const int groups = cin / VEC;                 // channel pieces per (cell, tap)
  const long c0 = (long)blockIdx.x * chunk;
  const long c1 = c0 + chunk < ncell ? c0 + chunk : ncell;
  // the K padding rows stay zero for the whole chunk
  for (int e = K * WG_PITCH + threadIdx.x; e < kpad * WG_PITCH; e += NT) pt[e] = 0;
  f32x4 acc[WG_MAXT][2];
#pragma unroll
  for (int t = 0; t < WG_MAXT; ++t) acc[t][0] = acc[t][1] = f32x4{0, 0, 0, 0};
  for (long s0 = c0; s0 < c1; s0 += WG_SUB) {
    // (piece, four cells, tap) items: consecutive threads take consecutive pieces of one neighbour
    for (int p = threadIdx.x; p < WG_SUB / 4 * taps * groups; p += NT) {
      const int gi = p % groups, rest = p / groups;
      const int c4 = rest % (WG_SUB / 4), tap = rest / (WG_SUB / 4);
      const int dx = tap % 3 - 1, dy = (tap / 3) % 3 - 1, dz = g.dim == 3 ? tap / 9 - 1 : 0;
      unsigned ic = (unsigned)(s0 + 4 * c4);   // ncell < 2^31 (checked by the caller)
      unsigned row = ic / (unsigned)g.nx;
      int x = (int)(ic - row * (unsigned)g.nx), y = (int)(row % (unsigned)g.ny), z = (int)(row / (unsigned)g.ny);
      uint16_t v[4][VEC];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int X = x + dx, Y = y + dy, Z = z + dz;
        const bool inside = s0 + 4 * c4 + i < c1 && (unsigned)X < (unsigned)g.nx && (unsigned)Y < (unsigned)g.ny &&
                            (unsigned)Z < (unsigned)g.nz;
        const uint16_t* src = in + ((long)X + (long)g.nx * (Y + (long)g.ny * Z)) * cin + gi * VEC;
        if constexpr (VEC == 8) {
          uint4 w = {0, 0, 0, 0};
          if (inside) w = *reinterpret_cast<const uint4*>(src);
          const unsigned u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
          for (int j = 0; j < 8; ++j) v[i][j] = (uint16_t)(j & 1 ? u[j / 2] >> 16 : u[j / 2] & 0xffffu);
        } else if constexpr (VEC == 4) {
          uint2 w = {0, 0};
          if (inside) w = *reinterpret_cast<const uint2*>(src);
          const unsigned u[2] = {w.x, w.y};
#pragma unroll
          for (int j = 0; j < 4; ++j) v[i][j] = (uint16_t)(j & 1 ? u[j / 2] >> 16 : u[j / 2] & 0xffffu);
        } else {
          v[i][0] = inside ? src[0] : (uint16_t)0;
        }
        if (++x == g.nx) {  // the next cell
          x = 0;
          if (++y == g.ny) {
            y = 0;
            ++z;
          }
        }
      }
      const int k0 = tap * cin + gi * VEC;
#pragma unroll
      for (int j = 0; j < VEC; ++j)
        *reinterpret_cast<bf16x4*>(&pt[(k0 + j) * WG_PITCH + 4 * c4]) =
            bf16x4{(short)v[0][j], (short)v[1][j], (short)v[2][j], (short)v[3][j]};
    }
    for (int e = threadIdx.x; e < npad * (WG_SUB / 4); e += NT) {
      const int co = e % npad, c4 = e / npad;
      bf16x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const long cell = s0 + 4 * c4 + i;
        v[i] = (co < cout && cell < c1) ? (short)gout[cell * cout + co] : (short)0;
      }
      *reinterpret_cast<bf16x4*>(&gt[co * WG_PITCH + 4 * c4]) = v;
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < WG_SUB; h += 16) {
      const bf16x4 b0 = *reinterpret_cast<const bf16x4*>(&gt[r * WG_PITCH + h + 4 * q]);
      bf16x4 b1 = {0, 0, 0, 0};
      if (ntiles > 1) b1 = *reinterpret_cast<const bf16x4*>(&gt[(16 + r) * WG_PITCH + h + 4 * q]);
#pragma unroll
      for (int t = 0; t < WG_MAXT; ++t) {
        const int kt = wave + WG_WAVES * t;
        if (kt < ktiles) {
          const bf16x4 a = *reinterpret_cast<const bf16x4*>(&pt[(kt * 16 + r) * WG_PITCH + h + 4 * q]);
          acc[t][0] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b0, acc[t][0], 0, 0, 0);
          if (ntiles > 1) acc[t][1] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b1, acc[t][1], 0, 0, 0);
        }
      }
    }
    __syncthreads();
  }
  const long len = (long)kpad * npad;
  float* P = partial + (long)blockIdx.x * (len + 32);
#pragma unroll
  for (int t = 0; t < WG_MAXT; ++t) {
    const int kt = wave + WG_WAVES * t;
    if (kt < ktiles) {
#pragma unroll
      for (int n = 0; n < 2; ++n)
        if (n < ntiles)
#pragma unroll
          for (int v = 0; v < 4; ++v) P[(long)(kt * 16 + 4 * q + v) * npad + n * 16 + r] = acc[t][n][v];
    }
  }
  if (!g32) return;
  // bias: thread t sums channel t % cout of every (NT / cout)-th cell, then a tree per channel
  float* red = (float*)lds;
  const int rows = NT / cout, co = threadIdx.x % cout, first = threadIdx.x / cout;
  float s = 0.f;
  if (first < rows)
    for (long c = c0 + first; c < c1; c += rows) s += g32[c * cout + co];
  red[threadIdx.x] = s;
  __syncthreads();
  if (threadIdx.x < 32) {
    float sum = 0.f;
    if ((int)threadIdx.x < cout)
      for (int i = 0; i < rows; ++i) sum += red[i * cout + threadIdx.x];
    P[len + threadIdx.x] = sum;
  }
}

// dW[e] (e < len), db[e - len] (or null) = sum_b partial[b][e]  (fixed order:
// deterministic).  64 entries per block, a quarter of the blocks' partials per wave.
__global__ __launch_bounds__(256) void k_sum_partials(int nb, long len, int cout, const float* __restrict__ partial,
                                                      float* __restrict__ dW, float* __restrict__ db) {
  __shared__ float sh[256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long e = blockIdx.x * 64L + lane, pitch = len + 32;
  float s = 0.f;
  if (e < (db ? pitch : len)) {
    const float* p = partial + e;
#pragma unroll 8
    for (int b = wave; b < nb; b += 4) s += p[b * pitch];
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  if (wave == 0) {
    s = (sh[lane] + sh[64 + lane]) + (sh[128 + lane] + sh[192 + lane]);
    if (e < len) dW[e] = s;
    else if (db && e - len < cout) db[e - len] = s;
  }
}

// g = 2 (y - t) / count ; partial[block] = sum (y - t)^2 over the block
__global__ __launch_bounds__(256) void k_mse(long n, const float* __restrict__ y, const float* __restrict__ t,
                                             float inv_count, float* __restrict__ g, float* __restrict__ partial) {
  __shared__ float sh[256];
  const long e = blockIdx.x * 256L + threadIdx.x;
  float d = 0.f;
  if (e < n) {
    d = y[e] - t[e];
    g[e] = 2.f * d * inv_count;
  }
  sh[threadIdx.x] = d * d;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = sh[0];
}

// gradient through ReLU given the layer's (post-ReLU) output act: g *= (act > 0);
// writes FP32 (bias gradient) and BF16 (GEMM operand) copies
__global__ __launch_bounds__(256) void k_relu_bwd(long n, const float* __restrict__ gin, const uint16_t* __restrict__ act,
                                                  int relu, float* __restrict__ g32, uint16_t* __restrict__ g16) {
  const long e = blockIdx.x * 256L + threadIdx.x;
  if (e >= n) return;
  float v = gin[e];
  if (relu && !(bf2f(act[e]) > 0.f)) v = 0.f;
  g32[e] = v;
  g16[e] = f2bf(v);
}

// FP32 master W [kpad][npad] (padded MFMA layout, zero padding) -> BF16 forward
// copy Wf [kpad][npad] and the backward-data copy Wt [kpad_t][npad_t] with
// Wt[tap' * cout + co][ci] = W[(taps-1-tap') * cin + ci][co] (flipped taps,
// transposed channels).
__global__ __launch_bounds__(256) void k_pack(int taps, int cin, int cout, int kpad, int npad, int kpad_t, int npad_t,
                                              const float* __restrict__ W, uint16_t* __restrict__ Wf,
                                              uint16_t* __restrict__ Wt) {
  const long e = blockIdx.x * 256L + threadIdx.x;
  if (e < (long)kpad * npad) {
    const int k = (int)(e / npad), co = (int)(e % npad);
    Wf[e] = (k < taps * cin && co < cout) ? f2bf(W[e]) : (uint16_t)0;
  }
  if (Wt && e < (long)kpad_t * npad_t) {
    const int k = (int)(e / npad_t), ci = (int)(e % npad_t);
    uint16_t v = 0;
    if (k < taps * cout && ci < cin) {
      const int tp = k / cout, co = k - tp * cout;
      v = f2bf(W[(long)((taps - 1 - tp) * cin + ci) * npad + co]);
    }
    Wt[e] = v;
  }
}

__global__ __launch_bounds__(256) void k_adam(long n, float* __restrict__ w, const float* __restrict__ g,
                                              float* __restrict__ m, float* __restrict__ v, float lr, float b1,
                                              float b2, float eps, float c1, float c2) {
  const long e = blockIdx.x * 256L + threadIdx.x;
  if (e >= n) return;
  const float gi = g[e];
  const float mi = b1 * m[e] + (1.f - b1) * gi;
  const float vi = b2 * v[e] + (1.f - b2) * gi * gi;
  m[e] = mi;
  v[e] = vi;
  w[e] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

__global__ __launch_bounds__(256) void k_to_bf16(long n, const float* __restrict__ x, float scale,
                                                 uint16_t* __restrict__ y) {
  const long e = blockIdx.x * 256L + threadIdx.x;
  if (e < n) y[e] = f2bf(x[e] * scale);
}

int check_layer(int dim, int cin, int cout, int kpad, int npad) {
  const int taps = dim == 3 ? 27 : 9;
  if (dim != 2 && dim != 3) return tf::fail("conv: dim must be 2 or 3");
  if (cin < 1 || cout < 1 || cout > 32) return tf::fail("conv: 1 <= cout <= 32 required");
  if (kpad % 16 || npad % 16 || kpad < taps * cin || npad < cout || npad > 32) return tf::fail("conv: bad padding");
  if ((long)kpad * npad > CONV_LDS) return tf::fail("conv: weights exceed the LDS stage");
  return 0;
}

}  // namespace

extern "C" {

// Forward of one layer.  in: BF16 [ncell][cin]; W: BF16 [kpad][npad]; bias FP32
// (may be null); out32 / out16 optional FP32 / BF16 [ncell][cout].
int tf_conv_fwd(int nx, int ny, int nz, int dim, int cin, int cout, int kpad, int npad, const void* in,
                const void* W, const float* bias, int relu, float* out32, void* out16, void* stream) {
  if (int e = check_layer(dim, cin, cout, kpad, npad)) return e;
  const long ncell = (long)nx * ny * nz;
  Grid3 g{nx, ny, nz, dim};
  hipStream_t st = (hipStream_t)stream;
  const uint16_t* in16 = (const uint16_t*)in;
  const uint16_t* W16 = (const uint16_t*)W;
  size_t lds = (sizeof(TapRow) + sizeof(uint16_t) * npad) * (size_t)kpad;
  if (cin % 4 == 0 && ((uintptr_t)in % 8) == 0 && ((uintptr_t)W % 4) == 0) {
    const int mt = conv_tiles(ncell);
    const dim3 grid((unsigned)((ncell + 128 * mt - 1) / (128 * mt)));
    lds = sizeof(uint16_t) * (size_t)(kpad + WPAD) * npad;
    auto go = [&](auto nt, auto tiles, auto c32) {
      hipLaunchKernelGGL((k_conv_fwd_v<decltype(nt)::value, decltype(tiles)::value, decltype(c32)::value>), grid,
                         dim3(512), lds, st, g, ncell, cin, cout, kpad, npad, in16, W16, bias, relu, out32,
                         (uint16_t*)out16);
    };
    auto with_tiles = [&](auto nt, auto c32) {
      if (mt == 1) go(nt, std::integral_constant<int, 1>(), c32);
      else go(nt, std::integral_constant<int, 4>(), c32);
    };
    auto with_channels = [&](auto nt) {
      if (cin == 32) with_tiles(nt, std::true_type());
      else with_tiles(nt, std::false_type());
    };
    if (npad == 16) with_channels(std::integral_constant<int, 1>());
    else with_channels(std::integral_constant<int, 2>());
  } else {
    TF_HIP(hipFuncSetAttribute((const void*)k_conv_fwd, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(k_conv_fwd, dim3((unsigned)((ncell + 63) / 64)), dim3(256), lds, st, g, ncell, cin, cout, kpad,
                       npad, in16, W16, bias, relu, out32, (uint16_t*)out16);
  }
  TF_PROF_WORK(tf::PROF_CONV, 2.0 * ncell * (dim == 3 ? 27 : 9) * cin * cout);
  TF_LAUNCH_CHECK("k_conv_fwd");
  return 0;
}

int tf_conv_wgrad_work_size(long ncell, int kpad, int npad) {
  const long n = wgrad_blocks(ncell) * ((long)kpad * npad + 32);
  return n > 2147483647L ? -1 : (int)n;
}

// dW [kpad][npad] FP32 = sum over cells of patch(in)^T gout; db[cout] = sum of g32 (db
// may be null: g32 is then not read).
// in: BF16 [ncell][cin]; gout16 / g32: BF16 / FP32 [ncell][cout]; work: FP32 of
// tf_conv_wgrad_work_size() elements.
int tf_conv_wgrad(int nx, int ny, int nz, int dim, int cin, int cout, int kpad, int npad, const void* in,
                  const void* gout16, const float* g32, float* work, float* dW, float* db, void* stream) {
  if (int e = check_layer(dim, cin, cout, kpad, npad)) return e;
  const long ncell = (long)nx * ny * nz;
  if (kpad > WG_KMAX || ncell >= (1L << 31)) return tf::fail("conv wgrad: K or the grid too large");
  if (nx < 1 || ny < 1 || nz < 1) return tf::fail("conv wgrad: empty grid");
  const long blocks = wgrad_blocks(ncell);
  const int chunk = (int)wgrad_chunk(ncell);
  hipStream_t st = (hipStream_t)stream;
  Grid3 g{nx, ny, nz, dim};
  const dim3 wg_grid((unsigned)blocks), wg_block(64 * WG_WAVES);
  const size_t lds = wgrad_lds(kpad, npad) < sizeof(float) * 64 * WG_WAVES ? sizeof(float) * 64 * WG_WAVES
                                                                         : wgrad_lds(kpad, npad);
  const uint16_t* in16 = (const uint16_t*)in;
  const uint16_t* g16 = (const uint16_t*)gout16;
  auto go = [&](auto vec) {
    constexpr int VEC = decltype(vec)::value;
    TF_HIP(hipFuncSetAttribute((const void*)k_conv_wgrad<VEC>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(k_conv_wgrad<VEC>, wg_grid, wg_block, lds, st, g, ncell, chunk, cin, cout, kpad, npad, in16,
                       g16, db ? g32 : nullptr, work);
    return 0;
  };
  int rc;
  if (cin % 8 == 0 && ((uintptr_t)in % 16) == 0) rc = go(std::integral_constant<int, 8>());
  else if (cin % 4 == 0 && ((uintptr_t)in % 8) == 0) rc = go(std::integral_constant<int, 4>());
  else rc = go(std::integral_constant<int, 1>());
  if (rc) return rc;
  const long len = (long)kpad * npad;
  hipLaunchKernelGGL(k_sum_partials, dim3((unsigned)((len + 32 + 63) / 64)), dim3(256), 0, st, (int)blocks, len, cout,
                     work, dW, db);
  TF_PROF_WORK(tf::PROF_CONV, 2.0 * ncell * (dim == 3 ? 27 : 9) * cin * cout);
  TF_LAUNCH_CHECK("conv wgrad");
  return 0;
}

// Loss work: partial sums per 256 elements -> loss_partial[(n+255)/256].
int tf_mse_grad(long n, const float* y, const float* t, float* g, float* loss_partial, void* stream) {
  hipLaunchKernelGGL(k_mse, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, n, y, t,
                     1.f / (float)n, g, loss_partial);
  TF_LAUNCH_CHECK("k_mse");
  return 0;
}

int tf_relu_bwd(long n, const float* gin, const void* act16, int relu, float* g32, void* g16, void* stream) {
  hipLaunchKernelGGL(k_relu_bwd, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, n, gin,
                     (const uint16_t*)act16, relu, g32, (uint16_t*)g16);
  TF_LAUNCH_CHECK("k_relu_bwd");
  return 0;
}

int tf_conv_pack(int dim, int cin, int cout, int kpad, int npad, int kpad_t, int npad_t, const float* W, void* Wf,
                 void* Wt, void* stream) {
  const int taps = dim == 3 ? 27 : 9;
  const long n = (long)kpad * npad > (long)kpad_t * npad_t ? (long)kpad * npad : (long)kpad_t * npad_t;
  hipLaunchKernelGGL(k_pack, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, taps, cin, cout,
                     kpad, npad, kpad_t, npad_t, W, (uint16_t*)Wf, (uint16_t*)Wt);
  TF_LAUNCH_CHECK("k_pack");
  return 0;
}

int tf_adam(long n, float* w, const float* g, float* m, float* v, float lr, float b1, float b2, float eps, int step,
            void* stream) {
  const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
  hipLaunchKernelGGL(k_adam, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, n, w, g, m, v, lr,
                     b1, b2, eps, c1, c2);
  TF_LAUNCH_CHECK("k_adam");
  return 0;
}

int tf_to_bf16(long n, const float* x, float scale, void* y, void* stream) {
  hipLaunchKernelGGL(k_to_bf16, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, n, x, scale,
                     (uint16_t*)y);
  TF_LAUNCH_CHECK("k_to_bf16");
  return 0;
}

}  // extern "C"
