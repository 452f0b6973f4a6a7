// FP64 hidden-layer products of the coefficient MLP for widths that are not whole 128 x 128 tiles, and
// its weight gradients up to h = 128.
//
// Layers: the weights of 64 output features stay in LDS as MFMA fragments while every wave streams rows
// of its own, 16 at a time: no barrier after the first, and each row is read once per 64 features.  The
// products are taken transposed (features are the rows of the MFMA), so that a lane holds four
// consecutive features of one row and reads and writes 32-byte pieces.
// Weight gradient: a block has a 64 x 64 tile of H^T G over its split of the rows, its four waves every
// fourth group of four rows, straight from memory: lane l holds features 4 l .. 4 l + 3 of a row, so
// that block J of an operand is the features 4 l + J.
//
// 73k rows, against guarded 128 x 128 and 64 x 64 tiles with scalar loads: h = 64 132 -> 34 us a layer
// (its bytes take 15, its products 8) and 132 -> 29 us a weight gradient; h = 96 177 -> 67 and 52,
// h = 192 488 -> 140 and 141, h = 240 601 -> 204 and 182.  The weight gradient of h = 128 takes 54 us
// here and 95 on a 128 x 128 tile, whose 128 splits leave half the CUs.
#pragma once
#include "gdx_common.h"
#include "gdx_gemm.h"

namespace gdx {

typedef double d2n __attribute__((ext_vector_type(2)));
constexpr int GN_F = 64;   // output features a block

// C (M x h) = A (M x h) . W (TB: W^T), EPI as in gdx_gemm.h; grid (persistent, ceil(h / 64)).
// KMAX: the width rounded up to 64, 128 or 256; WAVES a block.
template <int KMAX, int WAVES, bool TB, int EPI>
__global__ __launch_bounds__(64 * WAVES) void gemm_narrow_kernel(int M, int h, const double* __restrict__ A,
                                                                 const double* __restrict__ W, double* __restrict__ C,
                                                                 const double* __restrict__ bias,
                                                                 const double* __restrict__ Y) {
  __shared__ d2n Ws[4 * (KMAX / 8) * 64];   // [block][k pair step][lane]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, r = lane & 15, n0 = blockIdx.y * GN_F, ks = h / 8;
  // lane l of a block: feature 4 (l % 4) + (l % 16) / 4 (row 4 q + g of the result is then 4 g + q)
  for (int i = tid; i < 4 * ks * 64; i += 64 * WAVES) {
    const int l = i & 15, k = i / 64 % ks * 8 + 2 * ((i & 63) >> 4), J = i / 64 / ks;
    const int n = n0 + J * 16 + 4 * (l & 3) + (l >> 2);
    d2n w = {0.0, 0.0};
    if (n < h) {
      w[0] = TB ? W[(size_t)n * h + k] : W[(size_t)k * h + n];
      w[1] = TB ? W[(size_t)n * h + k + 1] : W[(size_t)(k + 1) * h + n];
    }
    Ws[(J * (KMAX / 8) + i / 64 % ks) * 64 + (i & 63)] = w;
  }
  __syncthreads();
  const int tiles = M / 16, step = gridDim.x * WAVES, nj = min(4, (h - n0) / 16), nc = (h + 63) / 64;
  int t = blockIdx.x * WAVES + wave;
  d2n x[8], nx[8];
  auto load = [&](int tile, int c) {   // 64 k of the tile's rows; past the row: the last pair (not used)
    const double* row = A + ((size_t)tile * 16 + r) * h;
#pragma unroll
    for (int s = 0; s < 8; ++s) nx[s] = *(const d2n*)(row + min(c * 64 + 8 * s + 2 * g, h - 2));
  };
  if (t < tiles) load(t, 0);
  for (; t < tiles; t += step) {
    d4 acc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = (d4){0, 0, 0, 0};
    for (int c = 0; c < nc; ++c) {
#pragma unroll
      for (int s = 0; s < 8; ++s) x[s] = nx[s];
      const bool last = c + 1 == nc;
      if (!last || t + step < tiles) load(last ? t + step : t, last ? 0 : c + 1);
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        const int sk = c * 8 + s;
        if (sk >= ks) break;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (j >= nj) break;
          const d2n w = Ws[(j * (KMAX / 8) + sk) * 64 + lane];
          acc[j] = MfmaT<double>::op(w[0], x[s][0], acc[j]);
          acc[j] = MfmaT<double>::op(w[1], x[s][1], acc[j]);
        }
      }
    }
    const size_t row = ((size_t)t * 16 + r) * h;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j >= nj) break;
      const int n = n0 + j * 16 + 4 * g;
      double v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        v[q] = acc[j][q];
        if (EPI == EPI_BIAS_ELU) v[q] = elu_d(v[q] + bias[n + q]);
        if (EPI == EPI_ELU_BWD) {
          const double y = Y[row + n + q];
          v[q] *= y > 0.0 ? 1.0 : y + 1.0;
        }
      }
      *(d2n*)(C + row + n) = (d2n){v[0], v[1]};
      *(d2n*)(C + row + n + 2) = (d2n){v[2], v[3]};
    }
  }
}

// part[z] (h x h) = H^T G over split z of the rows, colsum[z] the column sums of G; grid (ceil(h / 64),
// ceil(h / 64), splits).  Splits are whole groups of 16 rows.
__global__ __launch_bounds__(256, 2) void wgrad_narrow_kernel(int h, const double* __restrict__ H,
                                                                     const double* __restrict__ G,
                                                                     double* __restrict__ part,
                                                                     double* __restrict__ colsum, int kchunk, int kseg,
                                                                     int sps) {
  __shared__ double red[64][64 + 2];
  __shared__ double csum[64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, l = lane & 15, i0 = blockIdx.x * 64, j0 = blockIdx.y * 64;
  int kbeg, kend;
  split_range(blockIdx.z, kchunk, kseg, sps, kbeg, kend);
  // features past the width repeat the last ones; their products are not written
  const double* hp = H + (size_t)(4 * wave + g) * h + min(i0 + 4 * l, h - 4);
  const double* gp = G + (size_t)(4 * wave + g) * h + min(j0 + 4 * l, h - 4);
  constexpr int DEPTH = 3;   // groups of 16 rows in flight
  d2n a[DEPTH][2], b[DEPTH][2];
  auto load = [&](d2n (&x)[2], d2n (&y)[2], int k) {
    const size_t at = (size_t)min(k, kend - 16) * h;
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      x[v] = *(const d2n*)(hp + at + 2 * v);
      y[v] = *(const d2n*)(gp + at + 2 * v);
    }
  };
  d4 acc[4][4];
  double cs[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = (d4){0, 0, 0, 0};
  if (kbeg < kend) {
#pragma unroll
    for (int p = 0; p < DEPTH; ++p) load(a[p], b[p], kbeg + 16 * p);
    for (int k = kbeg; k < kend; k += 16 * DEPTH) {
#pragma unroll
      for (int p = 0; p < DEPTH; ++p) {
        if (k + 16 * p >= kend) break;
        const d2n xa[2] = {a[p][0], a[p][1]}, xb[2] = {b[p][0], b[p][1]};
        load(a[p], b[p], k + 16 * (p + DEPTH));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          cs[j] += xb[j / 2][j % 2];
#pragma unroll
          for (int i = 0; i < 4; ++i)
            acc[i][j] = MfmaT<double>::op(xa[i / 2][i % 2], xb[j / 2][j % 2], acc[i][j]);
        }
      }
    }
  }
  // the waves' sums, in order
  for (int w = 0; w < 4; ++w) {
    if (wave == w) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            double* at = &red[4 * (4 * q + g) + i][4 * l + j];
            *at = w == 0 ? acc[i][j][q] : *at + acc[i][j][q];
          }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        double c = cs[j];
        c += __shfl_xor(c, 16, 64);
        c += __shfl_xor(c, 32, 64);
        if (g == 0) csum[4 * l + j] = w == 0 ? c : csum[4 * l + j] + c;
      }
    }
    __syncthreads();
  }
  double* out = part + (size_t)blockIdx.z * h * h;
  for (int e = tid; e < 64 * 64; e += 256) {
    const int i = i0 + (e >> 6), j = j0 + (e & 63);
    if (i < h && j < h) out[(size_t)i * h + j] = red[e >> 6][e & 63];
  }
  if (colsum != nullptr && blockIdx.x == 0 && tid < 64 && j0 + tid < h) colsum[(size_t)blockIdx.z * h + j0 + tid] = csum[tid];
}

}  // namespace gdx
