// Hidden-layer products of the coefficient MLP for FP32 activations on bf16 MFMA
// (v_mfma_f32_16x16x32_bf16, 16 times the FP32 MFMA rate).
//
// Every FP32 value x is split into three bf16 terms
//   h = bf16(x), m = bf16(x - h), l = bf16(x - h - m)      (|x - h - m - l| <~ 2^-27 |x|)
// and a product a.b is formed from the six terms whose order is >= 2^-18 of it:
//   a_h b_h + a_h b_m + a_m b_h + a_h b_l + a_m b_m + a_l b_h,
// accumulated in FP32.  The dropped terms (2^-27) are below FP32's own rounding (2^-24), and an
// MFMA adds 32 products at a time where the FP32 instruction adds four, so the sums round less often,
// though not to nearest (mfma_split): dE/dtheta of the 3 x 256 network on benzene is 6e-8 from FP64 (FP32
// MFMA 2.5e-7), dE/dD 4.2e-8 (3.9e-8: the rounding of D); total energies of 32 batches of alkanes, all
// widths, are 4e-10 (rms, at most 1e-9) from FP64, half of them up and half down, where FP32 MFMA in the
// layers and the densities left 8e-9.  A two-term split with three products is not enough (E_xc moves by
// 5e-6 Ha).
//
// The weights are split from their FP64 masters once per evaluation (pack_weights_kernel), in the
// order a wave reads them as MFMA operands, and stay in L2; activations are split once per block
// while they are staged into LDS, as fragments of 8 consecutive k so that a lane's operand is one
// 16-byte read.  Blocks cover all h output features, so no activation is split twice.
//
// 135k rows, h = 256, against 128 x 128 FP32 MFMA tiles: forward 177 -> 139 us (124 without the leading
// product's own sum), backward 190 -> 135, weight gradient 162 -> 117 (the bytes take 53 us, 80 with the ELU outputs, the six products 47 at
// the MFMA rate): two waves a SIMD do not hide all of the LDS and L2 latency between barriers.
#pragma once
#include "gdx_common.h"
#include "gdx_gemm.h"

namespace gdx {

typedef float f2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));

// three-term split of 8 consecutive values
__device__ __forceinline__ void split8(const float* x, bf8& h, bf8& m, bf8& l) {
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    const f2v v = {x[e], x[e + 1]};
    const bf2 hv = __builtin_convertvector(v, bf2);
    const f2v r1 = v - __builtin_convertvector(hv, f2v);
    const bf2 mv = __builtin_convertvector(r1, bf2);
    const f2v r2 = r1 - __builtin_convertvector(mv, f2v);
    const bf2 lv = __builtin_convertvector(r2, bf2);
    h[e] = hv[0]; h[e + 1] = hv[1];
    m[e] = mv[0]; m[e + 1] = mv[1];
    l[e] = lv[0]; l[e + 1] = lv[1];
  }
}

// acc[i] += the six products of 16 x 16 x 32 steps a . b[i] for NI blocks.  A block's products are
// summed from zero and added to the running sum once: every MFMA rounds its whole accumulator, so a
// chain of all six through acc would round it six times a step, as often as FP32 MFMAs do.  The blocks'
// chains are interleaved (an MFMA waits for the previous one of its chain).
// LEAD: the leading product has a sum of its own.  An MFMA aligns its addends to the largest and cuts
// towards minus infinity what is below: for normally distributed factors -0.19 x 2^-24 of the largest
// product on average where the leading product joins the chain of the small ones, 0.004 where it does
// not.  In the layers of the energy that is a shift of every unit alike at all points, which moves E_xc
// by 5e-9 of itself; gradients, rounded to 4e-8 anyway, are spared its registers (3% of a benzene
// 6-31G* step).
template <int NI, bool LEAD>
__device__ __forceinline__ void mfma_split(const bf8 (&a)[3], const bf8 (&b)[NI][3], f4 (&acc)[NI]) {
  constexpr int PA[6] = {2, 1, 0, 1, 0, 0}, PB[6] = {0, 1, 2, 0, 1, 0};
  f4 t[NI], lead[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) t[i] = (f4)0.f;
#pragma unroll
  for (int p = 0; p < (LEAD ? 5 : 6); ++p)
#pragma unroll
    for (int i = 0; i < NI; ++i) t[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[PA[p]], b[i][PB[p]], t[i], 0, 0, 0);
  if (LEAD) {
#pragma unroll
    for (int i = 0; i < NI; ++i) lead[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[i][0], (f4)0.f, 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < NI; ++i) acc[i] += LEAD ? lead[i] + t[i] : t[i];
}

// the same chain of one block through c (which FP64 accumulators then take)
__device__ __forceinline__ void mfma_chain(const bf8 (&a)[3], const bf8 (&b)[3], f4& c) {
  constexpr int PA[6] = {2, 1, 0, 1, 0, 0}, PB[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
  for (int p = 0; p < 6; ++p) c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[PA[p]], b[PB[p]], c, 0, 0, 0);
}

// Packed weights of one hidden layer and direction: [k step of 32][16-feature block][term][lane][8],
// zero past h; lane l of a block holds feature l % 16, k = 8 (l / 16) + e.
__host__ __device__ inline int split_ksteps(int h) { return (h + 31) / 32; }
inline size_t split_pack_elems(int h) { return (size_t)split_ksteps(h) * (h / 16) * 3 * 64 * 8; }

// All parameters to FP32 (the hidden biases and the rows formed again read that copy), then for each hidden layer
// l = 1 .. nl-1 the packed W_l (forward: feature = output, k = input) and W_l^T (backward) at
// pack + (2 (l - 1) + direction) * split_pack_elems(h).  w1 = offset of W_1, layer stride h h + h.
__global__ void pack_weights_kernel(const double* __restrict__ params, long nparam, float* __restrict__ lowp,
                                    int h, int nhid, long w1, int nk, __bf16* __restrict__ pack) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nparam) {
    lowp[i] = (float)params[i];
    return;
  }
  i -= (nparam + blockDim.x - 1) / blockDim.x * blockDim.x;   // whole blocks for each part
  if (i < 0) return;
  const int nb = h / 16, lane = (int)(i & 63);
  long rest = i >> 6;
  const int b = (int)(rest % nb);
  rest /= nb;
  const int kt = (int)(rest % nk);
  rest /= nk;
  const int dir = (int)(rest & 1), l = (int)(rest >> 1);
  if (l >= nhid) return;
  const double* W = params + w1 + (long)l * ((long)h * h + h);
  const int f = b * 16 + (lane & 15), k0 = kt * 32 + 8 * (lane >> 4);
  bf8 t[3];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int k = k0 + e;
    const double w = k < h ? (dir ? W[(size_t)f * h + k] : W[(size_t)k * h + f]) : 0.0;
    const __bf16 hh = (__bf16)(float)w;
    const double r1 = w - (double)(float)hh;
    const __bf16 mm = (__bf16)(float)r1;
    const __bf16 ll = (__bf16)(float)(r1 - (double)(float)mm);
    t[0][e] = hh; t[1][e] = mm; t[2][e] = ll;
  }
  bf8* out = (bf8*)pack + ((((size_t)l * 2 + dir) * nk + kt) * nb + b) * 3 * 64 + lane;
#pragma unroll
  for (int p = 0; p < 3; ++p) out[(size_t)p * 64] = t[p];
}

// C (M x h) = epi(A (M x h) . W), W packed.  Block = 64 rows x all h features, four waves of
// 64 rows x NB 16-feature blocks (h <= 64 NB).  The MFMA rows are features and its columns grid
// rows, so a lane ends with four consecutive features of one row (16-byte stores, bias and Y
// loads).  Blocks are persistent; A is loaded one k step ahead and split into double-buffered LDS; a weight fragment (L2) is
// loaded for the next step as soon as its registers have been read.
//   EPI_BIAS_ELU    C = ELU(A W + bias)
//   EPI_ELU_BWD     C = (A W) elu'(Y), Y = the ELU output
//   EPI_STORE       C = A W
// An infinity, or a number past bf16's largest (3.39e38), has no split: its terms add up to NaN.  Such a
// result is formed again from the FP32 operands (W at stride wk along k and wf along the features): a
// unit saturated by it, ELU(-inf) = -1 or a coefficient of 0 or 2, is a finite answer.
constexpr int GS_ROWS = 64;

template <int NB, int EPI>
__global__ __launch_bounds__(256, 2) void gemm_split_kernel(int M, int h, const float* __restrict__ A,
                                                            const __bf16* __restrict__ Wp,
                                                            const float* __restrict__ W, int wk, int wf,
                                                            float* __restrict__ C, const float* __restrict__ bias,
                                                            const float* __restrict__ Y) {
  // fragments [k-group][row], rows xored by twice the k-group: four lanes of a row store to different
  // banks, and a wave's reads stay conflict-free
  __shared__ __align__(16) __bf16 As[2][3][4 * GS_ROWS * 8];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, r = lane & 15;
  const int nk = split_ksteps(h), nblk = h / 16;
  const int ntile = (M + GS_ROWS - 1) / GS_ROWS;
  const int jb0 = wave * NB, njv = max(0, min(NB, nblk - jb0));   // feature blocks of this wave
  // staging: row tid / 4 of the tile, k-group tid % 4 (a row's 32 k are one 128-byte line)
  // (no branch around a load anywhere in the loop: the compiler counts outstanding loads, and behind
  // a branch it waits for all of them, the weight fragments just requested among them)
  const int srow = tid >> 2, skg = tid & 3;
  f4 ra[2];
  auto gload = [&](int tile, int kt) {
    const int k = kt * 32 + 8 * skg;
    const float* p = A + (size_t)min(tile * GS_ROWS + srow, M - 1) * h + min(k, h - 8);
    ra[0] = *(const f4*)p;
    ra[1] = *(const f4*)(p + 4);
    if (k >= h) ra[0] = ra[1] = (f4)0.f;
  };
  auto lstore = [&](int buf) {
    const float x[8] = {ra[0][0], ra[0][1], ra[0][2], ra[0][3], ra[1][0], ra[1][1], ra[1][2], ra[1][3]};
    bf8 t[3];
    split8(x, t[0], t[1], t[2]);
#pragma unroll
    for (int p = 0; p < 3; ++p) *(bf8*)&As[buf][p][(skg * GS_ROWS + (srow ^ (2 * skg))) * 8] = t[p];
  };
  // (feature blocks past the last one repeat it; their results are not stored)
  const bf8* wp = (const bf8*)Wp + lane;
  auto wload = [&](int kt, int j, bf8 (&w)[3]) {
    const bf8* q = wp + ((size_t)kt * nblk + min(jb0 + j, nblk - 1)) * 3 * 64;
#pragma unroll
    for (int p = 0; p < 3; ++p) w[p] = q[p * 64];
  };
  bf8 w[NB][3];
#pragma unroll
  for (int j = 0; j < NB; ++j) wload(0, j, w[j]);
  gload(blockIdx.x, 0);
  lstore(0);
  __syncthreads();
  int cur = 0;
  for (int tile = blockIdx.x; tile < ntile; tile += gridDim.x) {
    const int m0 = tile * GS_ROWS;
    f4 acc[NB][4];
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[j][i] = (f4)0.f;
    for (int kt = 0; kt < nk; ++kt) {
      const int nxt = kt + 1 < nk ? kt + 1 : 0;   // past the tile: the first step of the block's next one
      gload(kt + 1 < nk ? tile : tile + (int)gridDim.x, nxt);
      bf8 hb[4][3];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int p = 0; p < 3; ++p) hb[i][p] = *(const bf8*)&As[cur][p][(g * GS_ROWS + i * 16 + (r ^ (2 * g))) * 8];
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        mfma_split<4, EPI == EPI_BIAS_ELU>(w[j], hb, acc[j]);
        wload(nxt, j, w[j]);   // the next step's fragments, into the registers just read
      }
      cur ^= 1;
      lstore(cur);
      __syncthreads();
    }
    f4 any = (f4)0.f;
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) any += acc[j][i];
    const float nan = (any[0] + any[1]) + (any[2] + any[3]);
    if (__any(nan != nan)) {
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            if (j >= njv || acc[j][i][q] == acc[j][i][q]) continue;
            const float* a = A + (size_t)min(m0 + i * 16 + r, M - 1) * h;
            const float* w = W + (size_t)((jb0 + j) * 16 + 4 * g + q) * wf;
            float s = 0.f;
#pragma unroll 1
            for (int k = 0; k < h; ++k) s = fmaf(a[k], w[(size_t)k * wk], s);
            acc[j][i][q] = s;
          }
    }
    // epilogue: feature f .. f + 3 of row m0 + 16 i + r
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      if (j >= njv) break;
      const int f = (jb0 + j) * 16 + 4 * g;
      f4 b4 = (f4)0.f;
      if (EPI == EPI_BIAS_ELU) b4 = *(const f4*)(bias + f);
      f4 y[4];
      if constexpr (EPI == EPI_ELU_BWD)
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] = *(const f4*)(Y + (size_t)min(m0 + i * 16 + r, M - 1) * h + f);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = m0 + i * 16 + r;
        f4 v = acc[j][i];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (EPI == EPI_BIAS_ELU) v[q] = elu_f(v[q] + b4[q]);
          if constexpr (EPI == EPI_ELU_BWD) v[q] *= (y[i][q] > 0.f ? 1.f : y[i][q] + 1.f);
        }
        if (row < M) {
          *(f4*)(C + (size_t)row * h + f) = v;
        }
      }
    }
  }
}

// Weight gradient of a hidden layer: part[split] (h x h) = sum over the split's rows r of
// Hin[r][i] G[r][f], colsum[split][f] = sum_r G[r][f].  Block = 128 inputs i x 32 NBF features f of
// one split, four waves of 64 x 16 NBF; a stage is 32 rows.  A staging thread reads 8 consecutive
// rows of one feature (coalesced across the lanes) -- the 8 k of a fragment -- so nothing is
// transposed.  Tiles of 128 x 128 (193 VGPRs, two blocks a CU, one's staging under the other's
// MFMAs) split each operand twice at h = 256; a 128 x 256 tile splits G once but spills.  The tiles
// of one split are placed on one XCD, whose L2 serves the second read.
constexpr int WG_I = 128, WG_K = 32;

template <int NBF>
__global__ __launch_bounds__(256, 2) void wgrad_split_kernel(int h, const float* __restrict__ Hin,
                                                             const float* __restrict__ G, float* __restrict__ part,
                                                             float* __restrict__ colsum, int kchunk, int kseg,
                                                             int sps) {
  static_assert(NBF % 2 == 0, "whole staging tasks a thread");
  constexpr int FT = 32 * NBF, NTB = FT * 4 / 256;
  __shared__ __align__(16) __bf16 As[3][4][WG_I * 8];
  __shared__ __align__(16) __bf16 Bs[3][4][FT * 8];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, r = lane & 15;
  int bx, ysplit;
  xcd_tile_split(gridDim.x, bx, ysplit);
  const int nft = (h + FT - 1) / FT;
  const int i0 = bx / nft * WG_I, f0 = bx % nft * FT;
  int kbeg, kend;
  split_range(ysplit, kchunk, kseg, sps, kbeg, kend);
  const int nst = (kend - kbeg) / WG_K;
  const int wi = (wave >> 1) * 64, wf = (wave & 1) * 16 * NBF;
  const int niv = max(0, min(4, (h - i0 - wi) / 16)), njv = max(0, min(NBF, (h - f0 - wf) / 16));
  float xa[2][8], xb[NTB][8];
  float cs[NTB];
#pragma unroll
  for (int u = 0; u < NTB; ++u) cs[u] = 0.f;
  auto gload = [&](int k0) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int t = tid + 256 * u, f = i0 + (t & (WG_I - 1)), kg = t / WG_I;
      const bool ok = f < h;
      const float* p = Hin + (size_t)(k0 + 8 * kg) * h + f;
#pragma unroll
      for (int e = 0; e < 8; ++e) xa[u][e] = ok ? p[(size_t)e * h] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < NTB; ++u) {
      const int t = tid + 256 * u, f = f0 + t % FT, kg = t / FT;
      const bool ok = f < h;
      const float* p = G + (size_t)(k0 + 8 * kg) * h + f;
#pragma unroll
      for (int e = 0; e < 8; ++e) xb[u][e] = ok ? p[(size_t)e * h] : 0.f;
    }
  };
  auto lstore = [&]() {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int t = tid + 256 * u, f = t & (WG_I - 1), kg = t / WG_I;
      bf8 s[3];
      split8(xa[u], s[0], s[1], s[2]);
#pragma unroll
      for (int p = 0; p < 3; ++p) *(bf8*)&As[p][kg][f * 8] = s[p];
    }
#pragma unroll
    for (int u = 0; u < NTB; ++u) {
      const int t = tid + 256 * u, f = t % FT, kg = t / FT;
      bf8 s[3];
      split8(xb[u], s[0], s[1], s[2]);
#pragma unroll
      for (int p = 0; p < 3; ++p) *(bf8*)&Bs[p][kg][f * 8] = s[p];
#pragma unroll
      for (int e = 0; e < 8; ++e) cs[u] += xb[u][e];
    }
  };
  f4 acc[NBF][4];
#pragma unroll
  for (int j = 0; j < NBF; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[j][i] = (f4)0.f;
  if (nst > 0) gload(kbeg);
  for (int st = 0; st < nst; ++st) {
    lstore();
    __syncthreads();
    if (st + 1 < nst) gload(kbeg + (st + 1) * WG_K);
    bf8 ha[4][3];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int p = 0; p < 3; ++p) ha[i][p] = *(const bf8*)&As[p][g][(wi + i * 16 + r) * 8];
#pragma unroll
    for (int j = 0; j < NBF; ++j) {
      if (j < njv) {
        bf8 gb[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) gb[p] = *(const bf8*)&Bs[p][g][(wf + j * 16 + r) * 8];
        // MFMA rows: features f; columns: inputs i (blocks past h only multiply zeros)
        if (niv > 0) mfma_split<4, false>(gb, ha, acc[j]);
      }
    }
    __syncthreads();
  }
  float* out = part + (size_t)ysplit * h * h;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < NBF; ++j)
      if (i < niv && j < njv)
        *(f4*)(out + (size_t)(i0 + wi + i * 16 + r) * h + f0 + wf + j * 16 + 4 * g) = acc[j][i];
  if (colsum != nullptr && i0 == 0) {
    // thread t summed its features over k-group kg of every stage: add the four k-groups
    float (*red)[FT] = (float (*)[FT])&Bs[0][0][0];
#pragma unroll
    for (int u = 0; u < NTB; ++u) {
      const int t = tid + 256 * u;
      red[t / FT][t % FT] = cs[u];
    }
    __syncthreads();
    if (tid < FT && f0 + tid < h)
      colsum[(size_t)ysplit * h + f0 + tid] = (red[0][tid] + red[1][tid]) + (red[2][tid] + red[3][tid]);
  }
}

}  // namespace gdx
