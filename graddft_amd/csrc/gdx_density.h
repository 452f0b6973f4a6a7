// Grid densities (grad_dft/molecule.py:388-502) for one molecule or a batch, FP64 and FP32:
//   X = phi D,  rho = X . phi,  grad_j = X . d_j phi,  L = X . lapl(phi),
//   T = sum_j (d_j phi U) . d_j phi,   U = D folded onto its upper 16 x 16 blocks (D_IJ + D_JI^T for
//   I < J, D_II, zero below): the form of T is symmetric, so 5/8 of the products of four full
//   d_c phi D are enough.  D need not be symmetric.
// Raw sums (rho, gx, gy, gz, T, L) are written; point_fwd applies grad = 2 g, tau = T / 2,
// lapl = 2 T + 2 L.
//
// Blocks of 64 grid points, 16 a wave, all waves on the same column chunk of 64.  The products are
// taken transposed, D's columns the rows of an MFMA: a lane then holds four consecutive columns of one
// point, so that the contraction reads AO values as vectors and keeps six sums.  AO fragments go from
// memory straight into the lanes that multiply them (each wave has its own points), one stage ahead; D
// and U are laid out beforehand as fragments (dens_pack_kernel) and staged through LDS for the four
// waves.  A stage is a panel of each where the derivatives take part, and D alone above the chunk's
// columns, where only phi does.  Both spins of a tile run on one XCD one after the other, so that the
// second finds the planes in L2.
//
// FP32 planes: X is formed in FP64 (AO values widened, D as it is), because rho is a sum that cancels;
// U and the derivatives are split into three bf16 terms (gdx_gemm_split.h).  With X on split products,
// too, the kernel is a third faster, but an MFMA aligns its 32 products to the largest and cuts what is
// below, which biases rho and moves dE/dD of n = 560 by 1e-7 .. 9e-7 (FP32 MFMA 5e-8 .. 4e-7, this way
// 2e-8 .. 3e-8).
// LOW: the FP32 planes come with d = phi - float(phi) in bf16, and rho = X . (float(phi) + 2 d), which
// is phi D phi to first order in d for a symmetric D.  All points of a shell around a nucleus have
// nearly the same core functions, so their rounding does not average out over the grid: without d, E_xc
// of water, alkanes and benzene (6-31G*, def2-SVP, levels 1 and 2, B3LYP and neural) moves by
// -1.7e-8 .. +1.4e-8 of itself, alike for all molecules of a basis and level.  With it 1e-9 remains, from
// phi in the gradients; the derivatives and the Laplacian, rounded too, move it by under 5e-10.
//
// Bound by the MFMA rate at FP64 (n = 190, 144k points, one spin: 1.02 -> 0.67 ms, 53% of it; the rest
// waits for loads with two waves a SIMD) and by load latency at FP32, where every chunk reads the planes
// again (n = 560, 427k points, one spin: 10.1 -> 8.5 ms; n = 102, 135k: 0.211 -> 0.19 ms).
#pragma once
#include "gdx_common.h"
#include "gdx_gemm.h"
#include "gdx_gemm_split.h"

namespace gdx {

struct DensMol {
  const void* ao;      // (5, npts_pad, nP) planes in the element type; LOW: then a bf16 plane phi - float(phi)
  void* pack;          // D and U fragments of the spins, dens_pack_bytes each
  long row0, dm_off;   // first row in the per-point arrays, first element in the density matrices
  int npts_pad, nP, n;
  int blk0, pblk0;     // first block in the density and the packing launch
};

constexpr int DN_PT = 64, DN_CB = 4;   // points a block, 16-wide column blocks a chunk
// k a step, 16-byte units a lane reads of a fragment of D, of U (FP32: three bf16 terms) and of an AO
// plane, and k steps a stage where only phi takes part; FP64 steps of 16 spill
typedef double d2v __attribute__((ext_vector_type(2)));
template <typename T> struct DensT;
template <> struct DensT<float> { static constexpr int KS = 32, ND = 4, NU = 3, NV = 2, STEPS = 1; };
template <> struct DensT<double> { static constexpr int KS = 8, ND = 1, NU = 1, NV = 1, STEPS = 2; };

__host__ __device__ inline int dens_chunks(int nP) { return (nP / 16 + DN_CB - 1) / DN_CB; }
template <typename T>
__host__ __device__ inline int dens_ksteps(int nP) { return (nP + DensT<T>::KS - 1) / DensT<T>::KS; }
// one spin: D as [chunk][k step][column block][unit][lane] of 16 bytes, then U
template <typename T>
__host__ __device__ inline size_t dens_panels(int nP) { return (size_t)dens_chunks(nP) * dens_ksteps<T>(nP); }
template <typename T>
__host__ __device__ inline size_t dens_pack_bytes(int nP) {
  return dens_panels<T>(nP) * DN_CB * (DensT<T>::ND + DensT<T>::NU) * 1024;
}
// threads of the packing: one a lane of every fragment
template <typename T>
inline long dens_pack_threads(int nP, int nspin) {
  return (long)nspin * 2 * dens_chunks(nP) * dens_ksteps<T>(nP) * DN_CB * 64;
}
inline int dens_blocks(int npts_pad, int nspin) { return (npts_pad / DN_PT + 7) / 8 * 8 * nspin; }

template <int DensMol::*FIRST>
__device__ __forceinline__ DensMol dens_find(const DensMol* __restrict__ mols, int nmol, const DensMol& one) {
  if (mols == nullptr) return one;
  int lo = 0, hi = nmol - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (mols[mid].*FIRST <= (int)blockIdx.x) lo = mid; else hi = mid - 1;
  }
  static_assert(sizeof(DensMol) % 4 == 0, "whole dwords");
  union U {
    DensMol m;
    int w[sizeof(DensMol) / 4];
    __device__ U() {}
  } u;
  const int* src = (const int*)&mols[lo];
#pragma unroll
  for (int k = 0; k < (int)(sizeof(DensMol) / 4); ++k) u.w[k] = __builtin_amdgcn_readfirstlane(src[k]);
  return u.m;
}

// Fragments of D (FP64) and U, zero past n.  Lane l of a column block holds k = KS / 4 (l / 16) + e of
// column l % 16 (bf16 terms), or of column 4 (l % 4) + (l % 16) / 4 (FP64: row 4 q + g of its MFMA's
// result is then column 4 g + q, as for bf16).
template <typename T>
__global__ __launch_bounds__(256) void dens_pack_kernel(const DensMol* __restrict__ mols, int nmol, const DensMol one,
                                                        int nspin, const double* __restrict__ rdm1) {
  constexpr int KS = DensT<T>::KS, ND = DensT<T>::ND, NU = DensT<T>::NU, NE = KS / 4;
  const DensMol M = dens_find<&DensMol::pblk0>(mols, nmol, one);
  const int nch = dens_chunks(M.nP), nks = dens_ksteps<T>(M.nP), n = M.n;
  const long i = (long)(blockIdx.x - M.pblk0) * 256 + threadIdx.x;
  const int lane = i & 63;
  long f = i >> 6;   // fragment
  const int j = f % DN_CB, ks = f / DN_CB % nks, m = f / DN_CB / nks % nch;
  const int tu = f / DN_CB / nks / nch;
  const int u = tu & 1, s = tu >> 1;
  if (s >= nspin) return;
  const int l = lane & 15, J = m * DN_CB + j;
  const bool f64 = sizeof(T) == 8 || !u;
  const int c = J * 16 + (f64 ? 4 * (l & 3) + (l >> 2) : l), k0 = ks * KS + (lane >> 4) * NE;
  const double* D = rdm1 + M.dm_off + (size_t)s * n * n;
  double x[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    const int k = k0 + e, I = k >> 4;
    double v = 0.0;
    if (k < n && c < n && !(u && I > J)) {
      v = D[(size_t)k * n + c];
      if (u && I < J) v += D[(size_t)c * n + k];
    }
    x[e] = v;
  }
  const size_t panel = (size_t)m * nks + ks;
  char* out = (char*)M.pack + s * dens_pack_bytes<T>(M.nP) + lane * 16 +
              (u ? dens_panels<T>(M.nP) * DN_CB * ND + (panel * DN_CB + j) * NU : (panel * DN_CB + j) * ND) * 1024;
  if (f64) {
#pragma unroll
    for (int p = 0; p < ND; ++p) *(d2v*)(out + p * 1024) = (d2v){x[2 * p], x[2 * p + 1]};
  } else {
    bf8 t[3];
#pragma unroll
    for (int e = 0; e < NE; ++e) {   // from the FP64 value: the terms hold 24 bits or more of it
      const __bf16 h = (__bf16)(float)x[e];
      const float r1 = (float)(x[e] - (double)(float)h);
      const __bf16 mm = (__bf16)r1;
      t[0][e] = h;
      t[1][e] = mm;
      t[2][e] = (__bf16)(r1 - (float)mm);
    }
#pragma unroll
    for (int p = 0; p < NU; ++p) *(bf8*)(out + p * 1024) = t[p % 3];
  }
}

// operands of one AO fragment (8 floats or 2 doubles a lane), and its product with a fragment of D or U:
// DensA in FP64, DensSplit as three bf16 terms
template <typename T> struct DensA {
  static constexpr int NV = DensT<T>::NV, ND = DensT<T>::ND, VE = 16 / sizeof(T);
  typedef T vec_t __attribute__((ext_vector_type(VE)));
  vec_t x[NV];
  __device__ __forceinline__ void set(const f4 (&raw)[NV]) {
#pragma unroll
    for (int v = 0; v < NV; ++v) x[v] = __builtin_bit_cast(vec_t, raw[v]);
  }
  __device__ __forceinline__ void mul(const f4* b, d4& acc) const {   // b: this lane's units, 64 apart
#pragma unroll
    for (int p = 0; p < ND; ++p) {
      const d2v d = __builtin_bit_cast(d2v, b[p * 64]);
#pragma unroll
      for (int e = 0; e < 2; ++e)
        acc = MfmaT<double>::op(d[e], (double)x[(2 * p + e) / VE][(2 * p + e) % VE], acc);
    }
  }
};
struct DensSplit {
  bf8 t[3];
  __device__ __forceinline__ void set(const f4 (&raw)[2]) {
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = raw[e / 4][e % 4];
    split8(x, t[0], t[1], t[2]);
  }
  __device__ __forceinline__ void mul(const f4 (&b)[3], f4& acc) const {
    bf8 d[3];
#pragma unroll
    for (int p = 0; p < 3; ++p) d[p] = __builtin_bit_cast(bf8, b[p]);
    // summed from zero, so that the running sum rounds once a step
    f4 sum = (f4)0.f;
    mfma_chain(d, t, sum);
    acc += sum;
  }
};
struct DensDouble {
  d2v x;
  __device__ __forceinline__ void set(const f4 (&raw)[1]) { x = __builtin_bit_cast(d2v, raw[0]); }
  __device__ __forceinline__ void mul(const f4 (&b)[1], d4& acc) const {
    const d2v d = __builtin_bit_cast(d2v, b[0]);
    acc = MfmaT<double>::op(d[0], x[0], acc);
    acc = MfmaT<double>::op(d[1], x[1], acc);
  }
};
// Grid: dens_blocks; dens_part rows are DENS_STRIDE doubles, out_rows a spin.
template <typename T, bool LOW>
__global__ __launch_bounds__(256, 2) void density_kernel(const DensMol* __restrict__ mols, int nmol, const DensMol one,
                                                         int nspin, size_t out_rows, double* __restrict__ dens_part) {
  typedef typename MfmaT<T>::acc_t acc_t;
  constexpr int KS = DensT<T>::KS, ND = DensT<T>::ND, NU = DensT<T>::NU, NV = DensT<T>::NV, STEPS = DensT<T>::STEPS;
  constexpr int PD = DN_CB * ND * 64, PU = DN_CB * NU * 64;   // 16-byte units of a panel
  constexpr int CV = sizeof(T) / 4;   // 16-byte vectors of four columns
  constexpr int NB = STEPS == 2 && ND > NU ? 2 * ND : ND + NU;   // units of a stage a thread copies
  __shared__ f4 Bs[2][256 * NB];
  const DensMol M = dens_find<&DensMol::blk0>(mols, nmol, one);
  const int local = blockIdx.x - M.blk0, slot = local >> 3, s = slot % nspin, tile = slot / nspin * 8 + (local & 7);
  if (tile >= M.npts_pad / DN_PT) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, r = lane & 15, nP = M.nP, nb = nP / 16;
  const int nch = dens_chunks(nP), nks = dens_ksteps<T>(nP);
  const size_t plane = (size_t)M.npts_pad * nP;
  const gptr<T> rows = (gptr<T>)M.ao + (size_t)(tile * DN_PT + wave * 16) * nP;   // this wave's 16 points
  static_assert(!LOW || sizeof(T) == 4, "the remainder of phi goes with FP32 planes");
  const gptr<char> lows = (gptr<char>)((gptr<T>)M.ao + 5 * plane) + (size_t)(tile * DN_PT + wave * 16) * nP * 2;
  const gptr<char> pack = (gptr<char>)M.pack + s * dens_pack_bytes<T>(nP);

  f4 ra[4][NV], rb[NB];
  auto load_a = [&](f4 (&x)[NV], int c, int ks) {   // past the row: any finite values, D is zero there
    const unsigned at = (r * nP + min(ks * KS + g * (KS / 4), nP - KS / 4)) * (unsigned)sizeof(T);
#pragma unroll
    for (int v = 0; v < NV; ++v) x[v] = row_load<f4>(rows + c * plane, at + 16 * v);
  };
  auto load_b = [&](int m, int ks, bool deriv) {
    const gptr<char> p0 = pack + ((size_t)m * nks + ks) * (PD * 16);
#pragma unroll
    for (int i = 0; i < ND; ++i) rb[i] = row_load<f4>(p0, tid * 16 + i * 4096);
    if (deriv) {
      const gptr<char> p1 = pack + dens_panels<T>(nP) * (PD * 16) + ((size_t)m * nks + ks) * (PU * 16);
#pragma unroll
      for (int i = 0; i < NU; ++i) rb[ND + i] = row_load<f4>(p1, tid * 16 + i * 4096);
    } else if (STEPS == 2) {
      const gptr<char> p1 = pack + ((size_t)m * nks + min(ks + 1, nks - 1)) * (PD * 16);
#pragma unroll
      for (int i = 0; i < ND; ++i) rb[ND + i] = row_load<f4>(p1, tid * 16 + i * 4096);
    }
  };
  double part[6];
#pragma unroll
  for (int v = 0; v < 6; ++v) part[v] = 0.0;
  int buf = 0;
  load_b(0, 0, true);
#pragma unroll
  for (int c = 0; c < 4; ++c) load_a(ra[c], c, 0);
  for (int m = 0; m < nch; ++m) {
    d4 acc0[DN_CB];
    acc_t acc[3][DN_CB];
#pragma unroll
    for (int j = 0; j < DN_CB; ++j) {
      acc0[j] = (d4){0, 0, 0, 0};
#pragma unroll
      for (int c = 0; c < 3; ++c) acc[c][j] = (acc_t){0, 0, 0, 0};
    }
    const int jn = min(DN_CB, nb - m * DN_CB), nd = min(nks, (m + 1) * DN_CB * 16 / KS);
    for (int ks = 0; ks < nks;) {
      const bool deriv = ks < nd;
      const int next = ks + (deriv ? 1 : STEPS);
      // the stage after this one, whose AO fragments are loaded as this one's have been taken
      const bool wrap = next >= nks, more = !wrap || m + 1 < nch, nderiv = wrap || next < nd;
      const int nk = wrap ? 0 : next;
#pragma unroll
      for (int i = 0; i < NB; ++i) Bs[buf][tid + 256 * i] = rb[i];
      const int j0 = ks * KS / 16 - m * DN_CB;   // U is zero in the column blocks before
      DensA<T> a;
      if constexpr (sizeof(T) == 8) {
        // the four components together, so that a fragment of U is read once
        DensA<T> a2;
        DensDouble b[3];
        auto mul_phi = [&](const DensA<T>& x, int panel) {
#pragma unroll
          for (int j = 0; j < DN_CB; ++j) {
            if (j >= jn) break;
            x.mul(&Bs[buf][panel + j * ND * 64 + lane], acc0[j]);
          }
        };
        a.set(ra[0]);
        if (deriv) {
#pragma unroll
          for (int c = 0; c < 3; ++c) b[c].set(ra[c + 1]);
        } else {
          a2.set(ra[1]);
        }
        __syncthreads();
        if (more) {
          load_b(wrap ? m + 1 : m, nk, nderiv);
          load_a(ra[0], 0, nk);
          if (nderiv) {
#pragma unroll
            for (int c = 1; c < 4; ++c) load_a(ra[c], c, nk);
          } else {
            load_a(ra[1], 0, min(nk + 1, nks - 1));
          }
        }
        if (deriv) {
#pragma unroll
          for (int j = 0; j < DN_CB; ++j) {
            if (j >= jn) break;
            a.mul(&Bs[buf][j * ND * 64 + lane], acc0[j]);
            const f4 u[1] = {Bs[buf][PD + j * NU * 64 + lane]};
            if (j >= j0)
#pragma unroll
              for (int c = 0; c < 3; ++c) b[c].mul(u, acc[c][j]);
          }
        } else {
          mul_phi(a, 0);
          if (ks + 1 < nks) mul_phi(a2, PD);
        }
      } else {
        // one component at a time, the next stage's load issued as it is taken: all four with their
        // splits do not fit beside the accumulators
        __syncthreads();
        if (more) load_b(wrap ? m + 1 : m, nk, nderiv);
        a.set(ra[0]);
        if (deriv) {
          if (more) load_a(ra[0], 0, nk);
#pragma unroll
          for (int j = 0; j < DN_CB; ++j) {
            if (j >= jn) break;
            a.mul(&Bs[buf][j * ND * 64 + lane], acc0[j]);
          }
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            DensSplit b;
            b.set(ra[c + 1]);
            if (more && nderiv) load_a(ra[c + 1], c + 1, nk);
#pragma unroll
            for (int j = 0; j < DN_CB; ++j) {
              if (j >= jn) break;
              if (j < j0) continue;
              f4 u[NU];
#pragma unroll
              for (int i = 0; i < NU; ++i) u[i] = Bs[buf][PD + (j * NU + i) * 64 + lane];
              b.mul(u, acc[c][j]);
            }
          }
        } else {
          if (more) {
            load_a(ra[0], 0, nk);
            if (nderiv) {
#pragma unroll
              for (int c = 1; c < 4; ++c) load_a(ra[c], c, nk);
            }
          }
#pragma unroll
          for (int j = 0; j < DN_CB; ++j) {
            if (j >= jn) break;
            a.mul(&Bs[buf][j * ND * 64 + lane], acc0[j]);
          }
        }
      }
      buf ^= 1;
      ks = next;
    }
    // contraction with the AO values at the chunk's columns, four a lane, one 16-byte vector of each
    // plane at a time and one ahead
    constexpr int VE = 16 / sizeof(T);   // columns a vector
    typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
    f4 rc[5];
    bf4 rl = (bf4)(__bf16)0.f;
    auto cload = [&](int v) {
      const unsigned at = r * nP + (m * DN_CB + v / CV) * 16 + 4 * g + v % CV * VE;
#pragma unroll
      for (int k = 0; k < 5; ++k) rc[k] = row_load<f4>(rows + k * plane, at * (unsigned)sizeof(T));
      if (LOW) rl = row_load<bf4>(lows, at * 2);
    };
    cload(0);
#pragma unroll
    for (int v = 0; v < DN_CB * CV; ++v) {
      const int j = v / CV;
      if (j >= jn) break;
      typedef T vec_t __attribute__((ext_vector_type(VE)));
      vec_t x[5];
#pragma unroll
      for (int k = 0; k < 5; ++k) x[k] = __builtin_bit_cast(vec_t, rc[k]);
      const bf4 xl = rl;
      if (v + 1 < jn * CV) cload(v + 1);
#pragma unroll
      for (int e = 0; e < VE; ++e) {
        const int q = v % CV * VE + e;
        const double x0 = acc0[j][q], gx = x[1][e], gy = x[2][e], gz = x[3][e];
        part[0] += x0 * (LOW ? (double)x[0][e] + 2.0 * (double)(float)xl[e] : (double)x[0][e]);
        part[1] += x0 * gx;
        part[2] += x0 * gy;
        part[3] += x0 * gz;
        part[4] += (double)acc[0][j][q] * gx + (double)acc[1][j][q] * gy + (double)acc[2][j][q] * gz;
        part[5] += x0 * (double)x[4][e];
      }
    }
  }
  double* out = dens_part + ((size_t)s * out_rows + M.row0 + tile * DN_PT + wave * 16 + r) * DENS_STRIDE;
#pragma unroll
  for (int v = 0; v < 6; ++v) {
    double t = part[v];
    t += __shfl_xor(t, 16, 64);
    t += __shfl_xor(t, 32, 64);
    if (g == 0) out[v] = t;
  }
}

}  // namespace gdx
