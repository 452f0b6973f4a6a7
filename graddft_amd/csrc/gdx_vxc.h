// The V_xc build, adjoint of the density kernel (grad_dft/train.py:86-121), for one molecule or a
// batch of them, FP64 and FP32:
//   V_s = phi^T Z_s + sum_j d_j phi^T (u_s d_j phi),   Z = v_rho phi + sum_j 2 v_grad_j d_j phi +
//   2 v_lapl lapl(phi),   u = v_tau / 2 + 2 v_lapl,
// a contraction over grid points (8 n^2 flop a point and spin), bound by the MFMA rate.
//
// The second term is symmetric: it is formed for the 16 x 16 blocks on and above the diagonal only
// and mirrored when the partial sums are added, so the build needs 5/8 of the products.
// Output tiles are 16 tb wide with tb <= 4: tiles of 128 were slower or level on every shape from n = 7
// to 560 (half the waves), and FP64 would not hold its accumulators.  Work items come in classes (below),
// whose point chunks are sized so that the items cost the same, and all items of one chunk run on one
// XCD (blocks L, L + 8, ... share it), whose L2 then serves the chunk's AO rows to every tile and both
// spins: tiles spread over the XCDs re-read them from HBM (n = 192, 9 tiles: 11 TB/s of cache traffic).
// Four waves take quadrants of at most 2 x 2 blocks, rotated with the block index so that the smaller
// quadrants of odd tiles and the empty one of a diagonal tile fall on every SIMD alike.
//
// Measured with the reduction, before (one tile an item, every tile forming its own operands, FP32 on
// the FP32 MFMA, full symmetric products) and now:
//   FP32, both spins: n = 560, 427k points 31.2 -> 13.0 ms; n = 102, 135k 0.38 -> 0.34 ms; a batch of
//   n = 28 .. 210, 820k 6.1 -> 3.2 ms
//   FP64: n = 190, 144k points, one spin 0.93 -> 0.65 ms (57% of the MFMA rate busy: stages wait for
//   their loads); n = 114, 44k, one spin 0.155 -> 0.128 ms; n = 82, 73k, both spins level at 0.29 ms
#pragma once
#include "gdx_common.h"
#include "gdx_gemm.h"
#include "gdx_gemm_split.h"

namespace gdx {

struct VxcMol {
  const void* ao;      // (5, npts_pad, nP) planes in the element type
  float* z;            // FP32: (nsv, slab, nP) Z of the current slab
  double* part;        // partial sums, (slots, nsv, nP, nP): see vxc_reduce_kernel
  long row0;           // first row of this molecule in every spin plane of the potentials
  long out_off;        // first element of its (2, n, n) output
  int npts_pad, nP, n;
  int slab;            // points a launch (FP32; a multiple of 64), all of them in FP64
  int tb, nf, rem;     // 16-wide blocks a tile, full tiles an edge, blocks of the last, ragged one
  int ch[4], nch[4];   // points per chunk and chunks a slab of the item classes
  int blk0, zblk0, rblk0;   // first block in the product, Z and reduction launches
};

// Item classes.  FP32: 0 general (one product phi^T Z, every tile), 1 symmetric (three products, tile
// row <= tile column).  FP64: tile pairs I < J (both general products and the symmetric one, five in
// all), 0 full and 1 with the ragged last tile, and diagonal tiles, 2 full and 3 the ragged one.
template <typename T>
__host__ __device__ inline int vxc_tiles(const VxcMol& M, int cls) {
  const int nt = M.nf + (M.rem != 0);
  if (sizeof(T) == 4) return cls == 0 ? nt * nt : cls == 1 ? nt * (nt + 1) / 2 : 0;
  const int ragged = M.rem != 0;
  return cls == 0 ? M.nf * (M.nf - 1) / 2 : cls == 1 ? M.nf * ragged : cls == 2 ? M.nf : ragged;
}
// cost of one item of a class a point: FP32 stages; FP64 products of the wave that has most, with two
// for staging a tile
template <typename T>
inline double vxc_cost(const VxcMol& M, int cls) {
  if (sizeof(T) == 4) return cls == 0 ? 1.0 : 3.0;
  const int hi = (M.tb + 1) / 2, hj = cls & 1 ? (M.rem + 1) / 2 : hi;
  return cls < 2 ? 4.0 + 5 * hi * hj : 2.0 + hj * hj + 3 * hj * (hj + 1) / 2;
}
template <typename T>
inline int vxc_blocks(const VxcMol& M, int nsv) {
  int b = 0;
  for (int c = 0; c < 4; ++c) b += (M.nch[c] + 7) / 8 * vxc_tiles<T>(M, c) * nsv;
  return 8 * b;
}
// partial slots: FP32 keeps the two classes' chunks one after the other; FP64 a general and a
// symmetric array of as many chunks as the largest class has
__host__ __device__ inline int vxc_max_chunks(const VxcMol& M) {
  const int a = M.nch[0] > M.nch[1] ? M.nch[0] : M.nch[1], b = M.nch[2] > M.nch[3] ? M.nch[2] : M.nch[3];
  return a > b ? a : b;
}
template <typename T>
inline long vxc_part_slots(const VxcMol& M) {
  return sizeof(T) == 4 ? M.nch[0] + M.nch[1] : 2L * vxc_max_chunks(M);
}

constexpr int VX_PTS = 32;   // chunk sizes are multiples of a stage
constexpr int VX_TB = 4;     // 16-wide blocks a tile at most
constexpr int VX_CP = 16 * VX_TB;

template <int VxcMol::*FIRST>
__device__ __forceinline__ VxcMol vxc_find(const VxcMol* __restrict__ mols, int nmol, const VxcMol& one, int blk) {
  if (mols == nullptr) return one;
  int lo = 0, hi = nmol - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (mols[mid].*FIRST <= blk) lo = mid; else hi = mid - 1;
  }
  // the same for the whole block: keep it in scalar registers
  static_assert(sizeof(VxcMol) % 4 == 0, "whole dwords");
  union U {
    VxcMol m;
    int w[sizeof(VxcMol) / 4];
    __device__ U() {}
  } u;
  const int* src = (const int*)&mols[lo];
#pragma unroll
  for (int k = 0; k < (int)(sizeof(VxcMol) / 4); ++k) u.w[k] = __builtin_amdgcn_readfirstlane(src[k]);
  return u.m;
}

// FP32: Z of every point of a slab, column and spin, once instead of once per tile row; four columns of a
// row a thread.  HBM-bound: reads the planes once, writes nsv.
// LOW: with d = phi - float(phi) behind the planes, v_rho enters with phi + 2 d, so that v_rho phi_a phi_a
// is right to first order in d where both factors would be rounded alike at every point of a shell (the
// core's diagonal), and so is their sum over (a, b) and (b, a) in V_xc + V_xc^T.  The bf16 plane costs 1%
// of dE/dD (B3LYP, n = 180: 447 against 438 us; n = 560: 6.70 against 6.60 ms; n = 43, 82, 102: 0 to 1 us).
template <bool LOW>
__global__ __launch_bounds__(256) void vxc_zform_kernel(const VxcMol* __restrict__ mols, int nmol,
                                                               const VxcMol one, const double* __restrict__ vpt,
                                                               size_t vpt_rows, int nsv, int slab) {
  const VxcMol M = vxc_find<&VxcMol::zblk0>(mols, nmol, one, blockIdx.x);
  const long i = ((long)(blockIdx.x - M.zblk0) * 256 + threadIdx.x) * 4;   // slab nP is a multiple of 1024
  const long plane = (long)M.npts_pad * M.nP, zplane = (long)M.slab * M.nP;
  const long r0 = (long)slab * M.slab, r = i / M.nP;
  if (r0 + r >= M.npts_pad) return;   // the last slab may be shorter
  const gptr<float> ao = (gptr<float>)M.ao + r0 * M.nP + i;
  const f4 p = *(gptr<f4>)ao, x = *(gptr<f4>)(ao + plane), y = *(gptr<f4>)(ao + 2 * plane),
           z = *(gptr<f4>)(ao + 3 * plane), l = *(gptr<f4>)(ao + 4 * plane);
  typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
  bf4 d = (bf4)(__bf16)0.f;
  if (LOW) d = *(gptr<bf4>)((gptr<__bf16>)((gptr<float>)M.ao + 5 * plane) + r0 * M.nP + i);
  for (int s = 0; s < nsv; ++s) {
    const double* v = vpt + ((size_t)s * vpt_rows + M.row0 + r0 + r) * VPT_STRIDE;
    const double v0 = v[0], v1 = v[1], v2 = v[2], v3 = v[3], v4 = v[4];
    f4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const double phi = LOW ? (double)p[e] + 2.0 * (double)(float)d[e] : (double)p[e];
      o[e] = (float)(v0 * phi + v1 * (double)x[e] + v2 * (double)y[e] + v3 * (double)z[e] + v4 * (double)l[e]);
    }
    *(gptr_w<f4>)((gptr_w<float>)M.z + s * zplane + i) = o;
  }
}

// One item: tile rows from a0, columns from b0 (16-wide blocks), points rbeg .. rend (multiples of
// VX_PTS), spin s, chunk number within its class.
struct VxcItem {
  int cls, a0, b0, rbeg, rend, s, chunk;
};

template <typename T>
__device__ __forceinline__ bool vxc_item(const VxcMol& M, int nsv, int slab, VxcItem& it) {
  const int local = blockIdx.x - M.blk0, xcd = local & 7;
  // selects of values: an indexed member would put the whole struct in scratch
  const int c0 = M.nch[0], c1 = M.nch[1], c2 = M.nch[2], c3 = M.nch[3];
  const int t0 = vxc_tiles<T>(M, 0), t1 = vxc_tiles<T>(M, 1), t2 = vxc_tiles<T>(M, 2), t3 = vxc_tiles<T>(M, 3);
  const int e0 = (c0 + 7) / 8 * t0 * nsv, e1 = e0 + (c1 + 7) / 8 * t1 * nsv, e2 = e1 + (c2 + 7) / 8 * t2 * nsv;
  int slot = local >> 3;
  it.cls = (slot >= e0) + (slot >= e1) + (slot >= e2);
  const int cls = it.cls;
  auto pick = [cls](int a, int b, int c, int d) { return cls == 0 ? a : cls == 1 ? b : cls == 2 ? c : d; };
  const int ntile = pick(t0, t1, t2, t3), nch = pick(c0, c1, c2, c3);
  const int ch = pick(+M.ch[0], +M.ch[1], +M.ch[2], +M.ch[3]);
  slot -= pick(0, e0, e1, e2);
  const int per = ntile * nsv;
  it.chunk = xcd + 8 * (slot / per);
  if (it.chunk >= nch) return false;
  slot %= per;
  it.s = slot / ntile;
  int col = slot % ntile, row = 0;
  if (sizeof(T) == 4 && it.cls == 0) {
    const int nt = M.nf + (M.rem != 0);
    row = col / nt;
    col %= nt;
  } else if (sizeof(T) == 8 && it.cls > 0) {
    row = it.cls == 3 ? M.nf : col;
    col = it.cls == 2 ? col : M.nf;
  } else {   // triangular: with the diagonal (FP32 symmetric), without (FP64 pairs)
    const int d = sizeof(T) == 8 ? 1 : 0, nt = sizeof(T) == 8 ? M.nf : M.nf + (M.rem != 0);
    while (col >= nt - d - row) col -= nt - d - row++;
    col += row + d;
  }
  it.a0 = row * M.tb;
  it.b0 = col * M.tb;
  const int r0 = slab * M.slab, r1 = min(M.npts_pad, r0 + M.slab);
  it.rbeg = r0 + it.chunk * ch;
  it.rend = min(r1, it.rbeg + ch);
  return it.rbeg < r1;   // a shorter last slab has fewer chunks
}

// Quadrant of this wave in a tile of tr x tc blocks: rows from wi, columns from wj, at most 2 x 2 blocks,
// and the mask of those that exist.  Waves rotate over the quadrants with the block index, so that the
// smaller ones of odd tiles fall on every SIMD alike; blocks 32 apart on an XCD tend to share a CU.
struct VxcQuad {
  int wi, wj;
  unsigned mask;
};
__device__ __forceinline__ int vxc_rotation(int wave) {
  const int slot = blockIdx.x >> 3;
  return (wave + slot + (slot >> 5)) & 3;
}
__device__ __forceinline__ VxcQuad vxc_quadrant(int q, int tr, int tc) {
  const int hi = (tr + 1) / 2, hj = (tc + 1) / 2;
  VxcQuad Q{(q >> 1) * hi, (q & 1) * hj, 0u};
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
      if (i < hi && j < hj && Q.wi + i < tr && Q.wj + j < tc) Q.mask |= 1u << (i * 2 + j);
  Q.mask = __builtin_amdgcn_readfirstlane(Q.mask);
  return Q;
}
// of those, the symmetric blocks this wave forms in a diagonal tile: on and above the diagonal, but of
// the upper right quadrant's every second block is taken, transposed, by the wave of the lower left
__device__ __forceinline__ unsigned vxc_sym_mask(const VxcQuad& Q, bool share) {
  unsigned m = 0;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const bool off = Q.wi != Q.wj;
      if (off && share ? (Q.wi < Q.wj) == (i == j) : Q.wi + i <= Q.wj + j) m |= 1u << (i * 2 + j);
    }
  return __builtin_amdgcn_readfirstlane(m & Q.mask);
}

__device__ __forceinline__ double readlane_f64(double x, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), lane),
                          __builtin_amdgcn_readlane(__double2loint(x), lane));
}

// FP32: both operands split into three bf16 terms while staged (gdx_gemm_split.h), a stage is 32
// points of one product.  A block's products are summed from zero in FP32 over VX_FL stages and then
// added to FP64 accumulators: the integrand cancels strongly near the nuclei (large Laplacian terms),
// and FP32 sums over hundreds of points degrade reverse mode through an SCF loop.  Staging takes as
// many issue slots as the products (28% MFMA, 50% VALU busy at n = 560): row addresses stay scalar, u is
// held one point a lane and read by lane index.  u d_j phi is an FP64 product rounded once (u as an FP32
// pair: the same time, a second rounding, and no value past FP32's range).
constexpr int VX_FL = 2;
// Z is formed and multiplied a slab of points at a time, whose sums add to the partials of the slab
// before (the same chunks of every slab, one launch after the other: a fixed order).  vxc_slabs has
// the sizes.

__global__ __launch_bounds__(256, 4) void vxc_f32_kernel(const VxcMol* __restrict__ mols, int nmol,
                                                                const VxcMol one, const double* __restrict__ vpt,
                                                                size_t vpt_rows, int nsv, int slab) {
  __shared__ __align__(16) __bf16 Ls[3][4][VX_CP * 8];
  __shared__ __align__(16) __bf16 Rs[3][4][VX_CP * 8];
  const VxcMol M = vxc_find<&VxcMol::blk0>(mols, nmol, one, blockIdx.x);
  VxcItem it;
  if (!vxc_item<float>(M, nsv, slab, it)) return;
  const bool sym = it.cls == 1;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, r = lane & 15, nP = M.nP;
  const size_t plane = (size_t)M.npts_pad * nP;
  const VxcQuad Q = vxc_quadrant(vxc_rotation(wave), min(M.tb, nP / 16 - it.a0), min(M.tb, nP / 16 - it.b0));
  const int wi = Q.wi, wj = Q.wj;
  const unsigned mask = sym && it.a0 == it.b0 ? vxc_sym_mask(Q, false) : Q.mask;
  // staging: lane = column, wave = group of 8 consecutive points, a fragment; columns past the matrix
  // repeat the last one (their blocks are not computed)
  const unsigned cl = 4 * min(it.a0 * 16 + lane, nP - 1), cr = 4 * min(it.b0 * 16 + lane, nP - 1);
  const gptr<float> lp = (gptr<float>)M.ao;
  const gptr<float> rp = sym ? lp : (gptr<float>)M.z + (size_t)it.s * M.slab * nP;
  const size_t rs = sym ? 0 : (size_t)slab * M.slab * nP;   // Z starts with the slab
  const gptr<double> up = (gptr<double>)vpt + ((size_t)it.s * vpt_rows + M.row0 + (lane & 31)) * VPT_STRIDE + 5;
  float xl[8], xr[8];
  double u = 0.0;   // u of point lane % 32 of the loaded stage
  auto gload = [&](int pt, int pl) {
    const size_t row = pl * plane + (size_t)(pt + 8 * wave) * nP;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      xl[e] = row_load<float>(lp + row + e * nP, cl);
      xr[e] = row_load<float>(rp + (row - rs) + e * nP, cr);
    }
    if (sym) u = up[(size_t)pt * VPT_STRIDE];
  };
  auto lstore = [&]() {
    bf8 f[3];
    split8(xl, f[0], f[1], f[2]);
#pragma unroll
    for (int p = 0; p < 3; ++p) *(bf8*)&Ls[p][wave][lane * 8] = f[p];
    if (sym)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        xr[e] = (float)(readlane_f64(u, 8 * wave + e) * (double)xr[e]);
    split8(xr, f[0], f[1], f[2]);
#pragma unroll
    for (int p = 0; p < 3; ++p) *(bf8*)&Rs[p][wave][lane * 8] = f[p];
  };
  double acc[2][2][4];
  f4 part[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      part[i][j] = (f4)0.f;
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[i][j][v] = 0.0;
    }
  const int pl0 = sym ? 1 : 0, pl1 = sym ? 3 : 0;
  int pt = it.rbeg, pl = pl0, st = 0;
  gload(pt, pl);
  while (pt < it.rend) {
    lstore();
    __syncthreads();
    if (++pl > pl1) {
      pl = pl0;
      pt += VX_PTS;
    }
    const bool more = pt < it.rend;
    if (more) gload(pt, pl);
    bf8 ha[2][3];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int p = 0; p < 3; ++p) ha[i][p] = *(const bf8*)&Ls[p][g][((wi + i) * 16 + r) * 8];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      bf8 hr[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) hr[p] = *(const bf8*)&Rs[p][g][((wj + j) * 16 + r) * 8];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        if (mask >> (i * 2 + j) & 1) mfma_chain(ha[i], hr, part[i][j]);
    }
    if (!more || ++st % VX_FL == 0) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
          for (int v = 0; v < 4; ++v) acc[i][j][v] += (double)part[i][j][v];
          part[i][j] = (f4)0.f;
        }
    }
    __syncthreads();
  }
  const int slot = it.chunk + (sym ? M.nch[0] : 0);
  const gptr_w<double> out = (gptr_w<double>)M.part + ((size_t)slot * nsv + it.s) * nP * nP;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
      if (mask >> (i * 2 + j) & 1)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const size_t at = (size_t)((it.a0 + wi + i) * 16 + mfma32_row(lane, v)) * nP + (it.b0 + wj + j) * 16 + r;
          out[at] = slab ? out[at] + acc[i][j][v] : acc[i][j][v];
        }
}

// FP64: an item is a pair of tiles (I, J), so that the planes of both are staged once for all five
// products: phi_I^T Z_J, phi_J^T Z_I and the three symmetric ones; a diagonal item has one tile, one
// general product and the upper half of the symmetric ones.  Z and u d_j phi are formed while staged, 8
// points at a time: FP64 vector operations share the matrix cores' issue (forming them again in every
// wave's operands: 0.74 ms at n = 192), and a pass over memory that stores Z costs 0.24 ms there.
constexpr int VXD_K = 8;
constexpr int VXD_LD = VX_CP + 16;

template <bool PAIR>
__device__ __forceinline__ void vxc_f64_item(const VxcMol& M, const VxcItem& it, const double* __restrict__ vpt,
                                             size_t vpt_rows, int nsv, double (*Is)[VXD_K][VXD_LD],
                                             double (*Js)[VXD_K][VXD_LD]) {
  typedef double v2 __attribute__((ext_vector_type(2)));
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, r = lane & 15, nP = M.nP;
  const size_t plane = (size_t)M.npts_pad * nP;
  const int ti = min(M.tb, nP / 16 - it.a0), tj = min(M.tb, nP / 16 - it.b0), q = vxc_rotation(wave);
  const VxcQuad Q = vxc_quadrant(q, ti, tj), R = vxc_quadrant(q, tj, ti);   // rows of I, of J
  const int wi = Q.wi, wj = Q.wj;
  const unsigned mij = Q.mask, mji = PAIR ? R.mask : 0u, msy = PAIR ? Q.mask : vxc_sym_mask(Q, true);
  // staging: columns sc, sc + 1 of point sp of both tiles, five planes
  const int sp = tid >> 5, sc = (tid & 31) * 2;
  const gptr<double> lp = (gptr<double>)M.ao;
  const unsigned ro = 8u * sp * nP, ca = ro + 8 * min(it.a0 * 16 + sc, nP - 2), cb = ro + 8 * min(it.b0 * 16 + sc, nP - 2);
  const gptr<double> vp = (gptr<double>)vpt + ((size_t)it.s * vpt_rows + M.row0 + sp) * VPT_STRIDE;
  v2 xa[5], xb[5], v[3];
  auto gload = [&](int pt) {
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      const gptr<double> row = lp + k * plane + (size_t)pt * nP;
      xa[k] = row_load<v2>(row, ca);
      if (PAIR) xb[k] = row_load<v2>(row, cb);
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) v[k] = *(gptr<v2>)(vp + (size_t)pt * VPT_STRIDE + 2 * k);
  };
  // a stage's products take about as long as a load from HBM: touch every 128-byte line of the stage
  // after the next one, so that its loads come from L2
  const int tk = min(tid >> 5, 4), tp = (tid >> 2) & 7, tq = (tid & 3) * 128;
  const unsigned to = 8u * tp * nP, ta = to + min(it.a0 * 128 + tq, 8 * nP - 128), tb = to + min(it.b0 * 128 + tq, 8 * nP - 128);
  int na = 0, nb = 0;
  auto touch = [&](int pt) {
    const gptr<double> row = lp + tk * plane + (size_t)pt * nP;
    na = *(gptr<int>)((gptr<char>)row + ta);
    if (PAIR) nb = *(gptr<int>)((gptr<char>)row + tb);
  };
  auto zform = [&](const v2* x) {
    return v[0][0] * x[0] + v[0][1] * x[1] + v[1][0] * x[2] + v[1][1] * x[3] + v[2][0] * x[4];
  };
  auto lstore = [&]() {
#pragma unroll
    for (int k = 0; k < 4; ++k) *(v2*)&Is[k][sp][sc] = xa[k];
    if (PAIR) {
      *(v2*)&Is[4][sp][sc] = zform(xa);
      *(v2*)&Js[0][sp][sc] = xb[0];
#pragma unroll
      for (int k = 1; k < 4; ++k) *(v2*)&Js[k][sp][sc] = v[2][1] * xb[k];
      *(v2*)&Js[4][sp][sc] = zform(xb);
    } else {
#pragma unroll
      for (int k = 1; k < 4; ++k) *(v2*)&Js[k][sp][sc] = v[2][1] * xa[k];
      *(v2*)&Js[4][sp][sc] = zform(xa);
    }
  };
  d4 gij[2][2], gji[2][2], sy[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) gij[i][j] = gji[i][j] = sy[i][j] = (d4){0, 0, 0, 0};
  const int last = it.rend - VXD_K;
  gload(it.rbeg);
  touch(min(it.rbeg + VXD_K, last));
  for (int pt = it.rbeg; pt <= last; pt += VXD_K) {
    lstore();
    __syncthreads();
    gload(min(pt + VXD_K, last));
    asm volatile("" ::"v"(na), "v"(nb));
    touch(min(pt + 2 * VXD_K, last));
#pragma unroll
    for (int kk = 0; kk < VXD_K / 4; ++kk) {
      const int p = kk * 4 + g;
      double a[4][2], b[5][2];   // rows of I, columns of J
#pragma unroll
      for (int e = 0; e < 2; ++e) {
#pragma unroll
        for (int k = 0; k < 4; ++k) a[k][e] = Is[k][p][(wi + e) * 16 + r];
#pragma unroll
        for (int k = 1; k < 5; ++k) b[k][e] = Js[k][p][(wj + e) * 16 + r];
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          if (mij >> (i * 2 + j) & 1) gij[i][j] = MfmaT<double>::op(a[0][i], b[4][j], gij[i][j]);
          if (msy >> (i * 2 + j) & 1)
#pragma unroll
            for (int k = 1; k < 4; ++k) sy[i][j] = MfmaT<double>::op(a[k][i], b[k][j], sy[i][j]);
        }
      if (mji) {   // rows of J, columns of I
        double c[2], z[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          c[e] = Js[0][p][(R.wi + e) * 16 + r];
          z[e] = Is[4][p][(R.wj + e) * 16 + r];
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            if (mji >> (i * 2 + j) & 1) gji[i][j] = MfmaT<double>::op(c[i], z[j], gji[i][j]);
      }
    }
    __syncthreads();
  }
  const size_t mat = (size_t)nP * nP, half = (size_t)vxc_max_chunks(M) * nsv * mat;
  const gptr_w<double> gen = (gptr_w<double>)M.part + ((size_t)it.chunk * nsv + it.s) * mat;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int lr = i * 16 + mfma64_row(lane, e), lc = j * 16 + r;
        const size_t row = it.a0 * 16 + wi * 16 + lr, col = it.b0 * 16 + wj * 16 + lc;
        if (mij >> (i * 2 + j) & 1) gen[row * nP + col] = gij[i][j][e];
        if (msy >> (i * 2 + j) & 1) gen[half + (row / 16 <= col / 16 ? row * nP + col : col * nP + row)] = sy[i][j][e];
        if (mji >> (i * 2 + j) & 1)
          gen[(size_t)(it.b0 * 16 + R.wi * 16 + lr) * nP + it.a0 * 16 + R.wj * 16 + lc] = gji[i][j][e];
      }
}

__global__ __launch_bounds__(256, 2) void vxc_f64_kernel(const VxcMol* __restrict__ mols, int nmol,
                                                                const VxcMol one, const double* __restrict__ vpt,
                                                                size_t vpt_rows, int nsv) {
  __shared__ __align__(16) double Is[5][VXD_K][VXD_LD];   // tile I: phi, its derivatives, Z
  __shared__ __align__(16) double Js[5][VXD_K][VXD_LD];   // tile J: phi, u d_j phi, Z
  const VxcMol M = vxc_find<&VxcMol::blk0>(mols, nmol, one, blockIdx.x);
  VxcItem it;
  if (!vxc_item<double>(M, nsv, 0, it)) return;
  if (it.cls < 2) vxc_f64_item<true>(M, it, vpt, vpt_rows, nsv, Is, Js);
  else vxc_f64_item<false>(M, it, vpt, vpt_rows, nsv, Is, Js);
}

// The partial sums of each molecule -> its (2, n, n) output (nsv = 1: the one spin written to both): an
// 8 x 8 patch of one spin a block, its waves take every fourth chunk with eight loads of a thread in
// flight and are added in a fixed order.  Symmetric partials hold the blocks on and above the diagonal;
// the others read the transposed patch, in 64-byte pieces either way.
inline long vxc_reduce_blocks(const VxcMol& M, int nsv) { return (long)nsv * (M.nP / 8) * (M.nP / 8); }

template <typename T>
__global__ __launch_bounds__(256) void vxc_reduce_kernel(const VxcMol* __restrict__ mols, int nmol, const VxcMol one,
                                                         int nsv, double* __restrict__ out) {
  const VxcMol M = vxc_find<&VxcMol::rblk0>(mols, nmol, one, blockIdx.x);
  __shared__ double red[4][64];
  const int c = threadIdx.x & 63, g = threadIdx.x >> 6, n = M.n, nP = M.nP, edge = nP / 8;
  const int patch = blockIdx.x - M.rblk0, s = patch / (edge * edge), pr = patch / edge % edge, pc = patch % edge;
  const int a = pr * 8 + (c >> 3), b = pc * 8 + (c & 7);
  const long stride = (long)nsv * nP * nP;
  double acc = 0.0;
  auto add = [&](gptr<double> p, int nch) {
    int k = g;
    for (; k + 28 < nch; k += 32) {
      double v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = p[(k + 4 * u) * stride];
#pragma unroll
      for (int u = 0; u < 8; ++u) acc += v[u];
    }
    for (; k < nch; k += 4) acc += p[k * stride];
  };
  const int I = a >> 4, J = b >> 4;
  const gptr<double> p = (gptr<double>)M.part + (long)s * nP * nP;
  const long at = (long)a * nP + b, up = I <= J ? at : (long)b * nP + a;
  if (sizeof(T) == 4) {
    add(p + at, M.nch[0]);
    add(p + M.nch[0] * stride + up, M.nch[1]);
  } else {
    const int ti = I / M.tb, tj = J / M.tb;
    const bool ragged = max(ti, tj) == M.nf;
    const int nch = ti == tj ? (ragged ? M.nch[3] : M.nch[2]) : (ragged ? M.nch[1] : M.nch[0]);
    add(p + at, nch);
    add(p + vxc_max_chunks(M) * stride + up, nch);
  }
  red[g][c] = acc;
  __syncthreads();
  if (g == 0 && a < n && b < n) {
    const double v = red[0][c] + red[1][c] + red[2][c] + red[3][c];
    double* o = out + M.out_off + (long)a * n + b;
    o[(long)s * n * n] = v;
    if (nsv == 1) o[(long)n * n] = v;
  }
}

}  // namespace gdx
