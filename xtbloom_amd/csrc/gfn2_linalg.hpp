// Dense FP64 linear algebra for the ragged batch: tiled GEMM over a tile
// queue, per-system Cholesky/inverse and the symmetric eigensolver (Householder
// tridiagonalization, Sturm bisection and Newton steps, twisted or inverse
// iteration, back-transformation).
#pragma once

#include <type_traits>

#include "gfn2_device.hpp"
#include "gfn2_occupation.hpp"

namespace xtb {

// One output tile of one system's GEMM; the queue is built on the host from the
// ragged sizes so that one launch covers every system.
struct TileTask {
  int sys;
  int ti;  // tile row
  int tj;  // tile column
};

constexpr int kTile = 64;
constexpr int kTileK = 16;

// C[sys] = sum_k opA(A)[i][k] * scale[k] * opB(B)[k][j]   (row-major n x n operands)
//   TA: A is read transposed (A[k][i]); TB: B is read transposed (B[j][k]).
//   K per system: kdim[sys] if given, else n.  ncol (optional): tiles whose
//   columns all lie at or past ncol[sys] are skipped.
//   SYMM: only tiles with ti >= tj are queued; the kernel mirrors them.
//   TRI: the K range a tile needs when an operand is upper triangular (its
//   strict lower part stored as zero, as for X = L^-T), so the skipped
//   products are exact zeros:
//     1  A read transposed and upper triangular (X^T H):  k < i0 + 64
//     2  B upper triangular (T X):                         k < j0 + 64
//     3  A upper triangular (X Y):                         k >= i0
// FP64 matrix-core product of one 16 x 16 x 4 step, v_mfma_f64_16x16x4f64:
// lane l supplies A[l % 16][l / 16] and B[l / 16][l % 16] and accumulates
// C[l / 16 + 4 r][l % 16], r = 0..3 (layout checked on gfx950).
typedef double mfma_d4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ mfma_d4 mfma_16x16x4(double a, double b, mfma_d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Systems whose density product runs in split-precision FP32 (k_gemm_split32):
// those in their first SCC round or with a mixer residual above kSplitResidual.
constexpr double kSplitResidual = 1e-3;
__device__ __forceinline__ bool split_round(const SysState& z) {
  return z.iterations == 0 || z.residual_rms > kSplitResidual;
}

template <bool TA, bool TB, bool SYMM, int TRI = 0>
__global__ __launch_bounds__(256) void k_gemm(Topo t, const TileTask* tasks, const double* A,
                                              const double* Bm, double* C, const double* scale,
                                              const int* kdim, const int* ncol,
                                              const unsigned char* active,
                                              const SysState* split = nullptr) {
  const TileTask task = tasks[blockIdx.x];
  const int s = task.sys;
  if (active && !active[s]) return;
  if (split && split_round(split[s])) return;  // computed by k_gemm_split32
  if (ncol && task.tj * kTile >= ncol[s]) return;  // columns past ncol are not needed
  const int n = t.ao_off[s + 1] - t.ao_off[s];
  const int64_t mo = t.mat_off[s];
  const double* a = A + mo;
  const double* b = Bm + mo;
  double* c = C + mo;
  const double* sc = scale ? scale + t.ao_off[s] : nullptr;
  const int K = kdim ? kdim[s] : n;
  const int i0 = task.ti * kTile, j0 = task.tj * kTile;
  __shared__ double As[2][kTileK][kTile + 1];  // two stages: one written while the other is read
  __shared__ double Bs[2][kTileK][kTile + 1];
  // wave w owns the 32 x 32 quadrant (w / 2, w % 2): 2 x 2 blocks of 16 x 16
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int qi = 32 * (w >> 1), qj = 32 * (w & 1);
  const int l16 = lane & 15, lk = lane >> 4;
  mfma_d4 acc[2][2];
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int q = 0; q < 2; ++q) acc[p][q] = mfma_d4{0.0, 0.0, 0.0, 0.0};
  int kbeg = 0, kend = K;
  if constexpr (TRI == 1) kend = min(K, i0 + kTile);
  if constexpr (TRI == 2) kend = min(K, j0 + kTile);
  if constexpr (TRI == 3) kbeg = i0;
  // Stage k0 of A and B is fetched into registers one step ahead: its global
  // loads are in flight while the matrix cores work on the previous stage.
  constexpr int kPer = kTile * kTileK / 256;  // elements of each operand per thread
  double pa[kPer], pb[kPer];
  auto fetch = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int idx = threadIdx.x + 256 * u;
      int kk, ii;
      if (TA) { ii = idx % kTile; kk = idx / kTile; } else { kk = idx % kTileK; ii = idx / kTileK; }
      const int gi = i0 + ii, gk = k0 + kk;
      double val = 0.0;
      if (gi < n && gk < K) {
        val = TA ? a[(int64_t)gk * n + gi] : a[(int64_t)gi * n + gk];
        if (sc) val *= sc[gk];
      }
      pa[u] = val;
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int idx = threadIdx.x + 256 * u;
      int kk, jj;
      if (TB) { kk = idx % kTileK; jj = idx / kTileK; } else { jj = idx % kTile; kk = idx / kTile; }
      const int gj = j0 + jj, gk = k0 + kk;
      pb[u] = (gj < n && gk < K) ? (TB ? b[(int64_t)gj * n + gk] : b[(int64_t)gk * n + gj]) : 0.0;
    }
  };
  // A tile rows i0..i0+63 -> As[buf][k][i], B tile -> Bs[buf][k][j]
  auto stash = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int idx = threadIdx.x + 256 * u;
      if (TA) As[buf][idx / kTile][idx % kTile] = pa[u]; else As[buf][idx % kTileK][idx / kTileK] = pa[u];
      if (TB) Bs[buf][idx % kTileK][idx / kTileK] = pb[u]; else Bs[buf][idx / kTile][idx % kTile] = pb[u];
    }
  };
  if (kbeg < kend) {
    fetch(kbeg);
    stash(0);
  }
  __syncthreads();
  int buf = 0;
  for (int k0 = kbeg; k0 < kend; k0 += kTileK, buf ^= 1) {
    const bool more = k0 + kTileK < kend;
    if (more) fetch(k0 + kTileK);
#pragma unroll
    for (int k4 = 0; k4 < kTileK; k4 += 4) {
      double af[2], bf[2];
#pragma unroll
      for (int p = 0; p < 2; ++p) af[p] = As[buf][k4 + lk][qi + 16 * p + l16];
#pragma unroll
      for (int q = 0; q < 2; ++q) bf[q] = Bs[buf][k4 + lk][qj + 16 * q + l16];
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q) acc[p][q] = mfma_16x16x4(af[p], bf[q], acc[p][q]);
    }
    // the other stage was last read before the previous barrier
    if (more) stash(buf ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int gi = i0 + qi + 16 * p + lk + 4 * r;
      if (gi >= n) continue;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int gj = j0 + qj + 16 * q + l16;
        if (gj >= n) continue;
        c[(int64_t)gi * n + gj] = acc[p][q][r];
        if (SYMM && task.ti != task.tj) c[(int64_t)gj * n + gi] = acc[p][q][r];
      }
    }
}

// Split-precision FP32 matrix-core form of the symmetric density products
// P = C diag(f) C^T and W = C diag(f eps) C^T (lower tiles of the tile queue,
// K = kocc, mirrored).  Each FP64 operand x is split into x_hi = fp32(x) and
// x_lo = fp32(x - x_hi), and a_hi b_hi + a_hi b_lo + a_lo b_hi run on
// v_mfma_f32_16x16x4f32 with FP32 accumulation over one 16-deep K stage; the
// stage sums are added in FP64.  The dropped a_lo b_lo term is below 2^-48 of
// a product; the FP32 accumulation bounds the result near 1e-7 relative to
// the stage sums.  `only_early` (P): systems still in their first SCC round
// or with a mixer residual above kSplitResidual; null (W): every system.
// k_gemm skips the same systems through its `split` argument.

typedef float mfma_f4 __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(256) void k_gemm_split32(Topo t, const TileTask* tasks, const double* A,
                                                      double* C, const double* scale, const int* kdim,
                                                      const SysState* only_early,
                                                      const unsigned char* active) {
  const TileTask task = tasks[blockIdx.x];
  const int s = task.sys;
  if (active && !active[s]) return;
  if (only_early && !split_round(only_early[s])) return;
  const int n = t.ao_off[s + 1] - t.ao_off[s];
  const int64_t mo = t.mat_off[s];
  const double* a = A + mo;
  double* c = C + mo;
  const double* sc = scale + t.ao_off[s];
  const int K = kdim[s];
  const int i0 = task.ti * kTile, j0 = task.tj * kTile;
  // operands of one K stage: A = C[i][k] f_k (rows i0..), B^T = C[j][k] (rows j0..)
  __shared__ float Ah[kTileK][kTile + 1], Al[kTileK][kTile + 1];
  __shared__ float Bh[kTileK][kTile + 1], Bl[kTileK][kTile + 1];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int qi = 32 * (w >> 1), qj = 32 * (w & 1);
  const int l16 = lane & 15, lk = lane >> 4;
  double acc[2][2][4];
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[p][q][r] = 0.0;
  constexpr int kPer = kTile * kTileK / 256;
  for (int k0 = 0; k0 < K; k0 += kTileK) {
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int idx = threadIdx.x + 256 * u;
      const int kk = idx % kTileK, ii = idx / kTileK;
      const int gk = k0 + kk;
      double va = 0.0, vb = 0.0;
      if (gk < K) {
        if (i0 + ii < n) va = a[(int64_t)(i0 + ii) * n + gk] * sc[gk];
        if (j0 + ii < n) vb = a[(int64_t)(j0 + ii) * n + gk];
      }
      const float ha = (float)va, hb = (float)vb;
      Ah[kk][ii] = ha;
      Al[kk][ii] = (float)(va - (double)ha);
      Bh[kk][ii] = hb;
      Bl[kk][ii] = (float)(vb - (double)hb);
    }
    __syncthreads();
    mfma_f4 part[2][2];
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int q = 0; q < 2; ++q) part[p][q] = mfma_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k4 = 0; k4 < kTileK; k4 += 4) {
      float ah[2], al[2], bh[2], bl[2];
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        ah[p] = Ah[k4 + lk][qi + 16 * p + l16];
        al[p] = Al[k4 + lk][qi + 16 * p + l16];
      }
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        bh[q] = Bh[k4 + lk][qj + 16 * q + l16];
        bl[q] = Bl[k4 + lk][qj + 16 * q + l16];
      }
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          part[p][q] = __builtin_amdgcn_mfma_f32_16x16x4f32(al[p], bh[q], part[p][q], 0, 0, 0);
          part[p][q] = __builtin_amdgcn_mfma_f32_16x16x4f32(ah[p], bl[q], part[p][q], 0, 0, 0);
          part[p][q] = __builtin_amdgcn_mfma_f32_16x16x4f32(ah[p], bh[q], part[p][q], 0, 0, 0);
        }
    }
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[p][q][r] += (double)part[p][q][r];
    __syncthreads();
  }
  // v_mfma_f32_16x16x4f32 leaves C[4 (l / 16) + r][l % 16] in lane l, item r
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int gi = i0 + qi + 16 * p + 4 * lk + r;
      if (gi >= n) continue;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int gj = j0 + qj + 16 * q + l16;
        if (gj >= n) continue;
        c[(int64_t)gi * n + gj] = acc[p][q][r];
        if (task.ti != task.tj) c[(int64_t)gj * n + gi] = acc[p][q][r];
      }
    }
}

// ---------------------------------------------------------------------------
// Symmetric eigensolver in three stages (all FP64):
//   reduction         Householder A = Q T Q^T; T's diagonal/off-diagonal go to d/e,
//                     the reflectors (H = I - 2 v v^T, |v| = 1) stay in A's strict
//                     lower triangle.  k_tridiag up to 256 AOs (a 512-thread block
//                     per system), k_tridiag_team up to kTeamN, k_tridiag_blocked
//                     above.
//   eigenpairs of T   k_tridiag_eigen, one block per system, or k_eig_values,
//                     _occupations and _vectors over the chip (257 to kEigSplitAO
//                     AOs): T is split where an off-diagonal is negligible, every
//                     eigenvalue is found by Sturm counts and Newton steps (a
//                     thread per eigenvalue), every eigenvector from its twisted
//                     factorization or, in a cluster of close eigenvalues, by
//                     inverse iteration with a partially pivoted tridiagonal LU and
//                     modified Gram-Schmidt (a thread per cluster).  Eigenvalues
//                     are ranked ascending (ties by index).
//   k_backtransform   Y = Q Z on column blocks, many blocks per system, on the
//                     matrix cores (k_backtransform_wy above 256 AOs).
// Layouts: Z and Y are row-major (row i = component i, column j = vector j).
// ---------------------------------------------------------------------------
constexpr double kEps = 2.220446049250313e-16;
constexpr double kSafeMin = 2.2250738585072014e-308;
constexpr double kClusterTol = 1e-6;  // relative gap (to the block 1-norm) below which vectors are orthogonalized
// Clusters of more than kSerialCluster eigenvalues go to k_cluster_vectors
// (a near-dependent basis inflates |T| and can chain hundreds of eigenvalues
// into one cluster, whose Gram-Schmidt is quadratic in its size)
constexpr int kSerialCluster = 8;
// Hand-over of those clusters, per system: flag[s] set when it has one; for
// a cluster of indices j .. g1-1 (block-local eigenvalue order), end[ao + j]
// = g1 and lam / rank[ao + jj] hold each member's eigenvalue and Z column.
// k_cluster_vectors clears end[] entries after use.
struct ClusterOut {
  int* flag;
  int* end;
  double* lam;
  int* rank;
};
constexpr int kInverseIterations = 3;

// Householder reduction for n > kTeamN in panels of kTriPanel reflectors, the
// arrangement of LAPACK's dsytrd/dlatrd.  Within a panel the trailing matrix
// is not written: after reflectors 0 .. j-1 of the panel it equals
//   A_j = A_0 - V W^T - W V^T,
// V holding the panel's unit reflectors v_i (H_i = I - 2 v_i v_i^T, stored
// in A's columns below the subdiagonal as the register path stores them) and
// W the vectors w_i = 2 (p_i - (v_i^T p_i) v_i), p_i = A_i v_i (in the
// scratch matrix W, same layout).  Reflector j therefore reads column k of A_0
// corrected by V and W, the lower triangle of A_0's trailing block once (the
// symmetric product), and V and W twice; the trailing lower triangle is
// rewritten once per panel, on the matrix cores.  Only the lower triangle of
// A is read or written.  512 threads.
//
// Every phase issues all of its global loads before the first use (fully
// unrolled, out-of-range lanes clamped to valid addresses and their values
// selected away), so that a wavefront waits once per column pair rather than
// once per 64-row slot.
constexpr int kTriPanel = 16;

// One unit of the symmetric product p = A v over an m x m trailing block
// (column-major at `blk`, leading dimension n, lower triangle): the columns
// c = cu .. cu + 2 kTriPairs - 1 (cu a multiple of 2 kTriPairs, so that all
// start in row slot cu / 64), rows 64 (tb + u) + lane, u < NS.  Column
// c adds a_rc x_c to the row partials (registers, flushed to the wavefront's
// row `prow` at the end) and its dot with x over the rows below the
// diagonal, plus the diagonal term, to pcol[c].  The next column pair is
// fetched while the current one is consumed.
//
// Rows past m read row m - 1 (a valid address) and meet x_r = 0, so they
// drop out of the dots without masks, and their row partials are never read;
// only slot 0, which holds the diagonal, is masked.  Column bases are
// wavefront-uniform and the row offsets 32-bit, so each load is one
// scalar-base instruction.
constexpr int kTriPairs = 8;

// Wavefront sums of two values at once: one exchange across the halves
// leaves column 0's partials in lanes 0..31 and column 1's in lanes 32..63,
// then five DPP steps sum each half (results in lanes 31 and 63).
__device__ __forceinline__ void wave_sum_pair(double d0, double d1, double& s0, double& s1) {
  const bool hi = (threadIdx.x & 32) != 0;
  double v = (hi ? d1 : d0) + __shfl_xor(hi ? d0 : d1, 32, 64);
  v += dpp_move<0xb1, 0xf>(v);   // quad_perm [1,0,3,2]
  v += dpp_move<0x4e, 0xf>(v);   // quad_perm [2,3,0,1]
  v += dpp_move<0x124, 0xf>(v);  // row_ror:4
  v += dpp_move<0x128, 0xf>(v);  // row_ror:8
  v += dpp_move<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  const long long b = __double_as_longlong(v);
  s0 = __longlong_as_double(((long long)__builtin_amdgcn_readlane((int)(b >> 32), 31) << 32) |
                            (unsigned int)__builtin_amdgcn_readlane((int)b, 31));
  s1 = __longlong_as_double(((long long)__builtin_amdgcn_readlane((int)(b >> 32), 63) << 32) |
                            (unsigned int)__builtin_amdgcn_readlane((int)b, 63));
}

template <int NS>
__device__ __forceinline__ void symv_fetch(const double* __restrict__ blk, int64_t n, int m, int c,
                                           const unsigned (&boff)[NS], double (&f0)[NS], double (&f1)[NS]) {
  const char* p0 = reinterpret_cast<const char*>(blk + (int64_t)min(c, m - 1) * n);
  const char* p1 = reinterpret_cast<const char*>(blk + (int64_t)min(c + 1, m - 1) * n);
#pragma unroll
  for (int u = 0; u < NS; ++u) {
    f0[u] = *reinterpret_cast<const double*>(p0 + boff[u]);
    f1[u] = *reinterpret_cast<const double*>(p1 + boff[u]);
  }
}

template <int NS>
__device__ __forceinline__ void symv_consume(int c, int m, int r0, const double* __restrict__ x,
                                             const double (&xr)[NS], const double (&f0)[NS],
                                             const double (&f1)[NS], double (&acc)[NS],
                                             double* __restrict__ pcol, bool add) {
  const double xc0 = c < m ? x[c] : 0.0;
  const double xc1 = c + 1 < m ? x[c + 1] : 0.0;
  // slot 0: strictly lower rows, and the diagonal on the lane that holds it
  const double e0 = r0 > c ? f0[0] : 0.0;
  const double e1 = r0 > c + 1 ? f1[0] : 0.0;
  double d0 = fma(e0, xr[0], r0 == c ? f0[0] * xc0 : 0.0);
  double d1 = fma(e1, xr[0], r0 == c + 1 ? f1[0] * xc1 : 0.0);
  acc[0] = fma(e0, xc0, fma(e1, xc1, acc[0]));
#pragma unroll
  for (int u = 1; u < NS; ++u) {
    d0 = fma(f0[u], xr[u], d0);
    d1 = fma(f1[u], xr[u], d1);
    acc[u] = fma(f0[u], xc0, fma(f1[u], xc1, acc[u]));
  }
  wave_sum_pair(d0, d1, d0, d1);
  if ((threadIdx.x & 63) == 0) {
    if (c < m) pcol[c] = add ? pcol[c] + d0 : d0;
    if (c + 1 < m) pcol[c + 1] = add ? pcol[c + 1] + d1 : d1;
  }
}

// tb: the first row slot of the unit's chunk, cu / 64 or more (row chunks of at
// most 16 slots); chunks after the first add their column dots to pcol, and
// their rows lie below every column of the unit.
template <int NS>
__device__ __forceinline__ void symv_unit(const double* __restrict__ blk, int64_t n, int m, int cu, int tb,
                                          const double* __restrict__ x, double* __restrict__ prow,
                                          double* __restrict__ pcol) {
  const int lane = threadIdx.x & 63;
  const bool add = tb != (cu >> 6);
  const int r0 = 64 * tb + lane;  // this lane's row in slot 0
  unsigned boff[NS];              // byte offsets of this lane's rows in a column
  double xr[NS], acc[NS];
#pragma unroll
  for (int u = 0; u < NS; ++u) {
    const int rr = r0 + 64 * u;
    const int rc = min(rr, m - 1);
    boff[u] = (unsigned)rc * 8u;
    xr[u] = rr < m ? x[rc] : 0.0;
    acc[u] = 0.0;
  }
  // two column pairs per trip, in two buffers: pair q + 1 is in flight while
  // pair q is consumed, with no register copies between trips
  double a0[NS], a1[NS], b0[NS], b1[NS];
  symv_fetch<NS>(blk, n, m, cu, boff, a0, a1);
#pragma unroll 1
  for (int q = 0; q < kTriPairs; q += 2) {
    const int c = cu + 2 * q;
    symv_fetch<NS>(blk, n, m, c + 2, boff, b0, b1);
    symv_consume<NS>(c, m, r0, x, xr, a0, a1, acc, pcol, add);
    if (q + 2 < kTriPairs) symv_fetch<NS>(blk, n, m, c + 4, boff, a0, a1);
    symv_consume<NS>(c + 2, m, r0, x, xr, b0, b1, acc, pcol, add);
  }
#pragma unroll
  for (int u = 0; u < NS; ++u) prow[r0 + 64 * u] += acc[u];
}

template <int NS>
__device__ __forceinline__ void dots_pair(const double* __restrict__ col0, const double* __restrict__ col1,
                                          int m, const double* __restrict__ x, double* __restrict__ out0,
                                          double* __restrict__ out1, bool add) {
  const int lane = threadIdx.x & 63;
  double a0[NS], a1[NS];
#pragma unroll
  for (int u = 0; u < NS; ++u) {
    const int rr = min(64 * u + lane, m - 1);
    a0[u] = col0[rr];
    a1[u] = col1[rr];
  }
  double d0 = 0.0, d1 = 0.0;
#pragma unroll
  for (int u = 0; u < NS; ++u) {
    const int rr = 64 * u + lane;
    const double xv = rr < m ? x[min(rr, m - 1)] : 0.0;
    d0 = fma(a0[u], xv, d0);
    d1 = fma(a1[u], xv, d1);
  }
  wave_sum_pair(d0, d1, d0, d1);
  if (lane == 0) {
    *out0 = add ? *out0 + d0 : d0;
    *out1 = add ? *out1 + d1 : d1;
  }
}

#define XTB_SLOT_SWITCH(NSV, CALL)                                                   \
  switch (NSV) {                                                                     \
    case 1: { constexpr int NS = 1; CALL; } break;                                   \
    case 2: { constexpr int NS = 2; CALL; } break;                                   \
    case 3: { constexpr int NS = 3; CALL; } break;                                   \
    case 4: { constexpr int NS = 4; CALL; } break;                                   \
    case 5: { constexpr int NS = 5; CALL; } break;                                   \
    case 6: { constexpr int NS = 6; CALL; } break;                                   \
    case 7: { constexpr int NS = 7; CALL; } break;                                   \
    case 8: { constexpr int NS = 8; CALL; } break;                                   \
    case 9: { constexpr int NS = 9; CALL; } break;                                   \
    case 10: { constexpr int NS = 10; CALL; } break;                                 \
    case 11: { constexpr int NS = 11; CALL; } break;                                 \
    case 12: { constexpr int NS = 12; CALL; } break;                                 \
    case 13: { constexpr int NS = 13; CALL; } break;                                 \
    case 14: { constexpr int NS = 14; CALL; } break;                                 \
    case 15: { constexpr int NS = 15; CALL; } break;                                 \
    case 16: { constexpr int NS = 16; CALL; } break;                                 \
    default: break;                                                                  \
  }

// v, pq, part and aux are global, with a row stride of `part` of n rounded up to
// 64; the symmetric product and the W^T v, V^T v dots run over row chunks of at
// most 16 slots.
__device__ __forceinline__ void tridiag_blocked(double* __restrict__ A, double* __restrict__ W, int n,
                                                double* d, double* e, double* v, double* pq,
                                                double* part, double* aux, double* red, double* bc) {
  const int tid = threadIdx.x, nt = blockDim.x;
  // the wavefront index is uniform: keep it (and the column indices derived
  // from it) in scalar registers
  const int lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), nw = nt >> 6;
  const int ldp = (n + 63) & ~63;
  double* pcol = aux;                   // [ldp] column dots of the symmetric product
  double* rowk = aux + ldp;             // [2 kTriPanel] row k of V, of W
  double* yv = rowk + 2 * kTriPanel;    // [2 kTriPanel] W^T v, V^T v
  double* prow = part + wv * ldp;       // this wavefront's row partials
  auto at = [n](int r, int c) __attribute__((always_inline)) { return (int64_t)r + (int64_t)c * n; };

  for (int k0 = 0; k0 + 2 < n; k0 += kTriPanel) {
    const int jn = min(kTriPanel, n - 2 - k0);
    for (int j = 0; j < jn; ++j) {
      const int k = k0 + j, b = k + 1, m = n - b;
      if (tid < kTriPanel) {
        const bool on = tid < j;
        const int ct = min(k0 + tid, n - 1);
        const double vk = A[at(k, ct)], wk = W[at(k, ct)];
        rowk[tid] = on ? vk : 0.0;
        rowk[kTriPanel + tid] = on ? wk : 0.0;
      }
      __syncthreads();
      // column k of A_j, rows k .. n-1 (the panel's later columns are read and
      // weighted by zero: one wait for all loads)
      double ss = 0.0;
      for (int r = k + tid; r < n; r += nt) {
        double av[kTriPanel], wv_[kTriPanel];
#pragma unroll
        for (int i = 0; i < kTriPanel; ++i) {
          av[i] = A[at(r, min(k0 + i, n - 1))];
          wv_[i] = W[at(r, min(k0 + i, n - 1))];
        }
        double x = A[at(r, k)];
#pragma unroll
        for (int i = 0; i < kTriPanel; ++i) {
          const bool on = i < j;
          x -= (on ? av[i] : 0.0) * rowk[kTriPanel + i] + (on ? wv_[i] : 0.0) * rowk[i];
        }
        if (r == k) {
          d[k] = x;
        } else {
          v[r - b] = x;
          ss += x * x;
        }
      }
      ss = block_sum(ss, red);
      if (tid == 0) {
        const double x0 = v[0];
        const double xn = sqrt(ss);
        if (xn == 0.0 || ss - x0 * x0 == 0.0) {
          e[k] = x0;  // already reduced: no reflection
          bc[0] = 0.0;
        } else {
          const double alpha = x0 >= 0.0 ? -xn : xn;
          const double v0 = x0 - alpha;
          const double vv = ss - x0 * x0 + v0 * v0;
          e[k] = alpha;
          v[0] = v0;
          bc[0] = 1.0 / sqrt(vv);
        }
      }
      __syncthreads();
      const double inv = bc[0];
      if (inv == 0.0) {
        for (int i = tid; i < m; i += nt) {
          A[at(b + i, k)] = 0.0;
          W[at(b + i, k)] = 0.0;
        }
        __syncthreads();
        continue;
      }
      const int tend = (m + 63) >> 6;
      for (int i = tid; i < m; i += nt) {
        const double vi = v[i] * inv;
        v[i] = vi;
        A[at(b + i, k)] = vi;
      }
      for (int i = lane; i < 64 * tend; i += 64) prow[i] = 0.0;
      __syncthreads();
      // p = A_0 v over the trailing block's lower triangle in units of
      // 2 kTriPairs columns, handed out in a snake over the wavefronts (the
      // units' work falls with their first column), then the 2j dots W^T v
      // and V^T v on the wavefront after the last unit's
      const int nunits = (m + 2 * kTriPairs - 1) / (2 * kTriPairs);
      for (int u0 = 0; u0 < nunits; u0 += nw) {
        const int u = u0 + (((u0 / nw) & 1) ? nw - 1 - wv : wv);
        if (u >= nunits) continue;
        const int cu = 2 * kTriPairs * u;
        const double* blk = A + at(b, b);
        for (int tb = cu >> 6; tb < tend; tb += 16)
          XTB_SLOT_SWITCH(min(16, tend - tb), (symv_unit<NS>(blk, n, m, cu, tb, v, prow, pcol)))
      }
      for (int q = (wv + nw - nunits % nw) % nw; q < j; q += nw) {
        for (int tb = 0; tb < tend; tb += 16)
          XTB_SLOT_SWITCH(min(16, tend - tb),
                          (dots_pair<NS>(W + at(b + 64 * tb, k0 + q), A + at(b + 64 * tb, k0 + q),
                                         m - 64 * tb, v + 64 * tb, yv + q, yv + kTriPanel + q, tb > 0)))
      }
      __syncthreads();
      // p_j = A_j v = p - V (W^T v) - W (V^T v);  K = v^T p_j
      double kp = 0.0;
      for (int i = tid; i < m; i += nt) {
        double av[kTriPanel], wv_[kTriPanel];
#pragma unroll
        for (int q = 0; q < kTriPanel; ++q) {
          av[q] = A[at(b + i, min(k0 + q, n - 1))];
          wv_[q] = W[at(b + i, min(k0 + q, n - 1))];
        }
        double p = pcol[i];
        for (int w = 0; w < nw; ++w) p += part[w * ldp + i];
#pragma unroll
        for (int q = 0; q < kTriPanel; ++q) {
          const bool on = q < j;
          p -= (on ? av[q] : 0.0) * (on ? yv[q] : 0.0) + (on ? wv_[q] : 0.0) * (on ? yv[kTriPanel + q] : 0.0);
        }
        pq[i] = p;
        kp += v[i] * p;
      }
      const double K = block_sum(kp, red);
      for (int i = tid; i < m; i += nt) W[at(b + i, k)] = 2.0 * (pq[i] - K * v[i]);
      __syncthreads();
    }
    // trailing lower triangle, rows and columns >= c0:
    //   A -= V W^T + W V^T = [V W] [W V]^T
    // in 16 x 16 tiles on the matrix cores (K = 2 kTriPanel).  The product is
    // formed transposed, so that a lane's outputs run along a column of A
    // (row = l16, column = lk + 4 r) and the update reads and writes whole
    // column segments.
    const int c0 = k0 + jn, mt = n - c0;
    const int nb16 = (mt + 15) >> 4;
    const int ntiles = nb16 * (nb16 + 1) / 2;
    const int l16 = lane & 15, lk = lane >> 4;
    for (int tile = wv; tile < ntiles; tile += nw) {
      // tile -> (TI, TJ), TI >= TJ, row-major over the lower triangle
      int TI = (int)((sqrt(8.0 * tile + 1.0) - 1.0) * 0.5);
      while (TI * (TI + 1) / 2 > tile) --TI;
      while ((TI + 1) * (TI + 2) / 2 <= tile) ++TI;
      const int TJ = tile - TI * (TI + 1) / 2;
      const int rr = 16 * TI + l16, cc = 16 * TJ + l16;  // this lane's operand row and column
      const int rrc = c0 + min(rr, mt - 1), ccc = c0 + min(cc, mt - 1);
      double xa[2 * kTriPanel / 4], xb[2 * kTriPanel / 4];
#pragma unroll
      for (int q = 0; q < kTriPanel / 4; ++q) {
        const int i = 4 * q + lk;
        const int ci = k0 + min(i, jn - 1);
        // A operand: column side [W V] at row cc; B operand: row side [V W] at row rr
        xa[q] = W[at(ccc, ci)];
        xa[kTriPanel / 4 + q] = A[at(ccc, ci)];
        xb[q] = A[at(rrc, ci)];
        xb[kTriPanel / 4 + q] = W[at(rrc, ci)];
      }
      mfma_d4 acc = mfma_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int q = 0; q < 2 * kTriPanel / 4; ++q) {
        const bool on = 4 * (q % (kTriPanel / 4)) + lk < jn;
        acc = mfma_16x16x4(on && cc < mt ? xa[q] : 0.0, on && rr < mt ? xb[q] : 0.0, acc);
      }
      // acc[r] = D[row = 16 TI + l16][col = 16 TJ + lk + 4 r]
      const int row = 16 * TI + l16;
      double old[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int col = 16 * TJ + lk + 4 * r;
        old[r] = A[at(c0 + min(row, mt - 1), c0 + min(col, mt - 1))];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int col = 16 * TJ + lk + 4 * r;
        if (row < mt && col < mt && row >= col) A[at(c0 + row, c0 + col)] = old[r] - acc[r];
      }
    }
    __syncthreads();
  }
  if (tid == 0) {
    if (n >= 2) {
      d[n - 2] = A[(n - 2) + (int64_t)(n - 2) * n];
      e[n - 2] = A[(n - 1) + (int64_t)(n - 2) * n];
    }
    d[n - 1] = A[(n - 1) + (int64_t)(n - 1) * n];
    e[n - 1] = 0.0;
  }
}

// Householder reduction with the lower triangle held in registers, n <= 16 NR,
// 512 threads.  Thread (lr, lc) = (tid / 32, tid % 32) owns element
// (16 TI + lr, 32 TJ + lc) of every 16 x 32 tile that meets the lower triangle
// (TJ <= TI / 2), so the symmetric matvec and the rank-2 update of each step
// never touch memory.  Only the reflector (LDS, and its column of A for the
// back-transformation), the matvec partials (LDS) and d/e leave the registers.
// Stored form: strictly-lower elements as is, diagonal elements halved, the
// strictly-upper part of tiles crossing the diagonal as zero.  Then every slot
// contributes x v_j to p_i and x v_i to p_j, which is the full symmetric
// product, and the rank-2 update keeps the form with factor 2 / 1 / 0.
constexpr int tri_slots(int NR) { return NR == 0 ? 0 : tri_slots(NR - 1) + (NR - 1) / 2 + 1; }
// slot -> (row tile, column tile) of the register layout; folded at compile time
constexpr int tri_row(int slot) {
  int TI = 0;
  while (tri_slots(TI + 1) <= slot) ++TI;
  return TI;
}
constexpr int tri_col(int slot) { return slot - tri_slots(tri_row(slot)); }
// tile entirely strictly below the diagonal (every row index > every column index)
constexpr bool tri_strict(int TI, int TJ) { return 16 * TI > 32 * TJ + 31; }

// compile-time loop: f(std::integral_constant<int, I>) for I in [B, E)
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

constexpr int kTriPad = 257;  // row stride of the partial-sum buffers (bank spread)
constexpr int kFullN = 192;  // columns reduced with both triangles in registers (tridiag_full)

template <int NR>
__device__ __forceinline__ void tridiag_registers(double* A, int n, double* d, double* e, double* v,
                                                  double* col, double* pq, double* rowpart,
                                                  double* colpart) {
  constexpr int NC = NR / 2;
  constexpr int NE = tri_slots(NR);
  const int tid = threadIdx.x, lr = tid >> 5, lc = tid & 31, lane = tid & 63;
  double a[NE];
  static_for<0, NE>([&](auto S) __attribute__((always_inline)) {
    constexpr int sl = decltype(S)::value;
    constexpr int TI = tri_row(sl), TJ = tri_col(sl);
    const int i = 16 * TI + lr, j = 32 * TJ + lc;
    // A is symmetric: lanes read row i along j contiguously
    const double x = (i < n && j < n) ? A[j + (int64_t)i * n] : 0.0;
    if constexpr (tri_strict(TI, TJ)) a[sl] = x;
    else a[sl] = i > j ? x : (i == j ? 0.5 * x : 0.0);
    // keep one row tile of loads in flight (address registers would spill the matrix)
    if constexpr (TJ == TI / 2) __builtin_amdgcn_sched_barrier(0);
  });
  // col holds column k of the reduced matrix (its owners publish column k+1
  // right after the update of step k); rows >= n stay zero.
  col[tid] = 0.0;
  __syncthreads();
  if (lc == 0) {
    static_for<0, NE>([&](auto S) __attribute__((always_inline)) {
      constexpr int sl = decltype(S)::value;
      constexpr int TI = tri_row(sl), TJ = tri_col(sl);
      if constexpr (TJ == 0) {
        const int i = 16 * TI + lr;
        if (i < n) col[i] = a[sl];
      }
    });
  }
  __syncthreads();
  int k = 0;
  for (; n - k > kFullN; ++k) {
    // Reflector of column k, formed redundantly (and identically) by every
    // wavefront: v = (x - alpha e_{k+1}) / |x - alpha e_{k+1}|.
    double part = 0.0;
    for (int i = k + 1 + lane; i < n; i += 64) {
      const double x = col[i];
      part = fma(x, x, part);
    }
    const double ss = wave_sum(part);
    const double x0 = col[k + 1];
    const double xn = sqrt(ss);
    const bool noref = xn == 0.0 || ss - x0 * x0 == 0.0;  // already reduced
    const double alpha = x0 >= 0.0 ? -xn : xn;
    const double v0 = x0 - alpha;
    const double inv = noref ? 0.0 : 1.0 / sqrt(ss - x0 * x0 + v0 * v0);
    if (tid == 0) {
      d[k] = 2.0 * col[k];
      e[k] = noref ? x0 : alpha;
    }
    // no reflection (inv = 0) runs the same path with v = 0: p, q and the
    // update vanish and the stored reflector is zero
    const double vi = (tid > k && tid < n) ? inv * (tid == k + 1 ? v0 : col[tid]) : 0.0;
    v[tid] = vi;
    if (tid > k && tid < n) A[tid + (int64_t)k * n] = vi;
    __syncthreads();
    // p = A v (v = 0 outside the trailing block), column tile by column tile:
    // a column tile whose columns are all <= k is frozen (v = p = 0 there) and
    // skipped, which leaves about (n-k)^2/2 elements of work per step.  Lane
    // partials go to LDS, transposed so that thread i sums its row's 32 + 16
    // partials without cross-lane shuffles: rowpart[lc][i] from x v_j,
    // colpart[lr][j] from x v_i.
    double vr[NR], pr[NR];
#pragma unroll
    for (int TI = 0; TI < NR; ++TI) {
      vr[TI] = v[16 * TI + lr];
      pr[TI] = 0.0;
    }
    static_for<0, NC>([&](auto CJ) __attribute__((always_inline)) {
      constexpr int TJ = decltype(CJ)::value;
      if (32 * TJ + 31 > k) {
        const double vj = v[32 * TJ + lc];
        double pc = 0.0;
        static_for<2 * TJ, NR>([&](auto CI) __attribute__((always_inline)) {
          constexpr int TI = decltype(CI)::value;
          constexpr int sl = tri_slots(TI) + TJ;
          const double x = a[sl];
          pr[TI] = fma(x, vj, pr[TI]);
          pc = fma(x, vr[TI], pc);
        });
        colpart[lr * kTriPad + 32 * TJ + lc] = pc;
      }
    });
#pragma unroll
    for (int TI = 0; TI < NR; ++TI) rowpart[lc * kTriPad + 16 * TI + lr] = pr[TI];
    __syncthreads();
    // only partials of live tiles are read: row i > k gets rowpart from its own
    // row tile (written every step) and colpart from column tiles TJ with
    // 32 TJ + 31 >= i > k, all of them live
    double p = 0.0;
    if (tid > k && tid < n) {
      // eight independent partial sums: the loads overlap and the add chain is short
      double ps[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
      for (int r = 0; r < 32; r += 8) {
#pragma unroll
        for (int u = 0; u < 8; ++u) ps[u] += rowpart[(r + u) * kTriPad + tid];
      }
      for (int r = 0; r < 16; r += 8) {
#pragma unroll
        for (int u = 0; u < 8; ++u) ps[u] += colpart[(r + u) * kTriPad + tid];
      }
      p = ((ps[0] + ps[1]) + (ps[2] + ps[3])) + ((ps[4] + ps[5]) + (ps[6] + ps[7]));
    }
    pq[tid] = p;
    __syncthreads();
    // K = v.p, again per wavefront; with q = p - K v,
    // v_i q_j + q_i v_j = v_i p_j + (p_i - 2 K v_i) v_j.
    part = 0.0;
    for (int i = k + 1 + lane; i < n; i += 64) part = fma(v[i], pq[i], part);
    const double K2 = 2.0 * wave_sum(part);
    double rr[NR];
#pragma unroll
    for (int TI = 0; TI < NR; ++TI) rr[TI] = fma(-K2, vr[TI], pq[16 * TI + lr]);
    // A -= 2 (v q^T + q v^T) over the live column tiles
    static_for<0, NC>([&](auto CJ) __attribute__((always_inline)) {
      constexpr int TJ = decltype(CJ)::value;
      if (32 * TJ + 31 > k) {
        const int j = 32 * TJ + lc;
        const double vj = v[j], pj = pq[j];
        const double vjm = -2.0 * vj, pjm = -2.0 * pj;  // strict tiles: two FMAs per element
        static_for<2 * TJ, NR>([&](auto CI) __attribute__((always_inline)) {
          constexpr int TI = decltype(CI)::value;
          constexpr int sl = tri_slots(TI) + TJ;
          const int i = 16 * TI + lr;
          if constexpr (tri_strict(TI, TJ)) {
            a[sl] = fma(rr[TI], vjm, fma(vr[TI], pjm, a[sl]));
          } else {
            const double u = fma(vr[TI], pj, rr[TI] * vj);
            a[sl] -= (i > j ? 2.0 : (i == j ? 1.0 : 0.0)) * u;
          }
        });
      }
    });
    // publish column k+1 for the next step
    const int Tk1 = (k + 1) >> 5, ck1 = (k + 1) & 31;
    if (lc == ck1) {
      static_for<0, NE>([&](auto S) __attribute__((always_inline)) {
        constexpr int sl = decltype(S)::value;
        constexpr int TI = tri_row(sl), TJ = tri_col(sl);
        if (TJ == Tk1) {
          const int i = 16 * TI + lr;
          if (i < n) col[i] = a[sl];
        }
      });
    }
    __syncthreads();
  }
  // the trailing kFullN x kFullN block goes back to A, both triangles with the
  // full diagonal, for tridiag_full.  The indices are opaque copies: addresses
  // shared with the loads at the top would stay live through the loop, in
  // scratch memory.
  int wr = lr, wc = lc;
  asm volatile("" : "+v"(wr), "+v"(wc));
  static_for<0, NE>([&](auto S) __attribute__((always_inline)) {
    constexpr int sl = decltype(S)::value;
    constexpr int TI = tri_row(sl), TJ = tri_col(sl);
    const int i = 16 * TI + wr, j = 32 * TJ + wc;
    if (j >= k && i < n && i >= j) {
      const double x = a[sl];
      if (i > j) {
        A[i + (int64_t)j * n] = x;
        A[j + (int64_t)i * n] = x;
      } else {
        A[i + (int64_t)i * n] = 2.0 * x;
      }
    }
  });
  __syncthreads();
}

// 1 / sqrt(x) for x > 0, finite and not subnormal: the hardware estimate y with
// one third-order correction y (1 + e / 2 + 3 e^2 / 8), e = 1 - x y^2 (within
// 1 ulp; a fraction of the IEEE square root's and division's instructions,
// which sit on the serial chain of a reduction step)
__device__ __forceinline__ double rsqrt_refined(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}

// Sums of R values over the 16 lanes of a DPP row, scattered: on return lane lc
// of the row holds the row's sum of value row16_index<R>(lc).  Four exchange
// stages (lane ^ 15, ^ 7, ^ 2, ^ 1); each of the first three halves the number
// of live values by sending away the one the partner keeps.
template <int CTRL, int M, int NV>
__device__ __forceinline__ void row16_stage(double (&v)[NV], bool hi) {
#pragma unroll
  for (int q = 0; q < (M + 1) / 2; ++q) {
    if (2 * q + 1 < M) {
      const double keep = hi ? v[2 * q + 1] : v[2 * q];
      const double send = hi ? v[2 * q] : v[2 * q + 1];
      v[q] = keep + dpp_permute<CTRL>(send);
    } else {
      v[q] = v[2 * q] + dpp_permute<CTRL>(v[2 * q]);
    }
  }
}
constexpr int half_up(int m) { return (m + 1) / 2; }
template <int R, int NV>
__device__ __forceinline__ double row16_sums(double (&v)[NV], int lc) {
  constexpr int M1 = half_up(R), M2 = half_up(M1), M3 = half_up(M2);
  static_assert(M3 == 1, "at most eight values");
  row16_stage<0x140, R>(v, (lc & 8) != 0);   // row_mirror: lane ^ 15
  row16_stage<0x141, M1>(v, (lc & 4) != 0);  // row_half_mirror: lane ^ 7
  row16_stage<0x4e, M2>(v, (lc & 2) != 0);   // quad_perm [2,3,0,1]: lane ^ 2
  return v[0] + dpp_permute<0xb1>(v[0]);     // quad_perm [1,0,3,2]: lane ^ 1
}
template <int R>
__device__ __forceinline__ int row16_index(int lc) {
  constexpr int M1 = half_up(R), M2 = half_up(M1);
  int q = 0;
  if (M2 > 1) q = (lc & 2) ? 1 : 0;
  if (M1 > 1) q = (2 * q + 1 < M1 && (lc & 4)) ? 2 * q + 1 : 2 * q;
  if (R > 1) q = (2 * q + 1 < R && (lc & 8)) ? 2 * q + 1 : 2 * q;
  return q;
}

// Householder reduction of an n x n symmetric matrix, n <= kFullN, with the
// whole matrix (both triangles) in registers: thread (lr, lc) = (tid / 16,
// tid % 16) of 512 owns the elements (32 TI + lr, 16 TJ + lc), 72 doubles.
// The indices are right-aligned (local index = global + kFullN - n), so that
// the last tiles are always full and one code sequence serves every n.
//
// Holding both triangles doubles the multiply-adds of a triangle, but every
// row of the product then ends inside the 16 lanes of one DPP row: no partial
// sum crosses wavefronts and a step needs two barriers instead of four.
//   1. (column k published in xb) A u is formed row by row; the 16 lanes of a
//      DPP row hold every column of u, so the norm of u and later u.p are row
//      sums too.  Only the entry k+1 of the reflector depends on the norm: its
//      column tile is multiplied last.  p = A u goes to pb.
//   2. (barrier) A -= beta u p^T + (beta p - beta^2 (u.p) u) u^T with
//      H = I - beta u u^T, u unnormalized; the owners of column k+1 publish it
//      (barrier).
// The steps run in twelve phases of 16, phase E with the row and column tiles
// below column 16 E dropped at compile time.
//
// Bound: the latency and instruction issue of one step (LDS round trips, row
// sums, reciprocal square roots, two barriers), about 0.75 us at 122 AOs.
// Measured against the triangle with four barriers a step (and the last 64
// columns on one wavefront): k_tridiag 233 -> 95 us for one system of 122 AOs,
// 648 -> 397 us a round for 512 systems of 14-235 AOs.
constexpr int kFullTI = kFullN / 32, kFullTJ = kFullN / 16;
constexpr double kTinyNorm = 1e-290;  // squared norms below it: already reduced

// column L of the local matrix (L in column tile TJ) goes to xb, zero above the
// subdiagonal, and its diagonal entry to d
template <int TJ>
__device__ __forceinline__ void full_publish(const double (&a)[kFullTI][kFullTJ], int lr, int lc, int L, double* dL,
                                             double* xb) {
  if (lc == (L & 15)) {
    static_for<TJ / 2, kFullTI>([&](auto CI) __attribute__((always_inline)) {
      constexpr int TI = decltype(CI)::value;
      const int row = 32 * TI + lr;
      if constexpr (TI == TJ / 2) {
        xb[row] = row > L ? a[TI][TJ] : 0.0;
        if (row == L) *dL = a[TI][TJ];
      } else {
        xb[row] = a[TI][TJ];
      }
    });
  }
}

// the reflectors k with k + 1 in column tile E
template <int E>
__device__ __forceinline__ void full_phase(double (&a)[kFullTI][kFullTJ], int& k, double* A, int64_t ld, int off,
                                           double* d, double* e, double* xb, double* pb) {
  constexpr int T0 = E / 2, R = kFullTI - T0;  // live row tiles
  const int tid = threadIdx.x, lc = tid & 15, lr = tid >> 4;
  const bool first = __builtin_amdgcn_readfirstlane(tid) < kFullN;  // a wavefront with rows tid < kFullN
  const int prow = 32 * (T0 + row16_index<R>(lc)) + lr;  // the row whose sum this lane ends with
  for (; k < 16 * E + 15 && k + 2 < kFullN; ++k) {
    double uj[kFullTJ], ui[kFullTI], p[R];
    const double x0 = xb[k + 1];
#pragma unroll
    for (int TJ = E; TJ < kFullTJ; ++TJ) uj[TJ] = xb[16 * TJ + lc];
#pragma unroll
    for (int TI = T0; TI < kFullTI; ++TI) ui[TI] = xb[32 * TI + lr];
    const bool at_j = 16 * E + lc == k + 1, at_i = 32 * T0 + lr == k + 1;
    const double xe = at_j ? 0.0 : uj[E];
    double part = xe * xe;
#pragma unroll
    for (int TJ = E + 1; TJ < kFullTJ; ++TJ) part = fma(uj[TJ], uj[TJ], part);
    const double tail = row16_sum(part);
    const double ss = fma(x0, x0, tail);
    const bool noref = tail == 0.0 || ss < kTinyNorm;  // already reduced: inv = beta = 0
    const double xn = ss * rsqrt_refined(fmax(ss, kTinyNorm));
    const double alpha = x0 >= 0.0 ? -xn : xn;
    const double v0 = x0 - alpha;
#pragma unroll
    for (int q = 0; q < R; ++q) p[q] = 0.0;
    static_for<E + 1, kFullTJ>([&](auto CJ) __attribute__((always_inline)) {
      constexpr int TJ = decltype(CJ)::value;
#pragma unroll
      for (int q = 0; q < R; ++q) p[q] = fma(a[T0 + q][TJ], uj[TJ], p[q]);
    });
    uj[E] = at_j ? v0 : uj[E];
    ui[T0] = at_i ? v0 : ui[T0];
#pragma unroll
    for (int q = 0; q < R; ++q) p[q] = fma(a[T0 + q][E], uj[E], p[q]);
    pb[prow] = row16_sums<R>(p, lc);
    // the unit reflector for the back-transformation (zero for no reflection)
    const double inv = noref ? 0.0 : rsqrt_refined(fmax(fma(v0, v0, tail), kTinyNorm));
    if (first) {
      if (tid > k) A[(tid - off) + (int64_t)(k - off) * ld] = (tid == k + 1 ? v0 : xb[tid]) * inv;
      if (tid == 0) e[k - off] = noref ? x0 : alpha;
    }
    const double beta = 2.0 * (inv * inv);
    __syncthreads();
    double pj[kFullTJ], pi[kFullTI];
#pragma unroll
    for (int TJ = E; TJ < kFullTJ; ++TJ) pj[TJ] = pb[16 * TJ + lc];
#pragma unroll
    for (int TI = T0; TI < kFullTI; ++TI) pi[TI] = pb[32 * TI + lr];
    double kp = uj[E] * pj[E];
#pragma unroll
    for (int TJ = E + 1; TJ < kFullTJ; ++TJ) kp = fma(uj[TJ], pj[TJ], kp);
    const double bK = beta * row16_sum(kp);
    double bu[kFullTI], rf[kFullTI];
#pragma unroll
    for (int TI = T0; TI < kFullTI; ++TI) {
      bu[TI] = -beta * ui[TI];
      static_for<E, kFullTJ>([&](auto CJ) __attribute__((always_inline)) {
        constexpr int TJ = decltype(CJ)::value;
        a[TI][TJ] = fma(bu[TI], pj[TJ], a[TI][TJ]);
      });
    }
#pragma unroll
    for (int TI = T0; TI < kFullTI; ++TI) {
      rf[TI] = -beta * fma(-bK, ui[TI], pi[TI]);
      static_for<E, kFullTJ>([&](auto CJ) __attribute__((always_inline)) {
        constexpr int TJ = decltype(CJ)::value;
        a[TI][TJ] = fma(rf[TI], uj[TJ], a[TI][TJ]);
      });
    }
    full_publish<E>(a, lr, lc, k + 1, d + (k + 1 - off), xb);
    __syncthreads();
  }
}

// A (leading dimension ld) is read whole; on return its column k holds the unit
// reflector k below the diagonal.  xb and pb hold kFullN doubles.
__device__ __forceinline__ void tridiag_full(double* A, int64_t ld, int n, double* d, double* e, double* xb,
                                             double* pb) {
  const int tid = threadIdx.x, lc = tid & 15, lr = tid >> 4;
  const int off = kFullN - n;
  double a[kFullTI][kFullTJ];
  static_for<0, kFullTI>([&](auto CI) __attribute__((always_inline)) {
    constexpr int TI = decltype(CI)::value;
    const int row = 32 * TI + lr - off;
#pragma unroll
    for (int TJ = 0; TJ < kFullTJ; ++TJ) a[TI][TJ] = 0.0;
    if (32 * TI + 31 >= off) {  // small systems: only the tiles they reach
      static_for<0, kFullTJ>([&](auto CJ) __attribute__((always_inline)) {
        constexpr int TJ = decltype(CJ)::value;
        const int col = 16 * TJ + lc - off;
        if (row >= 0 && col >= 0) a[TI][TJ] = A[col + row * ld];
      });
    }
    // keep one row tile of loads in flight (address registers would spill the matrix)
    __builtin_amdgcn_sched_barrier(0);
  });
  // every wavefront's loads are done before the first reflector is stored to A
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (tid < kFullN) {
    xb[tid] = 0.0;
    pb[tid] = 0.0;
  }
  __syncthreads();
  static_for<0, kFullTJ>([&](auto CJ) __attribute__((always_inline)) {
    constexpr int TJ = decltype(CJ)::value;
    if (TJ == off >> 4) full_publish<TJ>(a, lr, lc, off, d, xb);
  });
  __syncthreads();
  int k = off;
  static_for<0, kFullTJ>([&](auto CE) __attribute__((always_inline)) {
    full_phase<decltype(CE)::value>(a, k, A, ld, off, d, e, xb, pb);
  });
  if (lr == 31 && lc == 15) d[n - 1] = a[kFullTI - 1][kFullTJ - 1];
  if (tid == 0) {
    if (n >= 2) e[n - 2] = xb[kFullN - 1];
    e[n - 1] = 0.0;
  }
}

// Householder reduction by a team of workgroups, one system of 257 .. kTeamN
// AOs, down to its last kFullN columns (k_tridiag finishes those).
//
// The whole matrix, both triangles, sits in the team's registers: member g of G
// holds the rows i = g (mod G), its wavefront w the rows (8 q + w) G + g, q <
// team_rows(n), lane l the columns l + 64 t.  A step k on every member:
//   pass     A -= u r^T + r u^T of step k - 1 and p = A u_k on the member's
//            rows, one sweep over the registers (u, r from LDS); row sums stay
//            inside a wavefront;
//   exchange the rows' p_i, and row k + 1 of A from its owner, through a ring
//            of buffers in global memory; every member reads all of both;
//   vectors  r = beta (p - beta (u.p) u / 2) and the next column
//            A_{k+1, :} - u_{k+1} r - r_{k+1} u, formed by every member for
//            itself (bit-identical: same data, same order).
// So a step has one exchange and two block barriers, no panels and no pass over
// memory.
//
// The exchanged words validate themselves: a buffer starts out filled with
// kTeamEmpty (a NaN no arithmetic produces) and a reader spins on each word
// until it is something else.  Slot k % kTeamRing is emptied in step k + 1, when
// every member has published that step and so has read slot k; it is written
// again in step k + kTeamRing, a row's slot by another member than the one that
// emptied it.  Emptying comes before that write: the emptying stores are waited
// for before the first barrier of step k + 2; behind it the member publishes p of
// step k + 3 (every member owns one of the last kFullN rows, so it always has one
// to publish); and the next writer has read that p, from every member, before it
// goes on to step k + kTeamRing.  The words are agent-scope stores, complete at the level
// that every member's loads read when the wait for them returns.
//
// Waiting is safe: no member writes anything before all G have met at the gate,
// so from then on every partner is resident and runs.  Members that do not all
// arrive within kTeamWaitTicks (the chip is held by something else) close the
// gate together and leave; k_tridiag_solo then does the same arithmetic.  After
// one such failure the call's teams wait kTeamRetryTicks only: above the 7 ms for
// which a running team can hold a partner's CU, and a call of ten rounds on a chip
// that stays held loses 0.4 s to waiting instead of 2 s.  A team larger than the
// device finds its gate closed from the start.  The spins are bounded too; one that
// runs out fails the system (status 8).
//
// Bound: the latency of a step, 4.1 us at 482 AOs (8 members) and 5.1 us at
// 1142 (36), most of it the exchange through memory.  Measured against one
// workgroup per system with panels of 16 reflectors (k_tridiag_blocked): 9.0 ->
// 1.2 + 0.4 ms a round for 14 systems of 258-482 AOs, 111 -> 4.8 ms at 1142.
// Members on one XCD (every eighth block) were 10 % slower than neighbours.
constexpr int kTeamN = 1280;
constexpr int kTeamRing = 8;
constexpr int team_own(int tiles) { return (64 * tiles + 511) / 512; }  // vector entries per thread
constexpr unsigned long long kTeamEmpty = 0xfff7a5a5c3c3e1e1ull;
constexpr long long kTeamWaitTicks = 20000000;  // 100 MHz counter: 0.2 s
constexpr long long kTeamRetryTicks = 2000000;
constexpr int kTeamSpins = 1 << 22;
constexpr unsigned kTeamClosed = 1u << 30;
constexpr unsigned kTeamNever = 1u << 29;  // a start value from which no count reaches G
// Rows of a wavefront: as many as about 80 doubles a lane hold, tiles of 64 columns
// for the largest n of the class.  Smaller teams leave CUs to other systems: with
// four rows for every n the teams of 256 systems of 482 AOs took 239 ms of a call
// (eleven rounds) and with eight 108, where one workgroup per system took 142; 256
// of 650 AOs 515 and 316 (six rows), 319 with one workgroup per system.
__host__ __device__ constexpr int team_rows(int n) { return n <= 640 ? 8 : n <= 832 ? 6 : n <= 1024 ? 5 : 4; }
__host__ __device__ constexpr int team_size(int n) { return (n + 8 * team_rows(n) - 1) / (8 * team_rows(n)); }
static_assert(team_size(kTeamN) <= kFullN && team_size(640) <= kFullN, "a row of the last kFullN for every member");
// f(rows of a wavefront, column tiles) of n's class
template <typename F>
__device__ __forceinline__ void team_class(int n, F&& f) {
  if (n <= 640)
    f(std::integral_constant<int, 8>{}, std::integral_constant<int, 10>{});
  else if (n <= 832)
    f(std::integral_constant<int, 6>{}, std::integral_constant<int, 13>{});
  else if (n <= 1024)
    f(std::integral_constant<int, 5>{}, std::integral_constant<int, 16>{});
  else
    f(std::integral_constant<int, 4>{}, std::integral_constant<int, 20>{});
}

// A system's exchange area (in the eigenvector matrix, free until the
// eigenvectors are written): p ring, row ring, then the gate and done words.
__device__ __forceinline__ unsigned* team_words(double* Z, int n) {
  return reinterpret_cast<unsigned*>(Z + 2 * kTeamRing * (int64_t)n);
}

// One step's arithmetic outside the product, the same instructions for a team and
// for k_tridiag_solo (contraction off: each kernel would otherwise fuse as its
// surroundings suggest), so that both leave the same bits.
struct TeamStep {
  double v0, alpha, inv, beta;  // noref (already reduced): inv = beta = 0
  bool noref;
};
__device__ __forceinline__ TeamStep team_step(const double* redn, double x0) {
#pragma clang fp contract(off)
  TeamStep z;
  const double tail = ((redn[0] + redn[1]) + (redn[2] + redn[3])) + ((redn[4] + redn[5]) + (redn[6] + redn[7]));
  const double ss = fma(x0, x0, tail);
  z.noref = tail == 0.0 || ss < kTinyNorm;
  const double xn = ss * rsqrt_refined(fmax(ss, kTinyNorm));
  z.alpha = x0 >= 0.0 ? -xn : xn;
  z.v0 = x0 - z.alpha;
  z.inv = z.noref ? 0.0 : rsqrt_refined(fmax(fma(z.v0, z.v0, tail), kTinyNorm));
  z.beta = 2.0 * (z.inv * z.inv);
  return z;
}
// Column 0: this thread's entries xo, the vectors and the norm's partial sums.
template <int TILES>
__device__ __forceinline__ void team_first(const double* A, int off, bool keeps_d, double* d,
                                           double (&xo)[team_own(TILES)], double* x, double* u, double* r,
                                           double* redn) {
  const int tid = threadIdx.x;
  double part = 0.0;
#pragma unroll
  for (int q = 0; q < team_own(TILES); ++q) {
    const int L = tid + 512 * q;
    double v = 0.0;
    if (L >= off && L < 64 * TILES) v = A[L - off];
    if (L == off && keeps_d) d[0] = v;
    xo[q] = L > off ? v : 0.0;
    if (L > off + 1) part = fma(xo[q], xo[q], part);
    if (L < 64 * TILES) {
      x[L] = xo[q];
      u[L] = 0.0;
      r[L] = 0.0;
    }
  }
  part = wave_sum(part);
  if ((tid & 63) == 0) redn[tid >> 6] = part;
}
// r of step K and the next column from this thread's entries of p and row k + 1;
// x: the vector of this step (its entry K + 1 becomes v0), xn: the next one.
// Returns the next column's diagonal on the thread that holds it.
template <int TILES>
__device__ __forceinline__ void team_vectors(const TeamStep& z, int K, const double* redk, double p1,
                                             const double (&po)[team_own(TILES)], const double (&ro)[team_own(TILES)],
                                             double (&xo)[team_own(TILES)], double* x, double* xn, double* rb,
                                             double* redn, double* dnext) {
#pragma clang fp contract(off)
  const int tid = threadIdx.x;
  const double hK = 0.5 * z.beta *
                    (((redk[0] + redk[1]) + (redk[2] + redk[3])) + ((redk[4] + redk[5]) + (redk[6] + redk[7])));
  const double r1 = z.beta * fma(-hK, z.v0, p1);
  double part = 0.0;
#pragma unroll
  for (int q = 0; q < team_own(TILES); ++q) {
    const int L = tid + 512 * q;
    const double r = z.beta * fma(-hK, xo[q], po[q]);
    const double y = fma(-z.v0, r, fma(-r1, xo[q], ro[q]));
    if (L == K + 1) {
      if (dnext) *dnext = y;
      x[L] = z.v0;
    }
    xo[q] = L > K + 1 ? y : 0.0;
    if (L > K + 2) part = fma(xo[q], xo[q], part);
    if (L < 64 * TILES) {
      rb[L] = r;
      xn[L] = xo[q];
    }
  }
  part = wave_sum(part);
  if ((tid & 63) == 0) redn[tid >> 6] = part;
}

__global__ __launch_bounds__(256) void k_team_init(Topo t, const int* order, const unsigned char* active,
                                                   double* Zall, int cus, unsigned start) {
  const int s = order[blockIdx.x];
  if (active && !active[s]) return;
  const int n = t.ao_off[s + 1] - t.ao_off[s];
  double* Z = Zall + t.mat_off[s];
  for (int i = threadIdx.x; i < 2 * kTeamRing * n; i += 256) Z[i] = __longlong_as_double((long long)kTeamEmpty);
  if (threadIdx.x < 2) team_words(Z, n)[threadIdx.x] = threadIdx.x != 0 ? 0u : team_size(n) > cus ? kTeamClosed : start;
}

__device__ __forceinline__ void team_put(double* p, double x) {
  unsigned long long b = (unsigned long long)__double_as_longlong(x);
  if (b == kTeamEmpty) b = 0x7ff8000000000000ull;
  __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void team_clear(double* p) {
  __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), kTeamEmpty, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long team_peek(const double* p) {
  return __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
}

// member g of G; xb: u of this step and of the last one, rb: r of the last step
template <int ROWS, int TILES>
__device__ __forceinline__ void team_member(int n, int G, int g, double* A, double* d, double* e, double* ring_p,
                                            int* status, int* failed, double (&xb)[2][kTeamN],
                                            double (&rb)[kTeamN]) {
  constexpr int N = 64 * TILES, OWN = team_own(TILES);
  double* ring_r = ring_p + (int64_t)kTeamRing * n;
  unsigned* gate = team_words(ring_p, n);
  __shared__ double redn[8], redk[8];
  __shared__ double sh_p;  // p at row k + 1
  __shared__ int sh_bad;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int off = N - n;  // local index = global + off: the last tiles are always full
  // the member's rows and column 0 (both read before the gate: from there on
  // the owner of row k overwrites that row with its reflector)
  double a[ROWS][TILES];
#pragma unroll
  for (int q = 0; q < ROWS; ++q) {
    const int i = (8 * q + w) * G + g;
    static_for<0, TILES>([&](auto CT) __attribute__((always_inline)) {
      constexpr int T = decltype(CT)::value;
      const int c = 64 * T + lane - off;
      a[q][T] = 0.0;
      if (i < n && c >= 0) a[q][T] = A[(int64_t)i * n + c];
    });
    __builtin_amdgcn_sched_barrier(0);
  }
  double xo[OWN];  // this thread's entries L = tid + 512 q of the current column
  team_first<TILES>(A, off, g == 0, d, xo, xb[0], xb[1], rb, redn);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  // the gate
  if (tid == 0) {
    unsigned old = __hip_atomic_fetch_add(gate, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    int closed = (old & kTeamClosed) != 0;
    const long long t0 = wall_clock64();
    old += 1;
    while (!closed && (old & ~kTeamClosed) != (unsigned)G) {
      __builtin_amdgcn_s_sleep(2);
      old = __hip_atomic_load(gate, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      closed = (old & kTeamClosed) != 0;
      const long long limit = __hip_atomic_load(failed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ? kTeamRetryTicks
                                                                                                    : kTeamWaitTicks;
      if (!closed && (old & ~kTeamClosed) != (unsigned)G && wall_clock64() - t0 > limit) {
        unsigned want = old;
        if (__hip_atomic_compare_exchange_strong(gate, &want, old | kTeamClosed, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT)) {
          closed = 1;
          __hip_atomic_store(failed, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
    }
    sh_bad = closed;
  }
  __syncthreads();
  if (sh_bad) return;
  const int kend = n - kFullN;  // columns reduced here
  int cur = 0;
  int k = 0;
  for (;; ++k) {
    const int K = k + off, slot = k & (kTeamRing - 1);
    double* pk = ring_p + (int64_t)slot * n;
    double* rk = ring_r + (int64_t)slot * n;
    const TeamStep z = team_step(redn, xb[cur][K + 1]);
    // one sweep over the registers: the pending update of step k - 1 (zero in
    // step 0) and p = A u.  Finished rows ride along: their entries of u and r
    // keep them finite, and the exchange hides them.
    double p[ROWS], ur[ROWS], rr[ROWS];
#pragma unroll
    for (int q = 0; q < ROWS; ++q) {
      const int L = min((8 * q + w) * G + g + off, N - 1);
      ur[q] = xb[cur ^ 1][L];
      rr[q] = rb[L];
      p[q] = 0.0;
    }
    static_for<0, TILES>([&](auto CT) __attribute__((always_inline)) {
      constexpr int T = decltype(CT)::value;
      if (64 * T + 63 >= K) {  // a column tile with a live column
        const int L = 64 * T + lane;
        const double x = L == K + 1 ? z.v0 : xb[cur][L], u = xb[cur ^ 1][L], r = rb[L];
#pragma unroll
        for (int q = 0; q < ROWS; ++q) {
          a[q][T] = fma(-ur[q], r, fma(-rr[q], u, a[q][T]));
          p[q] = fma(a[q][T], x, p[q]);
        }
      }
    });
    if (k == kend) break;  // the last update is in: the trailing block is done
    // publish row k + 1 and the rows' p
    // (opaque lane: addresses kept from step to step would live in scratch)
    int ln = lane;
    asm volatile("" : "+v"(ln));
    double* rl0 = rk + (ln - off);  // this lane's column of tile 0
#pragma unroll
    for (int q = 0; q < ROWS; ++q) {
      if ((8 * q + w) * G + g == k + 1) {
        static_for<0, TILES>([&](auto CT) __attribute__((always_inline)) {
          constexpr int T = decltype(CT)::value;
          if (64 * T + ln > K) team_put(rl0 + 64 * T, a[q][T]);
        });
      }
    }
    {
      double r = row16_sums<ROWS>(p, lane & 15);
      r += __shfl_xor(r, 16, 64);
      r += __shfl_xor(r, 32, 64);
      const int i = (8 * row16_index<ROWS>(lane & 15) + w) * G + g;
      if (lane < 16 && (lane & 1) == 0 && i > k && i < n) team_put(pk + i, r);
    }
    if (g == k % G) {  // this member keeps column k's unit reflector (zero for no reflection)
#pragma unroll
      for (int q = 0; q < OWN; ++q) {
        const int L = tid + 512 * q;
        if (L > K && L < N) A[(L - off) + (int64_t)k * n] = (L == K + 1 ? z.v0 : xo[q]) * z.inv;
      }
      if (tid == 0) e[k] = z.noref ? xb[cur][K + 1] : z.alpha;
    }
    // everybody's p and the row
    double po[OWN], ro[OWN];
    {
      int bad = 0;
      unsigned long long bp[OWN], br[OWN];
#pragma unroll
      for (int q = 0; q < OWN; ++q) {
        bp[q] = 0;
        br[q] = 0;
      }
      for (int spin = 0;; ++spin) {
        bool wait = false;
#pragma unroll
        for (int q = 0; q < OWN; ++q) {
          const int L = tid + 512 * q;
          if (L > K && L < N) {
            bp[q] = team_peek(pk + (L - off));
            br[q] = team_peek(rk + (L - off));
          }
        }
#pragma unroll
        for (int q = 0; q < OWN; ++q) wait = wait || bp[q] == kTeamEmpty || br[q] == kTeamEmpty;
        if (!wait) break;
        if (spin >= kTeamSpins) {
          bad = 1;
          break;
        }
      }
      if (bad) sh_bad = 1;
      double kp = 0.0;
#pragma unroll
      for (int q = 0; q < OWN; ++q) {
        const int L = tid + 512 * q;
        po[q] = __longlong_as_double((long long)bp[q]);  // 0 where L <= K
        ro[q] = __longlong_as_double((long long)br[q]);
        if (L == K + 1) {
          xo[q] = z.v0;
          sh_p = po[q];
        }
        kp = fma(xo[q], po[q], kp);
      }
      kp = wave_sum(kp);
      if (lane == 0) redk[w] = kp;
    }
    // the stores that emptied a slot in the last step are done (nothing to wait
    // for: they were issued a whole exchange ago)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (sh_bad) {
      if (tid == 0) *status = 8;
      return;
    }
    team_vectors<TILES>(z, K, redk, sh_p, po, ro, xo, xb[cur], xb[cur ^ 1], rb, redn,
                 g == 0 && k + 1 < kend ? d + k + 1 : nullptr);
    // every member has published step k, so it has read step k - 1: empty that slot
    if (k > 0) {
      double* pl = ring_p + (int64_t)((k - 1) & (kTeamRing - 1)) * n;
      double* rl = ring_r + (int64_t)((k - 1) & (kTeamRing - 1)) * n;
      if (lane < ROWS) {
        const int i = (8 * lane + w) * G + g;
        if (i >= k && i < n) team_clear(pl + i);
      }
      if (g == k % G && w == (k / G) % 8)
        for (int c = k + lane; c < n; c += 64) team_clear(rl + c);
    }
    __syncthreads();
    cur ^= 1;
  }
  // the trailing block, both triangles, for k_tridiag
  int ln = lane;
  asm volatile("" : "+v"(ln));
#pragma unroll
  for (int q = 0; q < ROWS; ++q) {
    const int i = (8 * q + w) * G + g;
    if (i >= kend && i < n)
      static_for<0, TILES>([&](auto CT) __attribute__((always_inline)) {
        constexpr int T = decltype(CT)::value;
        // columns >= kend are the last kFullN local ones
        if constexpr (64 * T >= N - kFullN) A[(int64_t)i * n + (64 * T + ln - off)] = a[q][T];
      });
  }
  if (g == 0 && tid == 0) gate[1] = 1u;  // done
}

__global__ __launch_bounds__(512) void k_tridiag_team(Topo t, const int* order, double* Aall, double* dall,
                                                      double* eall, double* Zall, const unsigned char* active,
                                                      SysState* st, int* failed) {
  const int s = order[blockIdx.y];
  if (active && !active[s]) return;
  const int n = t.ao_off[s + 1] - t.ao_off[s];
  const int G = team_size(n), g = blockIdx.x;
  if (g >= G) return;
  __shared__ double xb[2][kTeamN], rb[kTeamN];
  const int64_t mo = t.mat_off[s], o = t.ao_off[s];
  team_class(n, [&](auto R, auto T) __attribute__((always_inline)) {
    team_member<decltype(R)::value, decltype(T)::value>(n, G, g, Aall + mo, dall + o, eall + o, Zall + mo,
                                                        &st[s].status, failed, xb, rb);
  });
}

// The team's reduction by one workgroup, for systems whose team left at the gate:
// the rows stay in A, a wavefront per row, and every sum is formed from the same
// terms in the same order, so that the results do not depend on whether a team
// could assemble.  Bound: the sweep over the trailing block (16 n^2 bytes a step
// through one CU): 205 ms at 1280 AOs (240 with four tiles in flight instead of
// ten), where the team takes 6 ms.
template <int TILES>
__device__ __forceinline__ void team_solo(int n, double* A, double* d, double* e, double (&xb)[2][kTeamN],
                                          double (&rb)[kTeamN], double (&pb)[kTeamN]) {
  constexpr int N = 64 * TILES, OWN = team_own(TILES);
  __shared__ double redn[8], redk[8];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int off = N - n;
  double xo[OWN];
  team_first<TILES>(A, off, true, d, xo, xb[0], xb[1], rb, redn);
  __syncthreads();
  const int kend = n - kFullN;
  int cur = 0;
  for (int k = 0;; ++k) {
    const int K = k + off;
    const TeamStep z = team_step(redn, xb[cur][K + 1]);
    // the pending update of step k - 1 and p = A u: rows past k (all that is left
    // of the trailing block after the last column), columns from K's tile on
    const int first = k < kend ? k + 1 : k, T0 = K >> 6;
    for (int i = first + ((w - first) & 7); i < n; i += 8) {
      const double ur = xb[cur ^ 1][i + off], rr = rb[i + off];
      double* row = A + (int64_t)i * n;
      double p[1] = {0.0};
      auto sweep = [&](auto U, int T) __attribute__((always_inline)) {
        constexpr int NU = decltype(U)::value;
        double a[NU];
#pragma unroll
        for (int v = 0; v < NU; ++v) {
          const int c = 64 * (T + v) + lane - off;
          a[v] = c >= 0 ? row[c] : 0.0;
        }
#pragma unroll
        for (int v = 0; v < NU; ++v) {
          const int L = 64 * (T + v) + lane;
          const double x = L == K + 1 ? z.v0 : xb[cur][L], u = xb[cur ^ 1][L], r = rb[L];
          a[v] = fma(-ur, r, fma(-rr, u, a[v]));
          p[0] = fma(a[v], x, p[0]);
          if (L >= off) row[L - off] = a[v];
        }
      };
      int T = T0;
      for (; T + 10 <= TILES; T += 10) sweep(std::integral_constant<int, 10>{}, T);
      for (; T + 4 <= TILES; T += 4) sweep(std::integral_constant<int, 4>{}, T);
      for (; T < TILES; ++T) sweep(std::integral_constant<int, 1>{}, T);
      double r = row16_sums<1>(p, lane & 15);
      r += __shfl_xor(r, 16, 64);
      r += __shfl_xor(r, 32, 64);
      if (lane == 0) pb[i + off] = r;
    }
    if (k == kend) break;
    __syncthreads();
    double po[OWN], ro[OWN], kp = 0.0;
#pragma unroll
    for (int q = 0; q < OWN; ++q) {
      const int L = tid + 512 * q;
      const bool live = L > K && L < N;
      po[q] = live ? pb[L] : 0.0;
      ro[q] = live ? A[(int64_t)(k + 1) * n + (L - off)] : 0.0;
      if (live) A[(L - off) + (int64_t)k * n] = (L == K + 1 ? z.v0 : xo[q]) * z.inv;
      if (L == K + 1) xo[q] = z.v0;
      kp = fma(xo[q], po[q], kp);
    }
    if (tid == 0) e[k] = z.noref ? xb[cur][K + 1] : z.alpha;
    kp = wave_sum(kp);
    if (lane == 0) redk[w] = kp;
    __syncthreads();
    team_vectors<TILES>(z, K, redk, pb[K + 1], po, ro, xo, xb[cur], xb[cur ^ 1], rb, redn,
                 k + 1 < kend ? d + k + 1 : nullptr);
    __syncthreads();
    cur ^= 1;
  }
}

__global__ __launch_bounds__(512) void k_tridiag_solo(Topo t, const int* order, double* Aall, double* dall,
                                                      double* eall, double* Zall, const unsigned char* active) {
  const int s = order[blockIdx.x];
  if (active && !active[s]) return;
  const int n = t.ao_off[s + 1] - t.ao_off[s];
  unsigned* words = team_words(Zall + t.mat_off[s], n);
  if (words[1] != 0u) return;  // reduced by its team
  __shared__ double xb[2][kTeamN], rb[kTeamN], pb[kTeamN];
  const int64_t mo = t.mat_off[s], o = t.ao_off[s];
  team_class(n, [&](auto, auto T) __attribute__((always_inline)) {
    team_solo<decltype(T)::value>(n, Aall + mo, dall + o, eall + o, xb, rb, pb);
  });
  if (threadIdx.x == 0) words[1] = 1u;
}

// The back-transformation applies the reflectors in compact WY blocks of
// kWyBlock:  H_{k_15} ... H_{k_0} = I - V T V^T,  V = [v_{k_0} .. v_{k_15}],
// k_u = n-3 - 16 ch - u, unit v, T lower triangular with
//   T_mm = 2,  T_mc = -2 sum_{l=c}^{m-1} (v_m . v_l) T_lc  (c < m),
// the inverse of 1/2 on the diagonal and the inner products below it.  Block
// ch's entries below the diagonal sit packed by rows at wy_offset + 120 ch
// (row m at m (m - 1) / 2); the last block holds the rows it has.  A system
// needs at most 7.5 n doubles.
constexpr int kWyBlock = 16;  // reflectors per WY block, one matrix-core tile
constexpr int kWyPacked = kWyBlock * (kWyBlock - 1) / 2;
constexpr int kWyPerAO = 8, kWyPerSys = 64;  // doubles reserved
__device__ __forceinline__ int64_t wy_offset(const Topo& t, int s) {
  return (int64_t)kWyPerAO * t.ao_off[s] + (int64_t)kWyPerSys * s;
}

// T factor of block ch by one wavefront: the inner products V^T V on the matrix
// cores (both operands of a step are the same registers), then lane c < 16 runs
// the recurrence of column c.  g: 256 doubles of LDS of this wavefront's own.
__device__ __forceinline__ void wy_factor(const double* A, int n, int ch, double* Ts, double* g) {
  const int lane = threadIdx.x & 63, l16 = lane & 15, lk = lane >> 4;
  const int kb = n - 3 - kWyBlock * ch, cnt = min(kWyBlock, kb + 1);
  const int ku = kb - l16;  // this lane's reflector
  const double* v = A + (int64_t)max(ku, 0) * n;
  mfma_d4 acc[2] = {mfma_d4{0.0, 0.0, 0.0, 0.0}, mfma_d4{0.0, 0.0, 0.0, 0.0}};
  for (int r0 = max(kb - (kWyBlock - 1), 0) + 1; r0 < n; r0 += 32) {
    double x[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) x[q] = v[min(r0 + 4 * q + lk, n - 1)];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int r = r0 + 4 * q + lk;
      const double xm = (ku >= 0 && r > ku && r < n) ? x[q] : 0.0;
      acc[q & 1] = mfma_16x16x4(xm, xm, acc[q & 1]);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) g[(lk + 4 * r) * kWyBlock + l16] = acc[0][r] + acc[1][r];
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  if (lane < kWyBlock) {
    double* To = Ts + (int64_t)kWyPacked * ch;
    double tc[kWyBlock];
#pragma unroll
    for (int m = 0; m < kWyBlock; ++m) {
      double s0 = 0.0, s1 = 0.0;  // tc[l] = 0 for l < c
#pragma unroll
      for (int l = 0; l < m; ++l) {
        if (l & 1) s1 = fma(g[m * kWyBlock + l], tc[l], s1);
        else s0 = fma(g[m * kWyBlock + l], tc[l], s0);
      }
      tc[m] = m == lane ? 2.0 : -2.0 * (s0 + s1);
      if (m > lane && m < cnt) To[m * (m - 1) / 2 + lane] = tc[m];
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// n <= 256, 512 threads per system (two waves per SIMD, 256 VGPRs per thread):
// the columns before the last kFullN from the triangle in registers, the rest
// with both triangles.  n > 256: the last kFullN columns of the systems that
// k_tridiag_team or k_tridiag_solo has reduced to them.
__global__ __launch_bounds__(512) void k_tridiag(Topo t, const int* order, double* Aall, double* dall,
                                                 double* eall, double* Tall, double* Zall,
                                                 const unsigned char* active) {
  const int s = order[blockIdx.x];
  if (active && !active[s]) return;
  const int n = t.ao_off[s + 1] - t.ao_off[s];
  double* A = Aall + t.mat_off[s];  // column-major view of the symmetric matrix
  double* d = dall + t.ao_off[s];
  double* e = eall + t.ao_off[s];
  __shared__ double v[512];
  __shared__ double pq[512];
  __shared__ double col[512];  // published column of the triangle
  __shared__ double rowpart[32 * kTriPad];
  __shared__ double colpart[16 * kTriPad];
  if (n > 256 && team_words(Zall + t.mat_off[s], n)[1] == 0u) return;
  int k0 = 0;
  if (n > 256) {
    k0 = n - kFullN;
  } else if (n > kFullN) {
    tridiag_registers<16>(A, n, d, e, v, col, pq, rowpart, colpart);
    k0 = n - kFullN;
  }
  tridiag_full(A + k0 + (int64_t)k0 * n, n, n - k0, d + k0, e + k0, v, pq);
  if (n > 256) return;
  // WY factors for the back-transformation; the stored reflectors must be
  // visible to the whole block first
  __syncthreads();
  const int wv = threadIdx.x >> 6;
  for (int ch = wv; kWyBlock * ch < n - 2; ch += 8)
    wy_factor(A, n, ch, Tall + wy_offset(t, s), rowpart + 256 * wv);
}

// n > kTeamN: the blocked reduction, one 512-thread block per system; W is
// per-system n x n scratch, the work vectors sit in the system's slice of `big`.
__global__ __launch_bounds__(512) void k_tridiag_blocked(Topo t, const int* order, double* Aall,
                                                         double* dall, double* eall, double* Wall,
                                                         const unsigned char* active, double* big) {
  const int s = order[blockIdx.x];
  if (active && !active[s]) return;
  const int n = t.ao_off[s + 1] - t.ao_off[s];
  static_assert(kTriPanel % 4 == 0, "panel in K steps of 4");
  __shared__ double red[16];
  __shared__ double bc[2];
  // 2 n + 8 ldp + ldp + 4 kTriPanel <= kBigPerAO n + kBigPerSys doubles
  const int ldp = (n + 63) & ~63;
  double* v = big + big_offset(t, s);
  double* pq = v + n;
  double* part = pq + n;
  double* aux = part + 8 * ldp;
  tridiag_blocked(Aall + t.mat_off[s], Wall + t.mat_off[s], n, dall + t.ao_off[s], eall + t.ao_off[s], v, pq, part,
                  aux, red, bc);
}

// Overlap Cholesky S = L L^T (L column-major into `L`) and X = L^{-T} (row-major,
// upper triangular, into `Xm`) with the lower triangle in registers (same
// 16 x 32 tile layout as tridiag_registers, 512 threads, n <= 16 NR):
//   factorization  per column k: the owners broadcast column k through LDS, the
//                  trailing lower triangle takes the rank-1 update l l^T / l_kk;
//   inverse        Gauss-Jordan on the identity: row k of L^{-1} is scaled by
//                  1/L_kk, then rows i > k lose L_ik times it.
template <int NR>
__device__ __forceinline__ void cholesky_registers(const double* Sm, double* L, double* Xm, int n,
                                                   double* lcol, double* xr, int& bad) {
  constexpr int NE = tri_slots(NR);
  const int tid = threadIdx.x, lr = tid >> 5, lc = tid & 31;
  double a[NE];
  static_for<0, NE>([&](auto S) __attribute__((always_inline)) {
    constexpr int sl = decltype(S)::value;
    constexpr int TI = tri_row(sl), TJ = tri_col(sl);
    const int i = 16 * TI + lr, j = 32 * TJ + lc;
    a[sl] = (i < n && j < n && i >= j) ? Sm[(int64_t)i * n + j] : 0.0;
    if constexpr (TJ == TI / 2) __builtin_amdgcn_sched_barrier(0);
  });
  // lcol is zero outside [k, n): the rank-1 update then needs no masks (column k
  // itself and the strict upper part of diagonal tiles take harmless updates
  // that are never read again)
  if (tid >= n) lcol[tid] = 0.0;
  for (int k = 0; k < n; ++k) {
    const int Tk = k >> 5, ck = k & 31;
    if (tid < k) lcol[tid] = 0.0;
    if (lc == ck) {
      static_for<0, NE>([&](auto S) __attribute__((always_inline)) {
        constexpr int sl = decltype(S)::value;
        constexpr int TI = tri_row(sl), TJ = tri_col(sl);
        if (TJ == Tk) {
          const int i = 16 * TI + lr;
          if (i >= k && i < n) lcol[i] = a[sl];
        }
      });
    }
    __syncthreads();
    double piv = lcol[k];
    if (!(piv > 0.0)) {
      if (tid == 0) bad = 1;
      piv = 1.0;
    }
    const double sq = sqrt(piv);
    if (tid >= k && tid < n) L[tid + (int64_t)k * n] = tid == k ? sq : lcol[tid] / sq;
    const double ip = 1.0 / piv;
    // column tiles entirely left of k are final (lcol is zero there): skipped
    static_for<0, NR / 2>([&](auto CJ) __attribute__((always_inline)) {
      constexpr int TJ = decltype(CJ)::value;
      if (32 * TJ + 31 >= k) {
        const double lj = lcol[32 * TJ + lc] * ip;
        static_for<2 * TJ, NR>([&](auto CI) __attribute__((always_inline)) {
          constexpr int TI = decltype(CI)::value;
          constexpr int sl = tri_slots(TI) + TJ;
          a[sl] -= lcol[16 * TI + lr] * lj;
        });
      }
    });
    __syncthreads();
  }
  // L^{-1} in the same registers
  static_for<0, NE>([&](auto S) __attribute__((always_inline)) {
    constexpr int sl = decltype(S)::value;
    constexpr int TI = tri_row(sl), TJ = tri_col(sl);
    const int i = 16 * TI + lr, j = 32 * TJ + lc;
    a[sl] = (i == j && i < n) ? 1.0 : 0.0;
  });
  // lcol holds column k of L below the diagonal (zero elsewhere), xr row k of
  // L^{-1} (zero right of the diagonal), so the update needs no masks either
  for (int k = 0; k < n; ++k) {
    if (tid < kMaxAO) {
      lcol[tid] = (tid > k && tid < n) ? L[tid + (int64_t)k * n] : 0.0;
      if (tid > k) xr[tid] = 0.0;
    }
    __syncthreads();
    const double il = 1.0 / L[k + (int64_t)k * n];
    const bool rowk = lr == (k & 15);
    static_for<0, NE>([&](auto S) __attribute__((always_inline)) {
      constexpr int sl = decltype(S)::value;
      constexpr int TI = tri_row(sl), TJ = tri_col(sl);
      const int j = 32 * TJ + lc;
      const bool own = rowk && TI == (k >> 4) && j <= k;
      const double nv = own ? a[sl] * il : a[sl];
      a[sl] = nv;  // select, not a branch: keeps the register array free of copies
      if (own) xr[j] = nv;
    });
    __syncthreads();
    // xr is zero right of column k: column tiles entirely right of k are skipped
    static_for<0, NR / 2>([&](auto CJ) __attribute__((always_inline)) {
      constexpr int TJ = decltype(CJ)::value;
      if (32 * TJ <= k) {
        const double xj = xr[32 * TJ + lc];
        static_for<2 * TJ, NR>([&](auto CI) __attribute__((always_inline)) {
          constexpr int TI = decltype(CI)::value;
          constexpr int sl = tri_slots(TI) + TJ;
          a[sl] -= lcol[16 * TI + lr] * xj;
        });
      }
    });
    __syncthreads();
  }
  // X[r][c] = Linv[c][r]: the registers hold Linv(i, j), i >= j; X's strict lower part is zero
  for (int64_t idx = tid; idx < (int64_t)n * n; idx += blockDim.x) {
    const int r = (int)(idx / n), c = (int)(idx - (int64_t)r * n);
    if (c < r) Xm[idx] = 0.0;
  }
  static_for<0, NE>([&](auto S) __attribute__((always_inline)) {
    constexpr int sl = decltype(S)::value;
    constexpr int TI = tri_row(sl), TJ = tri_col(sl);
    const int i = 16 * TI + lr, j = 32 * TJ + lc;
    if (i >= j && i < n) Xm[(int64_t)j * n + i] = a[sl];
    if constexpr (TJ == TI / 2) __builtin_amdgcn_sched_barrier(0);  // one row tile of stores in flight
  });
  __syncthreads();
}

// Per-system overlap factorization, n <= 256, 512 threads: X = L^{-T} with L in `work`
// (column-major).  status = 8 on a non-positive pivot; the conditioning gate
// follows in k_overlap_rcond.
__global__ __launch_bounds__(512) void k_cholesky_inverse(Topo t, const int* order, const double* S,
                                                          double* work, double* X, SysState* status) {
  const int s = order[blockIdx.x];
  const int n = t.ao_off[s + 1] - t.ao_off[s];
  const int64_t mo = t.mat_off[s];
  const double* Sm = S + mo;
  double* L = work + mo;
  double* Xm = X + mo;
  __shared__ double lcol[kMaxAO];
  __shared__ double xr[kMaxAO];
  __shared__ int bad;
  if (threadIdx.x == 0) bad = 0;
  __syncthreads();
  if (n <= 64) cholesky_registers<4>(Sm, L, Xm, n, lcol, xr, bad);
  else if (n <= 128) cholesky_registers<8>(Sm, L, Xm, n, lcol, xr, bad);
  else if (n <= 192) cholesky_registers<12>(Sm, L, Xm, n, lcol, xr, bad);
  else cholesky_registers<16>(Sm, L, Xm, n, lcol, xr, bad);
  if (threadIdx.x == 0 && bad) status[s].status = 8;
}

// Overlap factorization for n > 256, X = L^{-T} as above (L in `work`,
// column-major lower; X row-major upper with its strict lower part zero), in
// launches that spread each system over the chip:
//   k_chol_start     L = S, X's strict lower part.
//   per panel of kCholPanel columns:
//   k_chol_panel     every block factors the diagonal block by itself (one
//                    wavefront, a row per lane in registers) and takes 256 rows
//                    below it, a row per thread, through the substitution.  Block
//                    0 leaves the diagonal factor in X, because the others read
//                    the unfactored one from L.
//   k_chol_trailing  A -= L21 L21^T on the lower triangle, a 16 x 16 tile per
//                    wavefront on the FP64 matrix cores; moves the diagonal
//                    factor into L.
//   k_chol_diagonal  the 16 x 16 diagonal blocks of L^{-1}, a thread per column.
//   k_chol_invert    a block per 16 columns J of L^{-1}, down the block rows:
//                      Linv_IJ = -Linv_II sum_{K=J}^{I-1} L_IK Linv_KJ,
//                    the sum over K split over eight wavefronts.
// Bound: two launches a panel (36 panels at 1142 AOs) and the chain of block rows
// of the inverse.  One 512-thread block per system took 21.2 ms at 1142 AOs and
// 2.5 ms for fourteen systems of 258 to 482; the launches take 1.5 and 0.6 ms.
// Matrix-core lane mapping (v_mfma_f64_16x16x4f64): for D = P Q^T over k,
// lane (l16, lk) supplies a = Q[l16][k], b = P[l16][k] for k = 4 q + lk and
// receives D[l16][lk + 4 r], r < 4.
constexpr int kCholPanel = 32;

__global__ __launch_bounds__(256) void k_chol_start(Topo t, const int* order, const double* S, double* work,
                                                    double* X) {
  const int s = order[blockIdx.x];
  const int n = t.ao_off[s + 1] - t.ao_off[s];
  const int64_t mo = t.mat_off[s], nn = (int64_t)n * n;
  for (int64_t idx = (int64_t)blockIdx.y * 256 + threadIdx.x; idx < nn; idx += (int64_t)gridDim.y * 256) {
    work[mo + idx] = S[mo + idx];
    const int r = (int)(idx / n), c = (int)(idx - (int64_t)r * n);
    if (c < r) X[mo + idx] = 0.0;
  }
}

__global__ __launch_bounds__(256) void k_chol_panel(Topo t, const int* order, double* work, double* X,
                                                    SysState* status, int k0) {
  const int s = order[blockIdx.x];
  const int n = t.ao_off[s + 1] - t.ao_off[s];
  const int r0 = k0 + kCholPanel + (int)blockIdx.y * 256;  // this block's first row
  if (k0 >= n || (blockIdx.y > 0 && r0 >= n)) return;
  double* __restrict__ L = work + t.mat_off[s];
  const int tid = threadIdx.x, jn = min(kCholPanel, n - k0);
  constexpr int P = kCholPanel;
  __shared__ double sL[P][P + 1];  // sL[c][r] = L11(r, c); diagonal: 1 / pivot
  // the row below the panel, in flight while the diagonal block is factored
  const int row = r0 + tid;
  double x[P];
  if (row < n) {
#pragma unroll
    for (int c = 0; c < P; ++c) x[c] = L[(int64_t)row + (int64_t)(k0 + c) * n];  // jn = P where rows follow
  }
  if (tid < 64) {
    // lane r < P: row r, identity past jn; entries above the diagonal are never used
    double a[P];
    const int r = min(tid, P - 1);
#pragma unroll
    for (int c = 0; c < P; ++c)
      a[c] = r < jn && c <= r ? L[(int64_t)(k0 + r) + (int64_t)(k0 + c) * n] : (r == c ? 1.0 : 0.0);
    bool bad = false;
    static_for<0, P>([&](auto J) __attribute__((always_inline)) {
      constexpr int j = decltype(J)::value;
      double d = lane_value(a[j], j);
      if (!(d > 0.0)) {
        bad = true;
        d = 1.0;
      }
      const double piv = sqrt(d), ipiv = 1.0 / piv;
      const double l = a[j] * ipiv;  // L(r, j) on lanes r > j
      if (tid > j && tid < P) sL[j][tid] = l;
      if (tid == j) {
        sL[j][j] = ipiv;
        a[j] = piv;
      } else {
        a[j] = l;
      }
      static_for<j + 1, P>([&](auto K) __attribute__((always_inline)) {
        constexpr int k = decltype(K)::value;
        a[k] = fma(-l, lane_value(l, k), a[k]);
      });
    });
    if (blockIdx.y == 0) {
      double* __restrict__ Xm = X + t.mat_off[s];
#pragma unroll
      for (int c = 0; c < P; ++c)
        if (tid < jn && c <= tid) Xm[(int64_t)(k0 + c) * n + k0 + tid] = a[c];
      if (bad && tid == 0) status[s].status = 8;
    }
  }
  __syncthreads();
  if (row < n) {
#pragma unroll
    for (int c = 0; c < P; ++c) {
      x[c] *= sL[c][c];
#pragma unroll
      for (int k = c + 1; k < P; ++k) x[k] = fma(-x[c], sL[c][k], x[k]);
    }
#pragma unroll
    for (int c = 0; c < P; ++c) L[(int64_t)row + (int64_t)(k0 + c) * n] = x[c];
  }
}

__global__ __launch_bounds__(256) void k_chol_trailing(Topo t, const int* order, double* work, const double* X,
                                                       int k0) {
  const int s = order[blockIdx.x];
  const int n = t.ao_off[s + 1] - t.ao_off[s];
  if (k0 >= n) return;
  double* __restrict__ L = work + t.mat_off[s];
  const int jn = min(kCholPanel, n - k0);
  auto at = [n](int r, int c) __attribute__((always_inline)) { return (int64_t)r + (int64_t)c * n; };
  if (blockIdx.y == 0)
    for (int idx = threadIdx.x; idx < jn * jn; idx += 256) {
      const int r = idx % jn, c = idx / jn;
      if (c <= r) L[at(k0 + r, k0 + c)] = X[t.mat_off[s] + (int64_t)(k0 + c) * n + k0 + r];
    }
  const int c0 = k0 + jn, mt = n - c0;  // rows and columns >= c0
  const int nb16 = (mt + 15) >> 4;
  const int ntiles = nb16 * (nb16 + 1) / 2;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, lk = lane >> 4;
  for (int tile = (int)blockIdx.y * 4 + wv; tile < ntiles; tile += (int)gridDim.y * 4) {
    int TI = (int)((sqrt(8.0 * tile + 1.0) - 1.0) * 0.5);
    while (TI * (TI + 1) / 2 > tile) --TI;
    while ((TI + 1) * (TI + 2) / 2 <= tile) ++TI;
    const int TJ = tile - TI * (TI + 1) / 2;
    const int rr = 16 * TI + l16, cc = 16 * TJ + l16;  // this lane's row of P (rows), of Q (columns)
    const int rrc = c0 + min(rr, mt - 1), ccc = c0 + min(cc, mt - 1);
    double xa[kCholPanel / 4], xb[kCholPanel / 4], old[4];
#pragma unroll
    for (int q = 0; q < kCholPanel / 4; ++q) {
      xa[q] = L[at(ccc, k0 + 4 * q + lk)];  // a panel with rows below it is full
      xb[q] = L[at(rrc, k0 + 4 * q + lk)];
    }
    // acc[r] = D[row = 16 TI + l16][col = 16 TJ + lk + 4 r]
#pragma unroll
    for (int r = 0; r < 4; ++r) old[r] = L[at(rrc, c0 + min(16 * TJ + lk + 4 * r, mt - 1))];
    mfma_d4 acc = mfma_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < kCholPanel / 4; ++q)
      acc = mfma_16x16x4(cc < mt ? xa[q] : 0.0, rr < mt ? xb[q] : 0.0, acc);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int col = 16 * TJ + lk + 4 * r;
      if (rr < mt && col < mt && rr >= col) L[at(c0 + rr, c0 + col)] = old[r] - acc[r];
    }
  }
}

__global__ __launch_bounds__(64) void k_chol_diagonal(Topo t, const int* order, const double* work, double* X) {
  const int s = order[blockIdx.x];
  const int n = t.ao_off[s + 1] - t.ao_off[s];
  const double* __restrict__ L = work + t.mat_off[s];
  double* __restrict__ Xm = X + t.mat_off[s];
  const int idx = (int)blockIdx.y * 64 + threadIdx.x;
  const int c = idx & 15, o = idx & ~15, b = min(16, n - o);
  if (c >= b) return;  // also where the block starts past n
  double y[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    y[r] = 0.0;
    if (r < c || r >= b) continue;
    double v = r == c ? 1.0 : 0.0;
#pragma unroll
    for (int k = 0; k < r; ++k)
      if (k >= c) v -= L[(int64_t)(o + r) + (int64_t)(o + k) * n] * y[k];
    y[r] = v / L[(int64_t)(o + r) + (int64_t)(o + r) * n];
    Xm[(int64_t)(o + c) * n + o + r] = y[r];
  }
}

__global__ __launch_bounds__(512) void k_chol_invert(Topo t, const int* order, const double* work, double* X) {
  const int s = order[blockIdx.x];
  const int n = t.ao_off[s + 1] - t.ao_off[s];
  const int NB = (n + 15) >> 4, J = (int)blockIdx.y;
  if (J >= NB) return;
  const double* __restrict__ L = work + t.mat_off[s];
  double* Xm = X + t.mat_off[s];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, lk = lane >> 4, oj = 16 * J;
  __shared__ double sP[8][16][17];
  for (int I = J + 1; I < NB; ++I) {
    const int oi = 16 * I;
    const int ri = oi + l16;  // this lane's row of block row I
    const bool rin = ri < n;
    const int ric = min(ri, n - 1);
    double bv[4];
    if (wv == 0) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int k = 4 * q + lk;
        // Linv(oi + l16, oi + k), zero above its diagonal
        bv[q] = rin && k <= l16 ? Xm[(int64_t)(oi + min(k, n - 1 - oi)) * n + ric] : 0.0;
      }
    }
    mfma_d4 acc = mfma_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll 2
    for (int K = J + wv; K < I; K += 8) {
      const int ok = 16 * K;
      double xa[4], xb[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int k = 4 * q + lk;
        // Linv(ok + k, oj + l16), zero above the diagonal of block J itself
        xa[q] = Xm[(int64_t)(oj + l16) * n + ok + k];
        xb[q] = L[(int64_t)ric + (int64_t)(ok + k) * n];  // L(oi + l16, ok + k)
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) acc = mfma_16x16x4(xa[q], rin ? xb[q] : 0.0, acc);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) sP[wv][l16][lk + 4 * r] = acc[r];
    __syncthreads();
    if (wv == 0) {
      const int nw = min(8, I - J);
      mfma_d4 acc2 = mfma_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int k = 4 * q + lk;
        double a = sP[0][k][l16];  // S[k][l16]
        for (int w = 1; w < nw; ++w) a += sP[w][k][l16];
        acc2 = mfma_16x16x4(a, bv[q], acc2);
      }
      if (rin) {
#pragma unroll
        for (int r = 0; r < 4; ++r) Xm[(int64_t)(oj + lk + 4 * r) * n + ri] = -acc2[r];
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Overlap conditioning gate of the reference (eigensolver.cpp:2388-2402):
// rcond_1 = 1 / (|S|_1 est(|S^{-1}|_1)) >= 1e-12, where est is LAPACK's
// Hager-Higham 1-norm estimate (dlacn2, the iteration dpocon runs; Higham,
// ACM TOMS 14 (1988) 381-396, Algorithm 4.1): at most five power steps
// x -> sign(S^{-1} x) -> S^{-1} sign(.) -> unit vector at the largest entry,
// stopped on a repeated sign vector, no increase, or a repeated index, then
// the alternating-sign test vector x_i = (-1)^i (1 + i/(n-1)) with estimate
// 2 |S^{-1} x|_1 / (3n).  Here S^{-1} v = X (X^T v) with X = L^{-T} (row-major,
// upper triangular) from k_cholesky_inverse.  One 512-thread block per system
// whose factorization succeeded.
// ---------------------------------------------------------------------------
constexpr double kMinOverlapRcond = 1e-12;

constexpr int kRcondThreads = 512;
constexpr int kRcondWaves = kRcondThreads / 64;

struct RcondShared {
  double x[kMaxAO];
  double y[kMaxAO];
  double part[kRcondWaves][kMaxAO];  // per-wave partial column sums of X^T x
  signed char sgn[kMaxAO];
  double red[kRcondWaves];
  int ired[kRcondWaves];
};

// The same vectors for systems above kMaxAO AOs, in their global slice (x, y:
// n doubles each, sgn: n bytes); red and ired stay in LDS.
struct RcondBig {
  double* x;
  double* y;
  signed char* sgn;
  double* red;
  int* ired;
};

// block sum of |v_i|
template <typename SH>
__device__ double rc_asum(const double* v, int n, SH& sh) {
  double a = 0.0;
  for (int i = threadIdx.x; i < n; i += blockDim.x) a += fabs(v[i]);
  a = wave_sum(a);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh.red[threadIdx.x >> 6] = a;
  __syncthreads();
  double t = 0.0;
  for (int w = 0; w < kRcondWaves; ++w) t += sh.red[w];
  __syncthreads();
  return t;
}

// first index of the largest |v_i| (LAPACK idamax)
template <typename SH>
__device__ int rc_iamax(const double* v, int n, SH& sh) {
  double best = -1.0;
  int bi = 0;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const double a = fabs(v[i]);
    if (a > best) { best = a; bi = i; }
  }
  for (int off = 32; off > 0; off >>= 1) {
    const double ob = __shfl_xor(best, off, 64);
    const int oi = __shfl_xor(bi, off, 64);
    if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
  }
  __syncthreads();
  if ((threadIdx.x & 63) == 0) { sh.red[threadIdx.x >> 6] = best; sh.ired[threadIdx.x >> 6] = bi; }
  __syncthreads();
  best = sh.red[0];
  bi = sh.ired[0];
  for (int w = 1; w < kRcondWaves; ++w)
    if (sh.red[w] > best || (sh.red[w] == best && sh.ired[w] < bi)) { best = sh.red[w]; bi = sh.ired[w]; }
  __syncthreads();
  return bi;
}

// sh.x <- S^{-1} sh.x  (y = X^T x, then x = X y); X row-major upper triangular
// with its strict lower part stored as zero.  Both products read X by rows,
// lanes along the row, 16 / KC rows per wave at a time (their loads are in
// flight together): X^T x as per-wave partial column sums (summed in
// a fixed order), X y as one wave per row.  KC = column chunks of 64.
template <int KC>
__device__ void rc_apply_k(const double* __restrict__ Xm, int n, RcondShared& sh) {
  constexpr int U = 16 / KC;  // rows in flight per wave: 16 loads per lane
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  __syncthreads();
  double acc[KC];
#pragma unroll
  for (int m = 0; m < KC; ++m) acc[m] = 0.0;
  for (int r0 = wv; r0 < n; r0 += U * kRcondWaves) {
    double xv[U], v[U][KC];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int r = r0 + u * kRcondWaves;
      xv[u] = r < n ? sh.x[r] : 0.0;
#pragma unroll
      for (int m = 0; m < KC; ++m) {
        const int c = lane + 64 * m;
        v[u][m] = (r < n && c >= r && c < n) ? Xm[(int64_t)r * n + c] : 0.0;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int m = 0; m < KC; ++m) acc[m] = fma(v[u][m], xv[u], acc[m]);
  }
#pragma unroll
  for (int m = 0; m < KC; ++m) {
    const int c = lane + 64 * m;
    if (c < n) sh.part[wv][c] = acc[m];
  }
  __syncthreads();
  for (int c = threadIdx.x; c < n; c += blockDim.x) {
    double t = 0.0;
    for (int w = 0; w < kRcondWaves; ++w) t += sh.part[w][c];
    sh.y[c] = t;
  }
  __syncthreads();
  for (int r0 = wv; r0 < n; r0 += U * kRcondWaves) {
    double a[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int r = r0 + u * kRcondWaves;
      a[u] = 0.0;
#pragma unroll
      for (int m = 0; m < KC; ++m) {
        const int c = lane + 64 * m;
        if (r < n && c >= r && c < n) a[u] = fma(Xm[(int64_t)r * n + c], sh.y[c], a[u]);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int r = r0 + u * kRcondWaves;
      const double t = wave_sum(a[u]);
      if (lane == 0 && r < n) sh.x[r] = t;
    }
  }
  __syncthreads();
}

__device__ void rc_apply(const double* __restrict__ Xm, int n, RcondShared& sh) {
  if (n <= 256) rc_apply_k<4>(Xm, n, sh);
  else if (n <= 512) rc_apply_k<8>(Xm, n, sh);
  else rc_apply_k<16>(Xm, n, sh);
}

// n > kMaxAO: y = X^T x with a thread per column (the column's entries of
// consecutive rows are adjacent across the threads), then x = X y with a
// wave per row
__device__ void rc_apply(const double* __restrict__ Xm, int n, RcondBig& sh) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  __syncthreads();
  for (int c = threadIdx.x; c < n; c += blockDim.x) {
    double a = 0.0;
    for (int r = 0; r <= c; ++r) a = fma(Xm[(int64_t)r * n + c], sh.x[r], a);
    sh.y[c] = a;
  }
  __syncthreads();
  for (int r = wv; r < n; r += kRcondWaves) {
    double a = 0.0;
    for (int c = r + lane; c < n; c += 64) a = fma(Xm[(int64_t)r * n + c], sh.y[c], a);
    a = wave_sum(a);
    if (lane == 0) sh.x[r] = a;
  }
  __syncthreads();
}

template <typename SH>
__device__ void overlap_rcond(const double* __restrict__ Sm, const double* __restrict__ Xm, int n, SH& sh,
                              SysState& status) {
  // |S|_1: S is symmetric, so the largest row sum (one wave per row, lanes
  // along the row)
  double anorm = 0.0;
  {
    const int lane = threadIdx.x & 63;
    double m = 0.0;
    for (int r = threadIdx.x >> 6; r < n; r += kRcondWaves) {
      double a = 0.0;
      for (int c = lane; c < n; c += 64) a += fabs(Sm[(int64_t)r * n + c]);
      m = fmax(m, wave_sum(a));
    }
    for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off, 64));
    if ((threadIdx.x & 63) == 0) sh.red[threadIdx.x >> 6] = m;
    __syncthreads();
    for (int w = 0; w < kRcondWaves; ++w) anorm = fmax(anorm, sh.red[w]);
    __syncthreads();
  }
  // estimate of |S^{-1}|_1
  for (int i = threadIdx.x; i < n; i += blockDim.x) sh.x[i] = 1.0 / n;
  rc_apply(Xm, n, sh);
  double est;
  if (n == 1) {
    est = fabs(sh.x[0]);
  } else {
    est = rc_asum(sh.x, n, sh);
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
      const signed char g = sh.x[i] >= 0.0 ? 1 : -1;
      sh.sgn[i] = g;
      sh.x[i] = g;
    }
    rc_apply(Xm, n, sh);
    int j = rc_iamax(sh.x, n, sh);
    for (int iter = 2;; ++iter) {
      for (int i = threadIdx.x; i < n; i += blockDim.x) sh.x[i] = i == j ? 1.0 : 0.0;
      rc_apply(Xm, n, sh);
      const double estold = est;
      est = rc_asum(sh.x, n, sh);
      __shared__ int differs;
      if (threadIdx.x == 0) differs = 0;
      __syncthreads();
      for (int i = threadIdx.x; i < n; i += blockDim.x)
        if ((sh.x[i] >= 0.0 ? 1 : -1) != sh.sgn[i]) differs = 1;
      __syncthreads();
      if (!differs || est <= estold) break;  // repeated sign vector, or no increase
      for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const signed char g = sh.x[i] >= 0.0 ? 1 : -1;
        sh.sgn[i] = g;
        sh.x[i] = g;
      }
      rc_apply(Xm, n, sh);
      const int jlast = j;
      j = rc_iamax(sh.x, n, sh);
      if (!(sh.x[jlast] != fabs(sh.x[j]) && iter < 5)) break;
    }
    // alternating-sign test vector
    for (int i = threadIdx.x; i < n; i += blockDim.x)
      sh.x[i] = (i & 1 ? -1.0 : 1.0) * (1.0 + (double)i / (double)(n - 1));
    rc_apply(Xm, n, sh);
    const double temp = 2.0 * (rc_asum(sh.x, n, sh) / (3.0 * n));
    if (temp > est) est = temp;
  }
  const double rcond = (est != 0.0 && anorm != 0.0) ? (1.0 / est) / anorm : 0.0;
  if (threadIdx.x == 0 && !(rcond >= kMinOverlapRcond && isfinite(rcond))) status.status = 8;
}

// BIG: the systems above kMaxAO AOs, with x, y and the signs in their global
// slice of `big`
template <bool BIG>
__global__ __launch_bounds__(kRcondThreads) void k_overlap_rcond(Topo t, const int* order, const double* S,
                                                       const double* X, SysState* status, double* big) {
  const int s = order[blockIdx.x];
  if (status[s].status != 0) return;
  const int n = t.ao_off[s + 1] - t.ao_off[s];
  const int64_t mo = t.mat_off[s];
  if constexpr (BIG) {
    __shared__ double red[kRcondWaves];
    __shared__ int ired[kRcondWaves];
    double* x = big + big_offset(t, s);
    RcondBig sh{x, x + n, reinterpret_cast<signed char*>(x + 2 * n), red, ired};
    overlap_rcond(S + mo, X + mo, n, sh, status[s]);
  } else {
    __shared__ RcondShared sh;
    overlap_rcond(S + mo, X + mo, n, sh, status[s]);
  }
}

// x / y via the hardware reciprocal refined by one Newton step (a few ulp,
// enough for the sign decisions of a Sturm count)
__device__ __forceinline__ double fast_div(double x, double y) {
  double r = __builtin_amdgcn_rcp(y);
  r = fma(r, fma(-y, r, 1.0), r);
  return x * r;
}

// Sturm count of T[b0:b1) - x I (the number of eigenvalues below x) together
// with L(x) = d/dx log|det(T - x I)| = sum_i 1/(x - lambda_i), from the
// three-term recurrence of the leading principal minors of T - x I
//   p_i = (d_i - x) p_{i-1} - e_{i-1}^2 p_{i-2},   p_{-1} = 1,
// and of their derivatives
//   p_i' = (d_i - x) p_{i-1}' - p_{i-1} - e_{i-1}^2 p_{i-2}',  p_{-1}' = 0.
// The count is the number of sign changes along p_{-1}, p_0, ..., p_{b-1}
// (a vanishing minor takes the sign opposite to its predecessor, as a
// vanishing pivot of T - x I = L D L^T counts as negative), and L = p'/p of
// the last minor.  The pivots of L D L^T are the ratios p_i / p_{i-1}, so this
// is the pivot count without a division per row: one FMA per row sits on the
// serial chain.  Every eight rows both minors and both derivatives are scaled
// by the same power of two (the exponent of the larger minor), which keeps
// them in range and changes neither a sign nor the ratio p'/p.
__device__ __forceinline__ int sturm_count_logd(const double* d, const double* e2, int b0, int b1,
                                                double x, double& L) {
  double pm2 = 1.0, pm1 = d[b0] - x;  // p_{i-2}, p_{i-1}
  double qm2 = 0.0, qm1 = -1.0;       // their derivatives
  int neg = pm1 <= 0.0 ? 1 : 0;       // sign of p_{i-1} (p_{-1} = 1 > 0)
  int c = neg;
  // sign bookkeeping on the bits (selects, no branches: the count must not
  // put control flow on the chain)
  auto step = [&](double di, double ei2) __attribute__((always_inline)) {
    const double dx = di - x;
    const double p = fma(dx, pm1, -ei2 * pm2);
    const double q = fma(dx, qm1, -fma(ei2, qm2, pm1));
    const unsigned long long bits = (unsigned long long)__double_as_longlong(p);
    const int sgn = (int)(bits >> 63);
    const int sn = (bits << 1) == 0ull ? (neg ^ 1) : sgn;  // a zero minor flips the sign
    c += sn ^ neg;
    neg = sn;
    pm2 = pm1;
    pm1 = p;
    qm2 = qm1;
    qm1 = q;
  };
  // load eight entries of d and e^2 ahead so that LDS latency stays off the chain
  int i = b0 + 1;
  for (; i + 7 < b1; i += 8) {
    double dv[8], ev[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      dv[u] = d[i + u];
      ev[u] = e2[i - 1 + u];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) step(dv[u], ev[u]);
    const int ex = __builtin_amdgcn_frexp_exp(fmax(fabs(pm1), fabs(pm2)));
    pm1 = ldexp(pm1, -ex);
    pm2 = ldexp(pm2, -ex);
    qm1 = ldexp(qm1, -ex);
    qm2 = ldexp(qm2, -ex);
  }
  for (; i < b1; ++i) step(d[i], e2[i - 1]);
  L = qm1 / pm1;
  return c;
}

// Eigenvalues of T by Sturm-count bracketing with Newton steps on
// det(T - x I) once a bracket isolates exactly its eigenvalue (a step outside
// the bracket falls back to bisection).  Converged when the bracket or the
// Newton step is below 2 eps |T_b| + pivmin, the accuracy of bisection.  A
// guess (the previous SCC round's eigenvalue) first narrows the bracket to
// [guess - delta, guess + delta] where the counts allow.
//
// The lanes of the block share the eigenvalues through an LDS counter: a lane
// whose eigenvalue converged takes the next index, so a wave's cost follows
// the total work instead of its slowest eigenvalue.  One trip of the loop is
// one pass over the block.
struct EigState {
  int j, b0, b1, k, it, phase;  // phase 0/1: guess bracket ends, 2: main iteration
  int clo, chi;
  double lo, hi, x, tol, guess, dl, dh;
  double dxo;  // size of the step before the last one (Newton acceptance)
};

// Gershgorin interval and tolerance of the unreduced block [b0, b1)
__device__ __forceinline__ void block_bounds(const double* d, const double* e, int b0, int b1,
                                             double pivmin, double& lo, double& hi, double& tol) {
  double gl = 1e300, gu = -1e300;
  for (int i = b0; i < b1; ++i) {
    const double off = (i > b0 ? fabs(e[i - 1]) : 0.0) + (i + 1 < b1 ? fabs(e[i]) : 0.0);
    gl = fmin(gl, d[i] - off);
    gu = fmax(gu, d[i] + off);
  }
  const double tnorm = fmax(fabs(gl), fabs(gu));
  const double fudge = 2.0 * kEps * tnorm * (b1 - b0) + 4.0 * pivmin;
  lo = gl - fudge;
  hi = gu + fudge;
  tol = 2.0 * kEps * tnorm + pivmin;
}

// starts eigenvalue j; when T is unsplit the whole-matrix bounds are passed in
__device__ __forceinline__ bool eig_start(EigState& st, int j, const double* d, const double* e,
                                          int n, double pivmin, bool unsplit, double glo,
                                          double ghi, double gtol, bool guess_ok, double guess,
                                          double gprev, double gnext, double delta, double* lam) {
  int b0 = 0, b1 = n;
  if (!unsplit) {
    b0 = j;
    b1 = j + 1;
    while (b0 > 0 && e[b0 - 1] != 0.0) --b0;
    while (b1 < n && e[b1 - 1] != 0.0) ++b1;
  }
  if (b1 - b0 == 1) {
    lam[j] = d[j];
    return false;
  }
  st.j = j; st.b0 = b0; st.b1 = b1; st.k = j - b0; st.it = 0;
  if (unsplit) {
    st.lo = glo; st.hi = ghi; st.tol = gtol;
  } else {
    block_bounds(d, e, b0, b1, pivmin, st.lo, st.hi, st.tol);
  }
  st.clo = 0;
  st.chi = b1 - b0;
  const bool g = guess_ok && guess > st.lo && guess < st.hi;
  st.guess = guess;
  // guess bracket: at most the largest change of the last round, and at most
  // half the distance to the neighbouring guesses, so that the bracket usually
  // isolates the eigenvalue at once (Newton then starts from the guess)
  const double dmin = 4.0 * st.tol;
  st.dl = fmax(fmin(delta, 0.5 * (guess - gprev)), dmin);
  st.dh = fmax(fmin(delta, 0.5 * (gnext - guess)), dmin);
  st.phase = g ? 0 : 2;
  st.x = g ? guess - st.dl : 0.5 * (st.lo + st.hi);
  st.dxo = st.hi - st.lo;
  return true;
}

// one pass at st.x; returns true (result in `out`) when the eigenvalue has converged
__device__ __forceinline__ bool eig_step(EigState& st, const double* d, const double* e2, double& out) {
  double L;
  const int c = sturm_count_logd(d, e2, st.b0, st.b1, st.x, L);
  if (st.phase < 2) {
    // guess bracket: only narrow where the count confirms the side
    if (st.x > st.lo && st.x < st.hi) {
      if (c <= st.k) { st.lo = st.x; st.clo = c; } else { st.hi = st.x; st.chi = c; }
    }
    if (st.phase == 0) {
      st.phase = 1;
      st.x = st.guess + st.dh;
      if (st.x < st.hi) return false;
    }
    st.phase = 2;
    st.x = (st.guess > st.lo && st.guess < st.hi) ? st.guess : 0.5 * (st.lo + st.hi);
    st.dxo = st.hi - st.lo;
    return false;
  }
  if (c <= st.k) { st.lo = st.x; st.clo = c; } else { st.hi = st.x; st.chi = c; }
  if (st.hi - st.lo <= st.tol || ++st.it >= 256) {
    out = 0.5 * (st.lo + st.hi);
    return true;
  }
  // Newton only on an isolating bracket and only while it converges: the step
  // must stay inside and be less than half the step before last (otherwise
  // bisect), which rules out slow one-sided creeping
  const double dxo = st.dxo;
  if (st.clo == st.k && st.chi == st.k + 1 && L != 0.0 && isfinite(L)) {
    const double step = -1.0 / L;
    if (fabs(step) <= st.tol) {
      out = st.x + step;
      return true;
    }
    const double xn = st.x + step;
    if (xn > st.lo && xn < st.hi && fabs(step) < 0.5 * dxo) {
      st.dxo = fabs(step);
      st.x = xn;
      return false;
    }
  }
  const double mid = 0.5 * (st.lo + st.hi);
  if (mid == st.lo || mid == st.hi) {
    out = mid;
    return true;
  }
  st.dxo = fabs(mid - st.x);
  st.x = mid;
  return false;
}

// deterministic start vector in [-1, 1)
__device__ __forceinline__ double start_component(int j, int i) {
  uint64_t z = (uint64_t)(j + 1) * 0x9E3779B97F4A7C15ull + (uint64_t)(i + 1) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  return (double)(z >> 11) * (2.0 / 9007199254740992.0) - 1.0;
}

// Per-system scratch for the LU factors of one shifted block, interleaved by
// vector (element i of vector j at [i * n + j]) so that a wavefront's threads
// touch consecutive addresses.
struct EigenScratch {
  double* u0;    // pivot row diagonal
  double* u1;    // first superdiagonal
  double* u2;    // second superdiagonal (fill-in from row interchanges)
  double* mult;  // elimination multipliers
  double* piv;   // 1.0 where rows k, k+1 were interchanged
};

// Eigenvector of an isolated eigenvalue x of the unreduced block T[b0:b1) from
// its twisted factorization: forward pivots D+ (in F0) and backward pivots D-
// (in F1) of T - x I, twist index r = argmin |D+_r + D-_r - (d_r - x)|, then
// z_r = 1, z_i = -(e_i / D+_i) z_{i+1} below r and z_i = -(e_{i-1} / D-_i) z_{i-1}
// above r.  Z receives the unnormalized vector and `scale` the factor that
// normalizes it with the largest component positive (applied when the vector
// is back-transformed).  Returns false (leaving Z to be overwritten) if the
// recurrences produced a non-finite value.
__device__ __forceinline__ bool twisted_vector(const double* d, const double* e, int b0, int b1,
                                               double x, double pivmin, int n, int jj,
                                               double* __restrict__ Dp, double* __restrict__ Dm,
                                               double* __restrict__ Z, double& scale) {
  // Every loop below is a serial chain; the entries it consumes (d, e from
  // LDS, pivots from global memory) are loaded eight at a time ahead of it.
  constexpr int U = 8;
  auto at = [&](int i) __attribute__((always_inline)) { return (int64_t)i * n + jj; };
  double q = d[b0] - x;
  if (fabs(q) < pivmin) q = -pivmin;
  Dp[at(b0)] = q;
  {
    auto step = [&](int i, double di, double ei) __attribute__((always_inline)) {
      q = (di - x) - fast_div(ei * ei, q);
      if (fabs(q) < pivmin) q = -pivmin;
      Dp[at(i)] = q;
    };
    int i = b0 + 1;
    for (; i + U - 1 < b1; i += U) {
      double dv[U], ev[U];
#pragma unroll
      for (int u = 0; u < U; ++u) { dv[u] = d[i + u]; ev[u] = e[i - 1 + u]; }
#pragma unroll
      for (int u = 0; u < U; ++u) step(i + u, dv[u], ev[u]);
    }
    for (; i < b1; ++i) step(i, d[i], e[i - 1]);
  }
  q = d[b1 - 1] - x;
  if (fabs(q) < pivmin) q = -pivmin;
  Dm[at(b1 - 1)] = q;
  int r = b1 - 1;
  double gmin = fabs(Dp[at(b1 - 1)] + q - (d[b1 - 1] - x));
  {
    auto step = [&](int i, double di, double ei, double dpi) __attribute__((always_inline)) {
      q = (di - x) - fast_div(ei * ei, q);
      if (fabs(q) < pivmin) q = -pivmin;
      Dm[at(i)] = q;
      const double g = fabs(dpi + q - (di - x));
      if (g < gmin) {
        gmin = g;
        r = i;
      }
    };
    int i = b1 - 2;
    for (; i - U + 1 >= b0; i -= U) {
      double dv[U], ev[U], pv[U];
#pragma unroll
      for (int u = 0; u < U; ++u) { dv[u] = d[i - u]; ev[u] = e[i - u]; pv[u] = Dp[at(i - u)]; }
#pragma unroll
      for (int u = 0; u < U; ++u) step(i - u, dv[u], ev[u], pv[u]);
    }
    for (; i >= b0; --i) step(i, d[i], e[i], Dp[at(i)]);
  }
  double z = 1.0, nrm = 1.0, big = 1.0;
  Z[at(r)] = 1.0;
  auto put = [&](int i, double ratio) __attribute__((always_inline)) {
    z = -ratio * z;
    Z[at(i)] = z;
    nrm += z * z;
    if (fabs(z) > fabs(big)) big = z;
  };
  {
    int i = r - 1;
    for (; i - U + 1 >= b0; i -= U) {
      double rv[U];
#pragma unroll
      for (int u = 0; u < U; ++u) rv[u] = e[i - u] / Dp[at(i - u)];
#pragma unroll
      for (int u = 0; u < U; ++u) put(i - u, rv[u]);
    }
    for (; i >= b0; --i) put(i, e[i] / Dp[at(i)]);
  }
  z = 1.0;
  {
    int i = r + 1;
    for (; i + U - 1 < b1; i += U) {
      double rv[U];
#pragma unroll
      for (int u = 0; u < U; ++u) rv[u] = e[i - 1 + u] / Dm[at(i + u)];
#pragma unroll
      for (int u = 0; u < U; ++u) put(i + u, rv[u]);
    }
    for (; i < b1; ++i) put(i, e[i - 1] / Dm[at(i)]);
  }
  if (!isfinite(nrm) || !(nrm > 0.0)) return false;
  scale = (big < 0.0 ? -1.0 : 1.0) / sqrt(nrm);
  return true;
}

// ---------------------------------------------------------------------------
// Fermi occupations of one spin channel (reference eigensolver.cpp:992-1161),
// FP64 bisection on the shifted frame; one wavefront.
// ---------------------------------------------------------------------------
__device__ double fermi_sum_wave(const double* eps, int n, double ref, double mu, double kt,
                                 bool holes) {
  double acc = 0.0;
  for (int i = threadIdx.x & 63; i < n; i += 64) {
    const double a = ((eps[i] - ref) - mu) / kt;
    double f;
    if (holes) f = a >= 0.0 ? 1.0 / (exp(-a) + 1.0) : exp(a) / (1.0 + exp(a));
    else f = a >= 0.0 ? exp(-a) / (1.0 + exp(-a)) : 1.0 / (exp(a) + 1.0);
    acc += f;
  }
  return wave_sum(acc);
}

// (h, l) += x in double-double (two-sum of the high parts, then renormalized)
__device__ __forceinline__ void dd_accumulate(double& h, double& l, double x) {
  const double sm = h + x, v = sm - h;
  const double err = (h - (sm - v)) + (x - v) + l;
  const double nh = sm + err;
  l = err - (nh - sm);
  h = nh;
}

// double-double sum over the wavefront, every lane receiving lane 0's result
__device__ __forceinline__ double dd_wave_excess(double h, double l, double qt) {
  for (int off = 32; off > 0; off >>= 1) {
    const double oh = __shfl_xor(h, off, 64), ol = __shfl_xor(l, off, 64);
    dd_accumulate(h, l, oh);
    dd_accumulate(h, l, ol);
  }
  h = __shfl(h, 0, 64);
  l = __shfl(l, 0, 64);
  dd_accumulate(h, l, -qt);
  return h + l;
}

// The counts of one spin channel at mu minus the target qt, both accumulated
// in double-double over the wavefront:
//   ideal  the occupations before rounding (holes: the hole occupations
//          1 / (e^-a + 1) as such), to the accuracy of exp and the division;
//   pub    the binary64 occupations f that are published (holes: 1 - f,
//          taken exactly).
// For electrons the two take the same terms.  The reference's long-double
// main path accepts its root when both lie within 64 eps qt of the target
// (eigensolver.cpp:1135-1161); with both counts this accurate the bisection
// below applies that same acceptance at every step, so the published count
// meets the target whenever a root is accepted.
__device__ __forceinline__ void fermi_counts_wave(const double* eps, int n, double ref, double mu,
                                                  double kt, bool holes, double qt, double& ideal,
                                                  double& pub) {
  double ih = 0.0, il = 0.0, ph = 0.0, pl = 0.0;
  for (int i = threadIdx.x & 63; i < n; i += 64) {
    const double a = ((eps[i] - ref) - mu) / kt;
    const double x = exp(-fabs(a));
    const double big = 1.0 / (x + 1.0), small = x / (1.0 + x);
    const double f = a >= 0.0 ? small : big;
    if (holes) {
      dd_accumulate(ih, il, a >= 0.0 ? big : small);
      const double h = 1.0 - f;
      dd_accumulate(ph, pl, h);
      pl += (1.0 - h) - f;  // the rounding error of 1 - f, exact for 0 <= f <= 1
    } else {
      dd_accumulate(ph, pl, f);
    }
  }
  pub = dd_wave_excess(ph, pl, qt);
  ideal = holes ? dd_wave_excess(ih, il, qt) : pub;
}

// Occupations of one spin channel on one wavefront.  Returns 0 when the
// occupations in `occ` are final, 1 when the rare path (fermi_policy) must
// publish them -- no binary64 chemical potential puts both the count before
// rounding and the published count within 64 eps of the target -- and 2 when
// the count is not bracketed (a data failure), as the reference's
// compute_occupations decides (eigensolver.cpp:1026-1161).  ideal_ok: the
// root met the count.
__device__ int fermi_wave(const double* eps, int n, double nel, double kt, double* occ,
                          double& entropy, bool& ideal_ok) {
  const int lane = threadIdx.x & 63;
  entropy = 0.0;
  ideal_ok = true;
  if (kt == 0.0) {
    const int full = (int)floor(nel);
    for (int i = lane; i < n; i += 64) occ[i] = i < full ? 1.0 : (i == full ? nel - full : 0.0);
    return 0;
  }
  if (nel == 0.0) {
    for (int i = lane; i < n; i += 64) occ[i] = 0.0;
    return 0;
  }
  if (nel == (double)n) {
    for (int i = lane; i < n; i += 64) occ[i] = 1.0;
    return 0;
  }
  const bool holes = nel > 0.5 * n;
  const double qt = holes ? n - nel : nel;
  const double steps = fmax(64.0, -log(qt / n) + 8.0);
  const double ref = holes ? eps[n - 1] : eps[0];
  const double lo0 = eps[0] - ref, hi0 = eps[n - 1] - ref;
  const double margin = steps * kt + 64.0 * 2.220446049250313e-16 * fmax(1.0, fabs(hi0 - lo0));
  double lo = lo0 - margin, hi = hi0 + margin;
  {
    const double ql = fermi_sum_wave(eps, n, ref, lo, kt, holes);
    const double qh = fermi_sum_wave(eps, n, ref, hi, kt, holes);
    const bool brk = holes ? (ql >= qt && qh <= qt) : (ql <= qt && qh >= qt);
    if (!isfinite(lo) || !isfinite(hi) || !(lo < hi) || !brk) return 2;
  }
  const double tol = 64.0 * 2.220446049250313e-16 * qt;
  double xi = 0.0, xp = 0.0;
  bool met = false;
  for (int it = 0; it < 4096; ++it) {
    const double mid = lo + 0.5 * (hi - lo);
    fermi_counts_wave(eps, n, ref, mid, kt, holes, qt, xi, xp);
    if (fabs(xi) <= tol && fabs(xp) <= tol) {
      lo = hi = mid;
      met = true;
      break;
    }
    if (mid == lo || mid == hi) break;
    if ((!holes && xi < 0.0) || (holes && xi > 0.0)) lo = mid; else hi = mid;
  }
  const double mu = lo + 0.5 * (hi - lo);
  if (!met) fermi_counts_wave(eps, n, ref, mu, kt, holes, qt, xi, xp);
  ideal_ok = fabs(xi) <= tol;
  const bool pub_ok = fabs(xp) <= tol;
  double sacc = 0.0;
  for (int i = lane; i < n; i += 64) {
    const double a = ((eps[i] - ref) - mu) / kt;
    const double x = exp(-fabs(a));
    const double f = a >= 0.0 ? x / (1.0 + x) : 1.0 / (x + 1.0);
    occ[i] = f;
    if (f > 0.0 && f < 1.0) sacc -= f * log(f) + (1.0 - f) * log(1.0 - f);
  }
  entropy = wave_sum(sacc);
  return ideal_ok && pub_ok ? 0 : 1;
}

// Occupations are negligible below kOccFloor: orbitals past the last one
// above it add less than 1e-30 of a unit occupation to P and W, far below
// FP64 resolution, and get no eigenvector.
constexpr double kOccFloor = 1e-30;

// Fermi outputs of the eigen kernel, per orbital in ascending eigenvalue order.
struct FermiOut {
  double* fa;    // alpha occupations
  double* fb;    // beta occupations
  double* occ;   // fa + fb
  double* fe;    // occ * eps
  SysState* st;  // entropy and kocc
  int* kocc;     // [B] leading orbitals with occ > kOccFloor
  double kt;
};

// T of one system into d, e and e2 = e^2 with the negligible off-diagonals
// zeroed, by the whole block; the pivot floor, and whether T did not split.
__device__ __forceinline__ bool eig_load(const double* dg, const double* eg, int n, double* d, double* e, double* e2,
                                         double* red, int& nsplit, double& pivmin) {
  const int tid = threadIdx.x, nt = blockDim.x;
  double emax2 = 0.0;
  for (int i = tid; i < n; i += nt) {
    d[i] = dg[i];
    e[i] = i + 1 < n ? eg[i] : 0.0;
  }
  if (tid == 0) nsplit = 0;
  __syncthreads();
  int cut = 0;
  for (int i = tid; i < n; i += nt) {
    double ei = e[i];
    if (i + 1 < n && ei * ei <= kEps * kEps * fabs(d[i] * d[i + 1]) + kSafeMin) ei = 0.0;
    if (i + 1 < n && ei == 0.0) ++cut;
    e2[i] = ei * ei;
    emax2 = fmax(emax2, ei * ei);
  }
  if (cut) atomicAdd(&nsplit, cut);
  __syncthreads();
  for (int i = tid; i < n; i += nt)
    if (e2[i] == 0.0) e[i] = 0.0;
  for (int off = 32; off > 0; off >>= 1) emax2 = fmax(emax2, __shfl_xor(emax2, off, 64));
  if ((tid & 63) == 0) red[tid >> 6] = emax2;
  __syncthreads();
  emax2 = 0.0;
  for (int w = 0; w < (nt >> 6); ++w) emax2 = fmax(emax2, red[w]);
  __syncthreads();
  pivmin = kSafeMin * fmax(1.0, emax2);
  return nsplit == 0;
}

// Whole-matrix Gershgorin bounds and tolerance of an unsplit T: gbound = lo, hi, tol
__device__ __forceinline__ void eig_bounds(const double* d, const double* e, int n, double pivmin, double* red,
                                           double* gbound) {
  const int tid = threadIdx.x, nt = blockDim.x;
  double gl = 1e300, gu = -1e300;
  for (int i = tid; i < n; i += nt) {
    const double off = (i > 0 ? fabs(e[i - 1]) : 0.0) + (i + 1 < n ? fabs(e[i]) : 0.0);
    gl = fmin(gl, d[i] - off);
    gu = fmax(gu, d[i] + off);
  }
  for (int off = 32; off > 0; off >>= 1) {
    gl = fmin(gl, __shfl_xor(gl, off, 64));
    gu = fmax(gu, __shfl_xor(gu, off, 64));
  }
  if ((tid & 63) == 0) { red[tid >> 6] = gl; red[8 + (tid >> 6)] = gu; }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < (nt >> 6); ++w) { gl = fmin(gl, red[w]); gu = fmax(gu, red[8 + w]); }
    const double tnorm = fmax(fabs(gl), fabs(gu));
    const double fudge = 2.0 * kEps * tnorm * n + 4.0 * pivmin;
    gbound[0] = gl - fudge;
    gbound[1] = gu + fudge;
    gbound[2] = 2.0 * kEps * tnorm + pivmin;
  }
  __syncthreads();
}

// 1-norm of T
__device__ __forceinline__ void eig_norm1(const double* d, const double* e, int n, double* red, double& tnorm1) {
  const int tid = threadIdx.x, nt = blockDim.x;
  double m = 0.0;
  for (int i = tid; i < n; i += nt)
    m = fmax(m, fabs(d[i]) + (i > 0 ? fabs(e[i - 1]) : 0.0) + (i + 1 < n ? fabs(e[i]) : 0.0));
  for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off, 64));
  if ((tid & 63) == 0) red[tid >> 6] = m;
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < (nt >> 6); ++w) m = fmax(m, red[w]);
    tnorm1 = m;
  }
  __syncthreads();
}

// Ascending ranks of the eigenvalues lam, the sorted spectrum (srt, w_out), the
// Fermi occupations and kocc, by a block of at least 128 threads; returns kocc.
__device__ __forceinline__ int eig_occupations(const Topo& t, int s, int n, const double* lam, int* rnk, double* srt,
                                               double* w_out, const FermiOut& fo) {
  const int tid = threadIdx.x, nt = blockDim.x;
  // ---- ascending rank (stable on ties) and the sorted spectrum ----
  __shared__ int kocc_sh;
  for (int j = tid; j < n; j += nt) {
    const double lj = lam[j];
    int r = 0;
    for (int i = 0; i < n; ++i) {
      const double li = lam[i];
      r += (li < lj) || (li == lj && i < j);
    }
    rnk[j] = r;
    srt[r] = lj;
    w_out[r] = lj;
  }
  __syncthreads();
  // ---- occupations: alpha on the first wavefront, beta on the second (a
  // closed shell solves once and copies) ----
  __shared__ int chan_r[2];
  __shared__ double chan_s[2];
  const bool same_channels = t.nalpha[s] == t.nbeta[s];
  if (tid < 128 && (tid < 64 || !same_channels)) {
    const int w = tid >> 6;
    const int o = t.ao_off[s];
    const double nel = w == 0 ? t.nalpha[s] : t.nbeta[s];
    double* f = (w == 0 ? fo.fa : fo.fb) + o;
    double sw;
    bool ideal;
    int r = fermi_wave(srt, n, nel, fo.kt, f, sw, ideal);
    // the reference's binary64 rare path, serial on lane 0
    if (r == 1) {
      if ((tid & 63) == 0) r = fermi_policy(srt, n, nel, fo.kt, f, sw) ? 0 : 2;
      __threadfence_block();
      r = __shfl(r, 0, 64);
      sw = __shfl(sw, 0, 64);
    }
    if ((tid & 63) == 0) {
      chan_r[w] = r;
      chan_s[w] = sw;
    }
  }
  __syncthreads();
  if (tid < 64) {
    const int o = t.ao_off[s];
    const int rb = same_channels ? chan_r[0] : chan_r[1];
    const double sb = same_channels ? chan_s[0] : chan_s[1];
    if ((chan_r[0] == 2 || rb == 2) && tid == 0) fo.st[s].status = 8;
    int last = 0;
    for (int i = tid; i < n; i += 64) {
      const double fa = fo.fa[o + i];
      const double fb = same_channels ? fa : fo.fb[o + i];
      if (same_channels) fo.fb[o + i] = fa;
      const double f = fa + fb;
      fo.occ[o + i] = f;
      fo.fe[o + i] = f * srt[i];
      if (f > kOccFloor) last = max(last, i + 1);
    }
    for (int off = 32; off > 0; off >>= 1) last = max(last, __shfl_xor(last, off, 64));
    if (tid == 0) {
      fo.st[s].entropy = chan_s[0] + sb;
      fo.st[s].kocc = last;
      fo.kocc[s] = last;
      kocc_sh = last;
    }
  }
  __syncthreads();
  return kocc_sh;
}

// Eigenvector of eigenvalue j below kocc, or of the cluster that j starts, by
// one thread.  A cluster is needed when its first (lowest) member is below
// kocc; every member of a needed cluster is computed so the cluster stays
// orthogonal.  An unsplit T is one block [0, n) of 1-norm tnorm1; split blocks
// are found and measured by the thread that needs them.
template <int U>
__device__ __forceinline__ void eig_vector(int j, int n, int kocc, const double* d, const double* e, const double* lam,
                                           const int* rnk, bool unsplit, double tnorm1, double pivmin,
                                           const EigenScratch& sc, int64_t mo, double* __restrict__ Z, double* zscale,
                                           const ClusterOut& co, int s, int o) {
  double* __restrict__ F0 = sc.u0 + mo;
  double* __restrict__ F1 = sc.u1 + mo;
  double* __restrict__ F2 = sc.u2 + mo;
  double* __restrict__ FM = sc.mult + mo;
  double* __restrict__ FP = sc.piv + mo;
  if (rnk[j] >= kocc) return;
  int b0 = j, b1 = j + 1;
  double onenrm = 0.0;
  if (unsplit) {
    b0 = 0;
    b1 = n;
    onenrm = tnorm1;
  } else {
    while (b0 > 0 && e[b0 - 1] != 0.0) --b0;
    while (b1 < n && e[b1 - 1] != 0.0) ++b1;
    for (int i = b0; i < b1; ++i)
      onenrm = fmax(onenrm, fabs(d[i]) + (i > b0 ? fabs(e[i - 1]) : 0.0) + (i + 1 < b1 ? fabs(e[i]) : 0.0));
  }
  const int bn = b1 - b0;
  const double gtol = kClusterTol * fmax(onenrm, kSafeMin);
  if (j > b0 && lam[j] - lam[j - 1] <= gtol) return;  // not a cluster start
  int g1 = j + 1;
  while (g1 < b1 && lam[g1] - lam[g1 - 1] <= gtol) ++g1;
  if (g1 - j > kSerialCluster) {  // the whole block orthogonalizes it (k_cluster_vectors)
    for (int jj = j; jj < g1; ++jj) {
      co.lam[o + jj] = lam[jj];
      co.rank[o + jj] = rnk[jj];
    }
    co.end[o + j] = g1;
    co.flag[s] = 1;
    return;
  }
  const double ptol = kEps * fmax(onenrm, kSafeMin);       // smallest admissible pivot
  const double pertol = 10.0 * kEps * fmax(onenrm, kSafeMin);
  double xprev = 0.0;
  for (int jj = j; jj < g1; ++jj) {
    const int cj = rnk[jj];  // Z column of eigenvalue jj
    // rows outside the block are zero
    for (int i = 0; i < b0; ++i) Z[(int64_t)i * n + cj] = 0.0;
    for (int i = b1; i < n; ++i) Z[(int64_t)i * n + cj] = 0.0;
    zscale[cj] = 1.0;
    if (bn == 1) {
      Z[(int64_t)b0 * n + cj] = 1.0;
      continue;
    }
    double x = lam[jj];
    if (jj > j && x - xprev < pertol) x = xprev + pertol;
    xprev = x;
    if (g1 - j == 1) {
      double f;
      if (twisted_vector(d, e, b0, b1, x, pivmin, n, cj, F0, F1, Z, f)) {
        zscale[cj] = f;
        continue;
      }
    }
    // LU with partial pivoting of T_b - x I
    double c0 = d[b0] - x, c1 = e[b0], c2 = 0.0;
    for (int k = 0; k < bn - 1; ++k) {
      const int gi = b0 + k;
      const double n0 = e[gi], n1 = d[gi + 1] - x, n2 = (k + 2 < bn) ? e[gi + 1] : 0.0;
      const int64_t at = (int64_t)gi * n + cj;
      if (fabs(c0) >= fabs(n0)) {
        const double m = c0 != 0.0 ? n0 / c0 : 0.0;
        F0[at] = c0; F1[at] = c1; F2[at] = c2; FM[at] = m; FP[at] = 0.0;
        c0 = n1 - m * c1;
        c1 = n2 - m * c2;
      } else {
        const double m = c0 / n0;
        F0[at] = n0; F1[at] = n1; F2[at] = n2; FM[at] = m; FP[at] = 1.0;
        const double t0 = c1 - m * n1, t1 = c2 - m * n2;
        c0 = t0;
        c1 = t1;
      }
      c2 = 0.0;
    }
    {
      const int64_t at = (int64_t)(b1 - 1) * n + cj;
      F0[at] = c0; F1[at] = 0.0; F2[at] = 0.0; FM[at] = 0.0; FP[at] = 0.0;
    }
    for (int i = b0; i < b1; ++i) Z[(int64_t)i * n + cj] = start_component(jj, i - b0);
    // The passes below read and write one column of global memory: U rows' loads
    // are in flight before the first of them is used.  k_eig_vectors takes eight:
    // close levels at 1142 AOs then hold its wavefront for 1.7 ms instead of 3.1.
    // k_tridiag_eigen takes one: eight cost it 90 VGPRs and a wavefront per SIMD
    // (1% of a call of 512 systems).
    auto scale_rows = [&](double f) __attribute__((always_inline)) {
      int i = b0;
      for (; i + U <= b1; i += U) {
        double v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = Z[(int64_t)(i + u) * n + cj];
#pragma unroll
        for (int u = 0; u < U; ++u) Z[(int64_t)(i + u) * n + cj] = v[u] * f;
      }
      for (; i < b1; ++i) Z[(int64_t)i * n + cj] *= f;
    };
    for (int it = 0; it <= kInverseIterations; ++it) {
      // orthogonalize against the cluster members already finished
      for (int p = j; p < jj; ++p) {
        const int cp = rnk[p];
        double dot = 0.0;
#pragma unroll U
        for (int i = b0; i < b1; ++i) dot += Z[(int64_t)i * n + cp] * Z[(int64_t)i * n + cj];
        int i = b0;
        for (; i + U <= b1; i += U) {
          double v[U], w[U];
#pragma unroll
          for (int u = 0; u < U; ++u) {
            v[u] = Z[(int64_t)(i + u) * n + cj];
            w[u] = Z[(int64_t)(i + u) * n + cp];
          }
#pragma unroll
          for (int u = 0; u < U; ++u) Z[(int64_t)(i + u) * n + cj] = v[u] - dot * w[u];
        }
        for (; i < b1; ++i) Z[(int64_t)i * n + cj] -= dot * Z[(int64_t)i * n + cp];
      }
      if (it == kInverseIterations) break;
      // scale to unit max-norm, then solve (T_b - x I) y = r
      double rmax = 0.0;
#pragma unroll U
      for (int i = b0; i < b1; ++i) rmax = fmax(rmax, fabs(Z[(int64_t)i * n + cj]));
      const double rs = rmax > 0.0 ? 1.0 / rmax : 1.0;
      // forward elimination; the running entry stays in a register (it is
      // the one stored one row earlier), so only independent loads remain
      {
        double cur = Z[(int64_t)b0 * n + cj] * rs;
        auto step = [&](int64_t at, double zn, double fp, double fm) __attribute__((always_inline)) {
          double rk = cur, rn = zn * rs;
          if (fp != 0.0) { const double tmp = rk; rk = rn; rn = tmp; }
          Z[at] = rk;
          cur = rn - fm * rk;
        };
        int k = 0;
        for (; k + U <= bn - 1; k += U) {
          double zn[U], fp[U], fm[U];
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const int64_t at = (int64_t)(b0 + k + u) * n + cj;
            zn[u] = Z[at + n];
            fp[u] = FP[at];
            fm[u] = FM[at];
          }
#pragma unroll
          for (int u = 0; u < U; ++u) step((int64_t)(b0 + k + u) * n + cj, zn[u], fp[u], fm[u]);
        }
        for (; k < bn - 1; ++k) {
          const int64_t at = (int64_t)(b0 + k) * n + cj;
          step(at, Z[at + n], FP[at], FM[at]);
        }
        Z[(int64_t)(b1 - 1) * n + cj] = cur;
      }
      // back substitution with the two entries below in registers (F1 of the
      // last row and F2 of the last two are zero)
      {
        double z1 = 0.0, z2 = 0.0;  // solution entries k + 1, k + 2
        auto step = [&](int64_t at, double r, double f0, double f1, double f2) __attribute__((always_inline)) {
          r -= f1 * z1;
          r -= f2 * z2;
          double u = f0;
          if (fabs(u) < ptol) u = u < 0.0 ? -ptol : ptol;
          const double zk = r / u;
          Z[at] = zk;
          z2 = z1;
          z1 = zk;
        };
        int k = bn - 1;
        for (; k - U + 1 >= 0; k -= U) {
          double r[U], f0[U], f1[U], f2[U];
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const int64_t at = (int64_t)(b0 + k - u) * n + cj;
            r[u] = Z[at];
            f0[u] = F0[at];
            f1[u] = F1[at];
            f2[u] = F2[at];
          }
#pragma unroll
          for (int u = 0; u < U; ++u) step((int64_t)(b0 + k - u) * n + cj, r[u], f0[u], f1[u], f2[u]);
        }
        for (; k >= 0; --k) {
          const int64_t at = (int64_t)(b0 + k) * n + cj;
          step(at, Z[at], F0[at], F1[at], F2[at]);
        }
      }
      // normalize
      double nrm = 0.0, ymax = 0.0;
#pragma unroll U
      for (int i = b0; i < b1; ++i) ymax = fmax(ymax, fabs(Z[(int64_t)i * n + cj]));
      const double ys = ymax > 0.0 ? 1.0 / ymax : 1.0;
#pragma unroll U
      for (int i = b0; i < b1; ++i) {
        const double y = Z[(int64_t)i * n + cj] * ys;
        nrm += y * y;
      }
      scale_rows(ys / sqrt(nrm));
    }
    // final normalization; sign: largest-magnitude component positive
    double nrm = 0.0, big = 0.0;
#pragma unroll U
    for (int i = b0; i < b1; ++i) {
      const double y = Z[(int64_t)i * n + cj];
      nrm += y * y;
      if (fabs(y) > fabs(big)) big = y;
    }
    scale_rows((big < 0.0 ? -1.0 : 1.0) / sqrt(nrm));
  }
}

// Eigenvalues of T (all), then the Fermi occupations, then eigenvectors for the
// kocc lowest eigenvalues only, written to Z column = ascending rank.
// From the second SCC round on, wall holds the previous round's ascending
// eigenvalues on entry; shift[s] carries the largest eigenvalue change of the
// system's previous round (written here for the next one).  BIG: the systems
// above kEigSplitAO AOs, with d, e, e^2, the eigenvalues and their ranks in their
// global slice of `big`.  Clusters of more than kSerialCluster close
// eigenvalues are left to k_cluster_vectors through `co`.
template <bool BIG>
__global__ __launch_bounds__(256) void k_tridiag_eigen(Topo t, const int* order,
                                                       const unsigned char* active,
                                                       const double* dall, const double* eall,
                                                       double* Zall, EigenScratch sc,
                                                       double* wall, double* shift, int round_arg,
                                                       const int* round_ptr,
                                                       double* zscale_all, FermiOut fo, double* big,
                                                       ClusterOut co) {
  const int s = order[blockIdx.x];
  if (active && !active[s]) return;
  const int n = t.ao_off[s + 1] - t.ao_off[s];
  const int64_t mo = t.mat_off[s];
  double* zscale = zscale_all + t.ao_off[s];
  __shared__ double d_l[BIG ? 1 : kMaxAO];
  __shared__ double e_l[BIG ? 1 : kMaxAO];   // split off-diagonal (negligible entries zeroed)
  __shared__ double e2_l[BIG ? 1 : kMaxAO];
  __shared__ double lam_l[BIG ? 1 : kMaxAO];
  double *d = d_l, *e = e_l, *e2 = e2_l, *lam = lam_l;
  if constexpr (BIG) {
    d = big + big_offset(t, s);  // d, e, e2, lam, rnk: 5 n <= kBigPerAO n doubles
    e = d + n;
    e2 = e + n;
    lam = e2 + n;
  }
  __shared__ double red[16];
  const int tid = threadIdx.x, nt = blockDim.x;
  if (tid == 0) co.flag[s] = 0;
  __shared__ int nsplit, next_j;
  if (tid == 0) next_j = 0;
  double pivmin;
  const bool unsplit = eig_load(dall + t.ao_off[s], eall + t.ao_off[s], n, d, e, e2, red, nsplit, pivmin);
  // the SCC round: the launch argument, or the device-resident counter of
  // rounds enqueued ahead of the host (graph-captured rounds)
  const int round = round_ptr ? *round_ptr : round_arg;
  const bool have_old = round >= 1 && unsplit;
  const bool guess_ok = round >= 2 && unsplit;
  const double delta = guess_ok ? 2.0 * shift[s] : 0.0;
  // whole-matrix Gershgorin bounds (used when T is unsplit)
  __shared__ double gbound[3];
  if (unsplit) eig_bounds(d, e, n, pivmin, red, gbound);
  double dmax = 0.0;
  {
    EigState st;
    bool busy = false;
    for (;;) {
      if (!busy) {
        const int j = atomicAdd(&next_j, 1);
        if (j >= n) break;
        const double* wo = wall + t.ao_off[s];
        const double g = have_old ? wo[j] : 0.0;
        const double gp = (have_old && j > 0) ? wo[j - 1] : -1e300;
        const double gn = (have_old && j + 1 < n) ? wo[j + 1] : 1e300;
        busy = eig_start(st, j, d, e, n, pivmin, unsplit, gbound[0], gbound[1], gbound[2], guess_ok,
                         g, gp, gn, delta, lam);
        if (!busy) continue;
      }
      double x;
      if (eig_step(st, d, e2, x)) {
        lam[st.j] = x;
        if (have_old) dmax = fmax(dmax, fabs(x - wall[t.ao_off[s] + st.j]));
        busy = false;
      }
    }
  }
  // largest eigenvalue change of this round (block max), for the next round's brackets
  for (int off = 32; off > 0; off >>= 1) dmax = fmax(dmax, __shfl_xor(dmax, off, 64));
  __syncthreads();
  if ((tid & 63) == 0) red[tid >> 6] = dmax;
  __syncthreads();
  if (tid == 0) {
    double m = 0.0;
    for (int w = 0; w < (nt >> 6); ++w) m = fmax(m, red[w]);
    // first round: no change measured yet, take a generous bracket
    shift[s] = have_old ? m : 1.0;
  }
  __syncthreads();

  __shared__ int rnk_l[BIG ? 1 : kMaxAO];
  int* rnk = BIG ? reinterpret_cast<int*>(lam + n) : rnk_l;
  double* srt = e2;  // e2 is not needed after the eigenvalues
  const int kocc = eig_occupations(t, s, n, lam, rnk, srt, wall + t.ao_off[s], fo);

  // ---- eigenvectors: thread per cluster start ----
  __shared__ double tnorm1;
  if (unsplit) eig_norm1(d, e, n, red, tnorm1);
  for (int j = tid; j < n; j += nt)
    eig_vector<1>(j, n, kocc, d, e, lam, rnk, unsplit, tnorm1, pivmin, sc, mo, Zall + mo, zscale, co, s, t.ao_off[s]);
}

// Block-wide maximum (blockDim.x <= 1024; red holds blockDim.x / 64 doubles).
__device__ __forceinline__ double block_max(double v, double* red) {
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  __syncthreads();
  if (lane == 0) red[wid] = v;
  __syncthreads();
  double m = red[0];
  for (int i = 1; i < nw; ++i) m = fmax(m, red[i]);
  __syncthreads();
  return m;
}

// 256 < n <= kEigSplitAO: the same three stages as launches of their own, so that
// a system's eigenvalues and vectors spread over the chip: one wavefront per 64
// eigenvalues, one block per system for ranks and occupations, one wavefront per
// 64 vectors.  Between the launches the eigenvalues (in T's order) and ranks sit
// in the system's slot of `lam_all` (the Y matrix, free until the
// back-transformation).  Larger systems run k_tridiag_eigen<true>.
//
// Bound: the serial chains of a lane (about nine Sturm passes, four recurrences
// of n rows).  Measured against one 256-thread block per system: 7.8 -> 1.5 ms
// a launch at 1142 AOs (eigenvalues 0.82, occupations 0.16, vectors 0.49; a
// geometry whose close eigenvalues need inverse iteration takes 1.7 for the
// vectors), 0.74 -> 0.45 ms for 14 systems of 258-482 AOs.
constexpr int kEigSplitAO = 2048;

__global__ __launch_bounds__(64) void k_eig_values(Topo t, const int* order, const unsigned char* active,
                                                   const double* dall, const double* eall, const double* wall,
                                                   const double* shift, int round_arg, const int* round_ptr,
                                                   double* lam_all) {
  const int s = order[blockIdx.y];
  if (active && !active[s]) return;
  const int n = t.ao_off[s + 1] - t.ao_off[s];
  if (64 * (int)blockIdx.x >= n) return;
  __shared__ double d[kEigSplitAO], e[kEigSplitAO], e2[kEigSplitAO];
  __shared__ double red[16], gbound[3];
  __shared__ int nsplit;
  double pivmin;
  const bool unsplit = eig_load(dall + t.ao_off[s], eall + t.ao_off[s], n, d, e, e2, red, nsplit, pivmin);
  if (unsplit) eig_bounds(d, e, n, pivmin, red, gbound);
  const int round = round_ptr ? *round_ptr : round_arg;
  const bool have_old = round >= 1 && unsplit, guess_ok = round >= 2 && unsplit;
  const double delta = guess_ok ? 2.0 * shift[s] : 0.0;
  double* lam = lam_all + t.mat_off[s];
  const int j = 64 * blockIdx.x + threadIdx.x;
  if (j >= n) return;
  const double* wo = wall + t.ao_off[s];
  EigState st;
  if (!eig_start(st, j, d, e, n, pivmin, unsplit, gbound[0], gbound[1], gbound[2], guess_ok, have_old ? wo[j] : 0.0,
                 have_old && j > 0 ? wo[j - 1] : -1e300, have_old && j + 1 < n ? wo[j + 1] : 1e300, delta, lam))
    return;
  double x;
  while (!eig_step(st, d, e2, x)) {}
  lam[j] = x;
}

__global__ __launch_bounds__(256) void k_eig_occupations(Topo t, const int* order, const unsigned char* active,
                                                         const double* dall, const double* eall, double* wall,
                                                         double* shift, int round_arg, const int* round_ptr,
                                                         double* lam_all, FermiOut fo, ClusterOut co) {
  const int s = order[blockIdx.x];
  if (active && !active[s]) return;
  const int n = t.ao_off[s + 1] - t.ao_off[s];
  const int tid = threadIdx.x, nt = blockDim.x;
  __shared__ double lam[kEigSplitAO], srt[kEigSplitAO];
  __shared__ int rnk[kEigSplitAO];
  __shared__ double red[16];
  double* lam_g = lam_all + t.mat_off[s];
  double* w = wall + t.ao_off[s];
  const double* dg = dall + t.ao_off[s];
  const double* eg = eall + t.ao_off[s];
  if (tid == 0) co.flag[s] = 0;
  const int round = round_ptr ? *round_ptr : round_arg;
  // the largest eigenvalue change of this round, for the next round's brackets;
  // a T that split gives none (its eigenvalues are not in ascending order)
  double dmax = 0.0;
  int cut = 0;
  for (int i = tid; i < n; i += nt) {
    lam[i] = lam_g[i];
    if (round >= 1) dmax = fmax(dmax, fabs(lam[i] - w[i]));
    if (i + 1 < n && eg[i] * eg[i] <= kEps * kEps * fabs(dg[i] * dg[i + 1]) + kSafeMin) cut = 1;
  }
  dmax = block_max(dmax, red);
  const bool unsplit = !__syncthreads_or(cut);
  if (tid == 0) shift[s] = round >= 1 && unsplit ? dmax : 1.0;
  __syncthreads();
  eig_occupations(t, s, n, lam, rnk, srt, w, fo);
  int* rnk_g = reinterpret_cast<int*>(lam_g + n);
  for (int i = tid; i < n; i += nt) rnk_g[i] = rnk[i];
}

__global__ __launch_bounds__(64) void k_eig_vectors(Topo t, const int* order, const unsigned char* active,
                                                    const double* dall, const double* eall, const double* lam_all,
                                                    double* Zall, EigenScratch sc, double* zscale_all,
                                                    const int* kocc_all, ClusterOut co) {
  const int s = order[blockIdx.y];
  if (active && !active[s]) return;
  const int n = t.ao_off[s + 1] - t.ao_off[s];
  if (64 * (int)blockIdx.x >= n) return;
  const int kocc = kocc_all[s];
  __shared__ double d[kEigSplitAO], e[kEigSplitAO], lam[kEigSplitAO];  // lam holds e^2 first
  __shared__ int rnk[kEigSplitAO];
  __shared__ double red[16], tnorm1;
  __shared__ int nsplit;
  double pivmin;
  const bool unsplit = eig_load(dall + t.ao_off[s], eall + t.ao_off[s], n, d, e, lam, red, nsplit, pivmin);
  if (unsplit) eig_norm1(d, e, n, red, tnorm1);
  const int64_t mo = t.mat_off[s];
  const double* lam_g = lam_all + mo;
  const int* rnk_g = reinterpret_cast<const int*>(lam_g + n);
  for (int i = threadIdx.x; i < n; i += 64) {
    lam[i] = lam_g[i];
    rnk[i] = rnk_g[i];
  }
  __syncthreads();
  const int j = 64 * blockIdx.x + threadIdx.x;
  if (j < n)
    eig_vector<8>(j, n, kocc, d, e, lam, rnk, unsplit, tnorm1, pivmin, sc, mo, Zall + mo, zscale_all + t.ao_off[s], co, s,
               t.ao_off[s]);
}

// Eigenvectors of the clusters k_tridiag_eigen hands over (more than
// kSerialCluster members), one 256-thread block per system with such a
// cluster.  The vectors follow the serial path's inverse iteration: the same
// shift perturbation, partially pivoted LU of T_b - x I and start vector, the
// same iteration count, normalization and sign.  The orthogonalization
// against the cluster's earlier vectors runs on the whole block as classical
// Gram-Schmidt applied twice, over chunks of kCoopChunk earlier vectors (their
// dots a thread per vector, the update a thread per row); only the LU and the
// two substitutions (O(n) per vector) stay on one thread.  T's splitting, the
// block norms are recomputed from d and e as k_tridiag_eigen forms them.
constexpr int kCoopChunk = 256;

__global__ __launch_bounds__(256) void k_cluster_vectors(Topo t, const int* order, const unsigned char* active,
                                                         const double* dall, const double* eall, double* Zall,
                                                         EigenScratch sc, double* zscale_all, ClusterOut co) {
  const int s = order[blockIdx.x];
  if ((active && !active[s]) || !co.flag[s]) return;
  const int o = t.ao_off[s], n = t.ao_off[s + 1] - o;
  const int64_t mo = t.mat_off[s];
  double* __restrict__ Z = Zall + mo;
  double* __restrict__ F0 = sc.u0 + mo;
  double* __restrict__ F1 = sc.u1 + mo;
  double* __restrict__ F2 = sc.u2 + mo;
  double* __restrict__ FM = sc.mult + mo;
  double* __restrict__ FP = sc.piv + mo;
  double* zscale = zscale_all + o;
  const double* d = dall + o;
  const int tid = threadIdx.x, nt = blockDim.x;
  __shared__ double red[16];
  __shared__ int ired[16];
  __shared__ double dots[kCoopChunk];
  // off-diagonal after the split (negligible entries zeroed)
  auto esp = [&](int i) -> double {
    if (i + 1 >= n) return 0.0;
    double ei = eall[o + i];
    if (ei * ei <= kEps * kEps * fabs(d[i] * d[i + 1]) + kSafeMin) ei = 0.0;
    return ei * ei == 0.0 ? 0.0 : ei;
  };
  double rows1 = 0.0, splits = 0.0;
  for (int i = tid; i < n; i += nt) {
    const double ei = esp(i), ep = i > 0 ? esp(i - 1) : 0.0;
    rows1 = fmax(rows1, fabs(d[i]) + fabs(ep) + fabs(ei));
    if (i + 1 < n && ei == 0.0) splits += 1.0;
  }
  const double tnorm1 = block_max(rows1, red);
  const bool unsplit = block_sum(splits, red) == 0.0;
  for (int j = 0; j < n; ++j) {
    const int g1 = co.end[o + j];
    if (g1 == 0) continue;
    int b0 = j, b1 = j + 1;
    double onenrm = 0.0;
    if (unsplit) {
      b0 = 0;
      b1 = n;
      onenrm = tnorm1;
    } else {
      while (b0 > 0 && esp(b0 - 1) != 0.0) --b0;
      while (b1 < n && esp(b1 - 1) != 0.0) ++b1;
      for (int i = b0; i < b1; ++i)
        onenrm = fmax(onenrm, fabs(d[i]) + (i > b0 ? fabs(esp(i - 1)) : 0.0) + (i + 1 < b1 ? fabs(esp(i)) : 0.0));
    }
    const int bn = b1 - b0;
    const double ptol = kEps * fmax(onenrm, kSafeMin);
    const double pertol = 10.0 * kEps * fmax(onenrm, kSafeMin);
    double xprev = 0.0;
    for (int jj = j; jj < g1; ++jj) {
      const int cj = co.rank[o + jj];
      for (int i = tid; i < n; i += nt)
        if (i < b0 || i >= b1) Z[(int64_t)i * n + cj] = 0.0;
      if (tid == 0) zscale[cj] = 1.0;
      double x = co.lam[o + jj];
      if (jj > j && x - xprev < pertol) x = xprev + pertol;
      xprev = x;
      if (bn == 1) {
        if (tid == 0) Z[(int64_t)b0 * n + cj] = 1.0;
        __syncthreads();
        continue;
      }
      if (tid == 0) {  // LU with partial pivoting of T_b - x I
        double c0 = d[b0] - x, c1 = esp(b0), c2 = 0.0;
        for (int k = 0; k < bn - 1; ++k) {
          const int gi = b0 + k;
          const double n0 = esp(gi), n1 = d[gi + 1] - x, n2 = (k + 2 < bn) ? esp(gi + 1) : 0.0;
          const int64_t at = (int64_t)gi * n + cj;
          if (fabs(c0) >= fabs(n0)) {
            const double m = c0 != 0.0 ? n0 / c0 : 0.0;
            F0[at] = c0; F1[at] = c1; F2[at] = c2; FM[at] = m; FP[at] = 0.0;
            c0 = n1 - m * c1;
            c1 = n2 - m * c2;
          } else {
            const double m = c0 / n0;
            F0[at] = n0; F1[at] = n1; F2[at] = n2; FM[at] = m; FP[at] = 1.0;
            const double t0 = c1 - m * n1, t1 = c2 - m * n2;
            c0 = t0;
            c1 = t1;
          }
          c2 = 0.0;
        }
        const int64_t at = (int64_t)(b1 - 1) * n + cj;
        F0[at] = c0; F1[at] = 0.0; F2[at] = 0.0; FM[at] = 0.0; FP[at] = 0.0;
      }
      for (int i = b0 + tid; i < b1; i += nt) Z[(int64_t)i * n + cj] = start_component(jj, i - b0);
      __syncthreads();
      for (int it = 0; it <= kInverseIterations; ++it) {
        // orthogonalize against the cluster members already finished (CGS twice)
        for (int pass = 0; pass < 2; ++pass)
          for (int p0 = j; p0 < jj; p0 += kCoopChunk) {
            const int pe = min(jj, p0 + kCoopChunk);
            for (int p = p0 + tid; p < pe; p += nt) {
              const int cp = co.rank[o + p];
              double dot = 0.0;
              for (int i = b0; i < b1; ++i) dot = fma(Z[(int64_t)i * n + cp], Z[(int64_t)i * n + cj], dot);
              dots[p - p0] = dot;
            }
            __syncthreads();
            for (int i = b0 + tid; i < b1; i += nt) {
              double z = Z[(int64_t)i * n + cj];
              for (int p = p0; p < pe; ++p) z = fma(-dots[p - p0], Z[(int64_t)i * n + co.rank[o + p]], z);
              Z[(int64_t)i * n + cj] = z;
            }
            __syncthreads();
          }
        if (it == kInverseIterations) break;
        // scale to unit max-norm, then solve (T_b - x I) y = r
        double rmax = 0.0;
        for (int i = b0 + tid; i < b1; i += nt) rmax = fmax(rmax, fabs(Z[(int64_t)i * n + cj]));
        rmax = block_max(rmax, red);
        const double rs = rmax > 0.0 ? 1.0 / rmax : 1.0;
        for (int i = b0 + tid; i < b1; i += nt) Z[(int64_t)i * n + cj] *= rs;
        __syncthreads();
        if (tid == 0) {
          double cur = Z[(int64_t)b0 * n + cj];
          for (int k = 0; k < bn - 1; ++k) {
            const int64_t at = (int64_t)(b0 + k) * n + cj;
            double rk = cur, rn = Z[at + n];
            if (FP[at] != 0.0) { const double tmp = rk; rk = rn; rn = tmp; }
            Z[at] = rk;
            cur = rn - FM[at] * rk;
          }
          Z[(int64_t)(b1 - 1) * n + cj] = cur;
          double z1 = 0.0, z2 = 0.0;
          for (int k = bn - 1; k >= 0; --k) {
            const int64_t at = (int64_t)(b0 + k) * n + cj;
            double r = Z[at];
            if (k + 1 < bn) r -= F1[at] * z1;
            if (k + 2 < bn) r -= F2[at] * z2;
            double u = F0[at];
            if (fabs(u) < ptol) u = u < 0.0 ? -ptol : ptol;
            const double zk = r / u;
            Z[at] = zk;
            z2 = z1;
            z1 = zk;
          }
        }
        __syncthreads();
        // normalize
        double ymax = 0.0;
        for (int i = b0 + tid; i < b1; i += nt) ymax = fmax(ymax, fabs(Z[(int64_t)i * n + cj]));
        ymax = block_max(ymax, red);
        const double ys = ymax > 0.0 ? 1.0 / ymax : 1.0;
        double nrm = 0.0;
        for (int i = b0 + tid; i < b1; i += nt) {
          const double y = Z[(int64_t)i * n + cj] * ys;
          nrm += y * y;
        }
        nrm = block_sum(nrm, red);
        const double sc2 = ys / sqrt(nrm);
        for (int i = b0 + tid; i < b1; i += nt) Z[(int64_t)i * n + cj] *= sc2;
        __syncthreads();
      }
      // final normalization; sign: the first largest-magnitude component positive
      double nrm = 0.0, big = 0.0;
      int bi = n;
      for (int i = b0 + tid; i < b1; i += nt) {
        const double y = Z[(int64_t)i * n + cj];
        nrm += y * y;
        if (fabs(y) > fabs(big)) { big = y; bi = i; }
      }
      nrm = block_sum(nrm, red);
      for (int off = 32; off > 0; off >>= 1) {
        const double ob = __shfl_xor(big, off, 64);
        const int oi = __shfl_xor(bi, off, 64);
        if (fabs(ob) > fabs(big) || (fabs(ob) == fabs(big) && oi < bi)) { big = ob; bi = oi; }
      }
      if ((tid & 63) == 0) { red[tid >> 6] = big; ired[tid >> 6] = bi; }
      __syncthreads();
      big = red[0];
      bi = ired[0];
      for (int w = 1; w < (nt >> 6); ++w)
        if (fabs(red[w]) > fabs(big) || (fabs(red[w]) == fabs(big) && ired[w] < bi)) { big = red[w]; bi = ired[w]; }
      __syncthreads();
      const double f = (big < 0.0 ? -1.0 : 1.0) / sqrt(nrm);
      for (int i = b0 + tid; i < b1; i += nt) Z[(int64_t)i * n + cj] *= f;
      __syncthreads();
    }
    if (tid == 0) co.end[o + j] = 0;  // consumed
  }
}

// One block's columns of the back-transformation, from j0 on; those at or past the
// system's kocc are left out (Z holds eigenvectors by ascending rank).
struct BackTask {
  int sys;
  int j0;
};

// T[m][u] of a WY block with the packed factor To (u, m < 16); rows past the
// block's last reflector are never used (their column of V is zero)
__device__ __forceinline__ double wy_entry(const double* To, int m, int u, int cnt) {
  const bool low = u < m && m < cnt;
  const double x = To[low ? m * (m - 1) / 2 + u : 0];
  return low ? x : (m == u ? 2.0 : 0.0);
}

// Y = Q Z, n <= 256, the occupied columns.  256 threads; each wavefront holds
// 16 columns whole in registers, tile t = rows 16 t .. 16 t + 15 in the
// accumulator layout of v_mfma_f64_16x16x4f64 (lane: column lane % 16, rows
// 16 t + lane / 16 + 4 r).  Register r of tile t is then exactly the B operand
// of the K step over rows 16 t + 4 r .. + 3, so
//   w = V^T z,  y = T w,  z -= V y
// run on the matrix cores with no data moved between lanes or wavefronts.  The
// block's four wavefronts share the WY block's reflectors, staged in LDS one
// block ahead (zero on and above their subdiagonal; row stride 260: the 16 x 4
// operand reads of w spread over all banks): one barrier per 16 reflectors.
//
// Bound: FP64 matrix cores (2 n^2 kocc flop, 16 x 16 tiles) for large batches,
// the serial chain of a wavefront's products for small ones.  Measured against
// blocks of eight reflectors on the vector units with four block barriers each:
// 74 -> 34 us for one system of 122 AOs, 314 -> 160 us a round for 512 systems
// of 14-235 AOs.
constexpr int kBackThreads = 256;
constexpr int kBackCols = 64;   // columns of one block
constexpr int kBackTiles = 16;  // row tiles (n <= 256)
constexpr int kBackLd = 260;

__global__ __launch_bounds__(kBackThreads, 2) void k_backtransform(Topo t, const BackTask* tasks,
                                                                   const double* Aall, const double* Zall,
                                                                   const double* Tall, double* Yall,
                                                                   const int* kocc_all,
                                                                   const double* zscale_all,
                                                                   const unsigned char* active) {
  __shared__ double vs[2][kWyBlock * kBackLd];
  const BackTask task = tasks[blockIdx.x];
  const int s = task.sys;
  if (active && !active[s]) return;
  const int n = t.ao_off[s + 1] - t.ao_off[s];
  const int kocc = kocc_all[s];
  if (task.j0 >= kocc) return;
  const int64_t mo = t.mat_off[s];
  const double* __restrict__ A = Aall + mo;
  const double* __restrict__ Z = Zall + mo;
  double* __restrict__ Y = Yall + mo;
  const double* __restrict__ Tf = Tall + wy_offset(t, s);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lk = lane >> 4;
  const int col = task.j0 + 16 * w + l16;
  const bool on = col < kocc, live = task.j0 + 16 * w < kocc;  // live: any column of the wavefront
  const int nt = (n + 15) >> 4;
  mfma_d4 z[kBackTiles];
  const double f = on ? zscale_all[t.ao_off[s] + col] : 0.0;
#pragma unroll
  for (int i = 0; i < kBackTiles; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * i + lk + 4 * r;
      z[i][r] = (on && row < n) ? f * Z[(int64_t)row * n + col] : 0.0;
      if (r == 3 && i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
  double fr[kWyBlock];  // the next block's reflectors, row tid
  auto fetch = [&](int ch) __attribute__((always_inline)) {
    const int kb = n - 3 - kWyBlock * ch;
#pragma unroll
    for (int u = 0; u < kWyBlock; ++u) {
      const int k = kb - u;
      fr[u] = (k >= 0 && tid > k && tid < n) ? A[tid + (int64_t)k * n] : 0.0;
    }
  };
  auto stage = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kWyBlock; ++u) vs[buf][u * kBackLd + tid] = fr[u];
  };
  const int nch = (n - 2 + kWyBlock - 1) / kWyBlock;  // n - 2 reflectors
  if (nch > 0) {
    fetch(0);
    stage(0);
  }
  __syncthreads();
  for (int ch = 0; ch < nch; ++ch) {
    const bool more = ch + 1 < nch;
    if (more) fetch(ch + 1);  // in flight while this block is applied
    if (live) {
      const double* hv = vs[ch & 1];
      const int kb = n - 3 - kWyBlock * ch, cnt = min(kWyBlock, kb + 1);
      const int t0 = (max(kb - (kWyBlock - 1), 0) + 1) >> 4;  // first row tile the block touches
      double tt[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) tt[q] = wy_entry(Tf + kWyPacked * ch, l16, 4 * q + lk, cnt);
      mfma_d4 wa = mfma_d4{0.0, 0.0, 0.0, 0.0}, wb = wa;
#pragma unroll
      for (int i = 0; i < kBackTiles; ++i) {
        if (i >= t0 && i < nt) {
          double a[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) a[r] = hv[l16 * kBackLd + 16 * i + 4 * r + lk];
          wa = mfma_16x16x4(a[0], z[i][0], wa);
          wb = mfma_16x16x4(a[1], z[i][1], wb);
          wa = mfma_16x16x4(a[2], z[i][2], wa);
          wb = mfma_16x16x4(a[3], z[i][3], wb);
        }
      }
      mfma_d4 y = mfma_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int q = 0; q < 4; ++q) y = mfma_16x16x4(-tt[q], wa[q] + wb[q], y);
#pragma unroll
      for (int i = 0; i < kBackTiles; ++i) {
        if (i >= t0 && i < nt) {
          double a[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) a[q] = hv[(4 * q + lk) * kBackLd + 16 * i + l16];
#pragma unroll
          for (int q = 0; q < 4; ++q) z[i] = mfma_16x16x4(a[q], y[q], z[i]);
        }
      }
    }
    if (more) stage((ch + 1) & 1);
    __syncthreads();
  }
  if (on) {
#pragma unroll
    for (int i = 0; i < kBackTiles; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * i + lk + 4 * r;
        if (row < n) Y[(int64_t)row * n + col] = z[i][r];
      }
  }
}

// T factors of the systems above 256 AOs (the register reduction forms its
// own) after the blocked reduction: blockIdx.y covers eight WY blocks, one per
// wavefront.
__global__ __launch_bounds__(512) void k_wy_factors(Topo t, const int* order, const double* Aall,
                                                    double* Tall, const unsigned char* active) {
  __shared__ double g[8][kWyBlock * kWyBlock];
  const int s = order[blockIdx.x];
  if (active && !active[s]) return;
  const int n = t.ao_off[s + 1] - t.ao_off[s];
  const int wv = threadIdx.x >> 6, ch = 8 * blockIdx.y + wv;
  if (kWyBlock * ch < n - 2) wy_factor(Aall + t.mat_off[s], n, ch, Tall + wy_offset(t, s), g[wv]);
}

// Y = Q Z, n > 256: the same products on 16 columns, whose row tiles are dealt
// to the block's eight wavefronts (tile w + 8 q).  The wavefronts' partial w
// meet in LDS: two barriers per WY block; y is formed redundantly.  Each
// wavefront reads only the reflector rows of its own tiles, straight from A
// (issued before the barriers, so that L2's latency overlaps the products).
// MT row tiles per wavefront in registers (n <= 128 MT); MT = 0 keeps the
// columns in Y.  Measured against eight reflectors at a time on the vector
// units: 10.6 -> 0.53 ms at 1142 AOs (0.70 with MT = 16, which spills twice as
// much as MT = 12), 375 -> 96 us for 14 systems of 258-482 AOs.
constexpr int kWyThreads = 512;
constexpr int kWyCols = 16;

template <int MT>
__global__ __launch_bounds__(kWyThreads) void k_backtransform_wy(Topo t, const BackTask* tasks,
                                                                 const double* Aall, const double* Zall,
                                                                 const double* Tall, double* Yall,
                                                                 const int* kocc_all, const double* zscale_all,
                                                                 const unsigned char* active) {
  __shared__ double part[8][kWyBlock * kWyCols];
  __shared__ double wsum[kWyBlock * kWyCols];
  const BackTask task = tasks[blockIdx.x];
  const int s = task.sys;
  if (active && !active[s]) return;
  const int n = t.ao_off[s + 1] - t.ao_off[s];
  const int kocc = kocc_all[s];
  if (task.j0 >= kocc) return;
  const int64_t mo = t.mat_off[s];
  const double* __restrict__ A = Aall + mo;
  const double* __restrict__ Z = Zall + mo;
  double* Y = Yall + mo;
  const double* __restrict__ Tf = Tall + wy_offset(t, s);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lk = lane >> 4;
  const int col = task.j0 + l16;
  const bool on = col < kocc;
  const int nt = (n + 15) >> 4;
  const double f = on ? zscale_all[t.ao_off[s] + col] : 0.0;
  constexpr int kQ = MT > 0 ? MT : 1;
  mfma_d4 z[kQ];
  auto at = [&](int i, int r) __attribute__((always_inline)) { return (int64_t)(16 * i + lk + 4 * r) * n + col; };
  if constexpr (MT > 0) {
#pragma unroll
    for (int q = 0; q < MT; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        z[q][r] = (on && 16 * (w + 8 * q) + lk + 4 * r < n) ? f * Z[at(w + 8 * q, r)] : 0.0;
        if (MT > 8 && r == 3 && q % 4 == 3) __builtin_amdgcn_sched_barrier(0);
      }
  } else {
    if (on)
      for (int i = w; i < nt; i += 8)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (16 * i + lk + 4 * r < n) Y[at(i, r)] = f * Z[at(i, r)];
  }
  const int nch = (n - 2 + kWyBlock - 1) / kWyBlock;
  for (int ch = 0; ch < nch; ++ch) {
    const int kb = n - 3 - kWyBlock * ch, cnt = min(kWyBlock, kb + 1);
    const int t0 = (max(kb - (kWyBlock - 1), 0) + 1) >> 4;
    // operand of w: V[row 16 i + 4 r + lk][u = l16]; of the update:
    // V[row 16 i + l16][u = 4 q + lk].  Addresses are clamped into A, values masked.
    const int ku = kb - l16;
    const double* vu = A + (int64_t)max(ku, 0) * n;
    auto w_op = [&](int i, double (&a)[4]) __attribute__((always_inline)) {
#pragma unroll
      for (int r = 0; r < 4; ++r) a[r] = vu[min(16 * i + 4 * r + lk, n - 1)];
    };
    auto w_mask = [&](int i, double (&a)[4]) __attribute__((always_inline)) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * i + 4 * r + lk;
        a[r] = (ku >= 0 && row > ku && row < n) ? a[r] : 0.0;
      }
    };
    auto u_op = [&](int i, double (&a)[4]) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < 4; ++q) a[q] = A[min(16 * i + l16, n - 1) + (int64_t)max(kb - (4 * q + lk), 0) * n];
    };
    auto u_mask = [&](int i, double (&a)[4]) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int k = kb - (4 * q + lk), row = 16 * i + l16;
        a[q] = (k >= 0 && row > k && row < n) ? a[q] : 0.0;
      }
    };
    double tt[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) tt[q] = wy_entry(Tf + (int64_t)kWyPacked * ch, l16, 4 * q + lk, cnt);
    mfma_d4 wa = mfma_d4{0.0, 0.0, 0.0, 0.0}, wb = wa;
    if constexpr (MT > 0) {
#pragma unroll
      for (int q = 0; q < MT; ++q) {
        const int i = w + 8 * q;
        if (i >= t0 && i < nt) {
          double a[4];
          w_op(i, a);
          w_mask(i, a);
          wa = mfma_16x16x4(a[0], z[q][0], wa);
          wb = mfma_16x16x4(a[1], z[q][1], wb);
          wa = mfma_16x16x4(a[2], z[q][2], wa);
          wb = mfma_16x16x4(a[3], z[q][3], wb);
        }
        if constexpr (MT > 8) {  // loads of four tiles in flight
          if (q % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
      }
    } else {
      for (int i = t0 + ((w - t0) & 7); i < nt; i += 8) {
        double a[4], zz[4];
        w_op(i, a);
#pragma unroll
        for (int r = 0; r < 4; ++r) zz[r] = (on && 16 * i + lk + 4 * r < n) ? Y[at(i, r)] : 0.0;
        w_mask(i, a);
        wa = mfma_16x16x4(a[0], zz[0], wa);
        wb = mfma_16x16x4(a[1], zz[1], wb);
        wa = mfma_16x16x4(a[2], zz[2], wa);
        wb = mfma_16x16x4(a[3], zz[3], wb);
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) part[w][(lk + 4 * r) * kWyCols + l16] = wa[r] + wb[r];
    __syncthreads();
    if (tid < kWyBlock * kWyCols) {
      double x = 0.0;
#pragma unroll
      for (int g = 0; g < 8; ++g) x += part[g][tid];
      wsum[tid] = x;
    }
    __syncthreads();
    mfma_d4 y = mfma_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < 4; ++q) y = mfma_16x16x4(-tt[q], wsum[(4 * q + lk) * kWyCols + l16], y);
    if constexpr (MT > 0) {
#pragma unroll
      for (int q = 0; q < MT; ++q) {
        const int i = w + 8 * q;
        if (i >= t0 && i < nt) {
          double a[4];
          u_op(i, a);
          u_mask(i, a);
#pragma unroll
          for (int r = 0; r < 4; ++r) z[q] = mfma_16x16x4(a[r], y[r], z[q]);
        }
        if constexpr (MT > 8) {
          if (q % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
      }
    } else {
      for (int i = t0 + ((w - t0) & 7); i < nt; i += 8) {
        double a[4];
        mfma_d4 zz;
        u_op(i, a);
#pragma unroll
        for (int r = 0; r < 4; ++r) zz[r] = (on && 16 * i + lk + 4 * r < n) ? Y[at(i, r)] : 0.0;
        u_mask(i, a);
#pragma unroll
        for (int r = 0; r < 4; ++r) zz = mfma_16x16x4(a[r], y[r], zz);
        if (on)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (16 * i + lk + 4 * r < n) Y[at(i, r)] = zz[r];
      }
    }
  }
  if constexpr (MT > 0) {
    if (on)
#pragma unroll
      for (int q = 0; q < MT; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (16 * (w + 8 * q) + lk + 4 * r < n) Y[at(w + 8 * q, r)] = z[q][r];
  }
}

}  // namespace xtb
