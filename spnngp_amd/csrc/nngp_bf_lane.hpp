// nngp_bf_lane.hpp — updateBF / updateConjBF (src/rNNGP.cpp:46-101,
// src/cNNGP.cpp:24-69) with one site per lane in FP64, for the sizes that a
// source instantiates.
#pragma once
#include "nngp_bf.hpp"

namespace nngp {

// One site per lane: B_i, F_i and the residual vector e of site i from its
// neighbor count, offset and index slots (slots past the count are not its
// neighbors; they are replaced by site 0 here, before any use).
// ZH > 0 stages the rows of Z (zs = 2 ZH doubles) of the M neighbor slots
// and of the site itself in LDS with the coordinate gathers, instead of
// gathering them into registers after the solve, where the wait for them
// would stall the wavefront: chunk h of slot k (slot M = the site) at
// stg[(k * ZH + h) * 64 + lane].  The residuals add the same terms in the
// same order either way.
template <int M, int COV, bool BATCH, int ZH = 0>
__device__ __forceinline__ void lane_site(const BfArgs &A, const BfProblem &P,
                                          const CovArgs &c, int i, int cnt,
                                          int off, int (&nb)[M], double &Fi,
                                          double (&e)[kMaxNZ],
                                          double2 *stg = nullptr) {
  if (cnt == 0) {  // site 0: F = s2 + t2, residual = the data
    Fi = c.diag;
#pragma unroll
    for (int j = 0; j < kMaxNZ; j++)
      if (j < A.nz) e[j] = P.Z[(size_t)i * A.zs + j];
    return;
  }
  if (cnt < M) {
#pragma unroll
    for (int k = 0; k < M; k++)
      if (k >= cnt) nb[k] = 0;
  }
  // The staged rows are requested before the coordinates: the hardware's
  // load counter retires in order, so the one wait for the coordinates
  // covers them too, and nothing waits on memory again until the residuals.
  if constexpr (ZH > 0) {
#pragma unroll
    for (int k = 0; k <= M; k++) {
      const double *zr = P.Z + (size_t)(k < M ? nb[k] : i) * (2 * ZH);
#pragma unroll
      for (int h = 0; h < ZH; h++)
        lds_load16(zr + 2 * h, stg + (k * ZH + h) * 64);
    }
  }
  // the site's own coordinates first, so that they arrive with the
  // neighbors' (one wait for both)
  const double2 s = P.xy[i];
  double px[M], py[M];
#pragma unroll
  for (int k = 0; k < M; k++) {
    const double2 q = P.xy[nb[k]];
    px[k] = q.x;
    py[k] = q.y;
  }
  if (cnt < M) {
#pragma unroll
    for (int k = 0; k < M; k++) {
      if (k >= cnt) {  // far away and far apart: zero correlation
        px[k] = 1e100 * (k + 1);
        py[k] = -1e100 * (k + 1);
      }
    }
  }
  // exponential, gaussian and the closed-form materns: neighbor offsets
  // from the site, in units where the exponential factor is 2^-d (2^-d^2),
  // see s2_exp2.  Offsetting first keeps large coordinate values (projected
  // systems) out of the rounding of the scaled coordinates.
  constexpr bool kBase2 = lane_base2<COV>();
  if constexpr (kBase2) {
#pragma unroll
    for (int k = 0; k < M; k++) {
      px[k] = (px[k] - s.x) * c.tsc;
      py[k] = (py[k] - s.y) * c.tsc;
    }
  }

  constexpr int T = M * (M + 1) / 2;
  double a[T];  // packed lower triangle
  double v[M];
#pragma unroll
  for (int k = 0; k < M; k++) {
    v[k] = lane_corr<COV>(kBase2 ? lane_d2<COV>(px[k], py[k])
                                 : sqdist(s.x, s.y, px[k], py[k]),
                          c);
#pragma unroll
    for (int l = 0; l < k; l++)
      a[tri(k, l)] = lane_corr<COV>(
          lane_d2<COV>(px[k] - px[l], py[k] - py[l]), c);
    a[tri(k, k)] = c.diag;
  }
  double vv;
  const bool ok = chol_solve<M>(a, v, vv);  // v <- B_i = C^-1 c
  if (!BATCH && A.B) {
#pragma unroll
    for (int k = 0; k < M; k++)
      if (k < cnt) A.B[off + k] = v[k];
  }
  Fi = c.diag - vv;
  // residual vectors; padded coefficients are exactly 0
  if constexpr (ZH > 0) {
    const int t = (int)threadIdx.x & 63;
#pragma unroll
    for (int h = 0; h < ZH; h++) {
      const double2 zi = stg[(M * ZH + h) * 64 + t];
      double e0 = zi.x, e1 = zi.y;
#pragma unroll
      for (int k = 0; k < M; k++) {
        const double2 z = stg[(k * ZH + h) * 64 + t];
        e0 = fma(-v[k], z.x, e0);
        e1 = fma(-v[k], z.y, e1);
      }
      e[2 * h] = e0;
      e[2 * h + 1] = e1;
    }
    if (!ok) atomicMin(P.err, i);
    return;
  }
#pragma unroll
  for (int j = 0; j < kMaxNZ; j++) {
    if (j < A.nz) {
      double ej = P.Z[(size_t)i * A.zs + j];
#pragma unroll
      for (int k = 0; k < M; k++)
        ej = fma(-v[k], P.Z[(size_t)nb[k] * A.zs + j], ej);
      e[j] = ej;
    }
  }
  if (!ok) atomicMin(P.err, i);
}

template <int M, int COV, bool BATCH>
__global__ __launch_bounds__(kLaneMaxThreads) void k_bf_lane(BfArgs A) {
  extern __shared__ double lane_red[];  // site_terms(nz) x 64 per wave
  const int nt = (int)blockDim.x;
  const int b = xcd_block((A.n + nt - 1) / nt);
  if (b < 0) return;  // whole padding block
  const BfProblem P = bf_problem<BATCH>(A);
  const CovArgs c = BATCH ? A.covs[(int)blockIdx.y % A.ng] : A.c;
  const int i = b * nt + (int)threadIdx.x;
  const bool valid = i < A.n;
  double Fi = 1.0;
  double e[kMaxNZ];
#pragma unroll
  for (int j = 0; j < kMaxNZ; j++) e[j] = 0.0;

  if (valid) {
    int cnt, off;
    if (A.lu_closed) {
      nn_closed(i, A.m, off, cnt);
    } else {
      cnt = P.lu[A.n + i];
      off = P.lu[i];
    }
    // The index array carries 64 padding entries, so off + k is in bounds.
    int nb[M];
#pragma unroll
    for (int k = 0; k < M; k++) nb[k] = P.nnIndx[off + k];
    lane_site<M, COV, BATCH>(A, P, c, i, cnt, off, nb, Fi, e);
    if (!BATCH && A.F) A.F[i] = Fi;
  }
  if (P.rows) {
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    block_site_terms_lds(A.nz, P.rows, A.rows_cap, valid, Fi, e, b,
                         lane_red + (size_t)w * site_terms(A.nz) * 64);
  }
}

// k_bf_lane with the covariate rows staged in LDS: the block's dynamic LDS
// holds, per wavefront, (M + 1) x ZH chunks of 64 x 16 bytes.  The launcher
// uses it only when Z is set, zs = 2 ZH and every problem's Z is 16-byte
// aligned.
template <int M, int COV, int ZH, bool BATCH>
__global__ __launch_bounds__(kLaneMaxThreads) void k_bf_lane_lds(BfArgs A) {
  extern __shared__ double2 zstage[];
  const int nt = (int)blockDim.x;
  const int b = xcd_block((A.n + nt - 1) / nt);
  if (b < 0) return;  // whole padding block
  const BfProblem P = bf_problem<BATCH>(A);
  const CovArgs c = BATCH ? A.covs[(int)blockIdx.y % A.ng] : A.c;
  const int i = b * nt + (int)threadIdx.x;
  const bool valid = i < A.n;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  double2 *stg = zstage + (size_t)w * (M + 1) * ZH * 64;
  double Fi = 1.0;
  double e[kMaxNZ];
#pragma unroll
  for (int j = 0; j < kMaxNZ; j++) e[j] = 0.0;

  if (valid) {
    int cnt, off;
    if (A.lu_closed) {
      nn_closed(i, A.m, off, cnt);
    } else {
      cnt = P.lu[A.n + i];
      off = P.lu[i];
    }
    int nb[M];
#pragma unroll
    for (int k = 0; k < M; k++) nb[k] = P.nnIndx[off + k];
    lane_site<M, COV, BATCH, ZH>(A, P, c, i, cnt, off, nb, Fi, e, stg);
    if (!BATCH && A.F) A.F[i] = Fi;
  }
  // the sums reuse the wave's staging area (the residuals have read it);
  // site_terms(nz) <= 11 doubles a lane fit in (M + 1) x ZH x 16 bytes
  if (P.rows)
    block_site_terms_lds(A.nz, P.rows, A.rows_cap, valid, Fi, e, b,
                         reinterpret_cast<double *>(stg));
}

template <int M, bool BATCH>
void launch_lane_m(const BfArgs &a, int variant, const dim3 &grid,
                          const dim3 &blk, hipStream_t st) {
  // LDS of the block sums: site_terms(nz) doubles a lane
  const size_t shm =
      a.rows ? (size_t)blk.x * site_terms(a.nz) * sizeof(double) : 0;
  switch (variant) {
    case 0: hipLaunchKernelGGL((k_bf_lane<M, 0, BATCH>), grid, blk, shm, st, a); break;
    case 1: hipLaunchKernelGGL((k_bf_lane<M, 1, BATCH>), grid, blk, shm, st, a); break;
    case kCovMatern15: hipLaunchKernelGGL((k_bf_lane<M, kCovMatern15, BATCH>), grid, blk, shm, st, a); break;
    case kCovMatern25: hipLaunchKernelGGL((k_bf_lane<M, kCovMatern25, BATCH>), grid, blk, shm, st, a); break;
    default: hipLaunchKernelGGL((k_bf_lane<M, 3, BATCH>), grid, blk, shm, st, a); break;
  }
}

template <int M, int ZH, bool BATCH>
static void launch_lane_lds_mh(const BfArgs &a, int variant, const dim3 &grid,
                               const dim3 &blk, size_t shm, hipStream_t st) {
  switch (variant) {
    case 0: hipLaunchKernelGGL((k_bf_lane_lds<M, 0, ZH, BATCH>), grid, blk, shm, st, a); break;
    case 1: hipLaunchKernelGGL((k_bf_lane_lds<M, 1, ZH, BATCH>), grid, blk, shm, st, a); break;
    case kCovMatern15: hipLaunchKernelGGL((k_bf_lane_lds<M, kCovMatern15, ZH, BATCH>), grid, blk, shm, st, a); break;
    case kCovMatern25: hipLaunchKernelGGL((k_bf_lane_lds<M, kCovMatern25, ZH, BATCH>), grid, blk, shm, st, a); break;
    default: hipLaunchKernelGGL((k_bf_lane_lds<M, 3, ZH, BATCH>), grid, blk, shm, st, a); break;
  }
}

template <int M>
void launch_lane_lds_m(const BfArgs &a, int variant, const dim3 &grid,
                              const dim3 &blk, size_t shm, hipStream_t st) {
  if (a.ng > 0) launch_lane_lds_mh<M, 2, true>(a, variant, grid, blk, shm, st);
  else if (a.zs == 2) launch_lane_lds_mh<M, 1, false>(a, variant, grid, blk, shm, st);
  else launch_lane_lds_mh<M, 2, false>(a, variant, grid, blk, shm, st);
}

}  // namespace nngp
