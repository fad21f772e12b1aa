// nngp_bf_lane.hpp — updateBF / updateConjBF (src/rNNGP.cpp:46-101,
// src/cNNGP.cpp:24-69) with one site per lane in FP64, for the sizes that a
// source instantiates.
#pragma once
#include "nngp_bf.hpp"

namespace nngp {

// Aligned pairs in a row of Z where the kernel can read it by pairs (one or
// two, every problem's Z 16-byte aligned), else 0.
inline int lane_zh(const BfArgs &a) {
  if (!a.Z || a.nz <= 0 || ((uintptr_t)a.Z & 15) != 0 ||
      (a.ng > 0 && a.fs_Z % 2 != 0))
    return 0;
  return a.zs == 2 ? 1 : a.zs == 4 ? 2 : 0;
}

// One site per lane: B_i, F_i and the residual vector e of site i from its
// neighbor count and offset.  K entries of the factor wait in LDS: pair q of
// them at keep[q * 64], `keep` the lane's slot in its wavefront's area.
//
// The lower triangle is built and factored column by column (left-looking),
// the covariance entries of a column evaluated when it is reached, so that
// the M x M system is never held whole: one wave a SIMD, with the whole
// triangle in registers, left the vector units idle for 30% of the time (the
// gathers at a wave's start and the chains of dependent instructions).  Each
// entry goes through the same operations in the same order as in a
// right-looking factorization, so the results are the same bit for bit.
// ZH > 0: the rows of Z are ZH aligned pairs (zs = 2 ZH).
template <int M, int COV, bool BATCH, int ZH, int K>
__device__ __forceinline__ void lane_site(const BfArgs &A, const BfProblem &P,
                                          const CovArgs &c, int i, int cnt,
                                          int off, double &Fi,
                                          double (&e)[kMaxNZ],
                                          double2 *keep) {
  if (cnt == 0) {  // site 0: F = s2 + t2, residual = the data
    Fi = c.diag;
#pragma unroll
    for (int j = 0; j < (ZH > 0 ? 2 * ZH : kMaxNZ); j++)
      if (ZH > 0 || j < A.nz) e[j] = P.Z[(size_t)i * A.zs + j];
    return;
  }
  // The index array carries 64 padding entries, so off + k is in bounds;
  // slots past the count are not the site's neighbors and read site 0.
  int nb[M];
#pragma unroll
  for (int k = 0; k < M; k++) nb[k] = P.nnIndx[off + k];
  if (cnt < M) {
#pragma unroll
    for (int k = 0; k < M; k++)
      if (k >= cnt) nb[k] = 0;
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
  double a[T];  // packed lower triangle, diagonal as 1 / L_jj
  double v[M];  // L^-1 c, then B_i
  double vv = 0.0;
  bool ok = true;
#pragma unroll
  for (int j = 0; j < M; j++) {
    v[j] = lane_corr<COV>(kBase2 ? lane_d2<COV>(px[j], py[j])
                                 : sqdist(s.x, s.y, px[j], py[j]),
                          c);
#pragma unroll
    for (int k = j + 1; k < M; k++)
      a[tri(k, j)] = lane_corr<COV>(
          lane_d2<COV>(px[k] - px[j], py[k] - py[j]), c);
    double piv = c.diag;
#pragma unroll
    for (int l = 0; l < j; l++) {
      const double ljl = a[tri(j, l)];
      piv = fma(-ljl, ljl, piv);
      v[j] = fma(-ljl, v[l], v[j]);
#pragma unroll
      for (int k = j + 1; k < M; k++)
        a[tri(k, j)] = fma(-a[tri(k, l)], ljl, a[tri(k, j)]);
    }
    ok = ok && (piv > 0.0);
    const double r = nn_rsqrt(piv);
    a[tri(j, j)] = r;
#pragma unroll
    for (int k = j + 1; k < M; k++) a[tri(k, j)] *= r;
    v[j] *= r;
    vv = fma(v[j], v[j], vv);
    // row j is finished: the kept pairs that end in it go to LDS
#pragma unroll
    for (int q = 0; q < K / 2; q++)
      if (2 * q + 1 >= tri(j, 0) && 2 * q + 1 <= tri(j, j))
        keep[q * 64] = make_double2(a[2 * q], a[2 * q + 1]);
    // no entry of a later column is evaluated before this column is done
    __builtin_amdgcn_sched_barrier(0);
  }
  Fi = c.diag - vv;
  // Going back up, the registers of the rows that are done with take what the
  // residuals need, so that nothing waits for memory after the solve: from
  // row M - 4 the neighbor slots (again, from cache, rather than held through
  // the factorization), from row kUp the kept entries and the covariate rows.
  // The empty asm stands behind the finished rows' work by v[k]; it also
  // keeps the kept entries from being held in registers since they were
  // stored, and the loads before it from sinking to their uses.
  constexpr int kUp = K > 0 ? 7 : M / 2 - 1;
  static_assert(K == 0 || K == tri(kUp, kUp) + 1, "whole rows are kept");
  const double2 *Z = reinterpret_cast<const double2 *>(P.Z);
  double2 z[ZH > 0 ? ZH : 1], zn[ZH > 0 ? M * ZH : 1];
#pragma unroll
  for (int k = M - 1; k >= 0; k--) {
    if (ZH > 0 && k == M - 4) {
      asm volatile("" : "+v"(v[k]) : : "memory");
#pragma unroll
      for (int q = 0; q < M; q++) nb[q] = P.nnIndx[off + q];
    }
    if ((K > 0 || ZH > 0) && k == kUp) {
      asm volatile("" : "+v"(v[k]) : : "memory");
#pragma unroll
      for (int q = 0; q < K / 2; q++) {
        const double2 x = keep[q * 64];
        a[2 * q] = x.x;
        a[2 * q + 1] = x.y;
      }
      if constexpr (ZH > 0) {
#pragma unroll
        for (int h = 0; h < ZH; h++) z[h] = Z[(size_t)i * ZH + h];
#pragma unroll
        for (int q = 0; q < M; q++) {
          const int id = q < cnt ? nb[q] : 0;
#pragma unroll
          for (int h = 0; h < ZH; h++) zn[q * ZH + h] = Z[(size_t)id * ZH + h];
        }
      }
    }
    const double t = v[k] * a[tri(k, k)];
    v[k] = t;
#pragma unroll
    for (int l = 0; l < k; l++) v[l] = fma(-a[tri(k, l)], t, v[l]);
  }
  if (ZH > 0) asm volatile("" : "+v"(v[0]) : : "memory");
  if (!BATCH && A.B) {
#pragma unroll
    for (int k = 0; k < M; k++)
      if (k < cnt) A.B[off + k] = v[k];
  }
  if (!ok) atomicMin(P.err, i);
  // residual vectors; padded coefficients are exactly 0
  if constexpr (ZH > 0) {
#pragma unroll
    for (int k = 0; k < M; k++) {
#pragma unroll
      for (int h = 0; h < ZH; h++) {
        z[h].x = fma(-v[k], zn[k * ZH + h].x, z[h].x);
        z[h].y = fma(-v[k], zn[k * ZH + h].y, z[h].y);
      }
    }
#pragma unroll
    for (int h = 0; h < ZH; h++) {
      e[2 * h] = z[h].x;
      e[2 * h + 1] = z[h].y;
    }
  } else if (A.nz > 0) {
#pragma unroll
    for (int k = 0; k < M; k++) nb[k] = k < cnt ? P.nnIndx[off + k] : 0;
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
  }
}

// The body of both per-lane kernels; `area` is the block's dynamic LDS, with
// K kept entries a lane and at least the block sums' terms, which overwrite
// them.
template <int M, int COV, bool BATCH, int ZH, int K>
__device__ __forceinline__ void lane_body(const BfArgs &A, double2 *area) {
  const int nt = (int)blockDim.x;
  const int b = xcd_block((A.n + nt - 1) / nt);
  if (b < 0) return;  // whole padding block
  const BfProblem P = bf_problem<BATCH>(A);
  const CovArgs c = BATCH ? cov_uniform(A.covs + P.point) : A.c;
  const int i = b * nt + (int)threadIdx.x;
  const bool valid = i < A.n;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  area += (size_t)w * (lane_wave_doubles(K, A.nz) / 2);
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
    lane_site<M, COV, BATCH, ZH, K>(A, P, c, i, cnt, off, Fi, e,
                                    area + ((int)threadIdx.x & 63));
    if (!BATCH && A.F) A.F[i] = Fi;
  }
  if (P.rows)
    block_site_terms_lds(A.nz, P.rows, A.rows_cap, valid, Fi, e, b,
                         reinterpret_cast<double *>(area));
}

// Mode 0: the whole factor in registers, one wave a SIMD from M = 15 on.
template <int M, int COV, bool BATCH>
__global__ __launch_bounds__(kLaneMaxThreads) void k_bf_lane(BfArgs A) {
  extern __shared__ double2 lane_lds[];
  lane_body<M, COV, BATCH, 0, 0>(A, lane_lds);
}

// Mode 2: two waves a SIMD, finished rows of the factor in LDS.  n = 1e6,
// m = 15, p = 3, exponential: 158 us a pass (20 iterations of a chain 3.71
// ms) against 200 us (4.61 ms) with the triangle in registers at one wave and
// the covariate rows staged in LDS; the vector units are busy 93% of the time
// against 70%, at 4,257 instructions a wave against 4,660 (no moves to and
// from the accumulation registers).  n = 4e5, mode 0 against 2: m = 9 57 and
// 42 us, m = 12 74 and 54, m = 15 127 and 78, m = 16 145 and 97.
template <int M, int COV, int ZH, bool BATCH>
__global__ __launch_bounds__(kLaneMaxThreads, 2) void k_bf_lane_lds(BfArgs A) {
  extern __shared__ double2 lane_lds[];
  lane_body<M, COV, BATCH, ZH, lane_lds_entries(M)>(A, lane_lds);
}

#define NNGP_LANE_COV(LAUNCH)                                         \
  switch (variant) {                                                  \
    case 0: LAUNCH(0); break;                                         \
    case 1: LAUNCH(1); break;                                         \
    case kCovMatern15: LAUNCH(kCovMatern15); break;                   \
    case kCovMatern25: LAUNCH(kCovMatern25); break;                   \
    default: LAUNCH(3); break;                                        \
  }

template <int M, bool BATCH>
void launch_lane_m(const BfArgs &a, int variant, const dim3 &grid,
                   const dim3 &blk, hipStream_t st) {
  const size_t shm =
      (size_t)(blk.x / 64) * lane_wave_doubles(0, a.nz) * sizeof(double);
#define LAUNCH(COV) \
  hipLaunchKernelGGL((k_bf_lane<M, COV, BATCH>), grid, blk, shm, st, a)
  NNGP_LANE_COV(LAUNCH)
#undef LAUNCH
}

template <int M, int ZH, bool BATCH>
static void launch_lane_lds_mz(const BfArgs &a, int variant, const dim3 &grid,
                               const dim3 &blk, hipStream_t st) {
  const size_t shm = lane_lds_shm(M, a.nz, (int)blk.x);
#define LAUNCH(COV) \
  hipLaunchKernelGGL((k_bf_lane_lds<M, COV, ZH, BATCH>), grid, blk, shm, st, a)
  NNGP_LANE_COV(LAUNCH)
#undef LAUNCH
}

template <int M, bool BATCH>
void launch_lane_lds_m(const BfArgs &a, int variant, const dim3 &grid,
                       const dim3 &blk, hipStream_t st) {
  switch (lane_zh(a)) {
    case 1: launch_lane_lds_mz<M, 1, BATCH>(a, variant, grid, blk, st); break;
    case 2: launch_lane_lds_mz<M, 2, BATCH>(a, variant, grid, blk, st); break;
    default: launch_lane_lds_mz<M, 0, BATCH>(a, variant, grid, blk, st); break;
  }
}
#undef NNGP_LANE_COV

}  // namespace nngp
