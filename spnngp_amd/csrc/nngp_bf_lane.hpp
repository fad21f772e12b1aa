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

  const double2 *Z = reinterpret_cast<const double2 *>(P.Z);
  double2 z[ZH > 0 ? ZH : 1], zn[ZH > 0 ? M * ZH : 1];
  double v[M];  // B_i
  double vv;
  const bool ok = lane_solve<M, K, (ZH > 0), ((BATCH && M > 8) || M > 15)>(
      c.diag,
      [&](int k, int l) {
        return lane_corr<COV>(lane_d2<COV>(px[k] - px[l], py[k] - py[l]), c);
      },
      [&](int k) {
        return lane_corr<COV>(kBase2 ? lane_d2<COV>(px[k], py[k])
                                     : sqdist(s.x, s.y, px[k], py[k]),
                              c);
      },
      keep, v, vv,
      [&] {  // the neighbor slots again (from cache), not held until now
#pragma unroll
        for (int q = 0; q < M; q++) nb[q] = P.nnIndx[off + q];
      },
      [&] {  // the covariate rows
        if constexpr (ZH > 0) {
#pragma unroll
          for (int h = 0; h < ZH; h++) z[h] = Z[(size_t)i * ZH + h];
#pragma unroll
          for (int q = 0; q < M; q++) {
            const int id = q < cnt ? nb[q] : 0;
#pragma unroll
            for (int h = 0; h < ZH; h++)
              zn[q * ZH + h] = Z[(size_t)id * ZH + h];
          }
        }
      });
  Fi = c.diag - vv;
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
    // the slots again (from cache), unless the registers held them: the second
    // read is a round trip that a pass of few waves waits for (M = 8, n = 5e4:
    // 11.7 us with it, 11.0 without; batched, 150 problems of 4e4 sites, spherical:
    // 338 and 302 us, at three waves a SIMD instead of four)
    if constexpr (!(M <= 8 || (M == 12 && !BATCH))) {
#pragma unroll
      for (int k = 0; k < M; k++) nb[k] = k < cnt ? P.nnIndx[off + k] : 0;
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
// against 70%, at 4,286 instructions a wave against 4,660 (no moves to and
// from the accumulation registers).  n = 4e5, mode 0 against 2: m = 9 57 and
// 42 us, m = 12 74 and 54, m = 15 127 and 78, m = 16 146 and 89.
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
