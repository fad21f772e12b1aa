// nngp_bf_mixed.hip — updateBF (src/rNNGP.cpp:46-101) with one site per lane
// in mixed precision.
#include "nngp_bf.hpp"

namespace nngp {

// ---------------------------------------------------------------------------
// mixed precision, one site per lane
// ---------------------------------------------------------------------------
// The covariance is built in FP32 from FP32 neighbor offsets (FP64
// differences to the site, rounded), factored and solved in FP32 for B0.
// One refinement step forms the residual r = c - C B0 of that FP32 system
// in FP64 arithmetic (each FP32 x FP64 product is exact before the sum),
// solves C d = r with the FP32 factor and sets B = B0 + d, which removes
// the factorization's error.  F = s2 + t2 - c.B and every sum stay in FP64.
// What remains is the FP32 rounding of the covariance entries themselves.
// COPY = true keeps C in LDS (lane-interleaved) for the residual; false
// evaluates the entries a second time (bit-identically) to save LDS.
template <int COV>
__device__ __forceinline__ float pair32(float dxk, float dyk, float dxl,
                                        float dyl, const CovArgs32 &c) {
  const float ex = dxk - dxl, ey = dyk - dyl;
  return s2_corr32<COV>(fmaf(ex, ex, ey * ey), c);
}

template <int M, int COV, bool COPY>
__global__ __launch_bounds__(kLaneMaxThreads, 2) void k_bf_mixed(BfArgs A) {
  // COPY: covariance entry t of lane L at cl[t*nt + L]; otherwise the
  // neighbor offsets dx_k at cl[k*nt + L], dy_k at cl[(M+k)*nt + L]
  extern __shared__ float cl[];
  const int nt = (int)blockDim.x;
  const int b = xcd_block((A.n + nt - 1) / nt);
  if (b < 0) return;
  const CovArgs &c = A.c;
  const CovArgs32 c32 = cov32(c);
  const int L = (int)threadIdx.x;
  const int i = b * nt + L;
  const bool valid = i < A.n;
  double Fi = 1.0;
  double e[kMaxNZ];  // set on every path just before use (no value is live
                     // through the factorization)

  if (valid) {
    int cnt, off;
    if (A.lu_closed) {
      nn_closed(i, A.m, off, cnt);
    } else {
      cnt = A.lu[A.n + i];
      off = A.lu[i];
    }
    if (cnt == 0) {
      Fi = c.diag;
#pragma unroll
      for (int j = 0; j < kMaxNZ; j++)
        e[j] = j < A.nz ? A.Z[(size_t)i * A.zs + j] : 0.0;
    } else {
      const double2 s = A.xy[i];
      // as in k_bf_lane: padding entries of the index read as site 0, then
      // replaced by far-away finite offsets (every product with one is +inf
      // or 0 in FP32, so its correlations are exactly 0)
      int nb[M];
#pragma unroll
      for (int k = 0; k < M; k++) nb[k] = A.nnIndx[off + k];
      if (cnt < M) {
#pragma unroll
        for (int k = 0; k < M; k++)
          if (k >= cnt) nb[k] = 0;
      }
      float dx[M], dy[M];
#pragma unroll
      for (int k = 0; k < M; k++) {
        const double2 q = A.xy[nb[k]];
        dx[k] = (float)(q.x - s.x);
        dy[k] = (float)(q.y - s.y);
      }
      if (cnt < M) {
#pragma unroll
        for (int k = 0; k < M; k++) {
          if (k >= cnt) {
            dx[k] = 1e30f * (k + 1);
            dy[k] = -1e30f * (k + 1);
          }
        }
      }
      if (!COPY) {  // read back by the residual; registers stay free
#pragma unroll
        for (int k = 0; k < M; k++) {
          cl[k * nt + L] = dx[k];
          cl[(M + k) * nt + L] = dy[k];
        }
      }
      constexpr int T = M * (M + 1) / 2;
      float a[T], v[M];
#pragma unroll
      for (int k = 0; k < M; k++) {
        if (COPY) {
          v[k] = s2_corr32<COV>(fmaf(dx[k], dx[k], dy[k] * dy[k]), c32);
          cl[(T + k) * nt + L] = v[k];
        }
#pragma unroll
        for (int l = 0; l < k; l++) {
          a[tri(k, l)] = pair32<COV>(dx[k], dy[k], dx[l], dy[l], c32);
          if (COPY) cl[tri(k, l) * nt + L] = a[tri(k, l)];
        }
        a[tri(k, k)] = c32.diag;
      }
      const bool ok = chol_factor32<M>(a);
      if (!COPY) {  // c after the factorization, from the offsets in LDS
#pragma unroll
        for (int k = 0; k < M; k++) {
          const float xk = cl[k * nt + L], yk = cl[(M + k) * nt + L];
          v[k] = s2_corr32<COV>(fmaf(xk, xk, yk * yk), c32);
        }
      }
      chol_apply32<M>(a, v);  // v <- B0
      // residual r = c - C B0 in FP64; B0 stays FP32 (converted where
      // used), so only r is an FP64 array while the factor is live
      double r[M];
      const double dg = (double)c32.diag;
#pragma unroll
      for (int k = 0; k < M; k++) {
        float ck;
        if (COPY) {
          ck = cl[(T + k) * nt + L];
        } else {
          const float xk = cl[k * nt + L], yk = cl[(M + k) * nt + L];
          ck = s2_corr32<COV>(fmaf(xk, xk, yk * yk), c32);
        }
        r[k] = fma(-dg, (double)v[k], (double)ck);
      }
#pragma unroll
      for (int k = 1; k < M; k++) {
        float xk = 0.0f, yk = 0.0f;
        if (!COPY) {
          xk = cl[k * nt + L];
          yk = cl[(M + k) * nt + L];
        }
#pragma unroll
        for (int l = 0; l < k; l++) {
          const double ckl =
              COPY ? (double)cl[tri(k, l) * nt + L]
                   : (double)pair32<COV>(xk, yk, cl[l * nt + L],
                                         cl[(M + l) * nt + L], c32);
          r[k] = fma(-ckl, (double)v[l], r[k]);
          r[l] = fma(-ckl, (double)v[k], r[l]);
        }
      }
      float d[M];
#pragma unroll
      for (int k = 0; k < M; k++) d[k] = (float)r[k];
      chol_apply32<M>(a, d);  // d <- C^-1 r
      double bd[M];
      double cb = 0.0;
#pragma unroll
      for (int k = 0; k < M; k++) {
        bd[k] = (double)v[k] + (double)d[k];
        float ck;
        if (COPY) {
          ck = cl[(T + k) * nt + L];
        } else {
          const float xk = cl[k * nt + L], yk = cl[(M + k) * nt + L];
          ck = s2_corr32<COV>(fmaf(xk, xk, yk * yk), c32);
        }
        cb = fma((double)ck, bd[k], cb);
      }
      if (A.B) {
#pragma unroll
        for (int k = 0; k < M; k++)
          if (k < cnt) A.B[off + k] = bd[k];
      }
      Fi = c.diag - cb;
      // the neighbor slots again (cache hits) rather than held in
      // registers through the factorization; padded coefficients are 0
#pragma unroll
      for (int k = 0; k < M; k++) nb[k] = k < cnt ? A.nnIndx[off + k] : 0;
#pragma unroll
      for (int j = 0; j < kMaxNZ; j++) {
        e[j] = 0.0;
        if (j < A.nz) {
          double ej = A.Z[(size_t)i * A.zs + j];
#pragma unroll
          for (int k = 0; k < M; k++)
            ej = fma(-bd[k], A.Z[(size_t)nb[k] * A.zs + j], ej);
          e[j] = ej;
        }
      }
      if (!ok || !(Fi > 0.0)) atomicMin(A.err, i);
    }
    if (A.F) A.F[i] = Fi;
  } else {
#pragma unroll
    for (int j = 0; j < kMaxNZ; j++) e[j] = 0.0;
  }
  if (A.rows) block_site_terms(A.nz, A.rows, A.rows_cap, valid, Fi, e, b);
}

// k_bf_mixed's scheme with a copy of C kept, so that no entry is evaluated
// twice: what of the copy the registers of W = 2 waves per SIMD cannot hold
// beside the factor waits in LDS for the residual (mixed_lds_entries, four
// entries a lane in each 16 bytes).  The arithmetic is k_bf_mixed's step for
// step, so B and F equal its results bit for bit.  With the whole copy in
// registers, one wave per SIMD and the covariate rows staged in LDS, a pass
// took 155 us at n = 1e6, m = 15 (the vector units busy 61% of the time);
// now 104 us.  ZH > 0: the rows of Z are ZH aligned pairs.
//
// At M = 16 two waves lack 29 registers (43 to 54 with the spherical's former
// branches), and LDS has no room for them.  With W = 1 nothing spills and
// the covariate rows can be requested with the coordinates.  W = 2 and 1, p =
// 3, exponential: n = 3,000 15.2 and 12.6 us, n = 2e5 45.2 and 43.7, n = 1e6
// 185 and 179.  Rows that are not pairs come after the solve, where a second
// wave covers their wait as soon as there is one (launch_mixed_reg_mh).
__host__ __device__ constexpr int mixed_lds_entries(int M, int W) {
  return M <= 12 || W == 1 ? 0 : 72;
}

template <int M, int COV, int ZH, int W>
__device__ __forceinline__ void mixed_reg_site(const BfArgs &A, int i,
                                               int cnt, int off,
                                               int (&nb)[M], double &Fi,
                                               double (&e)[kMaxNZ],
                                               float4 *keep) {
  constexpr int K = mixed_lds_entries(M, W);
  constexpr bool kEarlyZ = ZH > 0 && W == 1;
  const double2 *Z = reinterpret_cast<const double2 *>(A.Z);
  double2 z[ZH > 0 ? ZH : 1], zn[kEarlyZ ? M * ZH : 1];
  const CovArgs &c = A.c;
  const CovArgs32 c32 = cov32(c);
  if (cnt == 0) {  // site 0: F = s2 + t2, residual = the data
    Fi = c.diag;
#pragma unroll
    for (int j = 0; j < (ZH > 0 ? 2 * ZH : kMaxNZ); j++)
      if (ZH > 0 || j < A.nz) e[j] = A.Z[(size_t)i * A.zs + j];
    return;
  }
  if (cnt < M) {
#pragma unroll
    for (int k = 0; k < M; k++)
      if (k >= cnt) nb[k] = 0;
  }
  const double2 s = A.xy[i];
  float dx[M], dy[M];
#pragma unroll
  for (int k = 0; k < M; k++) {
    const double2 q = A.xy[nb[k]];
    dx[k] = (float)(q.x - s.x);
    dy[k] = (float)(q.y - s.y);
  }
  if constexpr (kEarlyZ) {
#pragma unroll
    for (int h = 0; h < ZH; h++) z[h] = Z[(size_t)i * ZH + h];
#pragma unroll
    for (int k = 0; k < M; k++) {
#pragma unroll
      for (int h = 0; h < ZH; h++) zn[k * ZH + h] = Z[(size_t)nb[k] * ZH + h];
    }
    asm volatile("" : : : "memory");
  }
  if (cnt < M) {  // far away and far apart: correlations exactly 0
#pragma unroll
    for (int k = 0; k < M; k++) {
      if (k >= cnt) {
        dx[k] = 1e30f * (k + 1);
        dy[k] = -1e30f * (k + 1);
      }
    }
  }
  constexpr int T = M * (M + 1) / 2;
  float a[T], v[M], cv[M];
  float ac[M * (M - 1) / 2];  // C below the diagonal, row by row
#pragma unroll
  for (int k = 0; k < M; k++) {
    v[k] = s2_corr32<COV>(fmaf(dx[k], dx[k], dy[k] * dy[k]), c32);
    cv[k] = v[k];
#pragma unroll
    for (int l = 0; l < k; l++) {
      const int q = k * (k - 1) / 2 + l;
      ac[q] = pair32<COV>(dx[k], dy[k], dx[l], dy[l], c32);
      a[tri(k, l)] = ac[q];
      if (q < K && q % 4 == 3)
        keep[q / 4 * 64] = make_float4(ac[q - 3], ac[q - 2], ac[q - 1], ac[q]);
    }
    a[tri(k, k)] = c32.diag;
  }
  const bool ok = chol_factor32<M>(a);
  chol_apply32<M>(a, v);  // v <- B0
  if constexpr (K > 0) {
    // the kept entries come from LDS, not from registers held until here
    asm volatile("" : "+v"(v[0]) : : "memory");
#pragma unroll
    for (int q = 0; q < K / 4; q++) {
      const float4 x = keep[q * 64];
      ac[4 * q] = x.x;
      ac[4 * q + 1] = x.y;
      ac[4 * q + 2] = x.z;
      ac[4 * q + 3] = x.w;
    }
  }
  // residual r = c - C B0 in FP64
  double r[M];
  const double dg = (double)c32.diag;
#pragma unroll
  for (int k = 0; k < M; k++) r[k] = fma(-dg, (double)v[k], (double)cv[k]);
#pragma unroll
  for (int k = 1; k < M; k++) {
#pragma unroll
    for (int l = 0; l < k; l++) {
      const double ckl = (double)ac[k * (k - 1) / 2 + l];
      r[k] = fma(-ckl, (double)v[l], r[k]);
      r[l] = fma(-ckl, (double)v[k], r[l]);
    }
  }
  // the neighbor slots again (from cache), in time for the covariate rows
  if constexpr (!kEarlyZ) {
    asm volatile("" : "+v"(r[0]) : : "memory");
#pragma unroll
    for (int k = 0; k < M; k++) nb[k] = A.nnIndx[off + k];
  }
  float d[M];
#pragma unroll
  for (int k = 0; k < M; k++) d[k] = (float)r[k];
  chol_apply32<M>(a, d);  // d <- C^-1 r
  double bd[M];
  double cb = 0.0;
#pragma unroll
  for (int k = 0; k < M; k++) {
    bd[k] = (double)v[k] + (double)d[k];
    cb = fma((double)cv[k], bd[k], cb);
  }
  if (A.B) {
#pragma unroll
    for (int k = 0; k < M; k++)
      if (k < cnt) A.B[off + k] = bd[k];
  }
  Fi = c.diag - cb;
  // residual vectors; padded coefficients are 0
#pragma unroll
  for (int k = 0; k < M; k++) nb[k] = k < cnt ? nb[k] : 0;
  if constexpr (ZH > 0) {
    if constexpr (!kEarlyZ) {
#pragma unroll
      for (int h = 0; h < ZH; h++) z[h] = Z[(size_t)i * ZH + h];
    }
#pragma unroll
    for (int k = 0; k < M; k++) {
#pragma unroll
      for (int h = 0; h < ZH; h++) {
        double2 q;
        if constexpr (kEarlyZ) q = zn[k * ZH + h];
        else q = Z[(size_t)nb[k] * ZH + h];
        z[h].x = fma(-bd[k], q.x, z[h].x);
        z[h].y = fma(-bd[k], q.y, z[h].y);
      }
    }
#pragma unroll
    for (int h = 0; h < ZH; h++) {
      e[2 * h] = z[h].x;
      e[2 * h + 1] = z[h].y;
    }
  } else {
#pragma unroll
    for (int j = 0; j < kMaxNZ; j++) {
      if (j < A.nz) {
        double ej = A.Z[(size_t)i * A.zs + j];
#pragma unroll
        for (int k = 0; k < M; k++)
          ej = fma(-bd[k], A.Z[(size_t)nb[k] * A.zs + j], ej);
        e[j] = ej;
      }
    }
  }
  if (!ok || !(Fi > 0.0)) atomicMin(A.err, i);
}

// Dynamic LDS of k_bf_mixed_reg a wavefront, in double2: the kept entries,
// which the block sums then overwrite, or the sums' terms.
__host__ __device__ inline int mixed_reg_wave_chunks(int M, int W, int nz) {
  const int sums = (site_terms(nz) * 64 + 1) / 2;
  const int keep = mixed_lds_entries(M, W) / 4 * 64;
  return keep > sums ? keep : sums;
}

// The body of both register-copy kernels; mstage: the block's dynamic LDS.
template <int M, int COV, int ZH, int W>
__device__ __forceinline__ void mixed_reg_body(const BfArgs &A,
                                               double2 *mstage) {
  const int nt = (int)blockDim.x;
  const int b = xcd_block((A.n + nt - 1) / nt);
  if (b < 0) return;  // whole padding block
  const int i = b * nt + (int)threadIdx.x;
  const bool valid = i < A.n;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  double2 *stg = mstage + (size_t)w * mixed_reg_wave_chunks(M, W, A.nz);
  double Fi = 1.0;
  double e[kMaxNZ];
#pragma unroll
  for (int j = 0; j < kMaxNZ; j++) e[j] = 0.0;
  if (valid) {
    int cnt, off;
    if (A.lu_closed) {
      nn_closed(i, A.m, off, cnt);
    } else {
      cnt = A.lu[A.n + i];
      off = A.lu[i];
    }
    int nb[M];
#pragma unroll
    for (int k = 0; k < M; k++) nb[k] = A.nnIndx[off + k];
    mixed_reg_site<M, COV, ZH, W>(
        A, i, cnt, off, nb, Fi, e,
        reinterpret_cast<float4 *>(stg) + ((int)threadIdx.x & 63));
    if (A.F) A.F[i] = Fi;
  }
  if (A.rows)
    block_site_terms_lds(A.nz, A.rows, A.rows_cap, valid, Fi, e, b,
                         reinterpret_cast<double *>(stg));
}

template <int M, int COV, int ZH>
__global__ __launch_bounds__(kLaneMaxThreads, 2) void k_bf_mixed_reg(BfArgs A) {
  extern __shared__ double2 mixed_lds[];
  mixed_reg_body<M, COV, ZH, 2>(A, mixed_lds);
}

template <int M, int COV, int ZH>
__global__ __launch_bounds__(kLaneMaxThreads, 1) void k_bf_mixed_one(BfArgs A) {
  extern __shared__ double2 mixed_lds[];
  mixed_reg_body<M, COV, ZH, 1>(A, mixed_lds);
}

// LDS of the mixed kernel's covariance copy: (M(M+1)/2 + M) floats a lane.
size_t mixed_copy_shm(int m, int threads) {
  const int M = lane_M(m);
  return (size_t)threads * (M * (M + 1) / 2 + M) * sizeof(float);
}

// LDS of the mixed per-lane kernel without the covariance copy: the
// neighbor offsets.
static size_t mixed_offsets_shm(int m, int threads) {
  return (size_t)threads * 2 * lane_M(m) * sizeof(float);
}

template <int M, bool COPY>
static void launch_mixed_mc(const BfArgs &a, int variant, const dim3 &grid,
                            const dim3 &blk, size_t shm, hipStream_t st) {
  switch (variant) {
    case 0: hipLaunchKernelGGL((k_bf_mixed<M, 0, COPY>), grid, blk, shm, st, a); break;
    case 1: hipLaunchKernelGGL((k_bf_mixed<M, 1, COPY>), grid, blk, shm, st, a); break;
    case kCovMatern15: hipLaunchKernelGGL((k_bf_mixed<M, kCovMatern15, COPY>), grid, blk, shm, st, a); break;
    case kCovMatern25: hipLaunchKernelGGL((k_bf_mixed<M, kCovMatern25, COPY>), grid, blk, shm, st, a); break;
    default: hipLaunchKernelGGL((k_bf_mixed<M, 3, COPY>), grid, blk, shm, st, a); break;
  }
}

// Aligned pairs in a row of Z that k_bf_mixed_reg reads (zs = 2 ZH, Z 16-byte
// aligned, m > 8), else 0: single values, as also for rows of two pairs in
// 256-thread blocks, a shape that smaller blocks beat.
static int mixed_reg_zh(const BfArgs &a, int threads) {
  if (!a.Z || a.nz <= 0 || a.m <= 8 || ((uintptr_t)a.Z & 15) != 0) return 0;
  return a.zs == 2 ? 1 : a.zs == 4 && threads <= 128 ? 2 : 0;
}

// Sites up to which no SIMD of the 1,024 has a second wave.
constexpr int kOneWaveSites = 1024 * 64;

template <int M, int ZH, int W>
static void launch_mixed_reg_mhw(const BfArgs &a, int variant,
                                 const dim3 &grid, const dim3 &blk,
                                 hipStream_t st) {
  // up to 72 KiB a block at 256 threads, which gfx950 grants (160 KiB a CU)
  const size_t shm = (size_t)(blk.x / 64) *
                     mixed_reg_wave_chunks(M, W, a.nz) * sizeof(double2);
  auto launch = [&](auto cov) {
    constexpr int COV = decltype(cov)::value;
    if constexpr (W == 2)
      hipLaunchKernelGGL((k_bf_mixed_reg<M, COV, ZH>), grid, blk, shm, st, a);
    else
      hipLaunchKernelGGL((k_bf_mixed_one<M, COV, ZH>), grid, blk, shm, st, a);
  };
  switch (variant) {
    case 0: launch(std::integral_constant<int, 0>()); break;
    case 1: launch(std::integral_constant<int, 1>()); break;
    case kCovMatern15:
      launch(std::integral_constant<int, kCovMatern15>());
      break;
    case kCovMatern25:
      launch(std::integral_constant<int, kCovMatern25>());
      break;
    default: launch(std::integral_constant<int, 3>()); break;
  }
}

// W = 2 up to M = 15, where everything fits; at M = 16 W = 1, but for rows of
// Z that are not pairs only while no SIMD has two waves (p = 5, W = 2 and 1: n
// = 3,000 15.1 and 14.4 us, n = 70,000 33.0 and 38.5).
template <int M, int ZH>
static void launch_mixed_reg_mh(const BfArgs &a, int variant, const dim3 &grid,
                                const dim3 &blk, hipStream_t st) {
  if constexpr (M <= 15) {
    launch_mixed_reg_mhw<M, ZH, 2>(a, variant, grid, blk, st);
  } else {
    if (ZH == 0 && a.n > kOneWaveSites)
      launch_mixed_reg_mhw<M, 0, 2>(a, variant, grid, blk, st);
    else
      launch_mixed_reg_mhw<M, ZH, 1>(a, variant, grid, blk, st);
  }
}

template <int M>
static void launch_mixed_reg(const BfArgs &a, int variant, const dim3 &grid,
                             const dim3 &blk, hipStream_t st) {
  switch (mixed_reg_zh(a, (int)blk.x)) {
    case 1: launch_mixed_reg_mh<M, 1>(a, variant, grid, blk, st); break;
    case 2: launch_mixed_reg_mh<M, 2>(a, variant, grid, blk, st); break;
    default: launch_mixed_reg_mh<M, 0>(a, variant, grid, blk, st); break;
  }
}

// mode 1: the covariance copy in LDS; 3: in registers, with what does not fit
// there in LDS; else re-evaluated
template <int M>
static void launch_mixed_m(const BfArgs &a, int variant, int mode,
                           const dim3 &grid, const dim3 &blk, hipStream_t st) {
  if (mode == 1)
    launch_mixed_mc<M, true>(a, variant, grid, blk,
                             mixed_copy_shm(a.m, (int)blk.x), st);
  else if (mode == 3)
    launch_mixed_reg<M>(a, variant, grid, blk, st);
  else
    launch_mixed_mc<M, false>(a, variant, grid, blk,
                              mixed_offsets_shm(a.m, (int)blk.x), st);
}

void launch_mixed(const BfArgs &a, int variant, int mode,
                         const dim3 &grid, const dim3 &blk, hipStream_t st) {
  switch (lane_M(a.m)) {
    case 4: launch_mixed_m<4>(a, variant, mode, grid, blk, st); break;
    case 8: launch_mixed_m<8>(a, variant, mode, grid, blk, st); break;
    case 10: launch_mixed_m<10>(a, variant, mode, grid, blk, st); break;
    case 12: launch_mixed_m<12>(a, variant, mode, grid, blk, st); break;
    case 15: launch_mixed_m<15>(a, variant, mode, grid, blk, st); break;
    default: launch_mixed_m<16>(a, variant, mode, grid, blk, st); break;
  }
}

}  // namespace nngp
