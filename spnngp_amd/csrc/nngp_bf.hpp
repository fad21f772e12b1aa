// nngp_bf.hpp — what the updateBF kernels' sources share: sizes, the
// problem a block works on, and wavefront sums.
#pragma once
#include "nngp_kernels.hpp"
#include "nngp_lane.hpp"
#include "nngp_wave.hpp"

namespace nngp {

constexpr int kLaneMaxThreads = 256;
constexpr int kCoopMaxWaves = 4;
constexpr int kCoopMaxM = 64;
constexpr int kCoopBlocks = 2048;  // logical blocks of the wavefront kernel
constexpr int kGrpMaxM = 32;       // the row kernel's largest system
// Waves of the row kernel for m > 16 or the matern: two a SIMD on 256 CUs, what
// the registers of its larger system allow.  In 256-thread blocks all are
// resident and copy the matern's 41 KB table once (in smaller ones the table
// takes the LDS: three of the eight blocks of 64 threads fit a CU).  With m <=
// 16 and no table four waves fit a SIMD, and the pass takes kCoopBlocks: n =
// 1e6, m = 15, exponential 1.09 ms on 2,048 waves, 0.90 ms.
constexpr int kGrpWaves = 2048;
constexpr int kRedThreads = 256;   // threads per block of the sum kernels
constexpr int kRowsThreads = 1024; // threads per column of k_rows_sum
constexpr int kRedBlocks = 1024;   // grid of the sum kernels (at most)

// DPP lane move of a double (two 32-bit moves); lanes outside ROWMASK get 0.
template <int CTRL, int ROWMASK>
__device__ __forceinline__ double dpp_mov(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL,
                                             ROWMASK, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL,
                                             ROWMASK, 0xF, false);
  return __hiloint2double(hi, lo);
}

// The same where lanes outside ROWMASK may receive anything (no value is
// prepared for them): for sums whose result is read in lanes the move
// reaches.
template <int CTRL, int ROWMASK>
__device__ __forceinline__ double dpp_mov_any(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, ROWMASK,
                                          0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, ROWMASK,
                                          0xF, false);
  return __hiloint2double(hi, lo);
}

// Sum over the 64 lanes with DPP moves only (no LDS round trips); the
// total is valid in lane 63 (other lanes hold partial or meaningless
// sums).  Fixed order: pairs, quads, half rows, rows, then rows 0+1 and
// 2+3, then all four.
__device__ __forceinline__ double wave_sum_to63(double x) {
  x += dpp_mov_any<0xB1, 0xF>(x);   // quad_perm [1,0,3,2]
  x += dpp_mov_any<0x4E, 0xF>(x);   // quad_perm [2,3,0,1]
  x += dpp_mov_any<0x141, 0xF>(x);  // row_half_mirror
  x += dpp_mov_any<0x140, 0xF>(x);  // row_mirror
  x += dpp_mov_any<0x142, 0xA>(x);  // row_bcast:15 into rows 1 and 3
  x += dpp_mov_any<0x143, 0xC>(x);  // row_bcast:31 into rows 2 and 3
  return x;
}

// ---------------------------------------------------------------------------
// problem view
// ---------------------------------------------------------------------------
struct BfProblem {
  const double2 *xy;
  const int *nnIndx;
  const int *lu;
  const double *Z;
  double *rows;
  int *err;
  int point = 0;  // batched passes: the problem's grid point
};

template <bool BATCH>
__device__ __forceinline__ BfProblem bf_problem(const BfArgs &A) {
  BfProblem P{A.xy, A.nnIndx, A.lu, A.Z, A.rows, A.err};
  if constexpr (BATCH) {
    const int j = (int)blockIdx.y;
    // the division's result is known to be uniform only after readfirstlane
    const int f = __builtin_amdgcn_readfirstlane(j / A.ng);
    P.point = j - f * A.ng;
    P.xy += (size_t)f * A.fs_xy;
    P.nnIndx += (size_t)f * A.fs_nn;
    P.lu += (size_t)f * A.fs_lu;
    if (P.Z) P.Z += (size_t)f * A.fs_Z;
    if (P.rows) P.rows += (size_t)j * A.ps_rows;
    P.err += j;
  }
  return P;
}

// ---------------------------------------------------------------------------
// per-block sums of the site terms
// ---------------------------------------------------------------------------
// The block's partial row: column 0 sum log F_i, column 1 zero (quadratic
// forms are formed from the cross-products), then the lower triangle of
// e e^T / F row by row.  Called by every thread of the block.
__device__ inline void block_site_terms(int nz, double *rows, int rows_cap,
                                        bool valid, double F,
                                        const double (&e)[kMaxNZ], int row) {
  __shared__ double red[kLaneMaxThreads / 64][kStatsMax];
  const int nw = (int)blockDim.x >> 6;
  const int w = (int)threadIdx.x >> 6, t = (int)threadIdx.x & 63;
  const double rf = valid ? 1.0 / F : 0.0;
  double x = wave_sum_to63(valid ? log(F) : 0.0);
  if (t == 63) red[w][0] = x;
  int g = 2;
#pragma unroll
  for (int p = 0; p < kMaxNZ; p++) {
    if (p < nz) {
#pragma unroll
      for (int q = 0; q <= p; q++) {
        x = wave_sum_to63(e[p] * e[q] * rf);
        if (t == 63) red[w][g + q] = x;
      }
    }
    g += p + 1;
  }
  __syncthreads();
  const int nv = 2 + nz * (nz + 1) / 2;
  const int k = (int)threadIdx.x;
  if (k < nv) {
    double s = 0.0;
    if (k != 1)
      for (int ww = 0; ww < nw; ww++) s += red[ww][k];
    rows[(size_t)k * rows_cap + row] = s;
  }
}

// Number of per-site terms of a partial row (column 1, always 0, aside):
// log F, then the nz(nz+1)/2 cross-products.
__host__ __device__ constexpr int site_terms(int nz) {
  return 1 + nz * (nz + 1) / 2;
}

// block_site_terms through LDS.  Each lane writes its terms to its wave's
// area `w` (term v of lane t at w[v * 64 + t], site_terms(nz) x 64 doubles),
// each quad of lanes then sums one term over 16 lanes apiece in lane order
// and combines its four partials (pairs, then the two pairs), and with more
// than one wave per block the wave sums meet in LDS and are added in wave
// order.  The order is fixed, so a launch shape's sums are reproducible.
// `w` may be memory the wave has finished reading (the kept entries of its
// factor); the barrier before the writes also keeps those reads first.
__device__ inline void block_site_terms_lds(int nz, double *rows,
                                            int rows_cap, bool valid,
                                            double F,
                                            const double (&e)[kMaxNZ],
                                            int row, double *w) {
  __shared__ double wsum[kLaneMaxThreads / 64][kStatsMax];
  const int nw = (int)blockDim.x >> 6;
  const int wv = (int)threadIdx.x >> 6, t = (int)threadIdx.x & 63;
  const int nt = site_terms(nz);
  const double rf = valid ? 1.0 / F : 0.0;
  __syncthreads();
  w[t] = valid ? log(F) : 0.0;
  int g = 1;
#pragma unroll
  for (int p = 0; p < kMaxNZ; p++) {
    if (p < nz) {
#pragma unroll
      for (int q = 0; q <= p; q++) w[(g + q) * 64 + t] = e[p] * e[q] * rf;
    }
    g += p + 1;
  }
  __syncthreads();
  for (int v0 = 0; v0 < nt; v0 += 16) {
    const int v = v0 + (t >> 2), qd = t & 3;
    double s = 0.0;
    if (v < nt) {
      const double2 *src = reinterpret_cast<const double2 *>(w + v * 64 +
                                                             qd * 16);
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const double2 x = src[u];
        s += x.x;
        s += x.y;
      }
    }
    s += dpp_mov_any<0xB1, 0xF>(s);  // quad_perm [1,0,3,2]
    s += dpp_mov_any<0x4E, 0xF>(s);  // quad_perm [2,3,0,1]
    if (qd == 0 && v < nt) {
      if (nw == 1)
        rows[(size_t)(v == 0 ? 0 : v + 1) * rows_cap + row] = s;
      else
        wsum[wv][v] = s;
    }
  }
  if (nw == 1) {
    if (t == 0) rows[(size_t)rows_cap + row] = 0.0;
    return;
  }
  __syncthreads();
  const int k = (int)threadIdx.x;
  if (k <= nt) {  // column k of the row: term k - 1 beyond column 1
    double s = 0.0;
    if (k != 1) {
      const int v = k == 0 ? 0 : k - 1;
      for (int ww = 0; ww < nw; ww++) s += wsum[ww][v];
    }
    rows[(size_t)k * rows_cap + row] = s;
  }
}

// Per-lane kernel size for m neighbors.
inline int lane_M(int m) {
  return m <= 4 ? 4 : m <= 8 ? 8 : m <= 10 ? 10 : m <= 12 ? 12 : m <= 15 ? 15
                                                                          : 16;
}

// LDS of one wavefront, in doubles: the kept entries or the block sums'
// terms, whichever is more.
__host__ __device__ constexpr int lane_wave_doubles(int keep, int nz) {
  const int sums = site_terms(nz);
  return 64 * (keep > sums ? keep : (sums + 1) / 2 * 2);
}

// Dynamic LDS of the per-lane kernel's mode 2, per block.
inline size_t lane_lds_shm(int M, int nz, int threads) {
  return (size_t)(threads / 64) * lane_wave_doubles(lane_lds_entries(M), nz) *
         sizeof(double);
}

// LDS of the mixed per-lane kernel's covariance copy, per block.
size_t mixed_copy_shm(int m, int threads);

// The per-lane kernels on a, by launch mode (nngp_bf_lane.hpp and
// nngp_bf_mixed.hip).
template <int M, bool BATCH>
void launch_lane_m(const BfArgs &a, int variant, const dim3 &grid,
                   const dim3 &blk, hipStream_t st);
template <int M, bool BATCH>
void launch_lane_lds_m(const BfArgs &a, int variant, const dim3 &grid,
                       const dim3 &blk, hipStream_t st);
void launch_mixed(const BfArgs &a, int variant, int mode, const dim3 &grid,
                  const dim3 &blk, hipStream_t st);

// The row kernel (nngp_bf_row.hip) on a's single FP64 problem; -2 when the
// pass's matern table is missing.
int bf_row_launch(const BfArgs &a, const dim3 &grid, const dim3 &blk,
                  hipStream_t st);

}  // namespace nngp
