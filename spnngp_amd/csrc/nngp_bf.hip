// nngp_bf.hip — neighbor-system kernels: updateBF / updateConjBF
// (src/rNNGP.cpp:46-101, src/cNNGP.cpp:24-69), the quadratic form Q
// (src/util.cpp:261-280) and the site sums the samplers and the conjugate
// grid need.
//
// The updateBF kernels add up their sites' terms in the same launch (log F_i
// and e_i e_i^T / F_i, with e_i the residual vector of X and y at site i), so
// one launch gives everything a Metropolis step or a conjugate grid point
// needs:
//  * one site per lane, 64 a wavefront, fully unrolled (M <= 16, closed-form
//    covariances): k_bf_lane, k_bf_lane_lds (nngp_bf_lane.hpp) and the mixed
//    k_bf_mixed, k_bf_mixed_reg (nngp_bf_mixed.hip).  Sites with fewer than M
//    neighbors (the first m sites of the NNGP order) are padded with far-away
//    points: their rows/columns of C are exactly zero off the diagonal, so the
//    real block factors bit-for-bit as if unpadded and the padded coefficients
//    come out exactly 0.  Block size 64, 128 or 256 threads.
//  * one site per 16-lane row, four a wavefront (m <= 32, single FP64
//    problems, any covariance): k_bf_grp (nngp_bf_row.hip).
//  * k_bf_coop<BATCH, MM> (here): one site per wavefront, the matrix built in
//    LDS and factored with one row per lane in registers (any m <= MM <= 64,
//    any covariance including the Bessel-K matern), 1, 2 or 4 wavefronts per
//    block walking a contiguous run of sites.
// All compute C = s2 R(N,N) + t2 I, c = s2 R(N,i), the Cholesky factor of C
// (pivots kept as reciprocal square roots), v = L^-1 c, B = L^-T v and
// F = s2 + t2 - v.v, i.e. the reference's potrf -> potri -> symv result
// without forming the inverse.
//
// BATCH = true runs many problems in one launch: gridDim.y problems, problem
// j is fold j / ng at grid point j % ng (the conjugate model's k-fold grid
// search); fold arrays sit at fixed strides and each problem has its own
// covariance parameters, partial rows and failure flag.
//
// Sums are deterministic for a given launch configuration: every thread
// adds a fixed set of sites in a fixed order, each block reduces with a
// fixed butterfly per wavefront and its wavefronts in order into one
// partial row, and k_rows_sum adds the rows of each column in a fixed order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdint>
#include <vector>

#include "nngp_bf.hpp"

namespace nngp {

int rows_capacity(int n) {
  const int lane_rows = (n + 63) / 64;  // smallest lane block is 64 threads
  return lane_rows > kCoopBlocks ? lane_rows : kCoopBlocks;
}

// ---------------------------------------------------------------------------
// one site per wavefront (generic m, generic covariance)
// ---------------------------------------------------------------------------
__device__ __forceinline__ int tri_row(int p) {
  // largest k with k(k+1)/2 <= p
  int k = (int)((sqrtf(8.0f * (float)p + 1.0f) - 1.0f) * 0.5f);
  while ((k + 1) * (k + 2) / 2 <= p) k++;
  while (k * (k + 1) / 2 > p) k--;
  return k;
}

// Per-wave LDS of the wavefront kernels, in doubles.
__host__ __device__ inline int coop_wave_doubles(int m) {
  return m * (m + 1) + 3 * m;
}

// Solve site i's system in the wave's LDS area Am; every lane returns F and
// the residual vector e (identical in all lanes); lane t < cnt returns its
// coefficient B_t in bcoef.  False when a pivot is not positive.
template <int MM>
__device__ inline bool coop_site(const BfArgs &A, const BfProblem &P,
                                 const CovArgs &c, const BesselTab &bt,
                                 const MaternTab &mt, double *Am, int i,
                                 double &F,
                                 double (&e)[kMaxNZ], double &bcoef,
                                 int &cnt_out, int &off_out) {
  const int t = lane_opaque((int)threadIdx.x & 63);
  const int ld = A.m + 1;
  double *cv = Am + A.m * ld;
  double *px = cv + A.m;
  double *py = px + A.m;
  // wave-uniform (one site per wavefront): scalar registers, so the
  // guards on cnt below are scalar branches, not exec-mask changes
  const int cnt = __builtin_amdgcn_readfirstlane(P.lu[A.n + i]);
  const int off = __builtin_amdgcn_readfirstlane(P.lu[i]);
  cnt_out = cnt;
  off_out = off;
  bcoef = 0.0;
  if (cnt == 0) {
    F = c.diag;
#pragma unroll
    for (int j = 0; j < kMaxNZ; j++)
      e[j] = j < A.nz ? P.Z[(size_t)i * A.zs + j] : 0.0;
    return true;
  }
  const double2 s = P.xy[i];
  int myid = 0;
  if (t < cnt) {
    myid = P.nnIndx[off + t];
    const double2 q = P.xy[myid];
    px[t] = q.x;
    py[t] = q.y;
  }
  wave_sync();
  // augmented lower triangle: rows 0..cnt-1 are C, row cnt is c
  const int np = (cnt + 1) * (cnt + 2) / 2 - 1;
  for (int p = t; p < np; p += 64) {
    const int k = tri_row(p);
    const int l = p - k * (k + 1) / 2;
    if (k < cnt && k == l) {
      Am[k * ld + k] = c.diag;
    } else {
      const double ax = k < cnt ? px[k] : s.x;
      const double ay = k < cnt ? py[k] : s.y;
      const double val = s2_corr_rt(sqdist(ax, ay, px[l], py[l]), c, bt, mt);
      if (k < cnt)
        Am[k * ld + l] = val;
      else
        cv[l] = val;
    }
  }
  wave_sync();
  double x, vv;
  if (!wave_chol_rows<MM>(Am, ld, cnt, t, t < cnt ? cv[t] : 0.0, x, vv)) {
    F = 1.0;  // keeps the sums finite; the pass reports the failure
#pragma unroll
    for (int j = 0; j < kMaxNZ; j++) e[j] = 0.0;
    wave_sync();
    return false;
  }
  bcoef = t < cnt ? x : 0.0;
  F = c.diag - vv;
#pragma unroll
  for (int j = 0; j < kMaxNZ; j++) {
    e[j] = 0.0;
    if (j < A.nz) {
      const double part =
          wave_sum(t < cnt ? x * P.Z[(size_t)myid * A.zs + j] : 0.0);
      e[j] = P.Z[(size_t)i * A.zs + j] - part;
    }
  }
  wave_sync();  // this LDS area is reused by the wave's next site
  return true;
}

// Per-wave LDS of the mixed wavefront kernel, in floats: C's lower triangle
// and then its factor (m rows of m + 1), the vector c and the neighbor
// offsets.
__host__ __device__ inline int coop_mixed_wave_floats(int m) {
  return m * (m + 1) + 3 * m;
}

// coop_site in mixed precision (the per-lane k_bf_mixed's scheme, one site
// per wavefront): neighbor offsets from site i and the covariance (any
// covModel, the matern by xnu_bessel_k32) in FP32, the FP32 factor one row
// per lane in registers, B0 = C32^-1 c32 in FP32, the residual
// r = c32 - C32 B0 of that FP32 system in FP64 (products of FP32 values are
// exact in FP64; lane t keeps its whole row of C32 in registers for it),
// one FP32 correction solve B = B0 + C32^-1 r, and F = s2 + t2 - c32.B and
// the residuals e in FP64.  False when a pivot or F is not positive.
template <int MM>
__device__ inline bool coop_site_mixed(const BfArgs &A, const BfProblem &P,
                                       const CovArgs &c,
                                       const CovArgs32 &c32,
                                       const BesselTab32 &bt, float *W, int i,
                                       double &F, double (&e)[kMaxNZ],
                                       double &bcoef, int &cnt_out,
                                       int &off_out) {
  const int t = lane_opaque((int)threadIdx.x & 63);
  const int ld = A.m + 1;
  float *Lm = W;
  float *cv = W + A.m * ld;
  float *px = cv + A.m;
  float *py = px + A.m;
  // wave-uniform (one site per wavefront): scalar registers, so the
  // guards on cnt below are scalar branches, not exec-mask changes
  const int cnt = __builtin_amdgcn_readfirstlane(P.lu[A.n + i]);
  const int off = __builtin_amdgcn_readfirstlane(P.lu[i]);
  cnt_out = cnt;
  off_out = off;
  bcoef = 0.0;
  if (cnt == 0) {
    F = c.diag;
#pragma unroll
    for (int j = 0; j < kMaxNZ; j++)
      e[j] = j < A.nz ? P.Z[(size_t)i * A.zs + j] : 0.0;
    return true;
  }
  const double2 s = P.xy[i];
  int myid = 0;
  if (t < cnt) {
    myid = P.nnIndx[off + t];
    const double2 q = P.xy[myid];
    px[t] = (float)(q.x - s.x);
    py[t] = (float)(q.y - s.y);
  }
  wave_sync();
  // augmented lower triangle: rows 0..cnt-1 are C, row cnt is c (site i
  // sits at the origin of the offsets)
  const int np = (cnt + 1) * (cnt + 2) / 2 - 1;
  for (int p = t; p < np; p += 64) {
    const int k = tri_row(p);
    const int l = p - k * (k + 1) / 2;
    if (k < cnt && k == l) {
      Lm[k * ld + k] = c32.diag;
    } else {
      const float ex = (k < cnt ? px[k] : 0.0f) - px[l];
      const float ey = (k < cnt ? py[k] : 0.0f) - py[l];
      const float val = s2_corr32_rt(fmaf(ex, ex, ey * ey), c32, bt);
      if (k < cnt)
        Lm[k * ld + l] = val;
      else
        cv[l] = val;
    }
  }
  wave_sync();
  float crow[MM], row[MM];
#pragma unroll
  for (int l = 0; l < MM; l++) {
    crow[l] = (t < cnt && l < cnt)
                  ? (l <= t ? Lm[t * ld + l] : Lm[l * ld + t])
                  : 0.0f;
    row[l] = l <= t ? crow[l] : 0.0f;
  }
  const float ct = t < cnt ? cv[t] : 0.0f;
  wave_sync();  // C is in registers now; the factor takes its place
  bool ok = wave_factor32<MM>(row, cnt, t);
  double x = 0.0;
  if (ok) {
#pragma unroll
    for (int l = 0; l < MM; l++)
      if (t < cnt && l <= t) Lm[t * ld + l] = row[l];
    wave_sync();
    const float x0 = wave_solve32<MM>(row, Lm, ld, cnt, t, ct);
    double r = (double)ct;
#pragma unroll
    for (int l = 0; l < MM; l++)
      if (l < cnt) r = fma(-(double)crow[l], (double)readlane_f(x0, l), r);
    const float d =
        wave_solve32<MM>(row, Lm, ld, cnt, t, t < cnt ? (float)r : 0.0f);
    x = t < cnt ? (double)x0 + (double)d : 0.0;
    F = c.diag - wave_sum((double)ct * x);
    ok = F > 0.0;
  }
  if (!ok) {
    F = 1.0;  // keeps the sums finite; the pass reports the failure
#pragma unroll
    for (int j = 0; j < kMaxNZ; j++) e[j] = 0.0;
    wave_sync();
    return false;
  }
  bcoef = x;
#pragma unroll
  for (int j = 0; j < kMaxNZ; j++) {
    e[j] = 0.0;
    if (j < A.nz) {
      const double part =
          wave_sum(t < cnt ? x * P.Z[(size_t)myid * A.zs + j] : 0.0);
      e[j] = P.Z[(size_t)i * A.zs + j] - part;
    }
  }
  wave_sync();  // this LDS area is reused by the wave's next site
  return true;
}

// The waves of the logical blocks of one XCD take that XCD's run of sites
// round robin (xcd_site_run).  A.coop_blocks logical blocks per problem.
// MIXED: the sites are solved by coop_site_mixed (single problem only).
// The block's matern tables: FP64 passes the Bessel-K loop divisors and the
// pass's correlation table, mixed passes the FP32 divisors.
template <bool MIXED>
struct CoopTabs {
  BesselTab bt;
  MaternTab mt;
};
template <>
struct CoopTabs<true> {
  BesselTab32 bt32;
};

template <bool BATCH, int MM, bool MIXED>
__global__ __launch_bounds__(64 * kCoopMaxWaves) void k_bf_coop(BfArgs A) {
  extern __shared__ double smem[];
  __shared__ double red[kCoopMaxWaves][kStatsMax];
  __shared__ CoopTabs<MIXED> tabs;
  const int nw = (int)blockDim.x >> 6;
  const int w = (int)threadIdx.x >> 6;
  const int t = (int)threadIdx.x & 63;
  const int b = xcd_block(A.coop_blocks);
  if (b < 0) return;
  const BfProblem P = bf_problem<BATCH>(A);
  const CovArgs c = BATCH ? A.covs[(int)blockIdx.y % A.ng] : A.c;
  if (c.cov == 2) {  // the matern's loop divisors for this block's mu
    if constexpr (MIXED) {
      bessel_tab_fill32(tabs.bt32, c);
      __syncthreads();
    } else {
      bessel_tab_fill(tabs.bt, c);
      __syncthreads();
      // and the pass's correlation table, built in the waves' system areas
      // (at least kMatScratch doubles, see the launcher) before their use
      matern_tab_fill(tabs.mt, c, tabs.bt, smem);
    }
  }
  double *Am = smem + (size_t)w * coop_wave_doubles(A.m);
  float *Wf = reinterpret_cast<float *>(smem) +
              (size_t)w * coop_mixed_wave_floats(A.m);
  const CovArgs32 c32 = cov32(c);
  const SiteRun run = xcd_site_run(A.coop_blocks, b, A.n, nw, w);
  // the wave's running sums live in LDS (lane 0 updates them), which keeps
  // this kernel's registers low enough for several waves per SIMD
  const int nv = 2 + A.nz * (A.nz + 1) / 2;
  for (int k = t; k < nv; k += 64) red[w][k] = 0.0;
  wave_sync();
  for (int i = run.first; i < run.end; i += run.stride) {
    double F, e[kMaxNZ], bcoef;
    int cnt, off;
    bool ok;
    if constexpr (MIXED)
      ok = coop_site_mixed<MM>(A, P, c, c32, tabs.bt32, Wf, i, F, e, bcoef,
                               cnt, off);
    else
      ok = coop_site<MM>(A, P, c, tabs.bt, tabs.mt, Am, i, F, e, bcoef, cnt,
                         off);
    if (!ok && t == 0) atomicMin(P.err, i);
    if (!BATCH) {
      if (A.B && ok && t < cnt) A.B[off + t] = bcoef;
      if (A.F && t == 0) A.F[i] = F;
    }
    if (t == 0) {
      const double rf = 1.0 / F;
      red[w][0] += log(F);
      int g = 2;
#pragma unroll
      for (int p = 0; p < kMaxNZ; p++) {
        if (p < A.nz) {
#pragma unroll
          for (int q = 0; q <= p; q++) red[w][g + q] += e[p] * e[q] * rf;
        }
        g += p + 1;
      }
    }
  }
  if (!P.rows) return;
  __syncthreads();
  const int k = (int)threadIdx.x;
  if (k < nv) {
    double s = 0.0;
    if (k != 1)
      for (int ww = 0; ww < nw; ww++) s += red[ww][k];
    P.rows[(size_t)k * A.rows_cap + b] = s;
  }
}

// ---------------------------------------------------------------------------
// sums
// ---------------------------------------------------------------------------
// Block (k, j): out[j*out_stride + k] = sum over rows r < nrows of column k
// of problem j's rows (fixed per-thread order, fixed butterfly).  Block
// (0, j) also hands over problem j's failure flag:
// err_out[j] = err[j], err[j] = INT_MAX.
__global__ __launch_bounds__(kRowsThreads) void k_rows_sum(
    const double *rows, int cap, int nrows, long long ps_rows, double *out,
    int out_stride, int *err, double *err_out, SumsSignal sig) {
  __shared__ double red[kRowsThreads / 64];
  const int k = (int)blockIdx.x, j = (int)blockIdx.y;
  const int w = (int)threadIdx.x >> 6, t = (int)threadIdx.x & 63;
  const double *col = rows + (size_t)j * ps_rows + (size_t)k * cap;
  // eight independent partial sums, so that a thread's loads are in flight
  // together; the order (per thread, then the fixed combination) is fixed
  constexpr int U = 8;
  double acc[U];
#pragma unroll
  for (int u = 0; u < U; u++) acc[u] = 0.0;
  int r = (int)threadIdx.x;
  for (; r + (U - 1) * kRowsThreads < nrows; r += U * kRowsThreads) {
#pragma unroll
    for (int u = 0; u < U; u++) acc[u] += col[r + u * kRowsThreads];
  }
#pragma unroll
  for (int u = 0; u < U; u++) {  // the tail: fewer than U rows left
    const int rr = r + u * kRowsThreads;
    if (rr < nrows) acc[u] += col[rr];
  }
  double s = ((acc[0] + acc[1]) + (acc[2] + acc[3])) +
             ((acc[4] + acc[5]) + (acc[6] + acc[7]));
  s = wave_sum(s);
  if (t == 0) red[w] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double tot = 0.0;
#pragma unroll
    for (int ww = 0; ww < kRowsThreads / 64; ww++) tot += red[ww];
    out[(size_t)j * out_stride + k] = tot;
    if (k == 0 && err) {
      err_out[j] = (double)err[j];
      err[j] = INT_MAX;
    }
    if (sig.flag) {  // the completion word, from the last block to finish
      __threadfence_system();  // this block's outputs, visible to the host
      const unsigned nb = gridDim.x * gridDim.y;
      if ((unsigned)atomicAdd(sig.done, 1) == nb - 1) {
        *sig.done = 0;
        __hip_atomic_store(sig.flag, sig.seq, __ATOMIC_RELEASE,
                           __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
  }
}

int rows_sum_launch(const double *rows, int cap, int nrows, long long ps_rows,
                    int nv, int nprob, double *out, int out_stride, int *err,
                    double *err_out, hipStream_t st, const SumsSignal *sig) {
  const SumsSignal none;
  hipLaunchKernelGGL(k_rows_sum, dim3(nv, nprob), dim3(kRowsThreads), 0, st,
                     rows, cap, nrows, ps_rows, out, out_stride, err,
                     err_out, sig ? *sig : none);
  return (int)hipGetLastError();
}

static int red_grid(int n) {
  const int b = (n + kRedThreads - 1) / kRedThreads;
  return b < 1 ? 1 : (b > kRedBlocks ? kRedBlocks : b);
}

// ---------------------------------------------------------------------------
// dispatch
// ---------------------------------------------------------------------------
bool bf_lane_ok(int m, int variant) { return m <= 16 && variant >= 0; }

// Scratch of matern_tab_fill, in doubles.
constexpr int kMatScratch = 2 * kMatPieces * kMatN + kMatN * kMatN;

// LDS per block of the wavefront kernel with `waves` waves (FP64; its
// system areas also hold the matern table's build).
static size_t coop_shm(int m, int waves) {
  const size_t d = (size_t)waves * coop_wave_doubles(m);
  return (d > (size_t)kMatScratch ? d : (size_t)kMatScratch) * sizeof(double);
}

bool bf_config_ok(const BfConfig &cfg, int m, int variant) {
  if (cfg.family == 0)
    return bf_lane_ok(m, variant) &&
           (cfg.threads == 64 || cfg.threads == 128 || cfg.threads == 256) &&
           (cfg.mode == 0 || cfg.mode == 2 || cfg.mode == 3 ||
            (cfg.mode == 1 && mixed_copy_shm(m, cfg.threads) <= 65536));
  if (cfg.family == 2)
    return m <= kGrpMaxM && cfg.mode == 0 &&
           (cfg.threads == 64 || cfg.threads == 128 || cfg.threads == 256);
  if (cfg.family != 1) return false;
  const int waves = cfg.threads / 64;
  return m <= kCoopMaxM && cfg.threads % 64 == 0 && waves >= 1 &&
         waves <= kCoopMaxWaves && coop_shm(m, waves) <= 65536;
}

// Untuned passes: per lane at 64 threads with finished rows of the factor
// in LDS where that applies (the fastest per-lane shape at n = 1e6, m = 15);
// else, for single FP64 problems with m <= 32, the row kernel at 256 threads
// (n = 4e6, m = 32, Bessel-K matern: 11 ms against 41 ms on the wavefront
// kernel); else the wavefront kernel.
BfConfig bf_default(int m, int variant, bool single_fp64) {
  BfConfig c;
  if (bf_lane_ok(m, variant)) {
    c.family = 0;
    c.threads = 64;
    c.mode = 2;
  } else if (single_fp64 && m <= kGrpMaxM) {
    c.family = 2;
    c.threads = 256;
  } else {
    c.family = 1;
    int w = kCoopMaxWaves;
    while (w > 1 && coop_shm(m, w) > 65536) w--;
    c.threads = 64 * w;
  }
  return c;
}

int bf_rows(const BfArgs &a, const BfConfig &cfg) {
  if (cfg.family == 0) return (a.n + cfg.threads - 1) / cfg.threads;
  const int waves = cfg.threads / 64;
  // the row kernel's waves take groups of four sites
  const int units = cfg.family == 2 ? (a.n + 3) / 4 : a.n;
  const int need = (units + waves - 1) / waves;
  const bool two = cfg.family == 2 && (a.m > 16 || a.c.cov == 2);
  const int most = two ? kGrpWaves / waves : kCoopBlocks;
  return need < most ? need : most;
}

// Whether an FP64 per-lane pass takes mode 2 (m > 8, where the system is
// large enough to matter, and the block's LDS within 64 KiB: 64 and 128
// threads from m = 13 on); where it does not, mode 2 runs the plain per-lane
// kernel, whose results are the same bit for bit.
static bool lane_lds_applies(const BfArgs &a, int threads) {
  return !a.mixed && a.m > 8 &&
         lane_lds_shm(lane_M(a.m), a.nz, threads) <= 65536;
}

template <bool BATCH>
static void launch_lane_lds(const BfArgs &a, int variant, const dim3 &grid,
                            const dim3 &blk, hipStream_t st) {
  switch (lane_M(a.m)) {
    case 10: launch_lane_lds_m<10, BATCH>(a, variant, grid, blk, st); break;
    case 12: launch_lane_lds_m<12, BATCH>(a, variant, grid, blk, st); break;
    case 15: launch_lane_lds_m<15, BATCH>(a, variant, grid, blk, st); break;
    default: launch_lane_lds_m<16, BATCH>(a, variant, grid, blk, st); break;
  }
}

template <bool BATCH>
static void launch_lane(const BfArgs &a, int variant, const dim3 &grid,
                        const dim3 &blk, hipStream_t st) {
  if (a.m <= 4) launch_lane_m<4, BATCH>(a, variant, grid, blk, st);
  else if (a.m <= 8) launch_lane_m<8, BATCH>(a, variant, grid, blk, st);
  else if (a.m <= 10) launch_lane_m<10, BATCH>(a, variant, grid, blk, st);
  else if (a.m <= 12) launch_lane_m<12, BATCH>(a, variant, grid, blk, st);
  else if (a.m <= 15) launch_lane_m<15, BATCH>(a, variant, grid, blk, st);
  else launch_lane_m<16, BATCH>(a, variant, grid, blk, st);
}

// The wavefront kernel's register-resident factor is sized by the smallest
// of 16, 32 and 64 rows that holds m.
template <bool BATCH, bool MIXED>
static void launch_coop(const BfArgs &a, const dim3 &grid, const dim3 &blk,
                        size_t shm, hipStream_t st) {
  switch (wave_rows_for(a.m)) {
    case 16:
      hipLaunchKernelGGL((k_bf_coop<BATCH, 16, MIXED>), grid, blk, shm, st, a);
      break;
    case 32:
      hipLaunchKernelGGL((k_bf_coop<BATCH, 32, MIXED>), grid, blk, shm, st, a);
      break;
    default:
      hipLaunchKernelGGL((k_bf_coop<BATCH, 64, MIXED>), grid, blk, shm, st, a);
  }
}

int bf_launch(const BfArgs &a0, const BfConfig &cfg, int nprob,
              hipStream_t st) {
  if (a0.n <= 0 || nprob <= 0) return 0;
  const bool batch = a0.ng > 0;
  if (!batch && nprob != 1) return -2;
  const int variant = a0.variant;
  if (!bf_config_ok(cfg, a0.m, variant)) return -1;
  BfArgs a = a0;
  const int nrows = bf_rows(a, cfg);
  if (a.rows && nrows > a.rows_cap) return -2;
  const dim3 grid(8 * ((nrows + 7) / 8), nprob);
  const dim3 blk(cfg.threads);
  if (cfg.family == 0) {
    const bool lds = cfg.mode == 2 && lane_lds_applies(a, cfg.threads);
    if (batch) {
      if (lds) launch_lane_lds<true>(a, variant, grid, blk, st);
      else launch_lane<true>(a, variant, grid, blk, st);
    }
    else if (a.mixed) launch_mixed(a, variant, cfg.mode, grid, blk, st);
    else if (lds) launch_lane_lds<false>(a, variant, grid, blk, st);
    else launch_lane<false>(a, variant, grid, blk, st);
  } else if (cfg.family == 2) {
    if (batch || a.mixed) return -1;  // single FP64 problems only
    a.coop_blocks = nrows;
    if (const int rc = bf_row_launch(a, grid, blk, st)) return rc;
  } else {
    a.coop_blocks = nrows;
    const int waves = cfg.threads / 64;
    if (batch)
      launch_coop<true, false>(a, grid, blk, coop_shm(a.m, waves), st);
    else if (a.mixed)
      launch_coop<false, true>(
          a, grid, blk,
          (size_t)waves * coop_mixed_wave_floats(a.m) * sizeof(float), st);
    else
      launch_coop<false, false>(a, grid, blk, coop_shm(a.m, waves), st);
  }
  return (int)hipGetLastError();
}

int bf_sums_launch(const BfArgs &a, const BfConfig &cfg, int nprob,
                   double *out, int out_stride, double *err_out,
                   hipStream_t st, const SumsSignal *sig) {
  const int nv = 2 + a.nz * (a.nz + 1) / 2;
  return rows_sum_launch(a.rows, a.rows_cap, bf_rows(a, cfg), a.ps_rows, nv,
                         nprob, out, out_stride, a.err, err_out, st, sig);
}

// ---------------------------------------------------------------------------
// autotuner
// ---------------------------------------------------------------------------
// Candidates: sites per wavefront (64: the per-lane kernel at 64, 128 or
// 256 threads per block; 1: the wavefront kernel with 1, 2 or 4 waves per
// block, i.e. LDS tiles of 1, 2 or 4 systems; 4: the row kernel).  Each is
// timed with HIP events on the caller's stream (one warm-up, then three
// launches; fewer where it is far behind) and the fastest kept.
int bf_autotune(const BfArgs &a, int nprob, hipStream_t st, BfConfig *best,
                BfTuneReport *rep) {
  const int variant = a.variant;
  std::vector<BfConfig> cand;
  if (a.mixed) {  // the per-lane mixed kernel: block size x covariance
                  // copy (none, LDS, registers); then the wavefront one
    for (int th : {64, 128, 256})
      for (int mode : {0, 1, 3}) cand.push_back(BfConfig{0, th, mode});
  } else {  // the per-lane kernel: block size x factor rows in LDS
    for (int th : {64, 128, 256}) {
      cand.push_back(BfConfig{0, th, 0});
      if (lane_lds_applies(a, th)) cand.push_back(BfConfig{0, th, 2});
    }
  }
  for (int w : {1, 2, 4}) cand.push_back(BfConfig{1, 64 * w, 0});
  if (!a.mixed && a.ng == 0)  // four sites per wavefront, one per row
    for (int th : {64, 128, 256}) cand.push_back(BfConfig{2, th, 0});
  hipEvent_t e0, e1;
  if (hipEventCreate(&e0) != hipSuccess) return -1;
  if (hipEventCreate(&e1) != hipSuccess) {
    (void)hipEventDestroy(e0);
    return -1;
  }
  // mean time of `reps` launches after one more
  auto timed = [&](const BfConfig &cfg, int np, int reps, double *per) -> int {
    int e = bf_launch(a, cfg, np, st);
    if (!e) e = (int)hipEventRecord(e0, st);
    for (int r = 0; r < reps && !e; r++) e = bf_launch(a, cfg, np, st);
    if (!e) e = (int)hipEventRecord(e1, st);
    if (!e) e = (int)hipEventSynchronize(e1);
    float ms = 0.0f;
    if (!e) e = (int)hipEventElapsedTime(&ms, e0, e1);
    *per = ms / reps;
    return e;
  };
  double best_ms = 1e300, best_few = 1e300;
  BfConfig pick = bf_default(a.m, variant, !a.mixed && a.ng == 0);
  int nc = 0;
  int rc = 0;
  for (const BfConfig &cfg : cand) {
    if (!bf_config_ok(cfg, a.m, variant)) continue;
    if (a.rows && bf_rows(a, cfg) > a.rows_cap) continue;
    double per = 0.0;
    // a candidate that a sixteenth of the problems (or the one problem) shows
    // to be half as fast as one before it is not timed further, nor kept; its
    // report is that one launch's time scaled to all problems.  The wavefront
    // shapes of a 250-problem grid cost 370 of its first run's 393 ms.  Few
    // problems leave part of the chip idle, which favors the shapes with more
    // waves; those stand behind the per-lane ones, so none is ruled out by it.
    const int few = std::max(1, nprob / 16);
    if ((rc = timed(cfg, few, 1, &per)) != 0) break;
    best_few = std::min(best_few, per);
    const bool whole = per < 2.0 * best_few;
    if (whole)
      rc = timed(cfg, nprob, 3, &per);
    else
      per *= (double)nprob / few;
    if (rc) break;
    if (rep && nc < NNGP_TUNE_MAX) {
      rep->family[nc] = cfg.family;
      rep->threads[nc] = cfg.threads;
      rep->mode[nc] = cfg.mode;
      rep->ms[nc] = per;
    }
    nc++;
    if (whole && per < best_ms) {
      best_ms = per;
      pick = cfg;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (rc) return rc;
  if (rep) {
    rep->n = nc < NNGP_TUNE_MAX ? nc : NNGP_TUNE_MAX;
    rep->best = pick;
    rep->best_ms = best_ms;
  }
  *best = pick;
  return 0;
}

// ---------------------------------------------------------------------------
// plain Q(u, v)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kRedThreads) void k_quadform(QArgs A) {
  __shared__ double red[kRedThreads / 64];
  double acc = 0.0;
  const int stride = (int)gridDim.x * kRedThreads;
  for (int i = blockIdx.x * kRedThreads + threadIdx.x; i < A.n; i += stride) {
    const int cnt = A.lu[A.n + i], off = A.lu[i];
    double a = 0.0, b = 0.0;
    for (int j = 0; j < cnt; j++) {
      const double bj = A.B[off + j];
      const int id = A.nnIndx[off + j];
      a += bj * A.u[id];
      b += bj * A.v[id];
    }
    acc += (A.u[i] - a) * (A.v[i] - b) / A.F[i];
  }
  const int w = (int)threadIdx.x >> 6, t = (int)threadIdx.x & 63;
  const double x = wave_sum(acc);
  if (t == 0) red[w] = x;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
#pragma unroll
    for (int ww = 0; ww < kRedThreads / 64; ww++) s += red[ww];
    A.rows[blockIdx.x] = s;
  }
}

static_assert(kRedBlocks == kQPartialRows,
              "k_quadform's grid bounds its partial sums");

int q_partial_rows(int n) { return red_grid(n); }

int q_launch(const QArgs &a, hipStream_t st) {
  const int nb = red_grid(a.n);
  hipLaunchKernelGGL(k_quadform, dim3(nb), dim3(kRedThreads), 0, st, a);
  return rows_sum_launch(a.rows, kRedBlocks, nb, 0, 1, 1, a.out, 1, nullptr,
                         nullptr, st);
}

__global__ void k_interleave(const double *cm, int n, double2 *xy) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) xy[i] = make_double2(cm[i], cm[(size_t)n + i]);
}

int interleave_launch(const double *coords_cm, int n, double2 *xy,
                      hipStream_t st) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(k_interleave, dim3((n + 255) / 256), dim3(256), 0, st,
                     coords_cm, n, xy);
  return (int)hipGetLastError();
}

}  // namespace nngp
