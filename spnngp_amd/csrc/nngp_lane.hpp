// nngp_lane.hpp — the neighbor system of one site (or of one site and sample)
// solved by one lane at two waves a SIMD: updateBF, the conjugate grid's
// held-out sites and kriging.
#pragma once
#include "nngp_device.hpp"

namespace nngp {

// The parameters at p, the same for every lane of the grid's row, by scalar
// loads: as an ordinary load they would fill 70 vector registers a lane.  p is
// not written while the kernel runs.
__device__ __forceinline__ CovArgs cov_uniform(const CovArgs *p) {
  static_assert(sizeof(CovArgs) % sizeof(double) == 0, "whole doubles");
  using Src = const __attribute__((address_space(4))) double *;
  const Src src = (Src)(uintptr_t)p;
  CovArgs c;
  double *d = reinterpret_cast<double *>(&c);
#pragma unroll
  for (int k = 0; k < (int)(sizeof(CovArgs) / sizeof(double)); k++)
    d[k] = src[k];
  return c;
}

// Entries of the factor, in packed order, that wait in LDS from the column
// that finishes their row to the back substitution (row k of L has its last
// use in the factorization in column k).  Two waves a SIMD leave 256 registers
// a lane.  Going down the columns, the rows still open, the finished rows, the
// right-hand side and the coordinates not yet used come to 135 doubles at
// M = 15 (153 at M = 16); with the first 36 entries in LDS, 99 (117),
// which fits beside the temporaries, at 18 KB a wave: eight waves take 144
// of a CU's 160 KB.  Up to M = 12 everything fits in registers.
// Whole rows: row 7 is the last one kept.
__host__ __device__ constexpr int lane_lds_entries(int M) {
  return M <= 12 ? 0 : 36;
}

// v = C^-1 c and vv = c^T C^-1 c of the M x M system with diagonal `diag`,
// entries entry(k, l), l < k, below it and right-hand side rhs(j).  False when
// a pivot is not positive (the reference's dpotrf failure).  K entries of the
// factor wait in LDS: pair q of them at keep[q * 64], `keep` the lane's slot
// in its wavefront's area.
//
// The lower triangle is built and factored column by column (left-looking),
// the covariance entries of a column evaluated when it is reached, so that
// the M x M system is never held whole: one wave a SIMD, with the whole
// triangle in registers, left the vector units idle for 30% of the time (the
// gathers at a wave's start and the chains of dependent instructions).  Each
// entry goes through the same operations in the same order as in a
// right-looking factorization (chol_solve), so the results are the same bit
// for bit.
//
// Going back up, the registers of the rows that are done with take what the
// caller needs next, so that nothing waits for memory after the solve: it asks
// for its first loads in mid() (behind row M - 4) and for those that depend on
// them in up() (behind row kUp, where the kept entries come back).  The empty
// asm stands behind the finished rows' work by v[k]; it also keeps the kept
// entries from being held in registers since they were stored, and the loads
// before it from sinking to their uses.
//
// EARLY: the pivots' signs are gathered in a scalar mask column by column.
// Without it the compiler may keep all M pivots and test them where the result
// is used, M spills: 140 B a lane in kriging at M = 15 (28 with the mask), 28
// B in the held-out sites and 36 B in the batched updateBF (none).  The single
// updateBF pass at M = 15 has no spills without the mask and 12 B with it; at M
// = 16 84 to 172 B without and 0 to 44 B with it (n = 3,000, p = 3, exponential:
// 17.1 us, now 15.8; n = 1e6 241 and 210).  Kriging at M = 8 takes 124 registers
// without the mask and 136 with it, three waves a SIMD for four (2,000 sites x
// 500 samples 59.9 and 63.0 us).
template <int M, int K, bool HOOKS, bool EARLY, class Entry, class Rhs,
          class Mid, class Up>
__device__ __forceinline__ bool lane_solve(double diag, Entry &&entry,
                                           Rhs &&rhs, double2 *keep,
                                           double (&v)[M], double &vv,
                                           Mid &&mid, Up &&up) {
  constexpr int T = M * (M + 1) / 2;
  constexpr int kUp = K > 0 ? 7 : M / 2 - 1;
  static_assert(K == 0 || K == tri(kUp, kUp) + 1, "whole rows are kept");
  double a[T];  // packed lower triangle, diagonal as 1 / L_jj
  vv = 0.0;
  bool ok = true;
  unsigned long long pos = ~0ull;
#pragma unroll
  for (int j = 0; j < M; j++) {
    v[j] = rhs(j);
#pragma unroll
    for (int k = j + 1; k < M; k++) a[tri(k, j)] = entry(k, j);
    double piv = diag;
#pragma unroll
    for (int l = 0; l < j; l++) {
      const double ljl = a[tri(j, l)];
      piv = fma(-ljl, ljl, piv);
      v[j] = fma(-ljl, v[l], v[j]);
#pragma unroll
      for (int k = j + 1; k < M; k++)
        a[tri(k, j)] = fma(-a[tri(k, l)], ljl, a[tri(k, j)]);
    }
    if (EARLY) {
      pos &= __ballot(piv > 0.0);
      asm volatile("" : "+s"(pos));
    } else {
      ok = ok && (piv > 0.0);
    }
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
#pragma unroll
  for (int k = M - 1; k >= 0; k--) {
    if (HOOKS && k == M - 4) {
      asm volatile("" : "+v"(v[k]) : : "memory");
      mid();
    }
    if ((K > 0 || HOOKS) && k == kUp) {
      asm volatile("" : "+v"(v[k]) : : "memory");
#pragma unroll
      for (int q = 0; q < K / 2; q++) {
        const double2 x = keep[q * 64];
        a[2 * q] = x.x;
        a[2 * q + 1] = x.y;
      }
      if (HOOKS) up();
    }
    const double t = v[k] * a[tri(k, k)];
    v[k] = t;
#pragma unroll
    for (int l = 0; l < k; l++) v[l] = fma(-a[tri(k, l)], t, v[l]);
  }
  if (HOOKS) asm volatile("" : "+v"(v[0]) : : "memory");
  return EARLY ? (pos >> (threadIdx.x & 63)) & 1 : ok;
}

}  // namespace nngp
