// nngp_bf_row.hip — updateBF (src/rNNGP.cpp:46-101) with one site per 16-lane
// row of a wavefront, four sites a wavefront, m <= 32, FP64: the general-nu
// matern, m > 16, and passes of few sites.
#include "nngp_bf.hpp"
#include "nngp_group.hpp"

namespace nngp {

// ---------------------------------------------------------------------------
// one site per 16-lane row (four sites per wavefront), m <= 32
// ---------------------------------------------------------------------------
constexpr int kGrpSlots = 4 * kCoopMaxWaves;  // sites a block works on at once

// Per-wave LDS of the row kernel, in doubles: each of its four rows'
// neighbor coordinates, x then y.
__host__ __device__ inline int grp_wave_doubles(int mm) { return 4 * 2 * mm; }

// The pass's matern table (matern_piece): block o fills the pieces of octave
// o from the series at their Chebyshev points; block 0 also writes the
// Bessel-K loop divisors behind the table, for the entries outside it.
// 36 blocks take about as long as one series evaluation; with every block of
// the row kernel building a table for itself (and 16 coefficients an entry) a
// pass took 261 us at n = 1e5, m = 15 and 1.99 ms at n = 5e5, m = 32; with
// this launch before it, 140 us and 1.53 ms.
constexpr int kMpThreads = 192;  // at least kMpSub * kMpN

__global__ __launch_bounds__(kMpThreads) void k_matern_pieces(CovArgs c,
                                                              double *out) {
  __shared__ BesselTab bt;
  __shared__ double fv[kMpSub * kMpN], cc[kMpSub * kMpN];
  bessel_tab_fill(bt, c);
  __syncthreads();
  const int q = (int)threadIdx.x, o = (int)blockIdx.x;
  const int pc = q / kMpN, j = q % kMpN;  // piece of the octave, node
  if (q < kMpSub * kMpN) {
    const double u = cospi((j + 0.5) / kMpN);
    const double m = 1.0 + (pc + 0.5 + 0.5 * u) / kMpSub;
    fv[q] = c.mnorm * xnu_bessel_k(ldexp(m, kMpOct0 + o), c, bt);
  }
  __syncthreads();
  if (q < kMpSub * kMpN) {  // Chebyshev coefficient j of the piece
    double s = 0.0;
    for (int k = 0; k < kMpN; k++)
      s = fma(fv[pc * kMpN + k], cospi(j * (k + 0.5) / kMpN), s);
    cc[q] = s * (j == 0 ? 1.0 / kMpN : 2.0 / kMpN);
  }
  __syncthreads();
  if (q < kMpSub * kMpN) {  // coefficient of (m - c)^j, u = 2 kMpSub (m - c)
    double s = 0.0;
    for (int k = j; k < kMpN; k++)
      s = fma(cc[pc * kMpN + k], kChebMono.t[k][j], s);
    out[(o * kMpSub + pc) * kMpN + j] = s * ldexp(1.0, 5 * j);
  }
  if (o == 0) {
    const double *src = reinterpret_cast<const double *>(&bt);
    for (int k = q; k < (int)(sizeof(BesselTab) / sizeof(double));
         k += kMpThreads)
      out[kMpLen + k] = src[k];
  }
}
static_assert(2 * kMpSub == 32, "u = 2^5 (m - c)");

// Covariance entries of the row kernel.  A lane evaluates about fifty per
// site in fully unrolled code, so only the common path is inline: for the
// matern (MAT) the pass's table, with coincident or nearly coincident sites
// and x >= 64 (outside the table) out of line; otherwise the exponential,
// spherical and gaussian.  The out-of-line series reads the parameters from
// the block's LDS copy `al` (a reference to the kernel argument would make
// the kernel keep a stack copy of it and read the inline path's fields from
// there).
__device__ __noinline__ double grp_matern_outside(double x, const CovArgs &al,
                                                  const BesselTab &bt) {
  if (!(x > 0.0)) return al.s2;
  if (x > 700.0) return 0.0;
  return al.mnorm * xnu_bessel_k(x, al, bt);
}

// Where the row kernel's entries come from: the parameters and, for the
// matern, their LDS copy, the table (LDS) and the divisors (device memory).
struct GrpCov {
  const CovArgs &a, &al;
  const double *T;
  const BesselTab &bt;
};

template <bool MAT>
__device__ __forceinline__ double grp_corr(double d2, const GrpCov &c) {
  if constexpr (MAT) {
    const double x = nn_sqrt(d2) * c.a.phi;
    const unsigned r = matern_piece(x);
    if (r >= (unsigned)kMpRows) return grp_matern_outside(x, c.al, c.bt);
    return matern_piece_at(x, r, c.T);
  } else {
    switch (c.a.cov) {
      case 0: return s2_corr<0>(d2, c.a);
      case 1: return s2_corr<1>(d2, c.a);
      default: return s2_corr<3>(d2, c.a);
    }
  }
}

// A site's inputs on its row: neighbor count and offset, the lane's two
// neighbor ids and coordinates, the site's coordinates.  The three loads
// depend on each other, so the row kernel fetches the next site's in three
// stages spread over the current site's work.
struct GrpIn {
  int cnt, off, ida, idb;
  double2 qa, qb, s;
};

__device__ __forceinline__ void grp_in_lu(const BfArgs &A, const BfProblem &P,
                                          int i, bool valid, GrpIn &in) {
  in.cnt = 0;
  in.off = 0;
  if (valid) {
    in.cnt = P.lu[A.n + i];
    in.off = P.lu[i];
  }
}

template <int R>
__device__ __forceinline__ void grp_in_ids(const BfProblem &P, int u,
                                           GrpIn &in) {
  in.ida = 0;
  in.idb = 0;
  if (u < in.cnt) in.ida = P.nnIndx[in.off + u];
  if (R == 2 && 31 - u < in.cnt) in.idb = P.nnIndx[in.off + 31 - u];
}

template <int R>
__device__ __forceinline__ void grp_in_xy(const BfProblem &P, int u, int i,
                                          bool valid, GrpIn &in) {
  in.qa = make_double2(0.0, 0.0);
  in.qb = in.qa;
  in.s = in.qa;
  if (u < in.cnt) in.qa = P.xy[in.ida];
  if (R == 2 && 31 - u < in.cnt) in.qb = P.xy[in.idb];
  if (valid) in.s = P.xy[i];
}

// The lane's rows of the system: the entries below the diagonal, the diagonal,
// zeros above.  Rows past the site's count are identity rows (with a zero
// right-hand side), so B and F are those of the cnt x cnt system.  An entry
// of the triangle costs an evaluation for all 16 lanes whether they need it
// or not, so the evaluations are shared out evenly:
//  * MM = 32: column l < 16 of row 31 - u is needed in every lane; column
//    14 - j of row u is needed where u > 14 - j, and column 16 + j of row
//    31 - u exactly in the other lanes, so one evaluation serves both: 31
//    for the 496 entries;
//  * MM = 16: column j < 7 of row u is needed where u > j; the other lanes
//    evaluate column 14 - j of row 15 - u for lane 15 - u, which takes it by
//    a row mirror: 8 for the 120 entries.
// With 46 and 15 evaluations, half of them idle, a pass took 1.53 ms at n =
// 5e5, m = 32 and 140 us at n = 1e5, m = 15 (matern); shared out, 1.38 ms and
// 129 us.  The vector units are then busy 80% of the time (m = 32: 4,414
// instructions for four sites, 33 of them table entries of 27 each).
template <int MM, bool MAT>
__device__ __forceinline__ void grp_build(GrpRows<MM> &S, const GrpCov &gc,
                                          const double *px, const double *py,
                                          int u, int cnt, double2 qa,
                                          double2 qb) {
  const double da = u < cnt ? gc.a.diag : 1.0;
  // entry (row r at q, column l), 0 where r is an identity row
  auto entry = [&](int r, double2 q, int l) {
    double v = 0.0;
    if (r < cnt) v = grp_corr<MAT>(sqdist(q.x, q.y, px[l], py[l]), gc);
    return v;
  };
  if constexpr (MM == 16) {
    const double2 qm = make_double2(px[15 - u], py[15 - u]);
    static_for<0, 7>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      const bool own = u > j;
      const double v = entry(own ? u : 15 - u, own ? qa : qm, own ? j : 14 - j);
      const double w = row_dpp<0x140>(v);  // row_mirror
      S.ra[j] = own ? v : (u == j ? da : 0.0);
      S.ra[14 - j] = u > 14 - j ? w : (u == 14 - j ? da : 0.0);
    });
    S.ra[7] = u == 7 ? da : 0.0;
    if (u > 7) S.ra[7] = entry(u, qa, 7);
    S.ra[15] = u == 15 ? da : 0.0;
  } else {
    const double db = 31 - u < cnt ? gc.a.diag : 1.0;
    static_for<0, 16>([&](auto lc) {
      constexpr int l = decltype(lc)::value;
      S.rb[l] = entry(31 - u, qb, l);
    });
    static_for<0, 15>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      const bool a = u > 14 - j;
      const double v =
          entry(a ? u : 31 - u, a ? qa : qb, a ? 14 - j : 16 + j);
      S.ra[14 - j] = a ? v : (u == 14 - j ? da : 0.0);
      S.rb[16 + j] = a ? (u == 15 - j ? db : 0.0) : v;
    });
    S.ra[15] = u == 15 ? da : 0.0;
    S.rb[31] = u == 0 ? db : 0.0;
  }
}

// Site i on the 16-lane row of lane u (valid: i < n), its inputs in `in`.
// The lane builds its rows of the site's system in registers from the
// neighbor coordinates the row stages in px/py (grp_build), then factor, forward and back substitution
// (nngp_group.hpp).  Meanwhile it fetches the inputs of the row's next site
// in2 (site i2, valid2).  Every lane of the row returns F and the residuals
// e; false when a pivot or F is not positive.
template <int MM, bool MAT>
__device__ inline bool grp_site(const BfArgs &A, const BfProblem &P,
                                const GrpCov &gc, double *px, double *py,
                                int i, bool valid, const GrpIn &in, int i2,
                                bool valid2, GrpIn &in2, int u, double &F,
                                double (&e)[kMaxNZ]) {
  constexpr int R = GrpRows<MM>::R;
  // opaque per site: the compares of u with every row number below would
  // otherwise be hoisted out of the caller's site loop as lane masks, more
  // than the SGPR file holds
  u = lane_opaque(u);
  const CovArgs &c = gc.a;
  const int cnt = in.cnt, off = in.off, ida = in.ida, idb = in.idb;
  const double2 qa = in.qa, qb = in.qb, s = in.s;
  const bool ina = u < cnt, inb = R == 2 && 31 - u < cnt;
  grp_in_lu(A, P, i2, valid2, in2);  // next site, stage 1
  px[u] = qa.x;
  py[u] = qa.y;
  if constexpr (R == 2) {
    px[31 - u] = qb.x;
    py[31 - u] = qb.y;
  }
  wave_sync();
  GrpRows<MM> S;
  grp_build<MM, MAT>(S, gc, px, py, u, cnt, qa, qb);
  const double ca =
      ina ? grp_corr<MAT>(sqdist(s.x, s.y, qa.x, qa.y), gc) : 0.0;
  const double cb =
      inb ? grp_corr<MAT>(sqdist(s.x, s.y, qb.x, qb.y), gc) : 0.0;
  wave_sync();  // the row's coordinates are read; the next site rewrites them
  grp_in_ids<R>(P, u, in2);  // next site, stage 2
  bool ok = grp_factor<MM>(S, u);
  grp_in_xy<R>(P, u, i2, valid2, in2);  // next site, stage 3
  double ya, yb, ba, bb;
  grp_forward<MM>(S, u, ca, cb, ya, yb);
  F = c.diag - row_sum16(ya * ya + yb * yb);
  grp_backward<MM>(S, u, ya, yb, ba, bb);
  ok = ok && F > 0.0;
  if (valid && A.B) {
    if (ina) A.B[off + u] = ba;
    if (inb) A.B[off + 31 - u] = bb;
  }
#pragma unroll
  for (int j = 0; j < kMaxNZ; j++) {
    e[j] = 0.0;
    if (j < A.nz) {
      double part = 0.0;
      if (ina) part = ba * P.Z[(size_t)ida * A.zs + j];
      if (inb) part = fma(bb, P.Z[(size_t)idb * A.zs + j], part);
      part = row_sum16(part);
      e[j] = valid ? P.Z[(size_t)i * A.zs + j] - part : 0.0;
    }
  }
  if (!ok) {
    F = 1.0;  // keeps the sums finite; the pass reports the failure
#pragma unroll
    for (int j = 0; j < kMaxNZ; j++) e[j] = 0.0;
  }
  return ok;
}

// Logical block b (xcd_block) takes groups of four consecutive sites from
// its XCD's run (xcd_site_run over the groups); each wave works on one
// group, row g of the wave on site 4 q + g.  Each row's running sums live
// in its own LDS slot (lane 0 of the row updates them); the block's row of
// partial sums adds the slots in a fixed order.  Single problem, FP64.
// MAT: the matern (c.cov == 2), by the pass's table.
template <int MM, bool MAT>
__global__ __launch_bounds__(64 * kCoopMaxWaves) void k_bf_grp(BfArgs A) {
  extern __shared__ double smem[];
  __shared__ double red[kGrpSlots][kStatsMax];
  __shared__ double2 tab[MAT ? kMpLen / 2 : 1];
  __shared__ CovArgs cl;  // for the out-of-line matern series
  const int nw = (int)blockDim.x >> 6;
  const int w = (int)threadIdx.x >> 6;
  const int t = (int)threadIdx.x & 63;
  const int g = t >> 4;
  const int u = t & 15;
  const int b = xcd_block(A.coop_blocks);
  if (b < 0) return;
  const BfProblem P = bf_problem<false>(A);
  const CovArgs c = A.c;
  if (MAT) {  // the pass's table
    if (threadIdx.x == 0) cl = c;
    const double2 *src = reinterpret_cast<const double2 *>(A.mtab);
    for (int k = (int)threadIdx.x; k < kMpLen / 2; k += (int)blockDim.x)
      tab[k] = src[k];
    __syncthreads();
  }
  const GrpCov gc{c, cl, reinterpret_cast<const double *>(tab),
                  *reinterpret_cast<const BesselTab *>(A.mtab + kMpLen)};
  double *px = smem + (size_t)w * grp_wave_doubles(MM) + (size_t)g * 2 * MM;
  double *py = px + MM;
  const int slot = 4 * w + g;
  const int nv = 2 + A.nz * (A.nz + 1) / 2;
  for (int k = u; k < nv; k += 16) red[slot][k] = 0.0;
  wave_sync();
  const SiteRun run = xcd_site_run(A.coop_blocks, b, (A.n + 3) >> 2, nw, w);
  GrpIn in;
  {  // the first site's inputs; later sites' arrive during their
     // predecessor's work
    const int i = 4 * run.first + g;
    const bool valid = run.first < run.end && i < A.n;
    grp_in_lu(A, P, i, valid, in);
    grp_in_ids<GrpRows<MM>::R>(P, u, in);
    grp_in_xy<GrpRows<MM>::R>(P, u, i, valid, in);
  }
  for (int q = run.first; q < run.end; q += run.stride) {
    const int i = 4 * q + g;
    const bool valid = i < A.n;
    const int q2 = q + run.stride, i2 = 4 * q2 + g;
    const bool valid2 = q2 < run.end && i2 < A.n;
    double F, e[kMaxNZ];
    GrpIn in2;
    const bool ok = grp_site<MM, MAT>(A, P, gc, px, py, i, valid, in, i2, valid2, in2, u, F, e);
    in = in2;
    if (valid && u == 0) {
      if (A.F) A.F[i] = F;
      if (!ok) atomicMin(P.err, i);
      const double rf = 1.0 / F;
      red[slot][0] += log(F);
      int gg = 2;
#pragma unroll
      for (int p = 0; p < kMaxNZ; p++) {
        if (p < A.nz) {
#pragma unroll
          for (int qq = 0; qq <= p; qq++)
            red[slot][gg + qq] += e[p] * e[qq] * rf;
        }
        gg += p + 1;
      }
    }
  }
  if (!P.rows) return;
  __syncthreads();
  const int k = (int)threadIdx.x;
  if (k < nv) {
    double sum = 0.0;
    if (k != 1)
      for (int sl = 0; sl < 4 * nw; sl++) sum += red[sl][k];
    P.rows[(size_t)k * A.rows_cap + b] = sum;
  }
}

int bf_row_launch(const BfArgs &a, const dim3 &grid, const dim3 &blk,
                  hipStream_t st) {
  const int waves = (int)blk.x / 64;
  const int mm = a.m <= 16 ? 16 : 32;
  const size_t shm = (size_t)waves * grp_wave_doubles(mm) * sizeof(double);
  const bool mat = a.c.cov == 2;
  if (mat) {
    if (!a.mtab) return -2;
    hipLaunchKernelGGL(k_matern_pieces, dim3(kMpOct), dim3(kMpThreads), 0, st,
                       a.c, a.mtab);
  }
  if (mm == 16) {
    if (mat) hipLaunchKernelGGL((k_bf_grp<16, true>), grid, blk, shm, st, a);
    else hipLaunchKernelGGL((k_bf_grp<16, false>), grid, blk, shm, st, a);
  } else {
    if (mat) hipLaunchKernelGGL((k_bf_grp<32, true>), grid, blk, shm, st, a);
    else hipLaunchKernelGGL((k_bf_grp<32, false>), grid, blk, shm, st, a);
  }
  return (int)hipGetLastError();
}

}  // namespace nngp
