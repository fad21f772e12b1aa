// nngp_knn.hip — exact nearest-neighbor search on gfx950.
//
// mkNNIndxCB (src/nn.cpp:128-257) finds, for every site i, the m nearest
// sites among its NNGP predecessors (index < i), ascending by the squared
// distance fl(fl(dx*dx) + fl(dy*dy)), then stores sqrt of it; mkNNIndx
// (src/nn.cpp:63-111) does the same by a scan, comparing the Euclidean
// distances.  The reference walks a u = x + y sorted list; this search uses
// a strip index (points sorted by x, cut into strips, each strip sorted by
// y) and one query per wavefront, or per lane for long lists and many nn2
// queries.  Every pruning test compares a rounded partial
// square (dx^2 of the strip gap, or dy^2 inside a strip) with the current
// worst distance; since fl(dx^2) + fl(dy^2) rounds monotonically, nothing
// that could enter the list is ever skipped, so the result is the exact set
// of smallest distances in the reference's own arithmetic.  Products and
// sums here must not contract into FMAs (the reference rounds dx*dx, dy*dy
// and their sum separately), so contraction is switched off for this file.
//
// Ties.  Where no two of a site's m+1 smallest distances are equal, every
// correct search gives the same list.  Where some are, the reference's
// result depends on the order its walk meets the candidates and on its
// unstable shell sort, and near-equal squared distances can also swap
// through the rounding of the walk's pruning test (du)^2 > 2 * worst.  The
// strip search therefore keeps m+1 candidates and flags a site when two
// consecutive ones are closer than that rounding can reach (code book) or
// have equal Euclidean distances (scan); the flagged sites are compacted
// and redone by k_knn_replay in the reference's own candidate order
// (nngp_knn_replay.hpp).  Continuous coordinates almost never flag a site;
// lattices, rounded coordinates and duplicated sites flag most of them.
//
// nn2 (RANN) orders equal distances by ascending fitted row: the candidate
// key is the pair (squared distance, row).
#include <hipcub/hipcub.hpp>

#include <vector>

#include "nngp_host.hpp"
#include "nngp_knn_replay.hpp"
#include "nngp_strips.hpp"

#pragma clang fp contract(off)

namespace nngp {

constexpr int kKnnBlock = 256;

template <int M>
struct TopM {
  // Sorted ascending, right-aligned: slots [0, M - cnt) hold -inf and never
  // move, so d[M-1] is always the current cnt-th smallest distance.
  double d[M];
  int id[M];
  __device__ __forceinline__ void init(int cnt) {
#pragma unroll
    for (int k = 0; k < M; k++) {
      d[k] = k < M - cnt ? -__builtin_inf() : __builtin_inf();
      id[k] = -1;
    }
  }
  __device__ __forceinline__ double worst() const { return d[M - 1]; }
  __device__ __forceinline__ int worst_id() const { return id[M - 1]; }
  // (distance, id) pairs ordered lexicographically: equal distances by id
  __device__ __forceinline__ void insert_lex(double x, int ix) {
#pragma unroll
    for (int k = M - 1; k >= 1; k--) {
      const bool sh = d[k - 1] > x || (d[k - 1] == x && id[k - 1] > ix);
      const bool here = d[k] > x || (d[k] == x && id[k] > ix);
      const double nd = sh ? d[k - 1] : (here ? x : d[k]);
      const int ni = sh ? id[k - 1] : (here ? ix : id[k]);
      d[k] = nd;
      id[k] = ni;
    }
    if (d[0] > x || (d[0] == x && id[0] > ix)) {
      d[0] = x;
      id[0] = ix;
    }
  }
  __device__ __forceinline__ void insert(double x, int ix) {
#pragma unroll
    for (int k = M - 1; k >= 1; k--) {
      const bool sh = d[k - 1] > x;
      const bool here = d[k] > x;
      const double nd = sh ? d[k - 1] : (here ? x : d[k]);
      const int ni = sh ? id[k - 1] : (here ? ix : id[k]);
      d[k] = nd;
      id[k] = ni;
    }
    if (d[0] > x) {
      d[0] = x;
      id[0] = ix;
    }
  }
};

__device__ __forceinline__ int lower_bound_y(const double *y, int len,
                                             double v) {
  int lo = 0, hi = len;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (y[mid] < v)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

// Scan strip t; `self` >= 0 restricts candidates to ids < self.  LEX keys
// candidates by (squared distance, id), else by the distance alone with
// strict insertion.
template <int M, bool LEX>
__device__ inline void scan_strip(const StripIndex &S, int t, double qx,
                                  double qy, int self, TopM<M> &top) {
  const int base = t * S.S;
  const int len = min(S.S, S.n - base);
  const double *sy = S.sy + base;
  const double *sx = S.sx + base;
  const int *sid = S.sid + base;
  const int p = lower_bound_y(sy, len, qy);
  // candidate j: squared distance rounded as the reference rounds it,
  // (x0-c0)^2 + (x1-c1)^2 with each square and the sum rounded; returns
  // false once dy^2 alone exceeds the current worst distance
  auto visit = [&](int j) {
    const double dy = qy - sy[j];
    const double dy2 = dy * dy;
    if (dy2 > top.worst()) return false;
    const int id = sid[j];
    if (self < 0 || id < self) {
      const double dx = qx - sx[j];
      const double dx2 = dx * dx;
      const double d2 = dx2 + dy2;
      if (LEX) {
        if (d2 < top.worst() || (d2 == top.worst() && id < top.worst_id()))
          top.insert_lex(d2, id);
      } else if (d2 < top.worst()) {
        top.insert(d2, id);
      }
    }
    return true;
  };
  for (int j = p; j < len; j++)
    if (!visit(j)) break;
  for (int j = p - 1; j >= 0; j--)
    if (!visit(j)) break;
}

template <int M, bool LEX>
__device__ inline void search(const StripIndex &S, int t0, double qx,
                              double qy, int self, bool left_only,
                              TopM<M> &top) {
  scan_strip<M, LEX>(S, t0, qx, qy, self, top);
  for (int t = t0 - 1; t >= 0; t--) {
    const double gap = qx - S.xhi[t];
    if (gap > 0.0 && gap * gap > top.worst()) break;
    scan_strip<M, LEX>(S, t, qx, qy, self, top);
  }
  if (left_only) return;
  for (int t = t0 + 1; t < S.nstrip; t++) {
    const double gap = S.xlo[t] - qx;
    if (gap > 0.0 && gap * gap > top.worst()) break;
    scan_strip<M, LEX>(S, t, qx, qy, self, top);
  }
}

// src/util.cpp:55-70 layout
__device__ __forceinline__ void nn_layout(int i, int m, int &off, int &cnt) {
  if (i == 0) {
    off = 0;
    cnt = 0;
  } else if (i < m) {
    off = (int)((double)i / 2 * (i - 1));
    cnt = i;
  } else {
    off = (int)((double)m / 2 * (m - 1) + (double)(i - m) * m);
    cnt = m;
  }
}

// One lane per site.  M >= m + 1 holds the cs = min(i, m + 1) smallest
// squared distances among the site's predecessors; the first cnt are the
// site's list, and all cs decide whether the site is flagged for replay:
//   code book (mode 0): two consecutive squared distances within
//     g = 2^-40 d + 2 sqrt(2 d) E + E^2 (d the largest of them).  The
//     reference's walk drops a direction when fl(du)^2 > 2 * worst; fl(du)
//     carries up to E = 2^-48 max(|x| + |y|) of absolute rounding, so a
//     candidate can be dropped, or a tie decided, against the exact order
//     only when its squared distance is within g of another's;
//   scan (mode 1): two consecutive Euclidean distances equal.
template <int M>
__global__ __launch_bounds__(kKnnBlock) void k_knn_pred(KnnArgs A) {
  const int i = blockIdx.x * kKnnBlock + (int)threadIdx.x;
  if (i >= A.n) return;
  int off, cnt;
  nn_layout(i, A.m, off, cnt);
  A.lu[i] = off;
  A.lu[A.n + i] = cnt;
  if (cnt == 0) {
    A.flag[i] = 0;
    return;
  }
  const int cs = min(i, A.m + 1);
  const double2 q = A.xy[i];
  TopM<M> top;
  top.init(cs);
  search<M, false>(A.s, A.strip_of[i], q.x, q.y, i, A.sorted != 0, top);
  // slots below M - cs hold -inf: their differences are NaN or +inf and
  // their square roots NaN, so they never flag
  bool flag = false;
  if (A.mode == 0) {
    const double dmax = top.d[M - 1];
    const double g =
        ldexp(dmax, -40) + 2.0 * sqrt(2.0 * dmax) * A.E + A.E * A.E;
#pragma unroll
    for (int k = 0; k + 1 < M; k++) flag |= top.d[k + 1] - top.d[k] <= g;
  } else {
#pragma unroll
    for (int k = 0; k + 1 < M; k++)
      flag |= sqrt(top.d[k + 1]) == sqrt(top.d[k]);
  }
  A.flag[i] = flag ? 1 : 0;
#pragma unroll
  for (int k = 0; k < M; k++) {
    const int r = k - (M - cs);  // rank among the site's candidates
    if (r >= 0 && r < cnt) {
      A.nnIndx[off + r] = top.id[k];
      if (A.nnDist) A.nnDist[off + r] = sqrt(top.d[k]);
    }
  }
}

// The flagged sites again, one lane each, in the reference's own candidate
// order (nngp_knn_replay.hpp): MODE 0 the code-book walk, MODE 1 the scan.
// Each lane's list sits in LDS, lane-interleaved (entry k at k * 64 + lane).
constexpr int kReplayBlock = 64;

template <int M, int MODE>
__global__ __launch_bounds__(kReplayBlock) void k_knn_replay(
    KnnReplayArgs A) {
  __shared__ double ld[M * kReplayBlock];
  __shared__ int li[M * kReplayBlock];
  const int t = blockIdx.x * kReplayBlock + (int)threadIdx.x;
  if (t >= A.nflag) return;
  const int site = A.list[t];
  int off, cnt;
  nn_layout(site, A.m, off, cnt);
  double *d = ld + threadIdx.x;
  int *id = li + threadIdx.x;
  if (MODE == 0)
    cb_walk(cnt, A.n, A.ux, A.uy, A.usid, A.upos[site], d, id, kReplayBlock);
  else
    brute_scan(site, cnt, A.x, A.y, d, id, kReplayBlock);
  for (int k = 0; k < cnt; k++) {
    A.nnIndx[off + k] = id[k * kReplayBlock];
    if (A.nnDist) {
      const double v = d[k * kReplayBlock];
      A.nnDist[off + k] = MODE == 0 ? sqrt(v) : v;
    }
  }
}

__device__ __forceinline__ int locate_strip(const StripIndex &S, double x) {
  int lo = 0, hi = S.nstrip - 1;  // last strip with xlo <= x
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (S.xlo[mid] <= x)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

template <int M>
__global__ __launch_bounds__(kKnnBlock) void k_nn2(Nn2Args A) {
  const int i = blockIdx.x * kKnnBlock + (int)threadIdx.x;
  if (i >= A.nq) return;
  const double2 q = A.q[i];
  TopM<M> top;
  top.init(A.k);
  search<M, true>(A.s, locate_strip(A.s, q.x), q.x, q.y, -1, false, top);
#pragma unroll
  for (int k = 0; k < M; k++) {
    if (k >= M - A.k) {
      const size_t o = (size_t)(k - (M - A.k)) * A.nq + i;
      A.idx[o] = top.id[k];
      if (A.dist) A.dist[o] = sqrt(top.d[k]);
    }
  }
}

// nn2 with one query a wavefront, any k <= 64: lane l holds the l-th smallest
// (squared distance, row) so far.  A strip is scanned 64 candidates at a time
// outward from the query's y, and the survivors enter the list one by one (a
// compare and a lane shift each), so the result is k_nn2's.
struct WaveList {
  double d;
  int id;
};

__device__ __forceinline__ bool lex_less(double d, int id, double e, int ie) {
  return d < e || (d == e && id < ie);
}

__device__ __forceinline__ double lane_value(double x, int lane) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(x), lane);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(x), lane);
  return __hiloint2double(hi, lo);
}

// Entries of the ascending a[0 .. len) for which below(a[j]) holds (a prefix),
// 64 probes at a time.
template <class Below>
__device__ __forceinline__ int wave_prefix(const double *a, int len, int t,
                                           Below below) {
  int lo = 0, hi = len;  // the answer is in [lo, hi]
  while (lo < hi) {
    const int step = (hi - lo + 63) / 64;
    const int j = lo + t * step;
    const int c = __popcll(__ballot(j < hi && below(a[min(j, len - 1)])));
    if (c == 0) return lo;
    const int last = lo + (c - 1) * step;  // below
    hi = min(hi, last + step);
    lo = last + 1;
  }
  return lo;
}

__device__ __forceinline__ void wave_scan_strip(const StripIndex &S, int strip,
                                                double qx, double qy, int self,
                                                int k, int t, WaveList &L,
                                                double &worst, int &wid) {
  const int base = strip * S.S;
  const int len = min(S.S, S.n - base);
  const double *sy = S.sy + base;
  const double *sx = S.sx + base;
  const int *sid = S.sid + base;
  // the 64 candidates from j0 on; returns the lanes whose candidate, in range,
  // has dy^2 within the worst distance
  auto batch = [&](int j0) {
    const int j = j0 + t;
    const bool in = j >= 0 && j < len;
    const int jc = in ? j : 0;
    const double dy = qy - sy[jc];
    const double dx = qx - sx[jc];
    const int id = sid[jc];
    const double dy2 = dy * dy, dx2 = dx * dx;
    const double d2 = dx2 + dy2;
    unsigned long long left = __ballot(in && (self < 0 || id < self) &&
                                       lex_less(d2, id, worst, wid));
    while (left) {
      const int c = __ffsll((long long)left) - 1;
      left &= left - 1;
      const double x = lane_value(d2, c);
      const int ix = __builtin_amdgcn_readlane(id, c);
      if (!lex_less(x, ix, worst, wid)) continue;  // the list moved on
      const bool gt = lex_less(x, ix, L.d, L.id);  // entries behind x
      const double pd = __shfl_up(L.d, 1);
      const int pi = __shfl_up(L.id, 1);
      const bool pgt = t > 0 && lex_less(x, ix, pd, pi);
      L.d = gt ? (pgt ? pd : x) : L.d;
      L.id = gt ? (pgt ? pi : ix) : L.id;
      worst = lane_value(L.d, k - 1);
      wid = __builtin_amdgcn_readlane(L.id, k - 1);
    }
    return __ballot(in && !(dy2 > worst));
  };
  const int p = wave_prefix(sy, len, t, [&](double y) { return y < qy; });
  // the first batch reaches to both sides, so that the worst distance is
  // small before either side goes on
  const int a = max(0, min(p - 32, len - 64));
  const unsigned long long first = batch(a);
  // each side ends where the farthest of a batch is out of reach (or out of
  // range, in the side's last batch)
  unsigned long long up = first, down = first;
  for (int j = a + 64; j < len && up >> 63; j += 64) up = batch(j);
  for (int j = a - 64; j > -64 && (down & 1); j -= 64) down = batch(j);
}

// The k nearest of the query (candidates below `self` only, when self >= 0)
// outward from strip t0.
__device__ __forceinline__ WaveList wave_search(const StripIndex &S, int t0,
                                                double qx, double qy, int self,
                                                int k, bool left_only, int t) {
  WaveList L{__builtin_inf(), -1};  // as TopM: unfilled places read -1
  // The worst distance is wave-uniform and lives in scalar registers; as a
  // constant, its start would become one s_mov_b64 of a 64-bit literal, which
  // this compiler emits and the encoding (32 bits) cuts to 0.
  asm volatile("" : "+v"(L.d), "+v"(L.id));
  double worst = lane_value(L.d, k - 1);
  int wid = __builtin_amdgcn_readlane(L.id, k - 1);
  wave_scan_strip(S, t0, qx, qy, self, k, t, L, worst, wid);
  for (int s = t0 - 1; s >= 0; s--) {
    const double gap = qx - S.xhi[s];
    if (gap > 0.0 && gap * gap > worst) break;
    wave_scan_strip(S, s, qx, qy, self, k, t, L, worst, wid);
  }
  if (left_only) return L;
  for (int s = t0 + 1; s < S.nstrip; s++) {
    const double gap = S.xlo[s] - qx;
    if (gap > 0.0 && gap * gap > worst) break;
    wave_scan_strip(S, s, qx, qy, self, k, t, L, worst, wid);
  }
  return L;
}

// Queries of one launch, a wavefront each: a grid holds fewer than 2^32
// threads, so 2^26 queries and more do not fit one.
constexpr int kWaveQueries = 1 << 25;
constexpr int kWaveBlock = kKnnBlock / 64;  // queries a block

// launch(first, blocks) for each launch over n queries
template <class Launch>
static int wave_launches(int n, Launch launch) {
  for (long long first = 0; first < n; first += kWaveQueries) {
    const int left = (int)std::min<long long>(n - first, kWaveQueries);
    launch((int)first, dim3((left + kWaveBlock - 1) / kWaveBlock));
    if (const hipError_t e = hipGetLastError()) return (int)e;
  }
  return 0;
}

// The wavefront's query, of those from `first` on.
__device__ __forceinline__ int wave_query(int first) {
  return first + (int)blockIdx.x * kWaveBlock +
         __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
}

__global__ __launch_bounds__(kKnnBlock) void k_nn2_wave(Nn2Args A, int first) {
  const int i = wave_query(first);
  const int t = (int)threadIdx.x & 63;
  if (i >= A.nq) return;
  const double2 q = A.q[i];
  // the last strip with xlo <= x, else the first
  const int t0 = max(0, wave_prefix(A.s.xlo, A.s.nstrip, t,
                                    [&](double x) { return x <= q.x; }) - 1);
  const WaveList L = wave_search(A.s, t0, q.x, q.y, -1, A.k, false, t);
  if (t < A.k) {
    const size_t o = (size_t)t * A.nq + i;
    A.idx[o] = L.id;
    if (A.dist) A.dist[o] = sqrt(L.d);
  }
}

// k_knn_pred with one site a wavefront (m + 1 <= 64 candidates, one a lane).
// n = 1e6, m = 15: 9.6 ms with one lane a site, whose every accepted candidate
// moves a 16-entry list of all 64 lanes; now 3.4 ms.  n = 5e5 clustered, m =
// 32: 9.7 and 2.7 ms.
__global__ __launch_bounds__(kKnnBlock) void k_knn_pred_wave(KnnArgs A,
                                                            int first) {
  const int i = wave_query(first);
  const int t = (int)threadIdx.x & 63;
  if (i >= A.n) return;
  int off, cnt;
  nn_layout(i, A.m, off, cnt);
  if (t == 0) {
    A.lu[i] = off;
    A.lu[A.n + i] = cnt;
    if (cnt == 0) A.flag[i] = 0;
  }
  if (cnt == 0) return;
  const int cs = min(i, A.m + 1);
  const double2 q = A.xy[i];
  const WaveList L = wave_search(A.s, A.strip_of[i], q.x, q.y, i, cs,
                                 A.sorted != 0, t);
  // k_knn_pred's rule for the replay, on lanes t and t + 1 < cs
  const double d = A.mode == 0 ? L.d : sqrt(L.d);
  const double nd = __shfl_down(d, 1);
  bool tie;
  if (A.mode == 0) {
    const double dmax = lane_value(L.d, cs - 1);
    const double g =
        ldexp(dmax, -40) + 2.0 * sqrt(2.0 * dmax) * A.E + A.E * A.E;
    tie = nd - d <= g;
  } else {
    tie = nd == d;
  }
  const bool flag = __ballot(t + 1 < cs && tie) != 0;
  if (t == 0) A.flag[i] = flag ? 1 : 0;
  if (t < cnt) {
    A.nnIndx[off + t] = L.id;
    if (A.nnDist) A.nnDist[off + t] = sqrt(L.d);
  }
}

int knn_launch(const KnnArgs &a, hipStream_t st) {
  const dim3 block(kKnnBlock);
  if (a.m < 64)
    return wave_launches(a.n, [&](int first, dim3 grid) {
      hipLaunchKernelGGL(k_knn_pred_wave, grid, block, 0, st, a, first);
    });
  if (a.m < 65)  // 65 candidates: one site a lane
    hipLaunchKernelGGL(k_knn_pred<65>, dim3((a.n + kKnnBlock - 1) / kKnnBlock),
                       block, 0, st, a);
  else
    return -1;
  return (int)hipGetLastError();
}

int knn_replay_launch(const KnnReplayArgs &a, hipStream_t st) {
  if (a.nflag <= 0) return 0;
  const dim3 grid((a.nflag + kReplayBlock - 1) / kReplayBlock),
      block(kReplayBlock);
  if (a.m <= 16) {
    if (a.mode == 0)
      hipLaunchKernelGGL((k_knn_replay<16, 0>), grid, block, 0, st, a);
    else
      hipLaunchKernelGGL((k_knn_replay<16, 1>), grid, block, 0, st, a);
  } else if (a.m <= 32) {
    if (a.mode == 0)
      hipLaunchKernelGGL((k_knn_replay<32, 0>), grid, block, 0, st, a);
    else
      hipLaunchKernelGGL((k_knn_replay<32, 1>), grid, block, 0, st, a);
  } else if (a.m <= 64) {
    if (a.mode == 0)
      hipLaunchKernelGGL((k_knn_replay<64, 0>), grid, block, 0, st, a);
    else
      hipLaunchKernelGGL((k_knn_replay<64, 1>), grid, block, 0, st, a);
  } else {
    return -1;
  }
  return (int)hipGetLastError();
}

// Compacts the sites with flag[i] != 0 into list[0 .. *count), ascending.
int knn_flagged(const unsigned char *flag, int n, int *list, int *count,
                DevBuf &tmp, hipStream_t st) {
  hipcub::CountingInputIterator<int> ids(0);
  size_t bytes = 0;
  NNGP_HIP(hipcub::DeviceSelect::Flagged(nullptr, bytes, ids, flag, list,
                                         count, n, st));
  NNGP_TRY(tmp.alloc(bytes));
  NNGP_HIP(hipcub::DeviceSelect::Flagged(tmp.p, bytes, ids, flag, list, count,
                                         n, st));
  return NNGP_OK;
}

// ---------------------------------------------------------------------------
// strip index
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kKnnBlock) void k_iota(int *p, int n) {
  const int i = blockIdx.x * kKnnBlock + (int)threadIdx.x;
  if (i < n) p[i] = i;
}

// The strip of the point at each rank of the x order (ord: nullptr when the
// points come x-ordered) and the x range of each strip.
__global__ __launch_bounds__(kKnnBlock) void k_strip_of(
    const int *ord, const double *x, int n, int S, int *strip_of, double *xlo,
    double *xhi) {
  const int r = blockIdx.x * kKnnBlock + (int)threadIdx.x;
  if (r >= n) return;
  const int id = ord ? ord[r] : r, t = r / S;
  strip_of[id] = t;
  if (r == t * S) xlo[t] = x[id];
  if (r == t * S + S - 1 || r == n - 1) xhi[t] = x[id];
}

__global__ __launch_bounds__(kKnnBlock) void k_gather_strip(
    const int *ids, const int *strip_of, int n, int *out) {
  const int k = blockIdx.x * kKnnBlock + (int)threadIdx.x;
  if (k < n) out[k] = strip_of[ids[k]];
}

__global__ __launch_bounds__(kKnnBlock) void k_gather_xy(
    const int *ids, const double *x, const double *y, int n, double *sx,
    double *sy) {
  const int k = blockIdx.x * kKnnBlock + (int)threadIdx.x;
  if (k >= n) return;
  const int id = ids[k];
  sx[k] = x[id];
  sy[k] = y[id];
}

// Of few points each finds its place by counting the points before it: two
// launches and one allocation for the sorts' ten and two.  A whole search of 20
// sites takes 194 us (227 with the sorts, 222 with the strips sorted on the
// host), nn2 of one query among 2,000 sites, k = 1, 179 us (250, 190), among
// 8,000 227 us (278, 420); at 12,000 the sorts are as fast.  The keys order all
// bit patterns, so that the places are a permutation whatever the coordinates.
constexpr int kCountPoints = 8192;

__device__ __forceinline__ unsigned long long order_key(double x) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(x);
  return b >> 63 ? ~b : b | (1ull << 63);
}

// Points of v[0 .. n) before point i in the order (value, index) for which
// in(j) holds; 64 at a time by the wavefront.
template <class In>
__device__ __forceinline__ int count_before(const double *__restrict__ v, int n,
                                            int i, In in) {
  const unsigned long long ki = order_key(v[i]);
  int r = 0;
  for (int j0 = 0; j0 < n; j0 += 64) {
    const int j = j0 + ((int)threadIdx.x & 63);
    const int jc = min(j, n - 1);
    const unsigned long long kj = order_key(v[jc]);
    r += __popcll(__ballot(j < n && in(jc) &&
                           (kj < ki || (kj == ki && j < i))));
  }
  return r;
}

// One wavefront a point.  Strip of point i, by its rank in x (i itself when the
// points come x-ordered), and the x range of each strip.
__global__ __launch_bounds__(kKnnBlock) void k_count_x(
    const double *__restrict__ x, int n, int S, int sorted, int *strip_of,
    double *xlo, double *xhi) {
  const int i = wave_query(0);
  if (i >= n) return;
  const int r = sorted ? i : count_before(x, n, i, [](int) { return true; });
  if ((threadIdx.x & 63) != 0) return;
  const double xi = x[i];
  const int t = r / S;
  strip_of[i] = t;
  if (r == t * S) xlo[t] = xi;
  if (r == t * S + S - 1 || r == n - 1) xhi[t] = xi;
}

// One wavefront a point: to its place in its strip, by its rank in y among the
// strip's points.
__global__ __launch_bounds__(kKnnBlock) void k_count_y(
    const double *__restrict__ x, const double *__restrict__ y,
    const int *__restrict__ strip_of, int n, int S, double *sx, double *sy,
    int *sid) {
  const int i = wave_query(0);
  if (i >= n) return;
  const int t = strip_of[i];
  const int p =
      t * S + count_before(y, n, i, [&](int j) { return strip_of[j] == t; });
  if ((threadIdx.x & 63) != 0) return;
  sx[p] = x[i];
  sy[p] = y[i];
  sid[p] = i;
}

int DevStrips::build(const double *coords, int n, int m, hipStream_t st) {
  const int S = strip_size(n, m), nstrip = (n + S - 1) / S;
  sorted = true;
  for (int i = 1; i < n; i++)
    if (coords[i] < coords[i - 1]) {
      sorted = false;
      break;
    }
  auto carve = [](size_t &at, size_t bytes) {
    const size_t o = at;
    at += (bytes + 255) / 256 * 256;
    return o;
  };
  const size_t nd = sizeof(double) * (size_t)n, ni = sizeof(int) * (size_t)n;
  const bool few = n <= kCountPoints;
  size_t keep = 0, work = 0;
  const size_t o_sx = carve(keep, nd), o_sy = carve(keep, nd),
               o_id = carve(keep, ni), o_of = carve(keep, ni),
               o_lo = carve(keep, sizeof(double) * nstrip),
               o_hi = carve(keep, sizeof(double) * nstrip);
  const size_t o_xy = few ? carve(keep, 2 * nd) : 0;
  NNGP_TRY(mem.alloc(keep));
  char *kp = mem.as<char>();
  double *sx = reinterpret_cast<double *>(kp + o_sx);
  double *sy = reinterpret_cast<double *>(kp + o_sy);
  int *sid = reinterpret_cast<int *>(kp + o_id);
  int *of = reinterpret_cast<int *>(kp + o_of);
  double *xlo = reinterpret_cast<double *>(kp + o_lo);
  double *xhi = reinterpret_cast<double *>(kp + o_hi);
  strip_of = of;
  idx.n = n;
  idx.S = S;
  idx.nstrip = nstrip;
  idx.sx = sx;
  idx.sy = sy;
  idx.sid = sid;
  idx.xlo = xlo;
  idx.xhi = xhi;
  const dim3 grid((n + kKnnBlock - 1) / kKnnBlock), block(kKnnBlock);
  if (few) {
    double *x = reinterpret_cast<double *>(kp + o_xy), *y = x + n;
    const dim3 waves((n + kWaveBlock - 1) / kWaveBlock);
    NNGP_HIP(hipMemcpyAsync(x, coords, 2 * nd, hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(k_count_x, waves, block, 0, st, (const double *)x, n, S,
                       sorted ? 1 : 0, of, xlo, xhi);
    hipLaunchKernelGGL(k_count_y, waves, block, 0, st, (const double *)x,
                       (const double *)y, (const int *)of, n, S, sx, sy, sid);
    NNGP_HIP(hipGetLastError());
    NNGP_HIP(hipStreamSynchronize(st));  // other streams may use the index
    return NNGP_OK;
  }
  // sizes of the sorts' workspaces
  hipcub::DoubleBuffer<double> kd(nullptr, nullptr);
  hipcub::DoubleBuffer<int> ki(nullptr, nullptr), vi(nullptr, nullptr);
  int bits = 1;
  while (bits < 31 && (1 << bits) < nstrip) bits++;
  size_t wd = 0, wi = 0;
  NNGP_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, wd, kd, vi, n, 0, 64, st));
  NNGP_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, wi, ki, vi, n, 0, bits, st));
  const size_t w_xy = carve(work, 2 * nd), w_k0 = carve(work, nd),
               w_k1 = carve(work, nd), w_v0 = carve(work, ni),
               w_v1 = carve(work, ni), w_tmp = carve(work, std::max(wd, wi));
  DevBuf scratch;
  NNGP_TRY(scratch.alloc(work));
  char *wp = scratch.as<char>();
  double *x = reinterpret_cast<double *>(wp + w_xy), *y = x + n;
  double *k0 = reinterpret_cast<double *>(wp + w_k0);
  double *k1 = reinterpret_cast<double *>(wp + w_k1);
  int *v0 = reinterpret_cast<int *>(wp + w_v0);
  int *v1 = reinterpret_cast<int *>(wp + w_v1);
  NNGP_HIP(hipMemcpyAsync(x, coords, 2 * nd, hipMemcpyHostToDevice, st));
  // ids by ascending key (one coordinate), ties by id
  auto by_coordinate = [&](const double *c, const int *&ids) -> int {
    hipLaunchKernelGGL(k_iota, grid, block, 0, st, v0, n);
    NNGP_HIP(hipMemcpyAsync(k0, c, nd, hipMemcpyDeviceToDevice, st));
    hipcub::DoubleBuffer<double> k(k0, k1);
    hipcub::DoubleBuffer<int> v(v0, v1);
    size_t b = wd;
    NNGP_HIP(hipcub::DeviceRadixSort::SortPairs(wp + w_tmp, b, k, v, n, 0, 64, st));
    ids = v.Current();
    return NNGP_OK;
  };
  const int *ids = nullptr;
  if (!sorted) NNGP_TRY(by_coordinate(x, ids));
  hipLaunchKernelGGL(k_strip_of, grid, block, 0, st, ids, (const double *)x, n,
                     S, of, xlo, xhi);
  // y order, then stably by strip
  NNGP_TRY(by_coordinate(y, ids));
  int *s0 = reinterpret_cast<int *>(k0), *s1 = reinterpret_cast<int *>(k1);
  hipLaunchKernelGGL(k_gather_strip, grid, block, 0, st, ids, (const int *)of,
                     n, s0);
  {
    int *cur = const_cast<int *>(ids), *alt = cur == v0 ? v1 : v0;
    hipcub::DoubleBuffer<int> k(s0, s1), v(cur, alt);
    size_t b = wi;
    NNGP_HIP(hipcub::DeviceRadixSort::SortPairs(wp + w_tmp, b, k, v, n, 0, bits, st));
    NNGP_HIP(hipMemcpyAsync(sid, v.Current(), ni, hipMemcpyDeviceToDevice, st));
  }
  hipLaunchKernelGGL(k_gather_xy, grid, block, 0, st, (const int *)sid,
                     (const double *)x, (const double *)y, n, sx, sy);
  NNGP_HIP(hipGetLastError());
  NNGP_HIP(hipStreamSynchronize(st));  // the scratch goes away
  return NNGP_OK;
}

int knn_build(const double *coords, int n, int m, int mode,
              const DevStrips &ds, const double2 *xy,
              int *nnIndx, double *nnDist, int *lu, hipStream_t st,
              int *nflag_out) {
  DevBuf dFlag, dList, dCount, tmp;
  NNGP_TRY(dFlag.alloc((size_t)n));
  NNGP_TRY(dList.alloc(sizeof(int) * (size_t)n));
  NNGP_TRY(dCount.alloc(sizeof(int)));
  double umax = 0.0;
  for (int i = 0; i < n; i++)
    umax = std::max(umax, std::fabs(coords[i]) + std::fabs(coords[n + i]));
  KnnArgs a;
  a.s = ds.idx;
  a.xy = xy;
  a.strip_of = ds.strip_of;
  a.n = n;
  a.m = m;
  a.sorted = ds.sorted ? 1 : 0;
  a.nnIndx = nnIndx;
  a.nnDist = nnDist;
  a.lu = lu;
  a.mode = mode;
  a.E = std::ldexp(umax, -48);
  a.flag = dFlag.as<unsigned char>();
  if (knn_launch(a, st)) return set_err(NNGP_ERR_HIP, "kNN launch failed");
  NNGP_TRY(knn_flagged(a.flag, n, dList.as<int>(), dCount.as<int>(), tmp, st));
  int nflag = 0;
  NNGP_HIP(hipMemcpyAsync(&nflag, dCount.p, sizeof(int), hipMemcpyDeviceToHost,
                          st));
  NNGP_HIP(hipStreamSynchronize(st));
  if (nflag_out) *nflag_out = nflag;
  if (nflag == 0) return NNGP_OK;
  KnnReplayArgs r{};
  r.n = n;
  r.m = m;
  r.mode = mode;
  r.nflag = nflag;
  r.list = dList.as<int>();
  r.nnIndx = nnIndx;
  r.nnDist = nnDist;
  DevBuf dux, duy, dus, dup, dc;
  std::vector<double> ux, uy;
  std::vector<int> us, up;
  if (mode == 0) {
    // R's u = x + y order: the permutation rsort_with_index gives
    // (src/nn.cpp:238-243), ties in u included
    std::vector<double> u(n);
    us.resize(n);
    for (int i = 0; i < n; i++) {
      us[i] = i;
      u[i] = coords[i] + coords[n + i];
    }
    r_rsort_with_index(u.data(), us.data(), n, 1);
    ux.resize(n);
    uy.resize(n);
    up.resize(n);
    for (int k = 0; k < n; k++) {
      ux[k] = coords[us[k]];
      uy[k] = coords[n + us[k]];
      up[us[k]] = k;
    }
    NNGP_TRY(dux.alloc(sizeof(double) * (size_t)n));
    NNGP_TRY(duy.alloc(sizeof(double) * (size_t)n));
    NNGP_TRY(dus.alloc(sizeof(int) * (size_t)n));
    NNGP_TRY(dup.alloc(sizeof(int) * (size_t)n));
    NNGP_HIP(hipMemcpyAsync(dux.p, ux.data(), dux.bytes, hipMemcpyHostToDevice,
                            st));
    NNGP_HIP(hipMemcpyAsync(duy.p, uy.data(), duy.bytes, hipMemcpyHostToDevice,
                            st));
    NNGP_HIP(hipMemcpyAsync(dus.p, us.data(), dus.bytes, hipMemcpyHostToDevice,
                            st));
    NNGP_HIP(hipMemcpyAsync(dup.p, up.data(), dup.bytes, hipMemcpyHostToDevice,
                            st));
    r.ux = dux.as<double>();
    r.uy = duy.as<double>();
    r.usid = dus.as<int>();
    r.upos = dup.as<int>();
  } else {
    NNGP_TRY(dc.alloc(sizeof(double) * 2 * (size_t)n));
    NNGP_HIP(hipMemcpyAsync(dc.p, coords, dc.bytes, hipMemcpyHostToDevice, st));
    r.x = dc.as<double>();
    r.y = dc.as<double>() + n;
  }
  if (knn_replay_launch(r, st))
    return set_err(NNGP_ERR_HIP, "kNN replay launch failed");
  // the staging vectors and buffers above must outlive the stream's work
  NNGP_HIP(hipStreamSynchronize(st));
  return NNGP_OK;
}

// Queries up to which nn2 gives each a wavefront when k <= 16.  That takes 17 us
// and 3.1 us a thousand queries whatever k; one query a lane takes about 30 + 13
// k us whatever their number (n = 2e3, 1e5 and 1e6: k = 1 42 to 64 us, k = 5 92
// to 144, k = 10 141 to 192, k = 15 217 to 254).  For k > 16 the lanes' 32- and
// 64-entry lists took 2 to 6 ms, against 7 us a thousand.
static int nn2_wave_queries(int k) { return std::min(4096 * (k + 1), 49152); }

int nn2_launch(const Nn2Args &a, hipStream_t st) {
  if (a.nq <= 0) return 0;
  if (a.k > 64) return -1;
  const dim3 block(kKnnBlock);
  if (a.k > 16 || a.nq <= nn2_wave_queries(a.k))
    return wave_launches(a.nq, [&](int first, dim3 grid) {
      hipLaunchKernelGGL(k_nn2_wave, grid, block, 0, st, a, first);
    });
  hipLaunchKernelGGL(k_nn2<16>, dim3((a.nq + kKnnBlock - 1) / kKnnBlock), block,
                     0, st, a);
  return (int)hipGetLastError();
}

}  // namespace nngp
