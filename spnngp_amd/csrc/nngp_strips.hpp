// nngp_strips.hpp — the strip index used by the neighbor searches
// (mkNNIndx(CB) and nn2): points sorted by x, cut into strips of S
// consecutive points, each strip sorted by y.
#pragma once
#include <algorithm>
#include <cmath>

#include "nngp_host.hpp"

namespace nngp {

// Strip length: the power of two >= sqrt(n m), so a query scans O(sqrt(n m))
// candidates in its own strip and about as many in each neighbor strip.
inline int strip_size(int n, int m) {
  double s = std::sqrt((double)n * (double)std::max(m, 1));
  int S = 64;
  while (S < s && S < (1 << 20)) S <<= 1;
  return std::min(S, std::max(n, 1));
}

// x ascending (ties by id), strips of S, y ascending inside (ties by id).
struct DevStrips {
  DevBuf mem;                     // every array below, one allocation
  const int *strip_of = nullptr;  // strip holding each point
  bool sorted = false;            // the points come x-ordered
  StripIndex idx;
  // From n points (host, column-major), sorted on the device by stable radix
  // sorts; returns after the stream has finished.  Sorting the strips on the
  // host took 55 of the 84 ms of a search over 1e6 sites.
  int build(const double *coords, int n, int m, hipStream_t st);
};

// Compacts the sites with flag[i] != 0 into list[0 .. *count) (device),
// ascending; tmp receives the scan's workspace.
int knn_flagged(const unsigned char *flag, int n, int *list, int *count,
                DevBuf &tmp, hipStream_t st);

// Neighbor lists of n sites (coords: column-major host copy; xy: the same
// on the device, interleaved) into device buffers in the reference layout:
// mode 0 the code-book search (src/nn.cpp:214-257), 1 the scan
// (src/nn.cpp:63-111).  The strip search flags the sites whose tied
// distances need the reference's own candidate order, and those are redone
// in that order.  nnDist may be nullptr; *nflag_out (optional) receives the
// number of redone sites.  Returns after the device work has finished.
int knn_build(const double *coords, int n, int m, int mode,
              const DevStrips &ds, const double2 *xy,
              int *nnIndx, double *nnDist, int *lu, hipStream_t st,
              int *nflag_out);

// Column-major n x 2 coordinates (host) to interleaved double2 (device).
inline int upload_xy(const double *cm, int n, DevBuf &xy, hipStream_t st) {
  DevBuf tmp;
  NNGP_TRY(tmp.alloc(sizeof(double) * 2 * (size_t)n));
  NNGP_HIP(hipMemcpyAsync(tmp.p, cm, tmp.bytes, hipMemcpyHostToDevice, st));
  NNGP_TRY(xy.alloc(sizeof(double2) * (size_t)n));
  if (interleave_launch(tmp.as<double>(), n, xy.as<double2>(), st))
    return set_err(NNGP_ERR_HIP, "coordinate upload kernel failed");
  NNGP_HIP(hipStreamSynchronize(st));
  return NNGP_OK;
}

}  // namespace nngp
