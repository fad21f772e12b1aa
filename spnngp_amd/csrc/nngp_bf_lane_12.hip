// nngp_bf_lane_12.hip — the per-lane kernels for M = 12.
#include "nngp_bf_lane.hpp"

namespace nngp {

template void launch_lane_m<12, false>(const BfArgs &, int, const dim3 &,
                                     const dim3 &, hipStream_t);
template void launch_lane_lds_m<12, false>(const BfArgs &, int, const dim3 &,
                                         const dim3 &, hipStream_t);
template void launch_lane_m<12, true>(const BfArgs &, int, const dim3 &,
                                     const dim3 &, hipStream_t);
template void launch_lane_lds_m<12, true>(const BfArgs &, int, const dim3 &,
                                         const dim3 &, hipStream_t);

}  // namespace nngp
