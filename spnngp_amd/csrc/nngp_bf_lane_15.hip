// nngp_bf_lane_15.hip — the per-lane kernels for M = 15.
#include "nngp_bf_lane.hpp"

namespace nngp {

template void launch_lane_m<15, false>(const BfArgs &, int, const dim3 &,
                                     const dim3 &, hipStream_t);
template void launch_lane_lds_m<15, false>(const BfArgs &, int, const dim3 &,
                                         const dim3 &, hipStream_t);
template void launch_lane_m<15, true>(const BfArgs &, int, const dim3 &,
                                     const dim3 &, hipStream_t);
template void launch_lane_lds_m<15, true>(const BfArgs &, int, const dim3 &,
                                         const dim3 &, hipStream_t);

}  // namespace nngp
