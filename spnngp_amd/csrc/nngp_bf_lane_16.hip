// nngp_bf_lane_16.hip — the per-lane kernels for M = 16.
#include "nngp_bf_lane.hpp"

namespace nngp {

template void launch_lane_m<16, false>(const BfArgs &, int, const dim3 &,
                                     const dim3 &, hipStream_t);
template void launch_lane_lds_m<16, false>(const BfArgs &, int, const dim3 &,
                                         const dim3 &, hipStream_t);
template void launch_lane_m<16, true>(const BfArgs &, int, const dim3 &,
                                     const dim3 &, hipStream_t);
template void launch_lane_lds_m<16, true>(const BfArgs &, int, const dim3 &,
                                         const dim3 &, hipStream_t);

}  // namespace nngp
