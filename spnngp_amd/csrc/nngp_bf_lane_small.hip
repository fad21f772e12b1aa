// nngp_bf_lane_small.hip — the per-lane kernels for M = 4, 8, 10.
#include "nngp_bf_lane.hpp"

namespace nngp {

template void launch_lane_m<4, false>(const BfArgs &, int, const dim3 &,
                                     const dim3 &, hipStream_t);
template void launch_lane_m<4, true>(const BfArgs &, int, const dim3 &,
                                     const dim3 &, hipStream_t);
template void launch_lane_m<8, false>(const BfArgs &, int, const dim3 &,
                                     const dim3 &, hipStream_t);
template void launch_lane_m<8, true>(const BfArgs &, int, const dim3 &,
                                     const dim3 &, hipStream_t);
template void launch_lane_m<10, false>(const BfArgs &, int, const dim3 &,
                                     const dim3 &, hipStream_t);
template void launch_lane_lds_m<10, false>(const BfArgs &, int, const dim3 &,
                                         const dim3 &, hipStream_t);
template void launch_lane_m<10, true>(const BfArgs &, int, const dim3 &,
                                     const dim3 &, hipStream_t);
template void launch_lane_lds_m<10, true>(const BfArgs &, int, const dim3 &,
                                         const dim3 &, hipStream_t);

}  // namespace nngp
