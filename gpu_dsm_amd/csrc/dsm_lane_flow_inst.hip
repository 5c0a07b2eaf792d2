// dsm_lane_flow_inst.hip -- instantiates the lane form under flow (dsm_lane_flow.h).
#include "dsm_lane_flow.h"

namespace dsm {

namespace {
template <int P>
hipError_t launch_p(const KmcArgs& a, int grid, hipStream_t st) {
  hipLaunchKernelGGL((kmc_lane_flow_kernel<P>), dim3(grid), dim3(64 * kFlowWaves),
                     sizeof(float) * (kLaneTabFloats + kFlowWaves * flow_wave_floats(P, a.lanes | 1)), st, a);
  return hipGetLastError();
}
}  // namespace

hipError_t launch_kmc_lane_flow(const KmcArgs& a, int cap, int grid, hipStream_t st) {
  if (grid <= 0) return hipSuccess;
  if (a.lanes < 1 || a.lanes > flow_max_lanes(cap)) return hipErrorInvalidValue;
  switch (cap) {
    case 8: return launch_p<8>(a, grid, st);
    case 12: return launch_p<12>(a, grid, st);
    case 16: return launch_p<16>(a, grid, st);
    case 20: return launch_p<20>(a, grid, st);
    case 24: return launch_p<24>(a, grid, st);
    case 28: return launch_p<28>(a, grid, st);
    case 32: return launch_p<32>(a, grid, st);
    case 36: return launch_p<36>(a, grid, st);
    case 40: return launch_p<40>(a, grid, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace dsm
