// dsm_lane_inst.hip -- instantiates the lane form of the KMC kernels (dsm_lane.h).
#include "dsm_lane.h"

namespace dsm {

namespace {
template <int NQ>
hipError_t launch_nq(const KmcArgs& a, int grid, hipStream_t st) {
  hipLaunchKernelGGL((kmc_lane_kernel<NQ>), dim3(grid), dim3(64 * kLaneWaves),
                     sizeof(float) * lane_lds_floats(NQ, a.lanes | 1), st, a);
  return hipGetLastError();
}
}  // namespace

hipError_t launch_kmc_lane(const KmcArgs& a, int quads, int grid, hipStream_t st) {
  if (grid <= 0) return hipSuccess;
  switch (quads) {
    case 8: return launch_nq<8>(a, grid, st);
    case 12: return launch_nq<12>(a, grid, st);
    case 16: return launch_nq<16>(a, grid, st);
    case 19: return launch_nq<19>(a, grid, st);
    case 24: return launch_nq<24>(a, grid, st);
    case 28: return launch_nq<28>(a, grid, st);
    case 32: return launch_nq<32>(a, grid, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace dsm
