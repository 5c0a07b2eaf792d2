// dsm_solo_inst.hip -- instantiates the solo form of the KMC kernels (dsm_solo.h).
#include "dsm_solo_flow.h"

namespace dsm {

namespace {
size_t solo_lds(int cap) { return sizeof(float) * (kLaneTabFloats + 4 * (size_t)cap); }
}  // namespace

int kmc_solo_occupancy(int cap) {
  int n = 0;
  const hipError_t rc =
      cap > 256 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kmc_solo_kernel<true>, 64, solo_lds(cap))
                : hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kmc_solo_kernel<false>, 64, solo_lds(cap));
  if (rc != hipSuccess) return 1;
  return n < 1 ? 1 : n;
}

hipError_t launch_kmc_solo(const KmcArgs& a, int cap, int grid, hipStream_t st) {
  if (grid <= 0) return hipSuccess;
  if (cap <= 0 || (cap & 3)) return hipErrorInvalidValue;
  KmcArgs b = a;
  b.cap = cap;
  if (cap > 256) hipLaunchKernelGGL((kmc_solo_kernel<true>), dim3(grid), dim3(64), solo_lds(cap), st, b);
  else hipLaunchKernelGGL((kmc_solo_kernel<false>), dim3(grid), dim3(64), solo_lds(cap), st, b);
  return hipGetLastError();
}

int kmc_solo_flow_occupancy(int cap) {
  int n = 0;
  const size_t lds = sizeof(float) * kLaneTabFloats;
  const hipError_t rc = cap > 256 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kmc_solo_flow_kernel<2>, 64, lds)
                                  : hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kmc_solo_flow_kernel<1>, 64, lds);
  if (rc != hipSuccess) return 1;
  return n < 1 ? 1 : n;
}

hipError_t launch_kmc_solo_flow(const KmcArgs& a, int cap, int grid, hipStream_t st) {
  if (grid <= 0) return hipSuccess;
  const size_t lds = sizeof(float) * kLaneTabFloats;
  if (cap == 512) hipLaunchKernelGGL((kmc_solo_flow_kernel<2>), dim3(grid), dim3(64), lds, st, a);
  else if (cap == 256) hipLaunchKernelGGL((kmc_solo_flow_kernel<1>), dim3(grid), dim3(64), lds, st, a);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace dsm
