// Launch wrappers of the ROS2 kernels (CHEMISTRY=3, chem_spack_ros_dyndt.f90).
#include <hip/hip_runtime.h>

#include "rodas3_launch.h"
#ifdef BRAMS_MECH_COOP
#include "rodas3_coop.h"
#else
#include "rodas3_lane.h"
#endif

namespace brams {

hipError_t launch_ros2(unsigned nblocks, const StepParams& p, int block0, hipStream_t st, [[maybe_unused]] int form) {
  if (nblocks == 0) return hipSuccess;
#ifdef BRAMS_MECH_COOP
  return coop_launch<kRos2, false, false>(nblocks, p, block0, st);
#else
  if (block_form(nblocks, form) == kFormFourWaves)
    hipLaunchKernelGGL((ros2_blocks<64, kLaneManyWaves>), dim3(nblocks), dim3(64), 0, st, p, block0);
  else
    hipLaunchKernelGGL((ros2_blocks<64, 1>), dim3(nblocks), dim3(64), 0, st, p, block0);
  return hipGetLastError();
#endif
}

hipError_t launch_ros2_big(unsigned nblocks, const StepParams& p, int block0, hipStream_t st) {
  if (nblocks == 0) return hipSuccess;
#ifdef BRAMS_MECH_COOP
  hipLaunchKernelGGL((coop_blocks<kRos2, false, true>), dim3(nblocks), dim3(kCoopLanes), 0, st, p, block0);
#else
  hipLaunchKernelGGL((ros2_blocks<128, 1>), dim3(nblocks), dim3(128), 0, st, p, block0);
#endif
  return hipGetLastError();
}

}  // namespace brams
