// Launch wrappers of the RODAS3 kernels of block 1 and of blocks of more than 64
// cells.
#include <hip/hip_runtime.h>

#include "rodas3_launch.h"
#ifdef BRAMS_MECH_COOP
#include "rodas3_coop.h"
#else
#include "rodas3_lane.h"
#endif

namespace brams {

hipError_t launch_rodas3_first(const StepParams& p, hipStream_t st) {
#ifdef BRAMS_MECH_COOP
  hipLaunchKernelGGL((coop_blocks<kRodas3, true, true>), dim3(1), dim3(kCoopLanes), 0, st, p, 0);
#else
  // a block 1 of at most 64 cells leaves the second wave idle
  hipLaunchKernelGGL((rodas3_blocks<128, true, 1>), dim3(1), dim3(128), 0, st, p, 0);
#endif
  return hipGetLastError();
}

hipError_t launch_rodas3_big(unsigned nblocks, const StepParams& p, int block0, hipStream_t st) {
  if (nblocks == 0) return hipSuccess;
#ifdef BRAMS_MECH_COOP
  hipLaunchKernelGGL((coop_blocks<kRodas3, false, true>), dim3(nblocks), dim3(kCoopLanes), 0, st, p, block0);
#else
  hipLaunchKernelGGL((rodas3_blocks<128, false, 1>), dim3(nblocks), dim3(128), 0, st, p, block0);
#endif
  return hipGetLastError();
}

}  // namespace brams
