// Launch wrappers of the RODAS3 kernel of blocks of at most 64 cells.
#include <hip/hip_runtime.h>

#include "rodas3_launch.h"
#ifdef BRAMS_MECH_COOP
#include "rodas3_coop.h"
#else
#include "rodas3_lane.h"
#endif

namespace brams {

hipError_t launch_rodas3(unsigned nblocks, const StepParams& p, int block0, hipStream_t st, [[maybe_unused]] int form) {
  if (nblocks == 0) return hipSuccess;
#ifdef BRAMS_MECH_COOP
  return coop_launch<kRodas3, false, false>(nblocks, p, block0, st);
#else
  if (p.cell_list) return hipErrorInvalidValue;
  if (block_form(nblocks, form) == kFormFourWaves)
    hipLaunchKernelGGL((rodas3_blocks<64, false, kLaneManyWaves>), dim3(nblocks), dim3(64), 0, st, p, block0);
  else
    hipLaunchKernelGGL((rodas3_blocks<64, false, 1>), dim3(nblocks), dim3(64), 0, st, p, block0);
  return hipGetLastError();
#endif
}

}  // namespace brams
