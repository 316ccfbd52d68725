// Launch wrapper of the multi-grid RODAS3 kernels (coop_grids in rodas3_coop.h):
// the nested grids of one model step in one launch per kind of block.
#include <hip/hip_runtime.h>

#include "rodas3_launch.h"
#ifndef BRAMS_MECH_LEAN
#include "rodas3_coop.h"
#endif

namespace brams {

hipError_t launch_rodas3_grids(bool first, bool big, unsigned nwork, const StepParams* grids, const int* work,
                               hipStream_t st) {
  if (nwork == 0) return hipSuccess;
  if (!grids || !work) return hipErrorInvalidValue;
#ifdef BRAMS_MECH_LEAN
  // a lean library (rodas3_launch.h) builds no coop_grids kernel
  (void)first, (void)big, (void)st;
  return hipErrorInvalidValue;
#else
  if (first) return coop_launch_grids<true, true>(nwork, grids, work, st);
  if (big) return coop_launch_grids<false, true>(nwork, grids, work, st);
  return coop_launch_grids<false, false>(nwork, grids, work, st);
#endif
}

}  // namespace brams
