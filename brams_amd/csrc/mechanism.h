// The chemical mechanism of this build.  BRAMS compiles one mechanism in
// (its chem1_list and SPACK kernels, src/brams/ccatt/<MECH>/); so does this
// library: BRAMS_MECH_GEN names the generated device functions,
// BRAMS_MECH_COOP the block kernels' wave programs, BRAMS_MECH_QSSA the QSSA
// kernel's and BRAMS_MECH_SLAB the slab-layout variants, all from
// brams_amd/codegen/gen_mech.py.  RELACS_TUV by default.
#pragma once
#ifndef BRAMS_MECH_GEN
#define BRAMS_MECH_GEN "generated/relacs_tuv_gen.h"
#define BRAMS_MECH_SLAB "generated/relacs_tuv_slab.h"
#define BRAMS_MECH_COOP "generated/relacs_tuv_coop.h"
#define BRAMS_MECH_QSSA "generated/relacs_tuv_qssa.h"
#endif
#include BRAMS_MECH_GEN
