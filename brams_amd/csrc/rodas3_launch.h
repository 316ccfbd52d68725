// Host entry of the RODAS3, ROS2 and QSSA kernels (rodas3_launch.hip,
// rodas3_grids.hip, ros2_launch.hip, qssa_launch.hip, split so the units
// compile in parallel).
#pragma once
#include <hip/hip_runtime.h>

#include "mechanism.h"

namespace brams {

struct StepParams;

// A library built with BRAMS_MECH_LEAN (the mechanisms other than RELACS_TUV)
// holds no several-grid kernels (rodas3_grids.hip; the entry launches grid by
// grid instead).
#ifdef BRAMS_MECH_LEAN
constexpr bool kLeanBuild = true;
#else
constexpr bool kLeanBuild = false;
#endif

// waves of a block's workgroup per SIMD, and the memory (StepParams.half_y)
// that one block of more than 64 cells takes
// (a mechanism without BRAMS_MECH_COOP runs one lane to a cell, rodas3_lane.h)
constexpr int kCoopWavesPerSimd = 2;
#ifdef BRAMS_MECH_COOP
constexpr size_t kHalfBytes = sizeof(double) * 4 * MECH_NS * 64;
#else
constexpr size_t kHalfBytes = 0;
#endif

// Kernel forms of the blocks of at most 64 cells, by the numbers that callers
// know (brams_chem_set_form).  0..2 were layouts that never ran, 3..5 register
// budgets of the one-lane-per-cell kernel (1, 2 and 4 waves per SIMD).  The
// cooperative kernel has one form, so there all of 3..5 run it.  A library
// without it holds 3 and 5.
constexpr int kFirstForm = 3;
constexpr int kFormFourWaves = 5;
constexpr int kForms = 6;
constexpr bool form_built(int f) { return f >= kFirstForm && f < kForms && (!kLeanBuild || f != kFirstForm + 1); }
#ifdef BRAMS_MECH_COOP
constexpr bool kOneForm = true;
#else
constexpr bool kOneForm = false;
// From this many blocks on, the one-lane-per-cell kernel takes the budget of
// four waves per SIMD: up to 1024 blocks run at once with one wave per SIMD
// and all of them sooner, then the waves that hide each other's spill traffic
// count.  Where the two meet depends on how alike the blocks' costs are.
// RACM_TUV, ms at one / four waves per SIMD (reference tolerances), a RODAS3
// step from an unbalanced state, where they are alike, and the third step, where
// a few long blocks decide:
//   blocks   2048      3072      4096      8192      12288     25000
//   first    212/218   285/268   345/295   585/434   910/588   1667/1029
//   third    109/143   134/178   132/163   198/229   251/277   427/390
// ROS2's steps meet at 2048 and between 6144 and 8192.  The line lies between.
constexpr unsigned kLaneManyBlocks = 4096;
#endif
// the form that nblocks blocks take: `forced` unless negative, else by their number
constexpr int block_form([[maybe_unused]] unsigned nblocks, int forced) {
#ifdef BRAMS_MECH_COOP
  return forced >= 0 ? forced : kFirstForm;
#else
  return forced >= 0 ? forced : nblocks >= kLaneManyBlocks ? kFormFourWaves : kFirstForm;
#endif
}

// block 1 of p alone: its mask is recomputed on every attempt and published
hipError_t launch_rodas3_first(const StepParams& p, hipStream_t st);
// nblocks blocks of 65..127 cells from block0 on; p.half_y holds kHalfBytes each
hipError_t launch_rodas3_big(unsigned nblocks, const StepParams& p, int block0, hipStream_t st);
// nblocks blocks of at most 64 cells: from block0 on, or p.block_order's, or
// the consecutive 64-entry runs of p.cell_list; form: block_form()'s `forced`
hipError_t launch_rodas3(unsigned nblocks, const StepParams& p, int block0, hipStream_t st, int form = -1);

// the same two for the ROS2 solver (no block-1 form)
hipError_t launch_ros2_big(unsigned nblocks, const StepParams& p, int block0, hipStream_t st);
hipError_t launch_ros2(unsigned nblocks, const StepParams& p, int block0, hipStream_t st, int form = -1);

// The QSSA solver (qssa_launch.hip): one lane per interior cell, itchim
// sub-steps; nfatal (device int, zeroed by the caller) counts the cells where
// a species reached 1e20.
hipError_t launch_qssa(const StepParams& p, int itchim, long long ncell, int* nfatal, hipStream_t st);

// Several grids in one launch (coop_grids): nwork workgroups, workgroup w on
// block work[w] & kGridBlockMask of grid work[w] >> kGridShift, whose
// parameters are grids[] (device memory).  first: block 1 of each grid; big:
// blocks of more than 64 cells (and block 1).
hipError_t launch_rodas3_grids(bool first, bool big, unsigned nwork, const StepParams* grids, const int* work,
                               hipStream_t st);

}  // namespace brams
