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

// block 1 of p alone: its mask is recomputed on every attempt and published
hipError_t launch_rodas3_first(const StepParams& p, hipStream_t st);
// nblocks blocks of 65..127 cells from block0 on; p.half_y holds kHalfBytes each
hipError_t launch_rodas3_big(unsigned nblocks, const StepParams& p, int block0, hipStream_t st);
// nblocks blocks of at most 64 cells: from block0 on, or p.block_order's, or
// the consecutive 64-entry runs of p.cell_list
hipError_t launch_rodas3(unsigned nblocks, const StepParams& p, int block0, hipStream_t st);

// the same two for the ROS2 solver (no block-1 form)
hipError_t launch_ros2_big(unsigned nblocks, const StepParams& p, int block0, hipStream_t st);
hipError_t launch_ros2(unsigned nblocks, const StepParams& p, int block0, hipStream_t st);

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
