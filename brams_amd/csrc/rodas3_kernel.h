// Parameters of the Rosenbrock block kernels (rodas3_coop.h) and of the other
// kernels that gather cells from the caller's Fortran arrays.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mechanism.h"

namespace brams {

struct StepParams {
  int m1, m2, m3, ia, iz, ja, jz;
  int nk, ni;                    // interior levels (m1-2) and columns in i
  float dtlt;
  int ndyn, split;
  float cp, cpor, p00;
  const float *pp, *pi0, *theta, *rv;
  const double* jphoto;          // (17, m1, m2, m3)
  const float* weight;           // [47]
  const int* transported;        // [47] 1/0
  float* sc_p;                   // [47][n3d]
  float* sc_t;                   // [47][n3d] or null
  const float* sc_t_dyn;         // [47][n3d] or null
  long long n3d;
  const int* block_start;        // [nob+1]
  double* last_dt;               // [nob]
  const double *atol, *rtol;     // [47]
  unsigned* mask;                // [MECH_MASK_WORDS]: block-1 mask, read by later blocks
  int* blk_attempts;             // [nob]
  int* blk_substeps;             // [nob]
  int* blk_failed;               // [nob]
  float* blk_forced;             // [nob] largest error of an acceptance forced at dt_min (0: none)
  int* blk_thresh;               // [nob] or null: pivots failing Sparse1.3's threshold rule, summed
                                 // over the block's cells and attempts
  int* order_thresh;             // [1] or null: the same count for cell 1 of block 1 (DYN kernel),
                                 // the matrix the reference orders on (rodas3:470-506)
  const int* cell_list;          // optional: blocks are consecutive WG-sized runs of this list
  const int* block_order;        // optional: workgroup w integrates block block_order[w]
  int list_n;                    // length of cell_list
  double* half_y;                // concentrations of the two halves of blocks of more than 64 cells
};

enum { kSplitSymmetric = 0, kSplitSequential = 1, kSplitParallel = 2 };
// Upper bound on attempts per block and call.  Each rejection shrinks dt by
// at least 10% until dt_min forces acceptance (rodas3:650-676), so a block
// needs far fewer (at most dtlt/dt_min accepted steps plus a few dozen
// rejections each); the bound only guards against a non-terminating wave.
constexpr int kMaxAttempts = 20000;

// The two Rosenbrock solvers of the reference on the same mechanism code:
// RODAS3 (chem_spack_rodas3_dyndt.f90, CHEMISTRY=4) and the two-stage ROS2
// (chem_spack_ros_dyndt.f90, CHEMISTRY=3).
enum { kRodas3 = 0, kRos2 = 1 };
// ROS2's gamma = 1 + 1/sqrt(2), with sqrt(2) written as the double value of
// its single-precision rounding, 1.4142135381698608 (ros_dyndt:130)
constexpr double kRos2Gamma = 1.0 + 1.0 / 1.4142135381698608;
constexpr double kRos2GammaInv = 1.0 / kRos2Gamma;

// Several grids in one launch (the nested grids of one model step, which the
// reference integrates one call per grid, chemistry.f90:313-320): workgroup
// w integrates block (work[w] & kGridBlockMask) of the grid whose parameters
// are grids[work[w] >> kGridShift].  Blocks never exchange data, so a block
// gives the same result here as in its own grid's launch.
constexpr int kGridShift = 24;
constexpr int kGridBlockMask = (1 << kGridShift) - 1;

}  // namespace brams
