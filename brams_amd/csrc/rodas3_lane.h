// Rosenbrock blocks with one lane to a cell, for mechanisms too large for the
// cooperative kernel (rodas3_coop.h): RACM_TUV's 1052 factors, 237 rate
// constants and stage vectors of 72 species exceed a CU's registers and LDS
// for 64 cells too, and its exchange between the waves exceeds the LDS.
//
// Mapping: one workgroup = one reference block (chem_spack_utils.f90:93-160),
// one lane = one cell.  Blocks of 64 cells are exactly one wave64; blocks of
// 65..127 cells run as a 128-lane workgroup.  The block-shared step size of
// the reference (rodas3:634-700) is a workgroup reduction of the per-cell
// error, so every lane takes the same accept/reject branch.  The Jacobian is
// not stored: each attempt rebuilds 1/(gamma h) I - J from y0 and rk inside
// the factorisation.
//
// A lane's state never fits the register file, so the compiler spills; what
// matters is how many waves hide the spill traffic.  WPS sets the register
// budget by the waves per SIMD it must allow.  RACM_TUV's step on 1.6M cells
// runs at 2.45e6 cell-steps/s with four and 1.67e6 with one; a launch of a few
// thousand blocks has too few waves to use the occupancy and runs faster with
// the whole register file.
#pragma once
#include <hip/hip_runtime.h>

#include "rodas3_kernel.h"

namespace brams {

constexpr int kLaneManyWaves = 4;        // WPS of large launches (form 5, rodas3_launch.h)

template <int WG>
__device__ __forceinline__ void block_reduce(double& errmax, int& rej, int& fail,
                                             double* s_err, int* s_rej, int* s_fail) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    errmax = fmax(errmax, __shfl_xor(errmax, off, 64));
    rej |= __shfl_xor(rej, off, 64);
    fail |= __shfl_xor(fail, off, 64);
  }
  if constexpr (WG > 64) {
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
      s_err[wave] = errmax;
      s_rej[wave] = rej;
      s_fail[wave] = fail;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < WG / 64; ++w) {
      errmax = fmax(errmax, s_err[w]);
      rej |= s_rej[w];
      fail |= s_fail[w];
    }
    __syncthreads();
  }
}

// DYN: block 1 of the call.  Its sparsity mask is recomputed from cell 1 on
// every attempt (rodas3:470-482) and the last one is published for the other
// blocks.  Otherwise the mask is read from p.mask.
// SOLVER kRos2: chem_ros_dyndt's integration, which uses the full structural
// Jacobian (no value mask, so no block-1 form) and no clipping.
template <int WG, bool DYN, int SOLVER = kRodas3>
__device__ __forceinline__ void integrate_block(const StepParams& p, int b) {
  static_assert(SOLVER == kRodas3 || !DYN, "ROS2 has no block-1 form");
  // Sparse1.3 applies its threshold rule only where it orders, on cell 1 of
  // block 1 (rodas3:470-506); the other blocks reuse that order unchecked.
  // Block 1 and the 65..127-cell blocks count failing pivots over all their
  // cells; the 64-cell blocks skip the count (it costs them a few
  // percent of their time).
  constexpr bool kCountThreshold = DYN || (WG > 64);
  const int start = p.block_start[b];
  const int ncell = p.block_start[b + 1] - start;
  const int c = threadIdx.x;
  const bool act = c < ncell;
  const long long g = (long long)(start + (act ? c : 0));  // idle lanes shadow cell 1

  // cell position, j -> i -> k order (chem_spack_utils.f90:144-160)
  const long long kk = 2 + g % p.nk;
  const long long t = g / p.nk;
  const long long ii = p.ia + t % p.ni;
  const long long jj = p.ja + t / p.ni;
  const long long o = (kk - 1) + (long long)p.m1 * (ii - 1) + (long long)p.m1 * p.m2 * (jj - 1);

  // ---- gather and unit conversion, rodas3:226-354
  const float exner = (p.pp[o] + p.pi0[o]) / p.cp;   // REAL arithmetic
  double press = (double)exner;
  const double temp = (double)p.theta[o] * press;
  press = pow(press, (double)p.cpor) * (double)p.p00;
  const double vapp = (double)p.rv[o];
  const double volmol = (6.02e23 * 1e-15 * 28.96) * press / (8.314 * temp);
  const double volmol_i = 1.0 / volmol;
  const bool par_n = (p.split == kSplitParallel) && (p.ndyn > 1);

  double y[MECH_NS];
#pragma unroll
  for (int s = 0; s < MECH_NS; ++s) {
    const float v = p.sc_p[(long long)s * p.n3d + o];
    if (!p.transported[s]) {
      y[s] = (double)v;
    } else if (par_n) {
      const float st = v - p.sc_t_dyn[(long long)s * p.n3d + o] * (float)p.ndyn * p.dtlt;
      y[s] = (double)st * volmol / (double)p.weight[s];
    } else {
      const double x = (double)v * volmol / (double)p.weight[s];
      y[s] = x > 0.0 ? x : 0.0;
    }
  }
  double rk[MECH_NR];
  {
    double J[MECH_NPHOT];
#pragma unroll
    for (int n = 0; n < MECH_NPHOT; ++n) J[n] = p.jphoto[n + (long long)MECH_NPHOT * o];
    mech_kinetic(temp, press, vapp, J, rk);
  }

  // ---- RODAS3 sub-steps, rodas3:413-705
  const double c83 = 8.0 / 3.0;
  const float tnf = p.dtlt * (float)p.ndyn;
  const double dt_min = fmax(1.0, 1.0e-2 * (double)tnf);
  const double dt_max = (double)tnf;
  const double time_f = (double)tnf;
  double dt = p.last_dt[b];
  double last_dt = dt;
  double time_c = 0.0;
  int natt = 0, nsub = 0, failed = 0, nviol = 0;
  float forced = 0.f;

  __shared__ unsigned s_mask[MECH_MASK_WORDS];
  __shared__ double s_err[WG / 64 + 1];
  __shared__ int s_rej[WG / 64 + 1], s_fail[WG / 64 + 1];
  unsigned mw[MECH_MASK_WORDS];
  if constexpr (SOLVER == kRos2) {
#pragma unroll
    for (int w = 0; w < MECH_MASK_WORDS; ++w) mw[w] = 0xffffffffu;   // every structural entry
  } else if constexpr (!DYN) {
#pragma unroll
    for (int w = 0; w < MECH_MASK_WORDS; ++w) mw[w] = p.mask[w];
  }

  while (time_c + 1.0e-8 < time_f) {
    double f0[MECH_NS];
    mech_fun(rk, y, f0);
    for (;;) {
      ++natt;
      // 1/(gamma h): RODAS3 gamma = 1/2 (rodas3:462), ROS2 ros_dyndt:387
      const double igdt = SOLVER == kRos2 ? 1.0 / (kRos2Gamma * dt) : 1.0 / (0.5 * dt);
      if constexpr (DYN) {
        // every lane evaluates the mask of its own cell, so the evaluation
        // is no divergent region; cell 1's is the one published
        unsigned m[MECH_MASK_WORDS];
        mech_mask(rk, y, igdt, m);
        if (c == 0) {
#pragma unroll
          for (int w = 0; w < MECH_MASK_WORDS; ++w) s_mask[w] = m[w];
        }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < MECH_MASK_WORDS; ++w) mw[w] = s_mask[w];
      }
      double lu[MECH_NLU];
      const int bad = mech_factor<kCountThreshold>(rk, y, igdt, mw, lu, &nviol);
      const double dti = 1.0 / dt;
      double yn[MECH_NS];
      double e = 0.0;
      if constexpr (SOLVER == kRos2) {
        // stage 1, ros_dyndt:404-424: k1 = (1/(gamma h) - J)^-1 f(y0)
        double k1[MECH_NS], k2[MECH_NS];
#pragma unroll
        for (int s = 0; s < MECH_NS; ++s) k1[s] = f0[s];
        mech_solve(lu, k1);
#pragma unroll
        for (int s = 0; s < MECH_NS; ++s) yn[s] = y[s] + kRos2GammaInv * k1[s];
        // stage 2, ros_dyndt:433-460: f(y0 + k1/gamma) - 2/(gamma h) k1
        mech_fun(rk, yn, k2);
#pragma unroll
        for (int s = 0; s < MECH_NS; ++s) k2[s] = k2[s] - 2.0 * kRos2GammaInv * dti * k1[s];
        mech_solve(lu, k2);
        // solution and error, ros_dyndt:463-498 (no clipping)
#pragma unroll
        for (int s = 0; s < MECH_NS; ++s) {
          const double v = y[s] + kRos2GammaInv * (1.5 * k1[s] + 0.5 * k2[s]);
          yn[s] = v;
          const double tol = p.atol[s] + p.rtol[s] * fmax(fabs(y[s]), fabs(v));
          const double q = (0.5 * kRos2GammaInv * (k1[s] + k2[s])) / tol;
          e = e + q * q;
        }
      } else {
      // stage 1, rodas3:523-527
      double k1[MECH_NS];
#pragma unroll
      for (int s = 0; s < MECH_NS; ++s) k1[s] = f0[s];
      mech_solve(lu, k1);
      // stage 2, rodas3:534-538
      double k2[MECH_NS];
#pragma unroll
      for (int s = 0; s < MECH_NS; ++s) k2[s] = (4.0 * dti) * k1[s] + f0[s];
      mech_solve(lu, k2);
      // stage 3 with clipping, rodas3:542-566
      double ft[MECH_NS];
#pragma unroll
      for (int s = 0; s < MECH_NS; ++s) {
        yn[s] = y[s] + 2.0 * k1[s];
        if (yn[s] < 0.0) {
          yn[s] = 0.0;
          k1[s] = 0.5 * (yn[s] - y[s]);
        }
      }
      mech_fun(rk, yn, ft);
      double k3[MECH_NS];
#pragma unroll
      for (int s = 0; s < MECH_NS; ++s) {
        k2[s] = k1[s] - k2[s];                    // k1 - k2, reused below
        k3[s] = ft[s] + dti * k2[s];
      }
      mech_solve(lu, k3);
      // stage 4 with clipping, rodas3:573-599
#pragma unroll
      for (int s = 0; s < MECH_NS; ++s) {
        yn[s] = y[s] + 2.0 * k1[s] + k3[s];
        if (yn[s] < 0.0) {
          yn[s] = 0.0;
          k3[s] = (yn[s] - y[s]) - 2.0 * k1[s];
        }
      }
      mech_fun(rk, yn, ft);
#pragma unroll
      for (int s = 0; s < MECH_NS; ++s) ft[s] = ft[s] + dti * (k2[s] - c83 * k3[s]);
      mech_solve(lu, ft);                          // ft now holds k4
      // solution and error, rodas3:609-648
#pragma unroll
      for (int s = 0; s < MECH_NS; ++s) {
        double v = y[s] + 2.0 * k1[s] + k3[s] + ft[s];
        v = fmax(v, 0.0);
        yn[s] = v;
        const double tol = p.atol[s] + p.rtol[s] * fmax(fabs(y[s]), fabs(v));
        const double q = ft[s] / tol;
        e = e + q * q;
      }
      }
      const double err = fmax(1.0e-15, sqrt(e / (double)MECH_NS));
      double errmax = act ? err : 0.0;
      int rej = (act && (err - 1.0e-8 > 1.0)) ? 1 : 0;
      // a zero pivot or a non-finite error sum ends the block (the reference
      // aborts the process there); kMaxAttempts bounds every wave's work
      int fail = (act && (bad || !isfinite(e))) ? 1 : 0;
      if (natt >= kMaxAttempts) fail = 1;
      block_reduce<WG>(errmax, rej, fail, s_err, s_rej, s_fail);
      // controller, rodas3:650-700 (error order 3) and ros_dyndt:501-551 (order 2)
      const double fac = fmin(6.0, fmax(0.2, 0.9 / pow(errmax, SOLVER == kRos2 ? 1.0 / 2.0 : 1.0 / 3.0)));
      double dt_new = dt * fac;
      dt_new = fmax(dt_min, fmin(dt_max, dt_new));
      if (fail) {
        failed = 1;
        time_c = time_f;
        break;
      }
      if (rej && dt_new > dt_min) {
        dt = dt_new;
        continue;
      }
      // an error above 1 accepted anyway: dt reached dt_min (rodas3:671-676)
      if (rej) forced = fmaxf(forced, (float)errmax);
      time_c = time_c + dt;
      dt = fmin(dt_new, time_f - time_c);
      if (time_c < time_f) last_dt = dt_new;
#pragma unroll
      for (int s = 0; s < MECH_NS; ++s) y[s] = yn[s];
      ++nsub;
      break;
    }
  }

  // ---- write-back, rodas3:713-798
  if (act) {
#pragma unroll
    for (int s = 0; s < MECH_NS; ++s) {
      const long long idx = (long long)s * p.n3d + o;
      if (!p.transported[s]) {
        const float v = (float)y[s];
        p.sc_p[idx] = v > 0.0f ? v : 0.0f;
        continue;
      }
      const double conv = y[s] * (double)p.weight[s] * volmol_i;
      if (par_n) {
        const float base = p.sc_t_dyn[idx] * (float)p.ndyn * p.dtlt;
        const float v = (float)((double)base + conv);
        p.sc_p[idx] = v > 0.0f ? v : 0.0f;
      } else if (p.split == kSplitParallel) {
        const double dti = 1.0 / (double)p.dtlt;
        p.sc_t[idx] = (float)((double)p.sc_t[idx] + (conv - (double)p.sc_p[idx]) * dti);
      } else {
        const float v = (float)conv;
        p.sc_p[idx] = v > 0.0f ? v : 0.0f;
      }
    }
  }
  // threshold-rule count of the block: sum over its cells (0 where not counted)
  if constexpr (!kCountThreshold) {
    if (c == 0 && p.blk_thresh) p.blk_thresh[b] = 0;
  } else {
    int v = act ? nviol : 0;
    if constexpr (DYN) {
      if (c == 0 && p.order_thresh) p.order_thresh[0] = nviol;
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    if constexpr (WG > 64) {
      __syncthreads();
      if ((threadIdx.x & 63) == 0) s_rej[threadIdx.x >> 6] = v;
      __syncthreads();
      v = 0;
#pragma unroll
      for (int w = 0; w < WG / 64; ++w) v += s_rej[w];
    }
    if (c == 0 && p.blk_thresh) p.blk_thresh[b] = v;
  }
  if (c == 0) {
    p.last_dt[b] = last_dt;
    p.blk_attempts[b] = natt;
    p.blk_substeps[b] = nsub;
    p.blk_failed[b] = failed;
    if (p.blk_forced) p.blk_forced[b] = forced;
    if constexpr (DYN) {
#pragma unroll
      for (int w = 0; w < MECH_MASK_WORDS; ++w) p.mask[w] = s_mask[w];
    }
  }
}

template <int WG, bool DYN, int WPS>
__global__ __launch_bounds__(WG, WPS) void rodas3_blocks(StepParams p, int block0) {
  const int b = p.block_order ? p.block_order[blockIdx.x] : block0 + blockIdx.x;
  integrate_block<WG, DYN>(p, b);
}

// CHEMISTRY=3: chem_ros_dyndt's blocks, all of one launch alike (no block-1 form)
template <int WG, int WPS>
__global__ __launch_bounds__(WG, WPS) void ros2_blocks(StepParams p, int block0) {
  const int b = p.block_order ? p.block_order[blockIdx.x] : block0 + blockIdx.x;
  integrate_block<WG, false, kRos2>(p, b);
}

}  // namespace brams
