// Batched FP64 Rosenbrock integration (RODAS3, ROS2) of one mechanism on
// CDNA4, one workgroup to a block.
//
// One reference block (chem_spack_utils.f90:93-160) is 64 cells that share
// the step size (rodas3:634-700).  A cell's working set (factors, rate
// constants, stage vectors) is about a thousand doubles: four times what a
// lane's registers hold, but what a CU's registers and LDS hold for one
// block.  So one workgroup of MECH_COOP_WAVES waves takes one block, lane l of
// every wave works on cell l, and each wave owns some species: their matrix
// rows, their rates, their entries of the stage vectors.  The waves'
// straight-line programs and the LDS exchange between them are generated
// (codegen/gen_coop.py); this file holds what is around them: gather, the
// sub-step loop, the step-size controller and the write-back.
//
// Bound: a block's attempt is a chain of phases between barriers, each as long
// as its busiest wave; one workgroup fills a CU (159 KB of LDS, 256 registers
// a lane at two waves per SIMD), so nothing overlaps another block's.
// Measured on 1.6M cells of RELACS_TUV, one step at the reference's
// tolerances (16.3 attempts a cell): 30.8 ms, 20.6 us or 49 000 clocks a
// block's attempt.  57 % of a wave's clocks are waits (barriers, LDS), 14 %
// waits for issue, 17 % FP64 and other vector instructions.  The attempt
// sweeps its straight-line code (385 KB for the eight waves) with 5 500
// fetches, of which 1.4 % miss the instruction cache or join a miss.  The
// generator's model (Layout.stats) gives 31 800 clocks; what the other 17 000
// are is not known.  A lane spills up to 176 bytes, which the caches hold:
// memory sees 1.3 KB a cell whatever the attempts.  The kernel it replaces
// kept one lane's whole state in registers and scratch: it read and wrote
// 63 KB of spilled state a cell-attempt and took 353 ms.
//
// Blocks of 65..127 cells (the first ones of a grid whose cell count is no
// multiple of 64) run as two halves in turn inside each attempt, with their
// concentrations in memory between them; the step size is the block's.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "coop_lane.h"
#include "rodas3_kernel.h"

namespace brams {

// ---- the pieces of an attempt that the generated code calls

// stage 3's point with clipping, rodas3:542-566
__device__ __forceinline__ void coop_stage3(double k1, double y, double& yn, double& k1c) {
  yn = y + 2.0 * k1;
  k1c = k1;
  if (yn < 0.0) {
    yn = 0.0;
    k1c = 0.5 * (yn - y);
  }
}

// stage 4's point with clipping, rodas3:573-599
__device__ __forceinline__ void coop_stage4(double k1, double k3, double y, double& yn, double& k3c) {
  yn = y + 2.0 * k1 + k3;
  k3c = k3;
  if (yn < 0.0) {
    yn = 0.0;
    k3c = (yn - y) - 2.0 * k1;
  }
}

// solution and error of one species, rodas3:609-648
__device__ __forceinline__ void coop_end_rodas3(double k1, double k3, double k4, double y, double atol, double rtol,
                                                double& yn, double& e) {
  const double v = fmax(y + 2.0 * k1 + k3 + k4, 0.0);
  yn = v;
  const double q = k4 / (atol + rtol * fmax(fabs(y), fabs(v)));
  e = fma(q, q, e);
}

// the same for ROS2 (no clipping), ros_dyndt:463-498
__device__ __forceinline__ void coop_end_ros2(double k1, double k2, double y, double atol, double rtol, double& yn,
                                              double& e) {
  const double v = y + kRos2GammaInv * (1.5 * k1 + 0.5 * k2);
  yn = v;
  const double q = (0.5 * kRos2GammaInv * (k1 + k2)) / (atol + rtol * fmax(fabs(y), fabs(v)));
  e = fma(q, q, e);
}

}  // namespace brams

namespace brams {
#include BRAMS_MECH_COOP

constexpr int kCoopLanes = 64 * MECH_COOP_WAVES;

// where cell `c` of block b lies, and its meteorology (rodas3:226-290)
struct CoopCell {
  long long o;
  double temp, press, vapp, volmol;
  bool act;
};

__device__ __forceinline__ CoopCell coop_cell(const StepParams& p, int start, int ncell, int c) {
  CoopCell q;
  q.act = c < ncell;
  const int at = start + (q.act ? c : 0);                 // idle lanes shadow cell 1
  const unsigned g = p.cell_list ? (unsigned)p.cell_list[at] : (unsigned)at;
  // cell position, j -> i -> k order (chem_spack_utils.f90:144-160)
  const unsigned t = g / (unsigned)p.nk;
  const unsigned k = g - t * (unsigned)p.nk;
  const unsigned jj = t / (unsigned)p.ni;
  const unsigned ii = t - jj * (unsigned)p.ni;
  q.o = (long long)(k + 1) + (long long)p.m1 * (p.ia - 1 + ii) + (long long)p.m1 * p.m2 * (p.ja - 1 + jj);
  const float exner = (p.pp[q.o] + p.pi0[q.o]) / p.cp;   // REAL arithmetic
  q.press = (double)exner;
  q.temp = (double)p.theta[q.o] * q.press;
  q.press = pow(q.press, (double)p.cpor) * (double)p.p00;
  q.vapp = (double)p.rv[q.o];
  q.volmol = (6.02e23 * 1e-15 * 28.96) * q.press / (8.314 * q.temp);
  return q;
}

// x^(-1/3) for x >= 1e-15: a 32-bit estimate and two Newton steps, each
// squaring the error (1e-7, 4e-14, below 1e-16).
__device__ __forceinline__ double coop_inv_cbrt(double x) {
#pragma clang fp contract(off)
  int ex;
  double m = frexp(x, &ex);                               // [0.5, 1)
  const int q = (ex + 3000) / 3 - 1000;                   // floor(ex / 3)
  m = ldexp(m, ex - 3 * q);                               // [0.5, 4)
  double r = (double)coop_exp2(coop_log2((float)m) * (-1.0f / 3.0f));
  r = fma(r * (1.0 / 3.0), fma(-m * r, r * r, 1.0), r);
  r = fma(r * (1.0 / 3.0), fma(-m * r, r * r, 1.0), r);
  return ldexp(r, -q);
}

// The next step size from the largest squared error sum of the block's cells
// (rodas3:650-700, error order 3; ros_dyndt:501-551, order 2).  Every wave
// evaluates it, and all must decide alike, so no operation here is left to
// the compiler's contraction.
template <int SOLVER>
__device__ __forceinline__ double coop_controller(double esum, double dt, double dt_min, double dt_max, double& err) {
#pragma clang fp contract(off)
  // the square root is monotonic: it can wait until after the maximum
  err = fmax(1.0e-15, sqrt(esum / (double)MECH_NS));
  const double grow = SOLVER == kRos2 ? 0.9 / sqrt(err) : 0.9 * coop_inv_cbrt(err);
  return fmax(dt_min, fmin(dt_max, dt * fmin(6.0, fmax(0.2, grow))));
}

// The program of wave WV.  lds: the workgroup's slots.
template <class WV, int SOLVER, bool DYN, bool COUNT>
__device__ __forceinline__ void coop_run(const StepParams& p, int b, int slot, double* lds, int wave, int lane) {
  const CoopLds S(lds + lane);
  int start, ncell;
  if (p.cell_list) {                                      // fallback blocks of listed cells
    start = b * 64;
    ncell = min(64, p.list_n - start);
  } else {
    start = coop_uniform(p.block_start[b]);
    ncell = coop_uniform(p.block_start[b + 1]) - start;
  }
  // COUNT kernels take the 65..127-cell blocks, in two halves
  const int halves = COUNT && ncell > 64 ? 2 : 1;
  const bool par_n = (p.split == kSplitParallel) && (p.ndyn > 1);
  int* vbits = reinterpret_cast<int*>(lds + MECH_COOP_VSLOT * 64) + lane;
  int* mbits = reinterpret_cast<int*>(lds + MECH_COOP_MSLOT * 64);
  (void)vbits;

  double y[WV::kOwn + 1], yn[WV::kOwn + 1];
  double* half = nullptr;                                 // [half][buffer][species][64]
  int cur = 0;
  if (COUNT && halves > 1) half = p.half_y + (long long)slot * (4 * MECH_NS * 64) + lane;

  CoopCell q;
  auto gather = [&](int h) {
    q = coop_cell(p, start, ncell, lane + 64 * h);
#pragma unroll
    for (int k = 0; k < WV::kOwn; ++k) {
      const int s = WV::own[k];
      const float v = p.sc_p[(long long)s * p.n3d + q.o];
      if (!p.transported[s]) {
        y[k] = (double)v;
      } else if (par_n) {
        const float st = v - p.sc_t_dyn[(long long)s * p.n3d + q.o] * (float)p.ndyn * p.dtlt;
        y[k] = (double)st * q.volmol / (double)p.weight[s];
      } else {
        const double x = (double)v * q.volmol / (double)p.weight[s];
        y[k] = x > 0.0 ? x : 0.0;
      }
    }
  };
  // the block's concentrations live in LDS, where every wave reads them
  auto publish = [&](const double* v) {
#pragma unroll
    for (int k = 0; k < WV::kOwn; ++k) S.put(WV::own[k], v[k]);
  };
  // rate coefficients of the cells in q, spread over the waves
  auto kinetic = [&]() {
    WV::kinetic(q.temp, q.press, q.vapp, p.jphoto + (long long)MECH_NPHOT * q.o, S);
    publish(y);
    coop_barrier();
  };

  const float tnf = p.dtlt * (float)p.ndyn;
  const double dt_min = fmax(1.0, 1.0e-2 * (double)tnf);
  const double dt_max = (double)tnf;
  const double time_f = (double)tnf;
  double dt = p.last_dt[b];
  double last_dt = dt;
  double time_c = 0.0;
  int natt = 0, nsub = 0, failed = 0;
  int nviol = 0, oviol = 0;
  float forced = 0.f;
  unsigned mw[MECH_MASK_WORDS];
#pragma unroll
  for (int k = 0; k < MECH_MASK_WORDS; ++k) mw[k] = (SOLVER == kRos2 || DYN) ? 0xffffffffu : (unsigned)coop_uniform((int)p.mask[k]);

  gather(0);
  if (COUNT && halves > 1) {
#pragma unroll
    for (int k = 0; k < WV::kOwn; ++k) half[WV::own[k] * 64] = y[k];
    gather(1);
#pragma unroll
    for (int k = 0; k < WV::kOwn; ++k) half[(2 * MECH_NS + WV::own[k]) * 64] = y[k];
  } else {
    kinetic();
  }

  while (coop_uniform(time_c + 1.0e-8 < time_f ? 1 : 0)) {
    ++natt;
    // 1/(gamma h): RODAS3 gamma = 1/2 (rodas3:462), ROS2 ros_dyndt:387
    const double igdt = SOLVER == kRos2 ? 1.0 / (kRos2Gamma * dt) : 1.0 / (0.5 * dt);
    const double dti = 1.0 / dt;
    double errmax = 0.0;
    bool fail = natt >= kMaxAttempts;
#pragma unroll
    for (int k = 0; k < MECH_MASK_WORDS; ++k)
      if (SOLVER != kRos2) coop_opaque(mw[k]);
    for (int h = 0; h < halves; ++h) {
      if (COUNT && halves > 1) {
        q = coop_cell(p, start, ncell, lane + 64 * h);
#pragma unroll
        for (int k = 0; k < WV::kOwn; ++k) y[k] = half[((2 * h + cur) * MECH_NS + WV::own[k]) * 64];
        kinetic();
      }
      double e = 0.0;
      unsigned viol[MECH_COOP_VWORDS] = {};
      if (COUNT) {
        if (wave == 0)
          for (int k = 0; k < MECH_COOP_VWORDS; ++k) vbits[k * 64] = 0;
      }
      if constexpr (SOLVER == kRos2)
        WV::template ros2<DYN, COUNT>(S, igdt, dti, mw, false, p.atol, p.rtol, yn, e, viol);
      else
        WV::template rodas3<DYN, COUNT>(S, igdt, dti, mw, DYN && h == 0, p.atol, p.rtol, yn, e, viol);
      if (COUNT) {
        for (int k = 0; k < MECH_COOP_VWORDS; ++k) atomicOr(&vbits[k * 64], (int)viol[k]);
        if (halves > 1) {
#pragma unroll
          for (int k = 0; k < WV::kOwn; ++k) half[((2 * h + (cur ^ 1)) * MECH_NS + WV::own[k]) * 64] = yn[k];
        }
      }
      // error over the species: every wave adds the waves' parts in the same order
      S.put(MECH_COOP_ESLOT + wave, e);
      coop_barrier();
      e = S.get(MECH_COOP_ESLOT);
#pragma unroll
      for (int w = 1; w < MECH_COOP_WAVES; ++w) e = e + S.get(MECH_COOP_ESLOT + w);
      // a zero pivot makes its species' error non-finite (its reciprocal
      // enters every solve), so this also ends a block there, where the
      // reference aborts the process
      fail = fail || coop_any(q.act && !isfinite(e));
      errmax = fmax(errmax, coop_wave_max(q.act ? e : 0.0));
      if (COUNT) {
        if (wave == 0 && q.act) {
          int n = 0;
          for (int k = 0; k < MECH_COOP_VWORDS; ++k) n += __popc((unsigned)vbits[k * 64]);
          nviol += n;
          if (h == 0 && lane == 0) oviol += n;
        }
        if (halves > 1) coop_barrier();                   // the error slots are read before the next half
      }
    }
    double err;
    const double dt_new = coop_controller<SOLVER>(errmax, dt, dt_min, dt_max, err);
    const bool rej = err - 1.0e-8 > 1.0;
    // One path for accepted and rejected attempts: a taken branch costs a
    // miss of the instruction cache, which the attempt's code has swept.  So a
    // rejected attempt evaluates the Jacobian and f(y0) again, to the same
    // values.
    const int act = coop_uniform(fail ? 2 : (rej && dt_new > dt_min) ? 1 : 0);
    if (__builtin_expect(act == 2, 0)) {
      failed = 1;
      break;
    }
    if (act == 0) {
      // an error above 1 accepted anyway: dt reached dt_min (rodas3:671-676)
      forced = rej ? fmaxf(forced, (float)err) : forced;
      time_c = time_c + dt;
      last_dt = time_c < time_f ? dt_new : last_dt;
      ++nsub;
      cur ^= 1;
      if (halves == 1) publish(yn);
    }
    dt = act == 0 ? fmin(dt_new, time_f - time_c) : dt_new;
    coop_barrier();
  }

  // ---- write-back, rodas3:713-798
  for (int h = 0; h < halves; ++h) {
    if (COUNT && halves > 1) {
      q = coop_cell(p, start, ncell, lane + 64 * h);
#pragma unroll
      for (int k = 0; k < WV::kOwn; ++k) y[k] = half[((2 * h + cur) * MECH_NS + WV::own[k]) * 64];
    } else {
#pragma unroll
      for (int k = 0; k < WV::kOwn; ++k) y[k] = S.get(WV::own[k]);
    }
    if (!q.act) continue;
    const double volmol_i = 1.0 / q.volmol;
#pragma unroll
    for (int k = 0; k < WV::kOwn; ++k) {
      const int s = WV::own[k];
      const long long idx = (long long)s * p.n3d + q.o;
      if (!p.transported[s]) {
        const float v = (float)y[k];
        p.sc_p[idx] = v > 0.0f ? v : 0.0f;
        continue;
      }
      const double conv = y[k] * (double)p.weight[s] * volmol_i;
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
  if constexpr (DYN) {
    // the call's mask: every wave holds the words of its own rows
    coop_barrier();
    if (wave == 0 && lane == 0)
      for (int k = 0; k < MECH_MASK_WORDS; ++k) mbits[k] = 0;
    coop_barrier();
    if (lane == 0)
      for (int k = 0; k < MECH_MASK_WORDS; ++k) atomicOr(&mbits[k], (int)(mw[k] & WV::mask_own[k]));
    coop_barrier();
    if (wave == 0 && lane == 0)
      for (int k = 0; k < MECH_MASK_WORDS; ++k) p.mask[k] = (unsigned)mbits[k];
  }
  if (wave == 0) {
    if (COUNT) nviol = coop_wave_sum(nviol);
    if (lane == 0) {
      if (COUNT && DYN && p.order_thresh) p.order_thresh[0] = oviol;
      if (p.blk_thresh) p.blk_thresh[b] = COUNT ? nviol : 0;
      p.last_dt[b] = last_dt;
      p.blk_attempts[b] = natt;
      p.blk_substeps[b] = nsub;
      p.blk_failed[b] = failed;
      if (p.blk_forced) p.blk_forced[b] = forced;
    }
  }
}

template <int SOLVER, bool DYN, bool COUNT>
__device__ __forceinline__ void coop_block(const StepParams& p, int b, int slot) {
  __shared__ double lds[MECH_COOP_SLOTS * 64];
  const int wave = coop_uniform(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  switch (wave) {
    case 0: coop_run<CoopWave0, SOLVER, DYN, COUNT>(p, b, slot, lds, 0, lane); break;
    case 1: coop_run<CoopWave1, SOLVER, DYN, COUNT>(p, b, slot, lds, 1, lane); break;
    case 2: coop_run<CoopWave2, SOLVER, DYN, COUNT>(p, b, slot, lds, 2, lane); break;
    case 3: coop_run<CoopWave3, SOLVER, DYN, COUNT>(p, b, slot, lds, 3, lane); break;
#if MECH_COOP_WAVES > 4
    case 4: coop_run<CoopWave4, SOLVER, DYN, COUNT>(p, b, slot, lds, 4, lane); break;
    case 5: coop_run<CoopWave5, SOLVER, DYN, COUNT>(p, b, slot, lds, 5, lane); break;
    case 6: coop_run<CoopWave6, SOLVER, DYN, COUNT>(p, b, slot, lds, 6, lane); break;
    default: coop_run<CoopWave7, SOLVER, DYN, COUNT>(p, b, slot, lds, 7, lane); break;
#endif
  }
}

// One launch of blocks: block0 + blockIdx.x of p, or, with p.block_order, in that order.
template <int SOLVER, bool DYN, bool COUNT>
__global__ __launch_bounds__(kCoopLanes, MECH_COOP_WAVES / 4) void coop_blocks(StepParams p, int block0) {
  const int b = p.block_order ? coop_uniform(p.block_order[blockIdx.x]) : block0 + (int)blockIdx.x;
  coop_block<SOLVER, DYN, COUNT>(p, b, (int)blockIdx.x);
}

// Several grids in one launch (kGridShift in rodas3_kernel.h).
template <bool DYN, bool COUNT>
__global__ __launch_bounds__(kCoopLanes, MECH_COOP_WAVES / 4) void coop_grids(const StepParams* __restrict__ grids,
                                                                              const int* __restrict__ work) {
  const int w = coop_uniform(work[blockIdx.x]);
  coop_block<kRodas3, DYN, COUNT>(grids[w >> kGridShift], w & kGridBlockMask, (int)blockIdx.x);
}

#ifdef __HIPCC__
// A dispatch counts its work-items in 32 bits, which 8M blocks exceed, so it
// takes at most half of that many.
constexpr unsigned kCoopMaxBlocks = 1u << 22;

template <int SOLVER, bool DYN, bool COUNT>
hipError_t coop_launch(unsigned nblocks, StepParams p, int block0, hipStream_t st) {
  while (nblocks > 0) {
    const unsigned n = nblocks < kCoopMaxBlocks ? nblocks : kCoopMaxBlocks;
    hipLaunchKernelGGL((coop_blocks<SOLVER, DYN, COUNT>), dim3(n), dim3(kCoopLanes), 0, st, p, block0);
    if (p.block_order) p.block_order += n;
    block0 += (int)n;
    nblocks -= n;
  }
  return hipGetLastError();
}

template <bool DYN, bool COUNT>
hipError_t coop_launch_grids(unsigned nwork, const StepParams* grids, const int* work, hipStream_t st) {
  while (nwork > 0) {
    const unsigned n = nwork < kCoopMaxBlocks ? nwork : kCoopMaxBlocks;
    hipLaunchKernelGGL((coop_grids<DYN, COUNT>), dim3(n), dim3(kCoopLanes), 0, st, grids, work);
    work += n;
    nwork -= n;
  }
  return hipGetLastError();
}
#endif

}  // namespace brams
