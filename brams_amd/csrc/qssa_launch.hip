// The QSSA solver of the reference (CHEMISTRY=1, chem_spack_qssa.f90:37-411)
// on CDNA4.
//
// Cells are independent: QSSA has no step-size control, so AllocIndex's
// blocks play no role.  A workgroup takes 64 cells of the interior, one to a
// lane, in the j -> i -> k order of the blocks (k fastest, so a wave's loads
// of one species coalesce along the column), and its eight waves share each
// cell's work (the generated qssa_program).  Per cell:
//   gather          chem_spack_qssa.f90:161-195 (every species from ppbm)
//   kinetic         the mechanism's rate laws (chem_spack_kinetic.f90)
//   P and L         rates, dratedc, fexprod, fexloss (:247-265): P the positive
//                   stoichiometric terms c w_r, L -c dw_rs over the negative
//                   ones, in reaction order; 0 where there is no term
//   itchim sub-steps of length dtlt/itchim with P and L held (solveur :343-348,
//                   qssa :368-411), negatives set to 0 (:352-354)
//   tendency        sc_t += (new - old) / dtlt for every species (:273-292)
// A cell where a species reaches 1e20 (solveur :357-361 stops the model) is
// counted and writes nothing.
//
// FP64 issue bounds it.  One lane with a whole cell (128 rate constants, 47
// concentrations, production and loss) filled the register file at one wave
// per SIMD, spilled, and waited on its own chains: 2.19 ms for 1.6M cells of
// RELACS_TUV, itchim 75, where memory needs 0.25 ms.  Shared out, a wave has
// 16 reactions and 6 species, and four waves fit a SIMD: 1.01 ms, with no
// register spilled.
#include <hip/hip_runtime.h>

#include "rodas3_kernel.h"
#include "coop_lane.h"
#include "rodas3_launch.h"

namespace brams {

// A divisor that many quotients share, with its reciprocal: n r, one
// correction by the exact remainder (P. Markstein, IBM J. Res. Dev. 34, 1990)
// and the hardware's treatment of zeros, infinities and NaN, four instructions
// where a division takes eleven.
struct QssaTemp {
  double t, r;
  __device__ __forceinline__ explicit QssaTemp(double d) : t(d), r(1.0 / d) {}
  __device__ __forceinline__ QssaTemp(double d, double reciprocal) : t(d), r(reciprocal) {}
};
__device__ __forceinline__ double operator/(double n, const QssaTemp& d) {
  double q = n * d.r;
  q = fma(fma(-d.t, q, n), d.r, q);
  return __builtin_amdgcn_div_fixup(q, d.t, n);
}
__device__ __forceinline__ double operator/(const QssaTemp& n, double d) { return n.t / d; }

// The sums are taken here, where what they read is at hand: the compiler would
// move them behind the sub-steps and keep, or spill, every value read instead.
__device__ __forceinline__ void qssa_here(double& P, double& L) {
  asm volatile("" : "+v"(P), "+v"(L));
  coop_fence();
}

// One lane's cell: its place in the arrays and what every wave derives alike.
struct QssaCell {
  const StepParams& p;
  long long o;            // the cell's offset in a 3-d field
  int lane, itchim;
  bool inside;            // a lane behind the last cell computes that cell again and writes nothing
  int* fatal;             // per lane: a species of the cell reached 1e20
  int* nfatal;
  const double2* weight;  // per species: 1 / weight and pmar / weight
  QssaTemp temp;

  // gather (:161-195): Exner in REAL, R and pmar as REAL literals, the REAL
  // product 6.02e23*1e-15; J for FAST-TUV as for FAST-JX
  __device__ __forceinline__ double exner() const {
    return (double)((p.pp[o] + p.pi0[o]) / p.cp);
  }
  __device__ __forceinline__ void pressure(const CoopLds& s, int slot) const {
    const double press = pow(exner(), (double)p.cpor) * (double)p.p00;
    const double vapp = (double)p.rv[o];
    const double volmol = press / ((double)8.314f * temp.t);
    const double M = press * 7.243e16 / temp;
    s.put(slot, M);
    s.put(slot + 1, 29.0 * M * vapp / (18.0 + 11.0 * vapp));
    s.put(slot + 2, (double)(6.02e23f * 1e-15f) * volmol);
  }
  __device__ __forceinline__ double photolysis(int n) const { return p.jphoto[n + (long long)MECH_NPHOT * o]; }
  __device__ __forceinline__ float load(int n) const { return p.sc_p[n * p.n3d + o]; }
  __device__ __forceinline__ double gather(float x, double av, int n) const {
    return (double)x * av * (double)28.96f / QssaTemp((double)p.weight[n], weight[n].x);
  }

  // itchim sub-steps (qssa :392-406) of N species, v becoming the new
  // concentrations; true if one reached 1e20.  Per species: ybid = L if L > 0,
  // else 1 (cvmgm_dp); the explicit step y + delt (P - L y) when L = 0, else
  // the steady state P/ybid when ybid delt >= 10, else P/ybid + (y - P/ybid)
  // exp(-ybid delt) (cvmgp_dp, cvmgz_dp; qssa:406 overrides the explicit
  // choice of :404).  The branch is fixed for the call, and all three are one
  // sub-step v <- (v - a) e + c with per-species coefficients:
  //   exponential  a = c = P/ybid, e = exp(-ybid delt)
  //   steady       a = c = P/ybid, e = 0 (v starts at P/ybid)
  //   explicit     a = 0, e = 1, c = delt P
  // and itchim of them are (v - a) e^itchim + c, c being itchim delt P in the
  // explicit one: the power by repeated squaring takes a dozen products where
  // the sub-steps one by one take 150 operations, and it is nearer to the
  // exact recurrence, whose rounding a sub-step adds to v instead of to e.
  // The power stays above zero, so that an infinite v stays infinite.
  template <int N>
  __device__ __forceinline__ bool advance(double* v, const double* P, const double* L) const {
    const double delt = (double)(p.dtlt / (float)itchim);
    double a[N], e[N], c[N], b[N];
#pragma unroll
    for (int q = 0; q < N; ++q) {
      const double l = L[q];
      const double ybid = (-l < 0.0) ? l : 1.0;
      const double pr = P[q] / ybid;
      const double arg = ybid * delt;
      const double ex = exp(-arg);
      const bool still = l == 0.0, steady = !still && arg - 10.0 >= 0.0;
      a[q] = still ? 0.0 : pr;
      b[q] = still ? 1.0 : steady ? 0.0 : ex;
      c[q] = still ? (double)itchim * (delt * (P[q] - l * v[q])) : pr;
      v[q] = steady ? pr : v[q];
      e[q] = 1.0;
      if (q & 1) coop_fence();
    }
    for (int n = itchim;;) {
      if (n & 1) {
#pragma unroll
        for (int q = 0; q < N; ++q) e[q] *= b[q];
      }
      if (!(n >>= 1)) break;
#pragma unroll
      for (int q = 0; q < N; ++q) b[q] *= b[q];
    }
    bool reached = false;
#pragma unroll
    for (int q = 0; q < N; ++q) {
      double r = fma(v[q] - a[q], fmax(e[q], 2.2250738585072014e-308), c[q]);
      if (r < 0.0) r = 0.0;
      if (r >= 1.0e20) reached = true;
      v[q] = r;
    }
    return reached;
  }

  // whether the lane writes its cell; one wave counts the cells that reached 1e20
  __device__ __forceinline__ bool store(bool count) const {
    const bool stop = fatal[lane] != 0;
    if (count && stop && inside) atomicAdd(nfatal, 1);
    return inside && !stop;
  }
  // tendency of a species (:273-292)
  __device__ __forceinline__ void tendency(int n, float x, double y, double av) const {
    const double fxc = 1.0 / (av * weight[n].y);
    const long long a = n * p.n3d + o;
    p.sc_t[a] = (float)((double)p.sc_t[a] + (y * fxc - (double)x) * (double)(1.0f / p.dtlt));
  }
};

#include BRAMS_MECH_QSSA

// Two workgroups to a CU, four waves to a SIMD, where LDS holds both.
constexpr int kQssaLds = MECH_QSSA_SLOTS * 64 * (int)sizeof(double) + MECH_NS * (int)sizeof(double2) + 64 * (int)sizeof(int);
constexpr int kQssaWaves = 2 * kQssaLds <= 160 * 1024 ? 4 : 2;
static_assert(MECH_QSSA_SLOTS <= 320 && kQssaLds <= 160 * 1024, "the exchange fits a CU's LDS");
static_assert(MECH_QSSA_WAVES * 64 >= MECH_NS, "one thread per weight");

__global__ __launch_bounds__(MECH_QSSA_WAVES * 64, kQssaWaves) void qssa_cells(StepParams p, int itchim, long long ncell,
                                                                              long long first, int* nfatal) {
  __shared__ double lds[MECH_QSSA_SLOTS * 64];
  __shared__ double2 weight[MECH_NS];
  __shared__ int fatal[64];
  const int lane = threadIdx.x & 63;
  const long long c = first + (long long)blockIdx.x * 64 + lane;
  const long long g = c < ncell ? c : ncell - 1;
  const int k = 1 + (int)(g % p.nk);
  const long long t = g / p.nk;
  const int i = p.ia - 1 + (int)(t % p.ni);
  const int j = p.ja - 1 + (int)(t / p.ni);
  const long long o = k + (long long)p.m1 * (i + (long long)p.m2 * j);
  if (threadIdx.x < 64) fatal[lane] = 0;
  if (threadIdx.x < MECH_NS) {
    const double w = (double)p.weight[threadIdx.x];
    weight[threadIdx.x] = make_double2(1.0 / w, (double)28.96f / w);
  }
  const double exner = (double)((p.pp[o] + p.pi0[o]) / p.cp);
  const QssaCell q{p, o, lane, itchim, c < ncell, fatal, nfatal, weight, QssaTemp((double)p.theta[o] * exner)};
  const CoopLds s(lds + lane);
  qssa_program(coop_uniform((int)threadIdx.x >> 6), q, s);
}

hipError_t launch_qssa(const StepParams& p, int itchim, long long ncell, int* nfatal, hipStream_t st) {
  // a dispatch counts its work-items in 32 bits: at most 2^31 of them
  constexpr long long kCells = (1ll << 31) / (MECH_QSSA_WAVES * 64) * 64;
  for (long long first = 0; first < ncell; first += kCells) {
    const long long n = ncell - first < kCells ? ncell - first : kCells;
    hipLaunchKernelGGL(qssa_cells, dim3((unsigned)((n + 63) / 64)), dim3(MECH_QSSA_WAVES * 64), 0, st, p, itchim, ncell,
                       first, nfatal);
  }
  return hipGetLastError();
}

}  // namespace brams
