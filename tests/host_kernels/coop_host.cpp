// Host emulation of the cooperative block kernels (rodas3_coop.h), for CPU
// tests: one thread for every lane of every wave, 64 lanes for a block of two
// halves and else two more than it has cells: the others shadow cell 1.  Barriers are barriers
// of the threads, the cross-lane operations go through shared arrays.
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

#include "hip/hip_runtime.h"

using std::fma;
using std::frexp;
using std::ldexp;
using std::fmaxf;
using std::fmin;
using std::isfinite;
using std::sqrt;
static int min(int a, int b) { return a < b ? a : b; }
#define __popc __builtin_popcount
#define __global__
#define __launch_bounds__(...)
#define __shared__ static
#define hipLaunchKernelGGL(...) ((void)0)

namespace {
struct Gate {                                   // reusable barrier of n threads
  std::mutex m;
  std::condition_variable c;
  int n = 0, at = 0;
  unsigned turn = 0;
  void wait() {
    std::unique_lock<std::mutex> l(m);
    const unsigned t = turn;
    if (++at == n) {
      at = 0;
      ++turn;
      c.notify_all();
    } else {
      c.wait(l, [&] { return turn != t; });
    }
  }
};
Gate g_group, g_wave[16];
double g_d[16][64];
int g_i[16][64], g_lanes = 1;
thread_local int t_wave, t_lane;
struct HostDim { int x; };
thread_local HostDim threadIdx, blockIdx;

template <class T, class F>
T across(T (*buf)[64], T v, F f) {              // f over the wave's lanes, the same result in each
  buf[t_wave][t_lane] = v;
  g_wave[t_wave].wait();
  T r = buf[t_wave][0];
  for (int l = 1; l < g_lanes; ++l) r = f(r, buf[t_wave][l]);
  g_wave[t_wave].wait();
  return r;
}
int atomicOr(int* p, int v) { return __atomic_fetch_or(p, v, __ATOMIC_SEQ_CST); }
}  // namespace

#define BRAMS_COOP_LANE_H
namespace brams {
struct CoopLds {
  double* column;
  explicit CoopLds(double* c) : column(c) {}
  double get(int slot) const { return column[slot * 64]; }
  void put(int slot, double v) const { column[slot * 64] = v; }
};
static void coop_fence() {}
static void coop_opaque(unsigned&) {}
static void coop_barrier() { g_group.wait(); }
static unsigned coop_lane0_nonzero(double v) {
  return (unsigned)across<int>(g_i, t_lane == 0 && v != 0.0, [](int a, int b) { return a | b; });
}
static bool coop_any(bool c) { return across<int>(g_i, c, [](int a, int b) { return a | b; }) != 0; }
static int coop_uniform(int v) { return v; }
static double coop_wave_max(double v) { return across<double>(g_d, v, [](double a, double b) { return fmax(a, b); }); }
static float coop_log2(float v) { return std::log2(v); }
static float coop_exp2(float v) { return std::exp2(v); }
static int coop_wave_sum(int v) { return across<int>(g_i, v, [](int a, int b) { return a + b; }); }
}  // namespace brams

#include "rodas3_coop.h"

using namespace brams;

// Every block of a grid with block_start[] of nblk + 1 entries, block 1 first
// (RODAS3: its mask).  counts: attempts, substeps, failed, thresh [nblk each],
// then order_thresh.  Blocks have 1..63 (one half) or 64 + 1..64 cells.
extern "C" void coop_step_host(int solver, int m1, int m2, int m3, float dtlt, int nblk, const int* block_start,
                               const float* pp, const float* pi0, const float* theta, const float* rv,
                               const double* jphoto, const float* weight, const int* transported, float* sc_p,
                               double* last_dt, const double* atol, const double* rtol, int* counts,
                               unsigned* mask) {
  std::vector<double> half((size_t)4 * MECH_NS * 64);
  StepParams p{};
  p.m1 = m1; p.m2 = m2; p.m3 = m3; p.ia = 2; p.iz = m2 - 1; p.ja = 2; p.jz = m3 - 1;
  p.nk = m1 - 2; p.ni = m2 - 2;
  p.dtlt = dtlt; p.ndyn = 1; p.split = 0;
  p.cp = 1004.0f; p.cpor = 1004.0f / 287.0f; p.p00 = 1.0e5f;
  p.pp = pp; p.pi0 = pi0; p.theta = theta; p.rv = rv; p.jphoto = jphoto;
  p.weight = weight; p.transported = transported; p.sc_p = sc_p;
  p.n3d = (long long)m1 * m2 * m3;
  p.block_start = block_start;
  p.last_dt = last_dt;
  p.atol = atol; p.rtol = rtol;
  p.mask = mask;
  p.blk_attempts = counts; p.blk_substeps = counts + nblk; p.blk_failed = counts + 2 * nblk;
  p.blk_thresh = counts + 3 * nblk; p.order_thresh = counts + 4 * nblk;
  p.half_y = half.data();
  for (int b = 0; b < nblk; ++b) {
    const int n = block_start[b + 1] - block_start[b];
    g_lanes = n + 2 < 64 ? n + 2 : 64;
    g_group.n = g_lanes * MECH_COOP_WAVES;
    std::vector<std::thread> th;
    for (int w = 0; w < MECH_COOP_WAVES; ++w) {
      g_wave[w].n = g_lanes;
      for (int l = 0; l < g_lanes; ++l)
        th.emplace_back([&, w, l] {
          t_wave = w;
          t_lane = l;
          threadIdx.x = 64 * w + l;
          if (solver == kRos2)
            coop_block<kRos2, false, true>(p, b, 0);
          else if (b == 0)
            coop_block<kRodas3, true, true>(p, b, 0);
          else if (n > 64)
            coop_block<kRodas3, false, true>(p, b, 0);
          else
            coop_block<kRodas3, false, false>(p, b, 0);
        });
    }
    for (auto& t : th) t.join();
  }
}
