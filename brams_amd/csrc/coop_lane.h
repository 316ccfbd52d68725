// Wave-level primitives of the cooperative block kernels (rodas3_coop.h).
#ifndef BRAMS_COOP_LANE_H
#define BRAMS_COOP_LANE_H
#include <hip/hip_runtime.h>

namespace brams {

// Workgroup barrier that orders LDS only: the waves exchange data through
// LDS alone, so global loads and stores in flight need no wait here.
__device__ __forceinline__ void coop_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// A lane's column of the LDS slots.  An LDS instruction reaches 64 KB from its
// address register, 128 slots, so the column has three of them.  They are
// kept opaque: told that they differ by constants, the compiler computes, and
// spills, an address for every slot instead.
typedef __attribute__((address_space(3))) double CoopLdsDouble;
struct CoopLds {
  CoopLdsDouble* base[3];
  __device__ __forceinline__ explicit CoopLds(double* column) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      base[k] = (CoopLdsDouble*)(column + k * 8192);
      asm volatile("" : "+v"(base[k]));
    }
  }
  // Volatile: a value that is read twice is meant to be read twice.  The
  // compiler would keep the first copy in a register (and spill it), and
  // would merge two reads into a ds_read2st64_b64, which moves 123 bytes a
  // clock where ds_read_b64 moves 184 (eight waves reading).
  __device__ __forceinline__ double get(int slot) const {
    return *(const volatile CoopLdsDouble*)&base[slot >> 7][(slot & 127) * 64];
  }
  __device__ __forceinline__ void put(int slot, double v) const { base[slot >> 7][(slot & 127) * 64] = v; }
};

// no instruction moves across this when the compiler schedules
__device__ __forceinline__ void coop_fence() { __builtin_amdgcn_sched_barrier(0); }

// v of a wave in which every lane has the same, in a scalar register
__device__ __forceinline__ int coop_uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Keeps what is computed from a wave-uniform v inside the loop: hoisted out, a
// test for every bit of the mask would fill the scalar registers.
__device__ __forceinline__ void coop_opaque(unsigned& v) {
  int s = coop_uniform((int)v);
  asm volatile("" : "+s"(s));
  v = (unsigned)s;
}

// 1 if v is nonzero (or NaN) in lane 0, else 0; the same in every lane
__device__ __forceinline__ unsigned coop_lane0_nonzero(double v) {
  return (unsigned)(__builtin_amdgcn_ballot_w64(v != 0.0) & 1ull);
}

__device__ __forceinline__ bool coop_any(bool c) { return __builtin_amdgcn_ballot_w64(c) != 0ull; }


template <int CTRL>
__device__ __forceinline__ double coop_dpp(double v) {
  union { double d; int i[2]; } a, b;
  a.d = v;
  b.i[0] = __builtin_amdgcn_update_dpp(a.i[0], a.i[0], CTRL, 0xf, 0xf, false);
  b.i[1] = __builtin_amdgcn_update_dpp(a.i[1], a.i[1], CTRL, 0xf, 0xf, false);
  return b.d;
}

// Largest v of the wave (NaNs left out, as fmax does), the same in every
// lane: four row shifts and two row broadcasts leave it in lane 63.
__device__ __forceinline__ double coop_wave_max(double v) {
  v = fmax(v, coop_dpp<0x111>(v));
  v = fmax(v, coop_dpp<0x112>(v));
  v = fmax(v, coop_dpp<0x114>(v));
  v = fmax(v, coop_dpp<0x118>(v));
  v = fmax(v, coop_dpp<0x142>(v));
  v = fmax(v, coop_dpp<0x143>(v));
  union { double d; int i[2]; } a;
  a.d = v;
  a.i[0] = __builtin_amdgcn_readlane(a.i[0], 63);
  a.i[1] = __builtin_amdgcn_readlane(a.i[1], 63);
  return a.d;
}

// base-2 logarithm and power at the rate of one instruction (about 1e-7)
__device__ __forceinline__ float coop_log2(float v) { return __builtin_amdgcn_logf(v); }
__device__ __forceinline__ float coop_exp2(float v) { return __builtin_amdgcn_exp2f(v); }

__device__ __forceinline__ int coop_wave_sum(int v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

}  // namespace brams
#endif
