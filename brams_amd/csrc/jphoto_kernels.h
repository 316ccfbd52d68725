// Photolysis rates on the device: the FAST-TUV output mapping of tuvDriver
// (ModTuvDriver2.7.f90:1302-1332) and the mechanism's J relations
// (:1333-1368; RELACS: J14 and J16, mech_j_relations of the generated code).
//
// tuvDriver gathers TUV's j-values into valJLoc(ia:iz, ja:jz, kj, kz) (double,
// :1263) and writes, for every TUV reaction k with xRef(k) /= 0 in ascending
// k, jphoto(xRef(k), m+1, i, j) = valJLoc(i, j, k, m) for m = 1..m1-1 and
// jphoto(xRef(k), 1, i, j) = jphoto(xRef(k), 2, i, j), over the interior
// columns.  RELACS then sets, at every point of the array,
//   J14 = 0.962055 J13 + 0.0106247 J9      J16 = 12 J13 + 208 J15
// with the constants as REAL literals, without FMA contraction (other
// mechanisms have their own relations, or none).
//
// The host resolves xRef into src[n]: the last k that writes jphoto index n
// (later reactions overwrite earlier ones), -1 where none does (that entry
// keeps its value).
#pragma once
#include <hip/hip_runtime.h>

#include "mechanism.h"

namespace brams {

struct TuvMapParams {
  int m1, m2, m3, ia, iz, ja, jz;
  int kj, kz;
  const double* valj;            // (iz-ia+1, jz-ja+1, kj, kz), Fortran order
  double* jphoto;                // (MECH_NPHOT, m1, m2, m3)
  int src[MECH_NPHOT];           // TUV reaction (0-based) that writes index n, -1: none
};

// Workgroups are dealt to the eight XCDs in turn (workgroup w on XCD w % 8),
// each with its own L2.  Workgroup w takes tile (w % 8) * chunk + w / 8, so
// every XCD works through one contiguous run of tiles, and neighbouring tiles,
// which share 128-byte lines of both arrays, go through one L2.
constexpr int kXcds = 8;
__device__ __forceinline__ unsigned xcd_tile(unsigned w, unsigned chunk) { return (w % kXcds) * chunk + w / kXcds; }

// valJLoc has the column fastest, jphoto the rate and then the level, so the
// mapping is a transpose.  A tile is kTuvCols consecutive interior columns (i,
// then j, as valJLoc has them without gaps, so that a narrow interior fills
// its tiles too) times kTuvLevels levels, one thread a point: a wave reads two
// runs of 256 bytes of valJLoc, the relations apply in registers, and the rates go through LDS to
// be written in runs of kTuvLevels * MECH_NPHOT values (1088 bytes).  The odd
// row length keeps the LDS columns on different banks.  HBM bound: 200x200x40
// (453 MB) takes 116 us with its launch, 3.9 TB/s where a large copy reaches
// 4.65; with a thread writing its 136 bytes directly, which touched 64 lines
// with every load and store, 170 us.  40000 columns as 2x20000 (whose frame
// has as many) take 209 us, 249 with a thread a point and 443 with tiles that
// end with the row of i.
constexpr int kTuvCols = 32, kTuvLevels = 8, kTuvRow = kTuvLevels * MECH_NPHOT + (MECH_NPHOT * kTuvLevels % 2 == 0);

struct TuvTiles {
  unsigned lev, tiles, chunk;          // tiles along the levels, in all, per XCD
};

__device__ __forceinline__ void tuv_relations_at(double* jp) {
  double v[MECH_NPHOT];
#pragma unroll
  for (int n = 0; n < MECH_NPHOT; ++n) v[n] = jp[n];
  mech_j_relations(v);
#pragma unroll
  for (int n = 0; n < MECH_NPHOT; ++n) jp[n] = v[n];
}

// Interior columns: the mapping, then the relations (kXcds * chunk
// workgroups).  The workgroups after them take the other columns, a thread a
// point: the relations alone, the entries they do not set unchanged.
__global__ __launch_bounds__(256) void tuv_map(TuvMapParams p, TuvTiles q) {
  __shared__ double s[kTuvCols * kTuvRow];
  __shared__ long long at[kTuvCols];                 // a column's first value in the tile's levels
  const int ni = p.iz - p.ia + 1, nj = p.jz - p.ja + 1;
  const unsigned w = blockIdx.y * gridDim.x + blockIdx.x;
  if (w >= kXcds * q.chunk) {
    const long long t = (long long)(w - kXcds * q.chunk) * 256 + threadIdx.x;
    long long c = t / p.m1;                          // column of the frame, j rows from the bottom
    const long long below = (long long)(p.ja - 1) * p.m2, side = p.m2 - ni;
    if (c >= (long long)p.m2 * p.m3 - (long long)ni * nj) return;
    if (c >= below) {
      const long long r = c - below;                 // beside the interior's rows, then above them
      if (r < side * nj) {
        const long long i = r % side;
        c = (p.ja - 1 + r / side) * p.m2 + (i < p.ia - 1 ? i : i + ni);
      } else {
        c = (long long)p.jz * p.m2 + (r - side * nj);
      }
    }
    tuv_relations_at(p.jphoto + (long long)MECH_NPHOT * (t % p.m1 + p.m1 * c));
    return;
  }
  const unsigned tile = xcd_tile(w, q.chunk);
  if (tile >= q.tiles) return;
  const int L0 = (int)(tile % q.lev) * kTuvLevels;
  const unsigned cols = (unsigned)ni * (unsigned)nj, c0 = tile / q.lev * kTuvCols;
  const int nl = min(kTuvLevels, p.m1 - L0);
  const unsigned nc = min((unsigned)kTuvCols, cols - c0);
  const unsigned c = threadIdx.x % kTuvCols, l = threadIdx.x / kTuvCols;
  if (c < nc && (int)l < nl) {
    const unsigned jj = (c0 + c) / (unsigned)ni, ii = c0 + c - jj * (unsigned)ni;
    const long long first =
        MECH_NPHOT * (L0 + (long long)p.m1 * ((p.ia - 1 + (int)ii) + (long long)p.m2 * (p.ja - 1 + (int)jj)));
    if (l == 0) at[c] = first;
    const int mz = L0 + l == 0 ? 0 : L0 + (int)l - 1;   // level 1 repeats level 2
    double v[MECH_NPHOT];
#pragma unroll
    for (int n = 0; n < MECH_NPHOT; ++n) {
      const int k = p.src[n];
      v[n] = k >= 0 ? p.valj[c0 + c + (long long)cols * (k + (long long)p.kj * mz)] : p.jphoto[first + l * MECH_NPHOT + n];
    }
    mech_j_relations(v);
#pragma unroll
    for (int n = 0; n < MECH_NPHOT; ++n) s[c * kTuvRow + l * MECH_NPHOT + n] = v[n];
  }
  __syncthreads();
  const unsigned run = (unsigned)nl * MECH_NPHOT, all = run * nc;
  for (unsigned e = threadIdx.x; e < all; e += 256) {
    const unsigned ec = e / run, er = e - ec * run;
    p.jphoto[at[ec] + er] = s[ec * kTuvRow + er];
  }
}

}  // namespace brams
