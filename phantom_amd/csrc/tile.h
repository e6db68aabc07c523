// tile.h -- a group's candidate particles staged once in LDS and shared by
// the wavefronts of one workgroup ("tile").
//
// The per-lane neighbour lists send every lane to its own cache line for
// every 16 bytes of every neighbour.  The texture-address unit takes one
// line per clock, so such a gather costs about 60 clocks of a whole CU per
// 16-byte load of one wavefront (measured: records of 16, 32, 64 and 128
// bytes gathered per lane take 139, 202, 306 and 551 clocks per wavefront),
// and it set the pace of the density and force pair loops.  64 neighbouring
// particles share about 400 (cubic) to 600 (quintic) candidate particles:
// staged in LDS once per group, the same reads are LDS reads of 128 bytes
// per clock.
//
// A tile is one workgroup for the active particles of one tree node of at most
// 64 or 80 particles (the highest such node of its branch), so that its
// particles are close together whatever the size of the set: 64 consecutive
// particles straddle nodes where leaves hold other than 8, and shared 950
// candidates on the average instead of 430 on the shock tube and the
// polytropes.  A wavefront takes 16 particles with four lanes per particle,
// so the list of a particle is summed by four lanes and no lane waits for a
// long list alone.
#pragma once

#include "stream.h"

constexpr int TILE_P = 16;  // particles per wavefront, TILE_L lanes each
constexpr int TILE_L = 4;
// Tiles of nodes of up to 64 particles have four wavefronts, of up to 80 five;
// TILE_BIG has the whole LDS of a CU for the groups that do not fit these.
enum { TILE_4 = 0, TILE_5 = 1, TILE_BIG = 2 };
// Limits of a tile by kernel: candidate particles of the group (NC) and list
// entries of a particle (LC, a multiple of 4).  A node of 64 particles of a
// uniform set needs 430 and 73 (cubic, search radius 1.03 R h) or 630 and 123
// (quintic).  The limits let the LDS of a CU hold 16 (cubic, TILE_4), 15
// (cubic, TILE_5), 12 (quintic, TILE_4) and 10 (quintic, TILE_5) wavefronts.
// TILE_BIG has two wavefronts that take 16 particles after 16 and keeps its
// lists in LDS only; what does not fit that goes to the list kernels.
template <int K, int V>
struct TileCap {
  static constexpr bool CU = K == PHSPH_KERNEL_CUBIC, BIG = V == TILE_BIG;
  static constexpr int W = BIG ? 2 : V == TILE_5 ? 5 : 4;
  static constexpr int NC = BIG ? 2560 : V == TILE_5 ? (CU ? 880 : 1280) : (CU ? 672 : 800);
  static constexpr int LC = BIG ? 1024 : CU ? 96 : 160;
  static constexpr int WPE = BIG ? 1 : V == TILE_5 ? (CU ? 3 : 2) : (CU ? 4 : 3);
};
constexpr int GBOX = 8;                  // doubles per group: bounding box, largest search h

// exchange within the four lanes of a particle
template <int CTRL>
__device__ __forceinline__ double dpp_quad(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
template <int CTRL>
__device__ __forceinline__ int dpp_quad_i(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
constexpr int DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E;  // quad_perm 1,0,3,2 and 2,3,0,1
// the four lanes add the same two pairs, so all four hold the same bits
__device__ __forceinline__ double quad_sum(double v) {
  v += dpp_quad<DPP_XOR1>(v);
  return v + dpp_quad<DPP_XOR2>(v);
}
__device__ __forceinline__ double quad_max(double v) {
  v = fmax(v, dpp_quad<DPP_XOR1>(v));
  return fmax(v, dpp_quad<DPP_XOR2>(v));
}
__device__ __forceinline__ int quad_sum_i(int v) {
  v += dpp_quad_i<DPP_XOR1>(v);
  return v + dpp_quad_i<DPP_XOR2>(v);
}
__device__ __forceinline__ int quad_max_i(int v) {
  v = max(v, dpp_quad_i<DPP_XOR1>(v));
  return max(v, dpp_quad_i<DPP_XOR2>(v));
}
