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
// Of five wavefronts two share a SIMD, so that its registers allow half as many
// workgroups as wavefronts: two with the cubic (109 registers) and one with the
// quintic kernel (145; 1.2 wavefronts per SIMD measured, 3.0 with TILE_4).
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
// adds the periodic offset of a separation code to a position (get_sep,
// kdtree.F90:1468-1501)
__device__ __forceinline__ void offset_pos(const DevConst &dc, int code, double &x, double &y, double &z) {
  if (code == SEP_PLAIN) return;
  int sx, sy, sz;
  off_decode(code, sx, sy, sz);
  if (sx) x = xadd(x, copysign(dc.dxbound, (double)sx));
  if (sy) y = xadd(y, copysign(dc.dybound, (double)sy));
  if (sz) z = xadd(z, copysign(dc.dzbound, (double)sz));
}

// A group whose box (half extents e) is too large beside the periodic box for
// one offset per leaf (dens_tile.hip), or beside its own search radius for FP32
// squares: rl is the search radius in units of h, hm the group's largest h, hmx
// that of its candidates too, smax the largest of their leaves' sizes.
__device__ __forceinline__ bool tile_unfit(const DevConst &dc, double ex, double ey, double ez, double rl, double hm,
                                           double hmx, double smax) {
  bool bad = !(ex + ey + ez + rl * hmx < 1e15 * (rl * hm));
  if (dc.periodic) {
    const double need = (rl * hmx + 3. * smax) * (1. + 1e-9);
    bad = bad || ex + need >= dc.hdlx || ey + need >= dc.hdly || ez + need >= dc.hdlz;
  }
  return bad;
}

// The lists that the density tile kernel leaves for the sums and for the force
// pass: the candidates of each group (tree position and offset code) and, per
// 16 particles (one wavefront), the entries of their lists as 16-bit slots of
// the group's candidates, entry k of the 16 particles in 32 consecutive bytes.
// Groups in the large form have arrays of their own, by position in big.
struct TileLists {
  const int32_t *gt;  // group ranges of the active list
  uint32_t *cand;     // ncap per group
  uint16_t *list;     // lw wavefronts of lc entries per group
  int32_t *nc;        // candidates per group; -1: large form, or handed back
  int ncap, lc, lw;
  int32_t *big, *nbig;  // groups in the large form
  uint32_t *bcand;
  uint16_t *blist;
  int32_t *bnc;
  int bncap, blc, bcap;  // bcap: groups the arrays hold (more are handed back)
};
constexpr int TILE_BW = 5;  // wavefronts of 16 particles of a group in the large form

// the group of a workgroup of a launch over all groups and the large ones
struct TileGroup {
  int g, t0, t1, nc, lc;
  const uint32_t *cand;
  const uint16_t *list;
  __device__ __forceinline__ bool find(const TileLists &tl, int ngroups) {
    const int ngr = (ngroups + 7) / 8 * 8;  // blocks of the ordinary groups
    if ((int)blockIdx.x < ngr) {
      g = xcd_block(blockIdx.x, ngr);
      if (g >= ngroups) return false;
      nc = tl.nc[g];
      lc = tl.lc;
      cand = tl.cand + (size_t)g * tl.ncap;
      list = tl.list + (size_t)g * tl.lw * tl.lc * TILE_P;
    } else {
      const int b = blockIdx.x - ngr;
      if (b >= *tl.nbig) return false;
      g = tl.big[b];
      nc = tl.bnc[b];
      lc = tl.blc;
      cand = tl.bcand + (size_t)b * tl.bncap;
      list = tl.blist + (size_t)b * TILE_BW * tl.blc * TILE_P;
    }
    t0 = tl.gt[g];
    t1 = tl.gt[g + 1];
    return nc >= 0 && t0 < t1;
  }
};
// the list buffers for the context's tile groups (dens_tile.hip)
int tile_lists(phsph_ctx *c, TileLists &tl);
static inline unsigned tile_grid(int ngroups, const TileLists &tl) { return xcd_grid(ngroups) + (unsigned)tl.bcap; }

// r and 1/(r + eps) of a squared separation, from a reciprocal square root
// estimate: one coupled Newton step for the root and its half reciprocal, the
// residual of the root, and one step for the reciprocal (each to about one unit
// in the last place; zero and denormal squares give about 1e-145, far below
// any h).  From 1/r that step leaves (eps/r)^2, so below 1e8 eps it starts from
// an estimate of 1/(r + eps).
__device__ __forceinline__ void sqrt_rsqrt_sep(double r2, double eps, double &r, double &r1) {
  const double a = fmax(r2, 1e-290);
  const double y = __builtin_amdgcn_rsq(a);
  double g = a * y, h = 0.5 * y;
  const double e = fma(-h, g, 0.5);
  g = fma(g, e, g);
  h = fma(h, e, h);
  const double d = fma(-g, g, a);
  r = fma(d, h, g);
  h = h + h;
  const double b = r + eps;
  if (eps > 0. && r < 1e8 * eps) {
    h = __builtin_amdgcn_rcp(b);
    h = fma(h, fma(-b, h, 1.), h);
  }
  const double e1 = fma(-b, h, 1.);
  r1 = fma(h, e1, h);
}

// 1/sqrt(x) for x >= 0 (below 1e-290: about 1e145), to about one unit in the
// last place
__device__ __forceinline__ double rsqrt_pos(double x) {
  const double a = fmax(x, 1e-290);
  const double y = __builtin_amdgcn_rsq(a);
  double g = a * y, h = 0.5 * y;
  const double e = fma(-h, g, 0.5);
  g = fma(g, e, g);
  h = fma(h, e, h);
  h = h + h;
  const double e1 = fma(-g, h, 1.);
  return fma(h, 0.5 * e1, h);
}

// dw/dq without branches: sums of max(k - q, 0)^n (kernel_cubic.f90:34-60,
// kernel_quintic.f90:34-75)
template <int K>
__device__ __forceinline__ double kern_grad(double q) {
  if (K == PHSPH_KERNEL_CUBIC) {
    const double a = fmax(2. - q, 0.), b = fmax(1. - q, 0.);
    return fma(-0.75 * a, a, 3. * (b * b));
  } else {
    const double a = fmax(3. - q, 0.), b = fmax(2. - q, 0.), c = fmax(1. - q, 0.);
    const double a2 = a * a, b2 = b * b, c2 = c * c;
    return fma(-5. * a2, a2, fma(30. * b2, b2, -75. * (c2 * c2)));
  }
}

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

template <int CTRL, class OP>
__device__ __forceinline__ double dpp_op(double v, OP op) { return op(v, dpp_quad<CTRL>(v)); }
// a reduction over the wavefront, the result in every lane
template <class OP>
__device__ __forceinline__ double wave_all(double v, OP op) {
  v = dpp_op<DPP_XOR1>(v, op);
  v = dpp_op<DPP_XOR2>(v, op);
  v = dpp_op<0x141>(v, op);  // row_half_mirror
  v = dpp_op<0x140>(v, op);  // row_mirror
  v = op(v, __shfl_xor(v, 16, 64));
  return op(v, __shfl_xor(v, 32, 64));
}
struct OpAdd { __device__ __forceinline__ double operator()(double a, double b) const { return a + b; } };
struct OpMin { __device__ __forceinline__ double operator()(double a, double b) const { return fmin(a, b); } };
struct OpMax { __device__ __forceinline__ double operator()(double a, double b) const { return fmax(a, b); } };
