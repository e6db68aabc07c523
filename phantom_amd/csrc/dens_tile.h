// dens_tile.h -- what the density list kernels and the tile kernels share.
#pragma once

#include "tile.h"

enum { DFL_CAND = 1, DFL_LIST = 2, DFL_REWALK = 4, DFL_NOCONV = 8, DFL_NEGH = 16, DFL_STACK = 32, DFL_TILE = 64 };

// outputs of the search and h iteration, by active slot (t_), tree position
// (p_, retry, htraj, hconv) and leaf
struct DensIterOut {
  uint32_t *nlist;  // list_at layout, capl entries per slot
  int capl;
  int32_t *t_nl, *t_nlj;
  double *t_hsum, *t_hfin;
  int32_t *p_nits, *leaf_nits, *retry, *nrewalk;
  double *htraj;
  size_t hstride;
  double *hconv;
  int32_t *big, *nbig;  // groups that need the large tile
};

// The kernels in the form w = sum_k c_k max(k - q, 0)^n (kernel_cubic.f90:34-60:
// (2-q)^3/4 - (1-q)^3; kernel_quintic.f90:34-75: (3-q)^5 - 6 (2-q)^5 +
// 15 (1-q)^5), which needs no branches.  With q = k - (k - q) the two sums of
// the h iteration, sum w and -sum (q w' + 3 w), are sums of two powers of each
// term, so a neighbour costs 8 (cubic) or 15 (quintic) instructions; the terms
// are scaled to 0..1 so that the lower bound is the instruction's clamp.
template <int K>
struct IterSums {
  static constexpr int NT = (K == PHSPH_KERNEL_CUBIC) ? 2 : 3;
  double lo[NT], hi[NT];
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int k = 0; k < NT; k++) lo[k] = hi[k] = 0.;
  }
  __device__ __forceinline__ void add(double r, const double (&mh)[NT]) {
#pragma unroll
    for (int k = 0; k < NT; k++) {
      const double a = fmin(fmax(fma(r, mh[k], 1.), 0.), 1.);
      const double a2 = a * a;
      if (K == PHSPH_KERNEL_CUBIC) {
        lo[k] += a2;
        hi[k] = fma(a2, a, hi[k]);
      } else {
        const double a4 = a2 * a2;
        lo[k] += a4;
        hi[k] = fma(a4, a, hi[k]);
      }
    }
  }
  // -1/(k h): the term's slope in r
  static __device__ __forceinline__ void slopes(double h1, double (&mh)[NT]) {
    if (K == PHSPH_KERNEL_CUBIC) {
      mh[0] = -0.5 * h1;
      mh[1] = -h1;
    } else {
      mh[0] = -h1 * (1. / 3.);
      mh[1] = -0.5 * h1;
      mh[2] = -h1;
    }
  }
  __device__ __forceinline__ void result(double &srho, double &sgh) const {
    if (K == PHSPH_KERNEL_CUBIC) {
      srho = 2. * hi[0] - hi[1];
      sgh = 6. * lo[0] - 12. * hi[0] - 3. * lo[1] + 6. * hi[1];
    } else {
      srho = 243. * hi[0] - 192. * hi[1] + 15. * hi[2];
      sgh = 1215. * lo[0] - 1944. * hi[0] - 960. * lo[1] + 1536. * hi[1] + 75. * lo[2] - 120. * hi[2];
    }
  }
};

// sqrt of a squared separation: reciprocal square root estimate and one
// coupled Newton step for the root and its half reciprocal, then the residual
// (to about one unit in the last place; zero and denormal squares give about
// 1e-145, far below any h)
__device__ __forceinline__ double sqrt_sep(double r2) {
  const double a = fmax(r2, 1e-290);
  const double y = __builtin_amdgcn_rsq(a);
  double g = a * y, h = 0.5 * y;
  const double e = fma(-h, g, 0.5);
  g = fma(g, e, g);
  h = fma(h, e, h);
  const double d = fma(-g, g, a);
  return fma(d, h, g);
}

void launch_dens_tile(phsph_ctx *c, int icall, double rfac, double lmargin, const double *hmax0,
                      const DensIterOut &out);
int dens_tile_list_cap(const phsph_ctx *c);
