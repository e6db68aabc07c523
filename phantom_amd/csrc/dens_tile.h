// dens_tile.h -- what the density list kernels and the tile kernels share.
#pragma once

#include "tile.h"

enum { DFL_CAND = 1, DFL_LIST = 2, DFL_REWALK = 4, DFL_NOCONV = 8, DFL_NEGH = 16, DFL_STACK = 32, DFL_TILE = 64,
       DFL_STACK_LO = 128 };
// c->counters: particles that outgrew their lists (tiles), groups that are no
// tiles (tile_unfit), and of one group in UNEVEN_STEP those whose largest h is
// more than 1.3 and more than 1.5 times the smallest
constexpr int CNT_REWALK = 8, CNT_UNFIT = 9, CNT_UNEVEN = 10, CNT_WALK = 12;  // CNT_WALK: words of a walk
constexpr int UNEVEN_STEP = 8;

struct DensIn {
  const double4 *tp;  // x, y, z (treecache) and h at entry
  const double4 *tv;  // vx, vy, vz
  const double4 *tf;  // fxyzu + fext (null: zero)
  const double4 *tB;  // Bevol x, y, z and rho(h at entry) (MHD)
};
struct DensOut {
  double *xyzh;  int ldx;
  float *divcurlv; int lddcv;
  float *divcurlB;
  float *alphaind;
  float *gradh; int ldgradh;
  float *dvdx;
};

// store_results (dens.F90:1511-1681) at the final h from the sums taken at
// the h of the last iteration
template <bool MHD>
__device__ __forceinline__ void dens_store(const DevConst &dc, int p, double hfin, double rs_rho, double rs_gh,
                                           double rs_gs, double rs_divv, double rs_divB, const double *dv,
                                           const double *da, const double *rr, const double *curlB,
                                           const int32_t *__restrict__ iparts, double *__restrict__ th_out,
                                           const DensOut &out, int32_t *__restrict__ p_nneigh, int nneigh,
                                           int32_t *__restrict__ flags) {
  const double pm = dc.pmass;
  const double hf1 = 1. / hfin, hf21 = hf1 * hf1, hf31 = hf1 * hf21, hf41 = hf21 * hf21;
  const double rhoi = dc.cnormk * (rs_rho + dc.wab0 * pm) * hf31;
  const double gradhs = dc.cnormk * (rs_gh + dc.gradh0 * pm) * hf41;
  const double dhdrhoi = -hfin / (3. * rhoh_d(hfin, dc.hfact, pm));
  const double omegai = 1. - dhdrhoi * gradhs;
  const double gradhi = 1. / omegai;
  const double gradsofti = ((rs_gs + dc.dphidh0 * pm) * hf21) * dhdrhoi;
  const double hnew = hrho_d(rhoi, dc.hfact, pm);
  if (hnew < 0.) atomicOr(flags, DFL_NEGH);
  const int o = abs(iparts[p]) - 1;
  out.xyzh[(size_t)o * out.ldx + 3] = hnew;
  th_out[p] = hnew;
  const float gh32 = (float)gradhi;
  out.gradh[(size_t)o * out.ldgradh] = gh32;
  if (dc.gravity && out.ldgradh > 1) out.gradh[(size_t)o * out.ldgradh + 1] = (float)gradsofti;
  const double rho1i = 1. / rhoi;
  const double term = dc.cnormk * (double)gh32 * rho1i * hf41;
  out.divcurlv[(size_t)o * out.lddcv] = (float)(-rs_divv * term);
  // exact-linear gradients (dens.F90:866-967, 997-1052, 1086-1101)
  const double rxx = rr[0], rxy = rr[1], rxz = rr[2], ryy = rr[3], ryz = rr[4], rzz = rr[5];
  const double denom = rxx * ryy * rzz + 2. * rxy * rxz * ryz - rxx * ryz * ryz - ryy * rxz * rxz - rzz * rxy * rxy;
  const double rm0 = ryy * rzz - ryz * ryz, rm1 = rxz * ryz - rzz * rxy, rm2 = rxy * ryz - rxz * ryy;
  const double rm3 = rzz * rxx - rxz * rxz, rm4 = rxy * rxz - rxx * ryz, rm5 = rxx * ryy - rxy * rxy;
  double gv[9], div_a;
  if (fabs(denom) > PH_TINY64) {
    const double dd = 1. / denom;
    for (int cpt = 0; cpt < 3; cpt++) {
      const double ax = dv[3 * cpt], ay = dv[3 * cpt + 1], az = dv[3 * cpt + 2];
      gv[3 * cpt] = -((ax * rm0 + ay * rm1 + az * rm2) * dd);
      gv[3 * cpt + 1] = -((ax * rm1 + ay * rm3 + az * rm4) * dd);
      gv[3 * cpt + 2] = -((ax * rm2 + ay * rm4 + az * rm5) * dd);
    }
    const double gax = (da[0] * rm0 + da[1] * rm1 + da[2] * rm2) * dd;
    const double gay = (da[3] * rm1 + da[4] * rm3 + da[5] * rm4) * dd;
    const double gaz = (da[6] * rm2 + da[7] * rm4 + da[8] * rm5) * dd;
    div_a = -(gax + gay + gaz);
  } else {
    for (int k = 0; k < 9; k++) gv[k] = -dv[k] * term;
    div_a = -term * (da[0] + da[4] + da[8]);
  }
  const double d5 = div_a - (gv[0] * gv[0] + gv[4] * gv[4] + gv[8] * gv[8] +
                             2. * (gv[1] * gv[3] + gv[2] * gv[6] + gv[5] * gv[7]));
  if (out.alphaind) out.alphaind[(size_t)o * 3 + 2] = (float)d5;
  if (out.dvdx)
    for (int k = 0; k < 9; k++) out.dvdx[(size_t)o * 9 + k] = (float)gv[k];
  if (MHD && out.divcurlB) {
    out.divcurlB[(size_t)o * 4 + 0] = (float)(-rs_divB * term);
    out.divcurlB[(size_t)o * 4 + 1] = (float)(-curlB[0] * term);
    out.divcurlB[(size_t)o * 4 + 2] = (float)(-curlB[1] * term);
    out.divcurlB[(size_t)o * 4 + 3] = (float)(-curlB[2] * term);
  }
  p_nneigh[p] = nneigh;
}

// outputs of the search and h iteration, by active slot (t_), tree position
// (p_, retry, htraj, hconv) and leaf
struct DensIterOut {
  int32_t *t_nl;
  double *t_hsum, *t_hfin;
  int32_t *p_nits, *leaf_nits, *retry, *nrewalk;
  double *htraj;
  size_t hstride;
  double *hconv;
  double2 *t_sums;  // sum of w m and of -(q w' + 3 w) m at the last iteration
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

void launch_dens_tile(phsph_ctx *c, int icall, double rfac, double lmargin, const double *hmax0,
                      const DensIterOut &out, const TileLists &tl);
void launch_dens_sums(phsph_ctx *c, const TileLists &tl, bool mhd, bool mixed, const DensIn &in, const DensOut &out);
size_t tile_list_bytes(const phsph_ctx *c);
