// force_tile.h -- what the list and the tile force kernels share: the sums of
// one particle and the end of its force evaluation.
#pragma once

#include "records.h"
#include "tile.h"

enum { FFL_LIST = 2, FFL_DTC = 32 };

// particle i as its pair terms and their end use it (force.F90:2172-2514)
struct ForceI {
  double h, h1, rho, rho1, pr, cs, vwave, en;
  double Bx, By, Bz, psi;  // MHD
  double eps, ts;          // dust
};
// its sums over the pairs (force.F90:1227-2056)
struct ForceSums {
  double fx, fy, fz, drhodt, dudtdiss, dendtdiss, vsigmax;
  double divBsym, dBx, dBy, dBz, divBdiff;     // MHD
  double ddust, dudtdust, dvx, dvy, dvz;       // dust
  int ibin_neigh;                              // largest bin of a neighbour
};

// finish_cell_and_store_results (force.F90:2649-3330) for particle o of the
// caller; dtc, dtf and bmax for the global reductions
template <bool MHD, bool DUST, bool THERMAL>
__device__ __forceinline__ void force_store(const DevConst &dc, const ForceIOArgs &out, int o, const ForceI &I,
                                            ForceSums S, int icall, double &dtc_o, double &dtf_o, int &bmax,
                                            int32_t *__restrict__ flags) {
  if (MHD) {
    const double B2i = I.Bx * I.Bx + I.By * I.By + I.Bz * I.Bz;
    double frac = 0.;
    if (B2i > 0.) {
      const double betai = 2. * I.pr / B2i;
      frac = (betai < 2.) ? 1. : (betai < 10.) ? (10. - betai) * 0.125 : 0.;
    }
    S.fx = S.fx - I.Bx * S.divBsym * frac;
    S.fy = S.fy - I.By * S.divBsym * frac;
    S.fz = S.fz - I.Bz * S.divBsym * frac;
    if (out.divBsymm) out.divBsymm[o] = (float)(I.rho * S.divBsym);
  }
  const double f2i = S.fx * S.fx + S.fy * S.fy + S.fz * S.fz;
  double *fo = out.fxyzu + (size_t)o * out.ldf;
  fo[0] = S.fx; fo[1] = S.fy; fo[2] = S.fz;
  const double drhodti = dc.pmass * S.drhodt;
  const double divvi = -drhodti * I.rho1;
  out.divcurlv[(size_t)o * out.lddcv] = (float)divvi;
  double dtc = dc.dtmax, dtf = PH_BIGNUMBER, dtclean = PH_BIGNUMBER, dtdusti = PH_BIGNUMBER;
  double fxyz4 = 0.;
  if (THERMAL) {
    const double rhogasi = DUST ? I.rho * (1. - I.eps) : I.rho;
    const double fac = (rhogasi > PH_TINY64) ? I.rho / rhogasi : 0.;
    const double pdv_work = fac * I.pr * I.rho1 * I.rho1 * drhodti;
    if (dc.ipdv_heating > 0) fxyz4 += pdv_work;
    if (dc.ishock_heating > 0) fxyz4 += fac * S.dudtdiss;
    fxyz4 += fac * S.dendtdiss;
    if (DUST) fxyz4 += 0.5 * fac * I.rho1 * S.dudtdust;
  }
  if (MHD) {
    double *dB = out.dBevol + (size_t)o * 4;
    dB[0] = S.dBx; dB[1] = S.dBy; dB[2] = S.dBz;
    if (dc.psidecayfac > 0.) {
      const double vclean = dc.overcleanfac * I.vwave;
      const double dtau = dc.psidecayfac * vclean * I.h1;
      dB[3] = -vclean * S.divBdiff * I.rho1 - I.psi * dtau - 0.5 * I.psi * divvi;
      dtclean = dc.C_cour * I.h / (vclean + PH_TINY64);
    }
  }
  if (DUST) {
    const double om = 1. - I.eps;
    out.ddustevol[o] = 0.5 * (S.ddust * I.rho1 / (om * om));
    out.deltav[(size_t)o * 3 + 0] = S.dvx;
    out.deltav[(size_t)o * 3 + 1] = S.dvy;
    out.deltav[(size_t)o * 3 + 2] = S.dvz;
    if (out.tstop) out.tstop[o] = I.ts;
    if (I.eps > 0. && I.cs > 0. && I.eps > PH_EPS64) {
      const double tseff = (1. - I.eps) / I.eps * (I.eps * I.ts);
      const double den = I.eps * tseff * I.cs * I.cs;
      if (den > PH_TINY64) dtdusti = dc.C_force * I.h * I.h / den;
    }
  }
  const double vsigdtc = fmax(S.vsigmax, I.vwave);
  if (vsigdtc > PH_TINY64) dtc = dc.C_cour * I.h / (vsigdtc * fmax(dc.alpha, 1.0));
  if (THERMAL) {
    if (I.en + dtc * fxyz4 < PH_EPS64 && I.en > PH_EPS64) fxyz4 = fxyz4 / (1. - dtc * fxyz4 / I.en);
    fo[3] = fxyz4;
  }
  if (fabs(f2i) > PH_EPS64) dtf = dc.C_force * sqrt(I.h / sqrt(f2i));
  if (!(dtc > PH_TINY64) || !(dtc < PH_HUGE64)) atomicOr(flags, FFL_DTC);
  dtc_o = dtc;
  dtf_o = fmin(fmin(dtf, dtdusti), dtclean);
  if (out.ibin) {
    // force.F90:3272-3310: the particle's own timestep and its new bin
    double dti = dtc;
    const double dtitmp = fmin(fmin(dtf, dtclean), dtdusti);
    if (dtitmp < dti + PH_TINY64 && dtitmp < dc.dtmax) dti = dtitmp;
    int b = get_newbin_d(dti, dc.dtmax, (int)out.ibin[o], icall < 2, out.nbinmax, out.istepfrac);
    b = max(b, S.ibin_neigh - 1);  // Saitoh-Makino limiter
    out.ibin[o] = (int8_t)b;
    bmax = b;
    dtc_o = PH_HUGE64;
    dtf_o = PH_HUGE64;
  }
}

struct ForceTileIn {
  const FRec *rec;
  const FRecB *recB;
  const FRecD *recD;
  const FRec32 *rec32;
  const double4 *fpos, *fvel;
};
void launch_force_tile(phsph_ctx *c, int icall, const ForceIOArgs &a, const TileLists &tl, const ForceTileIn &in,
                       bool mixed, bool mhd, bool dust, const int32_t *skip);
