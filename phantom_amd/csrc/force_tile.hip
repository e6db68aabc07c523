// force_tile.hip -- the force pair loop of dense active sets over the lists
// that the density tile kernel left (tile.h): the pair terms of k_force and
// k_force_mixed (force.hip) with the candidates' records in LDS.
#include "force_tile.h"

// Record of a candidate in LDS, 16 bytes at a time:
//   x y | z 1/h | vx vy | vz u | c/h^4 gradh, 1/rho | P, P/rho^2 | v_wave, alpha v_wave
//   and with MHD Bx By | Bz psi, with dust eps sqrt(eps/(1-eps)) | t_s (1-eps)
// (mixed precision: the FP32 1/rho and rho share a word, P and P/rho^2 are the
// sums of their FP32 pairs).
template <bool MHD, bool DUST>
struct ForceCap {
  static constexpr int NP = 7 + (MHD ? 2 : 0) + (DUST ? 2 : 0);  // 16-byte pieces
  static constexpr int PB = 7, PD = MHD ? 9 : 7;                 // first MHD and dust piece
  static constexpr int NC = (MHD && DUST) ? 448 : (MHD || DUST) ? 544 : 464;  // candidates staged at a time
  static constexpr int WPE = (MHD || DUST) ? 2 : 3;  // wavefronts per SIMD that LDS and registers hold
};

// One workgroup per group as in k_dens_tile, four lanes per particle, the
// candidates staged in chunks of equal length (k_dens_sums).  A pair reads 112
// bytes (MHD + dust 176) from LDS instead of eight (thirteen) 16-byte loads
// whose 64 lanes go to 64 cache lines each.  FP64 records are staged by eight
// lanes each, one 128-byte line per record and load.
// Wavefronts wait 60 to 70 % of their time (the records of a chunk and the
// barriers around them) at two to three a SIMD; FP64 vector instructions take
// 42 to 58 % of the issue cycles.  8M-particle box 4.7 ms (8.1
// ms as a list kernel, which its gathers bound), 2M particles with MHD and
// dust 5.1 ms (8.2), 1M quintic 2.6 ms (3.35), 850k mixed 0.66 ms (0.92; the
// mixed form reads its FP32 records into FP64 ones and is no faster than FP64).
template <int K, int W, bool MHD, bool DUST, bool THERMAL, bool MIXED>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu((ForceCap<MHD, DUST>::WPE))))
k_force_tile(DevConst dc, int ngroups, const int32_t *__restrict__ act, TileLists tl, const int32_t *__restrict__ t_nl,
             const int32_t *__restrict__ skip, const int32_t *__restrict__ iparts, ForceTileIn in, ForceIOArgs out,
             const int8_t *__restrict__ tbin_old, int icall, unsigned long long *__restrict__ dtred,
             int32_t *__restrict__ flags) {
  using Cap = ForceCap<MHD, DUST>;
  constexpr int NP = Cap::NP, NC = Cap::NC;
  __shared__ double2 rec[NC * NP];
  TileGroup G;
  if (!G.find(tl, ngroups)) return;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int pi = lane / TILE_L, sl = lane % TILE_L;
  const int t = G.t0 + w * TILE_P + pi;
  const int pt = (t < G.t1) ? act[t] : -1;
  const bool live = pt >= 0 && !(skip && skip[pt]);
  const int p = live ? pt : act[G.t0];
  const double pm = dc.pmass, R2 = dc.radkern2;
  const FRec Ri = in.rec[p];
  const double xi = Ri.x, yi = Ri.y, zi = Ri.z;
  ForceI I;
  I.h = Ri.h;
  // rhoanddhdrho (part.F90:805-816)
  I.h1 = 1. / fabs(I.h);
  const double tt = dc.hfact * I.h1;
  I.rho = pm * (tt * tt * tt);
  const double rhoi = I.rho, rho1i = 1. / rhoi;
  I.rho1 = rho1i;
  const double hi1 = I.h1, hi21 = xmul(hi1, hi1);
  double gradhi = (double)Ri.gradh;
  if (!(gradhi > 0.)) gradhi = 1.;  // force.F90:2616-2621
  const double hfac = hi21 * hi21 * dc.cnormk * gradhi;
  const double vxi = Ri.vx, vyi = Ri.vy, vzi = Ri.vz, eni = Ri.u, pri = Ri.pr;
  I.en = eni; I.pr = pri; I.cs = Ri.cs;
  I.vwave = Ri.cs;
  double pro2i = pri * rho1i * rho1i;
  I.Bx = I.By = I.Bz = I.psi = I.eps = I.ts = 0.;
  if constexpr (MHD) {
    const FRecB Mi = in.recB[p];
    I.Bx = Mi.Bex * rhoi; I.By = Mi.Bey * rhoi; I.Bz = Mi.Bez * rhoi;
    I.psi = Mi.psi;
    const double Brx = I.Bx * rho1i, Bry = I.By * rho1i, Brz = I.Bz * rho1i;
    const double Bro2 = Brx * Brx + Bry * Bry + Brz * Brz;
    I.vwave = sqrt(I.cs * I.cs + Bro2 * rhoi);
    pro2i += 0.5 * Bro2;
  }
  double sqepsi = 0., tsgi = 0., tsfac = 0.;
  if constexpr (DUST) {
    I.eps = in.recD[p].eps;
    I.ts = get_ts_d(dc, rhoi * (1. - I.eps), rhoi * I.eps, I.cs);
    if (dc.ilimitdustflux) I.ts = fmin(I.ts, I.h / I.cs);
    sqepsi = sqrt(I.eps / (1. - I.eps));
    tsgi = I.ts - I.eps * I.ts;
    tsfac = (I.eps < 1.) ? I.ts / (1. - I.eps) * pm : 0.;
  }
  const double vwi = I.vwave, avwi = (double)Ri.alpha * vwi;
  const float pmf = (float)pm, rhoif = (float)rhoi, autermf = (float)(0.5 * pm * rho1i * dc.alphau),
              alphauf = (float)dc.alphau;
  ForceSums S;
  S.fx = S.fy = S.fz = S.drhodt = S.dudtdiss = S.dendtdiss = S.vsigmax = 0.;
  S.divBsym = S.dBx = S.dBy = S.dBz = S.divBdiff = 0.;
  S.ddust = S.dudtdust = S.dvx = S.dvy = S.dvz = 0.;
  S.ibin_neigh = 0;
  const bool ind = out.ibin != nullptr;
  const int8_t ibinnow_m1 = (int8_t)(out.ibinnow - 1);
  int npair = 0;
  const int n = live ? t_nl[t] : 0;
  const uint16_t *L = G.list + (size_t)w * G.lc * TILE_P + pi;
  // entries are read two steps ahead
  int k = sl, s0 = 0xffff, s1 = 0xffff;
  if (k < n) s0 = L[k * TILE_P];
  if (k + TILE_L < n) s1 = L[(k + TILE_L) * TILE_P];
  const int nch = (G.nc + NC - 1) / NC, cs = nch > 0 ? (G.nc + nch - 1) / nch : 0;
#pragma unroll 1
  for (int c0 = 0; c0 < G.nc; c0 += cs) {
    const int c1 = min(G.nc, c0 + cs), m = c1 - c0;
    if (c0 > 0) __syncthreads();
    if constexpr (MIXED) {
#pragma unroll 1
      for (int c = tid; c < m; c += 64 * W) {
        const uint32_t e = G.cand[c0 + c];
        const int j = cand_node(e);
        const double4 r = in.fpos[j], v = in.fvel[j];
        const FRec32 A = in.rec32[j];
        double x = r.x, y = r.y, z = r.z;
        offset_pos(dc, cand_code(e), x, y, z);
        const double h21 = xmul(r.w, r.w), vw = (double)A.vwave;
        double2 *R = rec + c * NP;
        R[0] = make_double2(x, y);
        R[1] = make_double2(z, r.w);
        R[2] = make_double2(v.x, v.y);
        R[3] = make_double2(v.z, v.w);
        R[4] = make_double2(h21 * h21 * dc.cnormk * (double)A.gradh,
                            __hiloint2double(__float_as_int(A.rho), __float_as_int(A.rho1)));
        R[5] = make_double2((double)A.pr + (double)A.prlo, (double)A.pro2 + (double)A.pro2lo);
        R[6] = make_double2(vw, (double)A.alpha * vw);
      }
    } else {
      // eight lanes per 128-byte record, the first seven pieces of which
      // become the candidate's in place
      const double2 *rsrc = reinterpret_cast<const double2 *>(in.rec);
#pragma unroll 4
      for (int q = tid; q < m * 8; q += 64 * W) {
        const int c = q >> 3, b = q & 7;
        const int j = cand_node(G.cand[c0 + c]);
        if (b < 7) rec[c * NP + b] = rsrc[(size_t)j * 8 + b];
      }
      if constexpr (MHD) {
        const double2 *bsrc = reinterpret_cast<const double2 *>(in.recB);
#pragma unroll 2
        for (int q = tid; q < m * 2; q += 64 * W)
          rec[(q >> 1) * NP + Cap::PB + (q & 1)] = bsrc[(size_t)cand_node(G.cand[c0 + (q >> 1)]) * 8 + (q & 1)];
      }
      if constexpr (DUST) {
        for (int c = tid; c < m; c += 64 * W) {
          const FRecD D = in.recD[cand_node(G.cand[c0 + c])];
          rec[c * NP + Cap::PD] = make_double2(D.eps, D.sqeps);
          rec[c * NP + Cap::PD + 1] = make_double2(D.ts - D.eps * D.ts, 0.);
        }
      }
      __syncthreads();
      // per candidate: the periodic offset, and what a pair would form from
      // rho, gradh and alpha
#pragma unroll 1
      for (int c = tid; c < m; c += 64 * W) {
        const int code = cand_code(G.cand[c0 + c]);
        double2 *R = rec + c * NP;
        if (code != SEP_PLAIN) {
          double x = R[0].x, y = R[0].y, z = R[1].x;
          offset_pos(dc, code, x, y, z);
          R[0] = make_double2(x, y);
          R[1].x = z;
        }
        const double h1 = R[1].y, h21 = xmul(h1, h1);
        const double2 v = R[6];
        const float2 ga = *reinterpret_cast<const float2 *>(&v.y);  // gradh, alpha
        R[4].x = h21 * h21 * dc.cnormk * (double)ga.x;
        R[6].y = (double)ga.y * v.x;
      }
    }
    __syncthreads();
#pragma unroll 1
    while (s0 < c1) {
      const double2 *R = rec + (s0 - c0) * NP;
      const double2 a0 = R[0], a1 = R[1];
      const double dx = xsub(xi, a0.x), dy = xsub(yi, a0.y), dz = xsub(zi, a1.x);
      const double rij2 = r2_exact(dx, dy, dz);
      const double hj1 = a1.y, hj21 = xmul(hj1, hj1);
      const double q2i = xmul(rij2, hi21), q2j = xmul(rij2, hj21);
      // the lists also hold particles that are not force neighbours
      if (q2i < R2 || q2j < R2) {
        npair++;
        const double2 a2 = R[2], a3 = R[3], a4 = R[4], a5 = R[5], a6 = R[6];
        if (ind) {
          // force.F90:1346-1352: every neighbour of an active particle is
          // flagged to be woken; the limiter needs the largest neighbour bin
          const int j = cand_node(G.cand[s0]);
          S.ibin_neigh = max(S.ibin_neigh, (int)tbin_old[j]);
          const int oj = abs(iparts[j]) - 1;
          if (out.ibin_wake[oj] < ibinnow_m1) out.ibin_wake[oj] = ibinnow_m1;
        }
        double rij, rij1;
        if constexpr (MIXED) {
          const float r2f = (float)rij2;
          rij1 = 0.;
          if (r2f > 0.f) {
            const double y = (double)rsqrtf(r2f);
            rij1 = y * (1.5 - 0.5 * rij2 * y * y);
          }
          rij = rij2 * rij1;
        } else {
          sqrt_rsqrt_sep(rij2, 0., rij, rij1);
        }
        const double gi = kern_grad<K>(rij * hi1) * hfac, gj = kern_grad<K>(rij * hj1) * a4.x;
        const double ux = dx * rij1, uy = dy * rij1, uz = dz * rij1;
        const double dvx = vxi - a2.x, dvy = vyi - a2.y, dvz = vzi - a3.x;
        const double projv = dvx * ux + dvy * uy + dvz * uz;
        const double bp = dc.beta * projv;
        const double vwj = a6.x;
        // j's wave speed counts where its own kernel reaches, and always with
        // MHD, dust or conductivity
        const bool usej = MHD || DUST || THERMAL || q2j < R2;
        S.vsigmax = fmax(S.vsigmax, (usej ? fmax(vwi, vwj) : vwi) - bp);
        const double rho1j = MIXED ? (double)__int_as_float(__double2loint(a4.y)) : a4.y;
        const double hp = -0.5 * fmin(projv, 0.);
        const double qi = hp * rho1i * fmax(avwi - bp, 0.), qj = hp * rho1j * fmax(a6.y - bp, 0.);
        const double gradp = pm * ((pro2i + qi) * gi + (a5.y + qj) * gj);
        S.drhodt = fma(projv, gi, S.drhodt);
        const double dpr = pri - a5.x;
        if constexpr (THERMAL) {
          S.dudtdiss = fma(pm * qi * projv, gi, S.dudtdiss);
          if constexpr (MIXED) {
            const float rhoj = __int_as_float(__double2hiint(a4.y));
            const float vsigu = sqrtf((float)fabs(dpr) * (2.f / (rhoif + rhoj)));
            const float denij = (float)(eni - a3.y);
            S.dendtdiss += (double)(vsigu * denij *
                                    (autermf * (float)gi + 0.5f * pmf * (float)rho1j * alphauf * (float)gj));
          } else {
            // sqrt(2 |dP| / (rho_i + rho_j)) from the reciprocal densities
            const double rr = rho1i * rho1j, a = 2. * fabs(dpr) * rr;
            const double vsigu = a * rsqrt_pos(a * (rho1i + rho1j));
            S.dendtdiss = fma(vsigu * (eni - a3.y), rho1i * gi + rho1j * gj, S.dendtdiss);
          }
        }
        double fx = ux * gradp, fy = uy * gradp, fz = uz * gradp;
        if constexpr (MHD) {
          const double2 b0 = R[Cap::PB], b1 = R[Cap::PB + 1];
          const double Bxj = b0.x, Byj = b0.y, Bzj = b1.x, psij = b1.y;
          const double dBx = I.Bx - Bxj, dBy = I.By - Byj, dBz = I.Bz - Bzj;
          const double projBi = I.Bx * ux + I.By * uy + I.Bz * uz;
          const double projBj = Bxj * ux + Byj * uy + Bzj * uz;
          const double projdB = dBx * ux + dBy * uy + dBz * uz;
          S.divBdiff = fma(-pm * projdB, gi, S.divBdiff);
          const double ax = dvx - projv * ux, ay = dvy - projv * uy, az = dvz - projv * uz;
          double vsigB, dum;
          sqrt_rsqrt_sep(ax * ax + ay * ay + az * az, 0., vsigB, dum);
          const double pmi = pm * rho1i * rho1i * gi, pmj = pm * rho1j * rho1j * gj;
          const double dis = 0.5 * dc.alphaB * (pmi + pmj) * vsigB;
          if (THERMAL && dc.iresistive_heating > 0)
            S.dudtdiss = fma(-0.5 * (dBx * dBx + dBy * dBy + dBz * dBz), dis, S.dudtdiss);
          // the stress -m B (B.r)/rho^2 of each particle along the pair
          const double termi = pmi * projBi, termj = pmj * projBj;
          S.divBsym += termi + termj;
          const double psit = dc.overcleanfac * (pmi * I.psi * vwi + pmj * psij * vwj);
          S.dBx += -termi * dvx + dis * dBx - psit * ux;
          S.dBy += -termi * dvy + dis * dBy - psit * uy;
          S.dBz += -termi * dvz + dis * dBz - psit * uz;
          fx -= I.Bx * termi + Bxj * termj;
          fy -= I.By * termi + Byj * termj;
          fz -= I.Bz * termi + Bzj * termj;
        }
        S.fx -= fx;
        S.fy -= fy;
        S.fz -= fz;
        if constexpr (DUST) {
          const double2 d0 = R[Cap::PD], d1 = R[Cap::PD + 1];
          if (I.eps > 0. || d0.x > 0.) {
            const double dft = pm * d0.y * rho1j * (tsgi + d1.x) * dpr * (0.5 * (gi + gj)) * rij1;
            S.ddust -= dft;
            if (THERMAL) S.dudtdust = fma(-sqepsi * dft, eni - a3.y, S.dudtdust);
          }
          const double term = tsfac * (pro2i * gi + a5.y * gj);
          S.dvx = fma(term, ux, S.dvx);
          S.dvy = fma(term, uy, S.dvy);
          S.dvz = fma(term, uz, S.dvz);
        }
      }
      k += TILE_L;
      s0 = s1;
      s1 = 0xffff;
      if (k + TILE_L < n) s1 = L[(k + TILE_L) * TILE_P];
    }
  }
  S.fx = quad_sum(S.fx); S.fy = quad_sum(S.fy); S.fz = quad_sum(S.fz);
  S.drhodt = quad_sum(S.drhodt);
  S.vsigmax = quad_max(S.vsigmax);
  if (THERMAL) {
    S.dudtdiss = quad_sum(S.dudtdiss);
    S.dendtdiss = quad_sum(S.dendtdiss);
    if (!MIXED) S.dendtdiss *= 0.5 * pm * dc.alphau;
  }
  if (MHD) {
    S.divBsym = quad_sum(S.divBsym); S.divBdiff = quad_sum(S.divBdiff);
    S.dBx = quad_sum(S.dBx); S.dBy = quad_sum(S.dBy); S.dBz = quad_sum(S.dBz);
  }
  if (DUST) {
    S.ddust = quad_sum(S.ddust); S.dudtdust = quad_sum(S.dudtdust);
    S.dvx = quad_sum(S.dvx); S.dvy = quad_sum(S.dvy); S.dvz = quad_sum(S.dvz);
  }
  if (ind) S.ibin_neigh = quad_max_i(S.ibin_neigh);
  double dtc_o = PH_HUGE64, dtf_o = PH_HUGE64;
  int bmax = -1;
  if (live && sl == 0)
    force_store<MHD, DUST, THERMAL>(dc, out, abs(iparts[p]) - 1, I, S, icall, dtc_o, dtf_o, bmax, flags);
  reduce_force_block(dtc_o, dtf_o, npair, bmax, dtred, flags);
}

void launch_force_tile(phsph_ctx *c, int icall, const ForceIOArgs &a, const TileLists &tl, const ForceTileIn &in,
                       bool mixed, bool mhd, bool dust, const int32_t *skip) {
  const int ng = c->ntg;
  const dim3 gr(tile_grid(ng, tl));
  const bool th = c->p.maxvxyzu >= 4, w4 = c->tg_max <= 4 * TILE_P;
#define FT(KK, WW, M, D, T, X)                                                                                    \
  hipLaunchKernelGGL((k_force_tile<KK, WW, M, D, T, X>), gr, dim3(64 * WW), 0, c->stream, c->dc, ng, c->act.p, tl, \
                     c->t_nl.p, skip, c->iparts.p, in, a, c->tbin_old.p, icall, c->dtred.p, c->counters.p)
#define FTW(KK, M, D, T, X) \
  if (w4) FT(KK, 4, M, D, T, X); else FT(KK, 5, M, D, T, X)
#define FTK(KK)                                                                                              \
  if (mixed) { if (th) FTW(KK, false, false, true, true); else FTW(KK, false, false, false, true); }         \
  else if (mhd && dust) { if (th) FTW(KK, true, true, true, false); else FTW(KK, true, true, false, false); } \
  else if (mhd) { if (th) FTW(KK, true, false, true, false); else FTW(KK, true, false, false, false); }      \
  else if (dust) { if (th) FTW(KK, false, true, true, false); else FTW(KK, false, true, false, false); }     \
  else { if (th) FTW(KK, false, false, true, false); else FTW(KK, false, false, false, false); }
  if (c->p.kernel == PHSPH_KERNEL_CUBIC) { FTK(PHSPH_KERNEL_CUBIC) } else { FTK(PHSPH_KERNEL_QUINTIC) }
#undef FTK
#undef FTW
#undef FT
}
