// dens_sums.hip -- the density sums of dense active sets: every sum of
// get_density_sums (dens.F90:578-857) at the h of the last iteration over the
// lists of the tile kernel (dens_tile.hip), and store_results
// (dens.F90:1511-1681) at the final h.
#include "dens_tile.h"

// FP64 records of a candidate in LDS, 16 bytes at a time: position with the
// offset, velocity, f + fext, and with MHD B = Bevol rho(h at entry)
template <int W, bool MHD>
struct SumCap {
  static constexpr int ND = MHD ? 12 : 10;  // doubles per record
  // candidates staged at a time, and wavefronts per SIMD that LDS and registers hold
  static constexpr int NC = MHD ? 544 : W == 4 ? 480 : 672;
  static constexpr int WPE = MHD ? 3 : 4;
};

// One workgroup per group as in k_dens_tile, four lanes per particle.  The
// candidates' records are staged in LDS in chunks of equal length (one
// chunk holds a node of 64 particles of a uniform set with the cubic kernel) and
// each lane sums every fourth entry of its particle's list, which is in
// candidate order, so that a chunk's entries are consecutive.
//
// A pair reads 72 bytes (MHD 96) from LDS instead of six 16-byte loads whose
// 64 lanes go to 64 cache lines each.  rho and its h derivative are the sums
// the last iteration ended with.  Wavefronts wait 60 to 70 % of their time (the
// records of a chunk and the barriers around them) at two to three and a half a
// SIMD; vector instructions take 67 % of the issue cycles on the 8M-particle box,
// LDS 42 % of the clocks, half of that bank conflicts.
// On the 8M-particle box 3.1 ms (6.7 ms as a list kernel; 3.8 ms with the ends
// in one lane of four and three wavefronts per SIMD), MHD 2M particles 2.1 ms
// (3.9), quintic 1M particles 1.9 ms (2.7; 2.9 where 135 registers let a SIMD
// hold three wavefronts of the 80-particle groups' five).
template <int K, int W, bool MHD, bool MIXED>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu((SumCap<W, MHD>::WPE))))
k_dens_sums(DevConst dc, int ngroups, const int32_t *__restrict__ act, TileLists tl, const int32_t *__restrict__ t_nl,
            const double *__restrict__ t_hsum, const double *__restrict__ t_hfin, const double2 *__restrict__ t_sums,
            const int32_t *__restrict__ retry, const int32_t *__restrict__ iparts, DensIn in,
            double *__restrict__ th_out, DensOut out, int32_t *__restrict__ p_nneigh, int32_t *__restrict__ flags) {
  constexpr int ND = SumCap<W, MHD>::ND, NC = SumCap<W, MHD>::NC;
  __shared__ double2 rec[NC * ND / 2];
  TileGroup G;
  if (!G.find(tl, ngroups)) return;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int pi = lane / TILE_L, sl = lane % TILE_L;
  const int t = G.t0 + w * TILE_P + pi;
  const int p = (t < G.t1) ? act[t] : -1;
  const bool live = p >= 0 && !retry[p];
  const bool have_f = in.tf != nullptr;
  const double pm = dc.pmass;
  double xi = 0., yi = 0., zi = 0., hi1 = 0., hi21 = 0., hi = 1.;
  double4 vi = make_double4(0., 0., 0., 0.), fi = vi;
  double Bxi = 0., Byi = 0., Bzi = 0.;
  int n = 0;
  if (live) {
    const double4 ri = in.tp[p];
    xi = ri.x; yi = ri.y; zi = ri.z;
    hi = t_hsum[t];
    hi1 = 1. / hi;
    hi21 = xmul(hi1, hi1);
    vi = in.tv[p];
    if (have_f) fi = in.tf[p];
    n = t_nl[t];
    if (MHD) {
      const double4 Bev = in.tB[p];
      const double rhoiB = rhoh_d(hi, dc.hfact, pm);
      Bxi = Bev.x * rhoiB; Byi = Bev.y * rhoiB; Bzi = Bev.z * rhoiB;
    }
  }
  const uint16_t *L = G.list + (size_t)w * G.lc * TILE_P + pi;
  double rs_gs = 0., rs_divv = 0.;
  double dv[9], da[9], rr[6], dB[9];
#pragma unroll
  for (int k = 0; k < 9; k++) dv[k] = da[k] = dB[k] = 0.;
#pragma unroll
  for (int k = 0; k < 6; k++) rr[k] = 0.;
  int nneigh = 0;
  // entries are read two steps ahead
  int k = sl, s0 = 0xffff, s1 = 0xffff;
  if (k < n) s0 = L[k * TILE_P];
  if (k + TILE_L < n) s1 = L[(k + TILE_L) * TILE_P];
  const int nch = (G.nc + NC - 1) / NC, cs = nch > 0 ? (G.nc + nch - 1) / nch : 0;
  for (int c0 = 0; c0 < G.nc; c0 += cs) {
    const int c1 = min(G.nc, c0 + cs);
    if (c0 > 0) __syncthreads();
#pragma unroll 1
    for (int c = c0 + tid; c < c1; c += 64 * W) {
      const uint32_t e = G.cand[c];
      const int j = cand_node(e);
      const double4 r = in.tp[j], v = in.tv[j];
      double4 f = make_double4(0., 0., 0., 0.);
      if (have_f) f = in.tf[j];
      double x = r.x, y = r.y, z = r.z;
      offset_pos(dc, cand_code(e), x, y, z);
      double2 *R = rec + (c - c0) * (ND / 2);
      R[0] = make_double2(x, y);
      R[1] = make_double2(z, v.x);
      R[2] = make_double2(v.y, v.z);
      R[3] = make_double2(f.x, f.y);
      if constexpr (MHD) {
        const double4 B = in.tB[j];  // rho_j from the h it had on entry
        R[4] = make_double2(f.z, B.x * B.w);
        R[5] = make_double2(B.y * B.w, B.z * B.w);
      } else {
        R[4] = make_double2(f.z, 0.);
      }
    }
    __syncthreads();
#pragma unroll 1
    while (s0 < c1) {
      const double2 *R = rec + (s0 - c0) * (ND / 2);
      const double2 a0 = R[0], a1 = R[1], a2 = R[2], a3 = R[3], a4 = R[4];
      const double dx = xsub(xi, a0.x), dy = xsub(yi, a0.y), dz = xsub(zi, a1.x);
      const double r2 = r2_exact(dx, dy, dz);
      const double q2 = xmul(r2, hi21);
      if (q2 < dc.radkern2) {
        nneigh++;
        const double dvx = vi.x - a1.y, dvy = vi.y - a2.x, dvz = vi.z - a2.y;
        if constexpr (MIXED) {
          // as the FP64 pass, with 1/r from an FP32 reciprocal square root
          // refined by one FP64 Newton step and the gradient-tensor
          // products in FP32, summed in FP64
          double rij1 = 0.;
          const float r2f = (float)r2;
          if (r2f > 0.f) {
            const double y = (double)rsqrtf(r2f);
            rij1 = y * (1.5 - 0.5 * r2 * y * y);
          }
          const double q = r2 * rij1 * hi1;
          if (dc.gravity) rs_gs += kern_dphidh<K, double>(q2, q) * pm;
          const float rg = (float)(kern_grad<K>(q) * rij1), pmf = (float)pm;
          const float ux = (float)dx * rg * pmf, uy = (float)dy * rg * pmf, uz = (float)dz * rg * pmf;
          const float gx = (float)dvx, gy = (float)dvy, gz = (float)dvz;
          rs_divv += (double)(gx * ux + gy * uy + gz * uz);
          dv[0] += (double)(gx * ux); dv[1] += (double)(gx * uy); dv[2] += (double)(gx * uz);
          dv[3] += (double)(gy * ux); dv[4] += (double)(gy * uy); dv[5] += (double)(gy * uz);
          dv[6] += (double)(gz * ux); dv[7] += (double)(gz * uy); dv[8] += (double)(gz * uz);
          const float ax = (float)(fi.x - a3.x), ay = (float)(fi.y - a3.y), az = (float)(fi.z - a4.x);
          da[0] += (double)(ax * ux); da[1] += (double)(ax * uy); da[2] += (double)(ax * uz);
          da[3] += (double)(ay * ux); da[4] += (double)(ay * uy); da[5] += (double)(ay * uz);
          da[6] += (double)(az * ux); da[7] += (double)(az * uy); da[8] += (double)(az * uz);
          const float xf = (float)dx, yf = (float)dy, zf = (float)dz;
          rr[0] -= (double)(xf * ux); rr[1] -= (double)(xf * uy); rr[2] -= (double)(xf * uz);
          rr[3] -= (double)(yf * uy); rr[4] -= (double)(yf * uz); rr[5] -= (double)(zf * uz);
        } else {
          double rij, rij1;
          sqrt_rsqrt_sep(r2, PH_EPS64, rij, rij1);
          const double q = rij * hi1;
          if (dc.gravity) rs_gs += kern_dphidh<K, double>(q2, q) * pm;
          const double rg = rij1 * kern_grad<K>(q) * pm;
          const double ux = dx * rg, uy = dy * rg, uz = dz * rg;
          dv[0] = fma(dvx, ux, dv[0]); dv[1] = fma(dvx, uy, dv[1]); dv[2] = fma(dvx, uz, dv[2]);
          dv[3] = fma(dvy, ux, dv[3]); dv[4] = fma(dvy, uy, dv[4]); dv[5] = fma(dvy, uz, dv[5]);
          dv[6] = fma(dvz, ux, dv[6]); dv[7] = fma(dvz, uy, dv[7]); dv[8] = fma(dvz, uz, dv[8]);
          const double ax = fi.x - a3.x, ay = fi.y - a3.y, az = fi.z - a4.x;
          da[0] = fma(ax, ux, da[0]); da[1] = fma(ax, uy, da[1]); da[2] = fma(ax, uz, da[2]);
          da[3] = fma(ay, ux, da[3]); da[4] = fma(ay, uy, da[4]); da[5] = fma(ay, uz, da[5]);
          da[6] = fma(az, ux, da[6]); da[7] = fma(az, uy, da[7]); da[8] = fma(az, uz, da[8]);
          rr[0] = fma(-dx, ux, rr[0]); rr[1] = fma(-dx, uy, rr[1]); rr[2] = fma(-dx, uz, rr[2]);
          rr[3] = fma(-dy, uy, rr[3]); rr[4] = fma(-dy, uz, rr[4]); rr[5] = fma(-dz, uz, rr[5]);
          if constexpr (MHD) {
            const double2 a5 = R[5];
            const double bx = Bxi - a4.y, by = Byi - a5.x, bz = Bzi - a5.y;
            dB[0] = fma(bx, ux, dB[0]); dB[1] = fma(bx, uy, dB[1]); dB[2] = fma(bx, uz, dB[2]);
            dB[3] = fma(by, ux, dB[3]); dB[4] = fma(by, uy, dB[4]); dB[5] = fma(by, uz, dB[5]);
            dB[6] = fma(bz, ux, dB[6]); dB[7] = fma(bz, uy, dB[7]); dB[8] = fma(bz, uz, dB[8]);
          }
        }
      }
      k += TILE_L;
      s0 = s1;
      s1 = 0xffff;
      if (k + TILE_L < n) s1 = L[(k + TILE_L) * TILE_P];
    }
  }
#pragma unroll
  for (int q = 0; q < 9; q++) {
    dv[q] = quad_sum(dv[q]);
    da[q] = quad_sum(da[q]);
    if (MHD) dB[q] = quad_sum(dB[q]);
  }
#pragma unroll
  for (int q = 0; q < 6; q++) rr[q] = quad_sum(rr[q]);
  if (dc.gravity) rs_gs = quad_sum(rs_gs);
  if (MIXED) rs_divv = quad_sum(rs_divv);
  else rs_divv = dv[0] + dv[4] + dv[8];
  nneigh = quad_sum_i(nneigh) + 1;
  // the ends of all particles by the first lanes of the workgroup, so that
  // they fill wavefronts (the ends are a fifth of the kernel in one lane of
  // four): sums through LDS, one row per sum
  constexpr int GP = W * TILE_P, NS = 27 + (MHD ? 4 : 0);
  static_assert(GP * NS <= NC * ND, "the sums of the workgroup fit the record buffer");
  double *R = reinterpret_cast<double *>(rec);
  __syncthreads();
  if (live && sl == 0) {
    double *o = R + w * TILE_P + pi;
#pragma unroll
    for (int q = 0; q < 9; q++) {
      o[q * GP] = dv[q];
      o[(9 + q) * GP] = da[q];
    }
#pragma unroll
    for (int q = 0; q < 6; q++) o[(18 + q) * GP] = rr[q];
    o[24 * GP] = rs_gs;
    o[25 * GP] = rs_divv;
    o[26 * GP] = (double)nneigh;
    if (MHD) {
      o[27 * GP] = dB[0] + dB[4] + dB[8];
      o[28 * GP] = dB[7] - dB[5];
      o[29 * GP] = dB[2] - dB[6];
      o[30 * GP] = dB[3] - dB[1];
    }
  }
  __syncthreads();
  const int te = G.t0 + tid;
  if (tid >= GP || te >= G.t1) return;
  const int pe = act[te];
  if (retry[pe]) return;
  const double *o = R + tid;
#pragma unroll
  for (int q = 0; q < 9; q++) {
    dv[q] = o[q * GP];
    da[q] = o[(9 + q) * GP];
  }
#pragma unroll
  for (int q = 0; q < 6; q++) rr[q] = o[(18 + q) * GP];
  double curl[3] = {0., 0., 0.};
  if (MHD)
    for (int q = 0; q < 3; q++) curl[q] = o[(28 + q) * GP];
  const double2 s = t_sums[te];
  dens_store<MHD>(dc, pe, t_hfin[te], s.x, s.y, o[24 * GP], o[25 * GP], MHD ? o[27 * GP] : 0., dv, da, rr, curl,
                  iparts, th_out, out, p_nneigh, (int)o[26 * GP], flags);
}

void launch_dens_sums(phsph_ctx *c, const TileLists &tl, bool mhd, bool mixed, const DensIn &in, const DensOut &out) {
  const int ng = c->ntg;
  const dim3 gr(tile_grid(ng, tl));
#define DS(KK, WW, MM, XX)                                                                                      \
  hipLaunchKernelGGL((k_dens_sums<KK, WW, MM, XX>), gr, dim3(64 * WW), 0, c->stream, c->dc, ng, c->act.p, tl,   \
                     c->t_nl.p, c->t_hsum.p, c->t_hfin.p, c->t_sums.p, c->tmpi.p, c->iparts.p, in, c->th.p, out,  \
                     c->p_nneigh.p, c->counters.p)
#define DSW(KK, WW) \
  if (mixed) DS(KK, WW, false, true); else if (mhd) DS(KK, WW, true, false); else DS(KK, WW, false, false);
#define DSK(KK) \
  if (c->tg_max <= 4 * TILE_P) { DSW(KK, 4) } else { DSW(KK, 5) }
  if (c->p.kernel == PHSPH_KERNEL_CUBIC) { DSK(PHSPH_KERNEL_CUBIC) } else { DSK(PHSPH_KERNEL_QUINTIC) }
#undef DSK
#undef DSW
#undef DS
}
