// dens_tile.hip -- neighbour search and h-rho iteration of dense active sets:
// one workgroup per tree node of at most 64 or 80 particles (tile.h).
//
// The neighbour sets, iteration counts and Newton steps are those of the list
// kernels (density.hip): k_dens_solo for sparse active sets and for the particles
// that are run again, k_dens_iter for dense sets that do not go by tile.
#include "dens_tile.h"

#include <algorithm>

// One particle's neighbour distances live in the registers of its four
// lanes, entry k in lane k mod 4, so a Newton iteration reads no memory.
//
//  1. stage: the group's candidate leaves (k_group_walk), one lane for each of
//     the up to 10 particles of a leaf, particles beyond the group's box plus
//     its search radius left out; the periodic offset of the leaf is added
//     here, once.
//  2. cull and test: each wavefront takes 64 candidates at a time, keeps those
//     that its own 16 particles can reach (about half) in FP32 relative to the
//     centre of these particles, and tests them 4 at a time against the 16
//     particles: with |x_j|^2 stored, three FMA and a compare.  The list may
//     hold more than the search sphere (the sums and the later passes make
//     their own exact tests), so FP32 with a margin above its rounding does.
//     Lengths there are in units of the group's search radius, so that no
//     square leaves the FP32 range whatever the unit of length; a group whose
//     box or neighbours' radii are 1e15 times its own goes to the list kernels.
//     Hits are packed into the particle's list in candidate order.
//  3. FP64 distances into registers, list to memory, Newton iterations.
//
// Bound by vector instructions in the four-wavefront form: 90 % of the issue
// cycles at 3600 per wavefront of 16 particles on the 8M-particle box, 3.9 ms
// (5.4 with an FP64 test and the kernel evaluated per neighbour, 10.6 as a
// search and iteration over per-lane lists).  The quintic five-wavefront form
// has one workgroup on a CU (tile.h) and 28 % of them: 2.9 ms on the 1.1M tube.
//
// Offsets.  get_sep (kdtree.F90:1468-1501) takes a leaf's offset from the two
// leaf centres.  Here it is taken from the group's box centre, which gives the
// same offset for every pair in reach when half the box exceeds the distance
// over which the leaf centres of the group spread plus the search radius plus
// the leaf sizes: a pair for which the two choices differ is then out of reach
// (and its separation under either is beyond the search radius), and no
// separation in reach needs a further minimum-image step.  Groups in boxes too
// small for that go to the list kernels (all of a set of which most are: dens_run).
template <int K, int V>
__global__ void __launch_bounds__((64 * TileCap<K, V>::W)) __attribute__((amdgpu_waves_per_eu(TileCap<K, V>::WPE)))
k_dens_tile(DevConst dc, int icall, double rfac, double lmargin, const int32_t *__restrict__ act, int ngroups,
            const int32_t *__restrict__ gt,
            const double *__restrict__ gbox, const int32_t *__restrict__ pleaf, const uint32_t *__restrict__ gcand,
            const int32_t *__restrict__ gncand, const int64_t *goff, int capg, const int32_t *__restrict__ nd_lo,
            const int32_t *__restrict__ nd_hi, const phsph_kdnode *__restrict__ nd, const double4 *__restrict__ tp,
            const double *__restrict__ hmax0, DensIterOut out, TileLists tl, int32_t *__restrict__ flags) {
  constexpr bool BIG = TileCap<K, V>::BIG;
  constexpr int W = TileCap<K, V>::W, NC = TileCap<K, V>::NC, LC = TileCap<K, V>::LC, NE = BIG ? 1 : LC / TILE_L;
  constexpr int LEAVES = 64 * W;  // leaves staged at a time
  __shared__ double cx[NC], cy[NC], cz[NC];  // position with the offset
  __shared__ float cr2[NC];                  // (list radius of j)^2 in units of the group's, rounded up
  __shared__ uint32_t cj[NC];                // tree position and offset code
  __shared__ float4 bxs[W][64];              // candidates under test: x, y, z about the centre and their square
  __shared__ uint2 brs[W][64];               // their cr2 and slot
  __shared__ union {
    struct {
      int lo[LEAVES], cc[LEAVES];  // first particle, count and code of the staged leaves
    } leaf;
    uint16_t list[W][LC + 1][TILE_P];  // the last row takes what does not fit
  } U;
  __shared__ int self[5 * TILE_P];  // slot of the group's own particles
  __shared__ int wcnt[2][W];
  __shared__ double wred[W][2];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  auto group = [&](const int g, const int b) {  // b: its place in the large arrays
  const int t0 = gt[g], t1 = gt[g + 1];
  if (t0 >= t1) {  // no active particle in the node
    if (!BIG && threadIdx.x == 0) tl.nc[g] = -1;
    return;
  }
  const double *gb = gbox + (size_t)g * GBOX;
  const double bx = 0.5 * (gb[0] + gb[3]), by = 0.5 * (gb[1] + gb[4]), bz = 0.5 * (gb[2] + gb[5]);
  const double ex = 0.5 * (gb[3] - gb[0]) * (1. + 1e-12) + 1e-300, ey = 0.5 * (gb[4] - gb[1]) * (1. + 1e-12) + 1e-300,
               ez = 0.5 * (gb[5] - gb[2]) * (1. + 1e-12) + 1e-300;
  const double rl = rfac * lmargin * dc.radkern;
  const double rg = rl * gb[6], rg2 = rg * rg;
  const double sc = 1. / rg, sc2 = sc * sc;  // to units of the group's search radius
  const uint32_t *gc = gcand + cand_base(goff, g, capg);
  const int nleaf = gncand[g];
  const int pfirst = act[t0], plast = act[t1 - 1];
  // --- stage ---
  int nc = 0, buf = 0;
  double smax = 0., hmx = gb[6];
  const int li = tid / PH_MINPART, lk = tid - li * PH_MINPART;
  constexpr int LR = LEAVES / PH_MINPART;  // leaves per pass
  for (int lb = 0; lb < nleaf; lb += LEAVES) {
    const int nb = min(LEAVES, nleaf - lb);
    if (tid < nb) {
      const int n = (int)gc[lb + tid];
      const int lo = nd_lo[n];
      const int cnt = min(nd_hi[n] - lo + 1, PH_MINPART);
      int sx = 0, sy = 0, sz = 0;
      if (dc.periodic) {
        const double dx = bx - nd[n].xcen[0], dy = by - nd[n].xcen[1], dz = bz - nd[n].xcen[2];
        if (fabs(dx) > dc.hdlx) sx = (dx > 0.) ? 1 : -1;
        if (fabs(dy) > dc.hdly) sy = (dy > 0.) ? 1 : -1;
        if (fabs(dz) > dc.hdlz) sz = (dz > 0.) ? 1 : -1;
        smax = fmax(smax, nd[n].size);
      }
      if (hmax0) hmx = fmax(hmx, hmax0[n]);
      U.leaf.lo[tid] = lo;
      U.leaf.cc[tid] = cnt | (off_code(sx, sy, sz) << 8);
    }
    __syncthreads();
    for (int r = 0; r < nb; r += LR) {
      bool in = false;
      double x = 0., y = 0., z = 0.;
      float rj2 = 0.f;
      uint32_t jc = 0u;
      if (li < LR && r + li < nb) {
        const int cc = U.leaf.cc[r + li];
        if (lk < (cc & 255)) {
          const int j = U.leaf.lo[r + li] + lk, code = cc >> 8;
          const double4 v = tp[j];
          x = v.x; y = v.y; z = v.z;
          offset_pos(dc, code, x, y, z);
          double rd2 = rg2;
          if (hmax0) {
            const double d2 = (rl * v.w) * (rl * v.w);
            rj2 = (float)(d2 * sc2 * (1. + 1.2e-7));
            rd2 = fmax(rd2, d2);
          }
          const double qx = fmax(fabs(x - bx) - ex, 0.), qy = fmax(fabs(y - by) - ey, 0.),
                       qz = fmax(fabs(z - bz) - ez, 0.);
          in = qx * qx + qy * qy + qz * qz < rd2 * (1. + 1e-9);
          jc = cand_pack(j, code);
        }
      }
      const unsigned long long m = __ballot(in);
      if (lane == 0) wcnt[buf][w] = __popcll(m);
      __syncthreads();
      int at = nc + __popcll(m & lanemask_lt());
      for (int k = 0; k < W; k++) {
        const int c = wcnt[buf][k];
        if (k < w) at += c;
        nc += c;
      }
      buf ^= 1;
      if (in && at < NC) {
        cx[at] = x; cy[at] = y; cz[at] = z; cr2[at] = rj2;
        cj[at] = jc;
        const int j = cand_node(jc);
        if (j >= pfirst && j <= plast && j - pfirst < 5 * TILE_P) self[j - pfirst] = at;
      }
    }
    __syncthreads();
  }
  // the list region is free of the leaves from here on
  bool bad = nc > NC || plast - pfirst >= 5 * TILE_P;
  smax = wave_max(smax);
  hmx = wave_max(hmx);
  if (lane == 0) { wred[w][0] = smax; wred[w][1] = hmx; }
  __syncthreads();
  for (int k = 0; k < W; k++) { smax = fmax(smax, wred[k][0]); hmx = fmax(hmx, wred[k][1]); }
  bad = bad || tile_unfit(dc, ex, ey, ez, rl, gb[6], hmx, smax);
  if (bad && !BIG && nc > NC && tid == 0) tl.big[atomicAdd(tl.nbig, 1)] = g;  // the large form next
  uint32_t *gcl = BIG ? tl.bcand + (size_t)b * tl.bncap : tl.cand + (size_t)g * tl.ncap;
  uint16_t *gll = BIG ? tl.blist + (size_t)b * TILE_BW * tl.blc * TILE_P : tl.list + (size_t)g * tl.lw * tl.lc * TILE_P;
  if (!bad)
    for (int k = tid; k < nc; k += 64 * W) gcl[k] = cj[k];
  if (tid == 0) (BIG ? tl.bnc[b] : tl.nc[g]) = bad ? -1 : nc;
  const int pi = lane / TILE_L, sl = lane % TILE_L;
  bool redo = false;  // a list of this group did not fit
  auto wave16 = [&](const int wt) {  // 16 particles of the wavefront
    const int t = wt + pi;
    const int p = (t < t1) ? act[t] : -1;
    const bool live = p >= 0;
    if (bad) {
      if (BIG || !(nc > NC)) {
        if (live && sl == 0) out.retry[p] = 1;
        if (lane == 0) atomicOr(flags, DFL_TILE);
      }
      return;
    }
    double xi = 0., yi = 0., zi = 0., h0 = 0.;
    double xl = PH_HUGE64, yl = PH_HUGE64, zl = PH_HUGE64, xh = -PH_HUGE64, yh = -PH_HUGE64, zh = -PH_HUGE64;
    int own = -1;
    if (live) {
      const double4 r = tp[p];
      xi = r.x; yi = r.y; zi = r.z; h0 = r.w;
      xl = xh = xi; yl = yh = yi; zl = zh = zi;
      own = self[p - pfirst];
    }
    // --- cull and test ---
    double hw = h0;
    for (int o = 32; o >= TILE_L; o >>= 1) {
      xl = fmin(xl, __shfl_xor(xl, o, 64)); yl = fmin(yl, __shfl_xor(yl, o, 64)); zl = fmin(zl, __shfl_xor(zl, o, 64));
      xh = fmax(xh, __shfl_xor(xh, o, 64)); yh = fmax(yh, __shfl_xor(yh, o, 64)); zh = fmax(zh, __shfl_xor(zh, o, 64));
      hw = fmax(hw, __shfl_xor(hw, o, 64));
    }
    const double wx = 0.5 * (xl + xh), wy = 0.5 * (yl + yh), wz = 0.5 * (zl + zh);
    const float fx = (float)(0.5 * (xh - xl) * sc) * 1.000001f, fy = (float)(0.5 * (yh - yl) * sc) * 1.000001f,
                fz = (float)(0.5 * (zh - zl) * sc) * 1.000001f;
    const float rw2 = (float)((rl * hw * sc) * (rl * hw * sc)) * 1.00001f;
    // particle i about the centre; the margin covers the FP32 rounding of the
    // separation (a few 2^-24 of (|x_i| + |x_j|)^2, |x_j| <= |x_i| + radius)
    const float xf = (float)((xi - wx) * sc), yf = (float)((yi - wy) * sc), zf = (float)((zi - wz) * sc);
    const float di2 = xf * xf + yf * yf + zf * zf;
    const float far = 2.f * sqrtf(di2) + (float)(rl * hmx * sc);
    const float rc2 = (float)((rl * h0 * sc) * (rl * h0 * sc)) * 1.000001f;
    const float ui = di2 - 2e-6f * far * far;
    const float mx = -2.f * xf, my = -2.f * yf, mz = -2.f * zf;
    uint16_t(*L)[TILE_P] = U.list[w];
    int n = 0;
    const bool upper = lane >= 32;
    const unsigned qsh = (unsigned)(lane & 31 & ~(TILE_L - 1)), qlt = (1u << sl) - 1u;
    for (int k0 = 0; k0 < nc; k0 += 64) {
      const int s = k0 + lane;
      bool in = false;
      float x = 0.f, y = 0.f, z = 0.f, rj2 = 0.f;
      if (s < nc) {
        x = (float)((cx[s] - wx) * sc); y = (float)((cy[s] - wy) * sc); z = (float)((cz[s] - wz) * sc);
        rj2 = cr2[s];
        const float qx = fmaxf(fabsf(x) - fx, 0.f), qy = fmaxf(fabsf(y) - fy, 0.f), qz = fmaxf(fabsf(z) - fz, 0.f);
        const float a2 = fabsf(x) + fabsf(y) + fabsf(z);
        in = qx * qx + qy * qy + qz * qz - 2e-6f * a2 * a2 <= fmaxf(rw2, rj2);
      }
      const unsigned long long m = __ballot(in);
      const int ns = __popcll(m);
      if (ns == 0) continue;
      if (in) {
        const int at = __popcll(m & lanemask_lt());
        bxs[w][at] = make_float4(x, y, z, x * x + y * y + z * z);
        brs[w][at] = make_uint2(__float_as_uint(rj2), (unsigned)s);
      }
      // the rest of the last four: farther than any radius
      if (lane < TILE_L - 1 && ns + lane < 64) {
        bxs[w][ns + lane] = make_float4(0.f, 0.f, 0.f, 3e38f);
        brs[w][ns + lane] = make_uint2(0u, 0u);
      }
      wave_lds_sync();
#pragma unroll 2
      for (int k = 0; k < ns; k += TILE_L) {
        const float4 c = bxs[w][k + sl];
        const uint2 rs = brs[w][k + sl];
        const float r2 = fmaf(mz, c.z, fmaf(my, c.y, fmaf(mx, c.x, ui + c.w)));
        const bool hit = r2 < fmaxf(rc2, __uint_as_float(rs.x)) && (int)rs.y != own && live;
        const unsigned long long hm = __ballot(hit);
        const unsigned q = ((upper ? (unsigned)(hm >> 32) : (unsigned)hm) >> qsh) & 15u;
        const int at = n + __popc(q & qlt);
        if (hit) L[min(at, LC)][pi] = (uint16_t)rs.y;
        n += __popc(q);
      }
      wave_lds_sync();
    }
    const bool full = n > LC;
    redo = redo || __ballot(full && !BIG) != 0ull;
    if (full && sl == 0 && BIG) {
      out.retry[p] = 1;
      atomicOr(flags, DFL_TILE);
    }
    // --- distances, list ---
    const int nl = full ? 0 : n;
    int nmax = nl;
    for (int o = 32; o >= TILE_L; o >>= 1) nmax = max(nmax, __shfl_xor(nmax, o, 64));
    nmax = __builtin_amdgcn_readfirstlane(nmax);
    auto dist = [&](int s) {
      const double dx = xi - cx[s], dy = yi - cy[s], dz = zi - cz[s];
      double rr, r1;
      sqrt_rsqrt_sep(dx * dx + dy * dy + dz * dz, 0., rr, r1);
      return rr;
    };
    double r[NE];
    if constexpr (BIG) {
      uint16_t *ll = gll + (size_t)((wt - t0) / TILE_P) * tl.blc * TILE_P;
      for (int k = sl; k < nl; k += TILE_L) ll[k * TILE_P + pi] = L[k][pi];
    } else {
      uint16_t *ll = gll + (size_t)w * LC * TILE_P;
#pragma unroll
      for (int e = 0; e < NE; e++) {
        r[e] = PH_HUGE64;
        if (TILE_L * e < nmax) {
          const int k = TILE_L * e + sl;
          if (k < nl) {
            const int s = L[k][pi];
            r[e] = dist(s);
            ll[k * TILE_P + pi] = (uint16_t)s;
          }
        }
      }
    }
    // --- Newton-Raphson on h (finish_cell, dens.F90:1382-1466) ---
    const double pm = dc.pmass;
    const double rcut = rfac * dc.radkern * h0;
    double hi = h0, hfin = h0;
    int it = 0;
    bool run = live && !full, ok = run;  // iterating; converged in the end
    while (__ballot(run) != 0ull) {
      it++;
      const double hi1 = 1. / hi;
      double mh[IterSums<K>::NT], srho, sgh;
      IterSums<K>::slopes(hi1, mh);
      IterSums<K> S;
      S.zero();
      if constexpr (BIG) {
        for (int k = sl; k < nl; k += TILE_L) S.add(dist(L[k][pi]), mh);
      } else {
#pragma unroll
        for (int e = 0; e < NE; e++)
          if (TILE_L * e < nmax) S.add(r[e], mh);
      }
      S.result(srho, sgh);
      srho = quad_sum(srho) * pm;
      sgh = quad_sum(sgh) * pm;
      if (run) {
        const double hi21 = hi1 * hi1, hi31 = hi1 * hi21, hi41 = hi21 * hi21;
        const double rhoi = dc.cnormk * (srho + dc.wab0 * pm) * hi31;
        const double gradhi = dc.cnormk * (sgh + dc.gradh0 * pm) * hi41;
        const double rhohi = rhoh_d(hi, dc.hfact, pm);
        const double dhdrhoi = -hi / (3. * rhohi);
        const double omegai = 1. - dhdrhoi * gradhi;
        const double func = rhohi - rhoi;
        const double dfdh1 = (omegai > PH_TINY64) ? dhdrhoi / omegai : dhdrhoi / fabs(omegai + PH_EPS64);
        double hnew = hi - func * dfdh1;
        if (hnew > 1.2 * hi) hnew = 1.2 * hi;
        else if (hnew < 0.8 * hi) hnew = 0.8 * hi;
        const bool conv = (fabs(hnew - hi) / h0 < dc.tolh) && omegai > 0. && hi > 0.;
        if (icall == 0) {  // one pass: store at hnew with the sums taken at h0 (dens.F90:341)
          hfin = conv ? hi : hnew;
          run = false;
        } else if (conv) {
          hfin = hi;
          run = false;
        } else if (it >= PH_MAXDENSITS) {
          if (sl == 0) {
            atomicOr(flags, DFL_NOCONV);
            out.retry[p] = 1;
          }
          run = ok = false;
        } else {
          hi = hnew;
          // iteration-major: neighbouring particles write adjacent words
          if (out.htraj && it <= HTRAJ && sl == 0) out.htraj[(size_t)(it - 1) * out.hstride + p] = hi;
          if (dc.radkern * hi * (1. + 1e-12) > rcut) {  // outgrew the list: run again with a wider one
            if (sl == 0) {
              atomicOr(flags, DFL_REWALK);
              // once, also in a group that runs again in the large form
              if (atomicExch(&out.retry[p], 1) == 0) atomicAdd(out.nrewalk, 1);
            }
            run = ok = false;
          }
        }
        if (!run && ok && sl == 0) {
          const int nit = (icall == 0) ? 1 : it;
          if (out.hconv) out.hconv[p] = hi;  // the h of the last summation (cell%h once converged)
          out.t_nl[t] = n;
          out.t_sums[t] = make_double2(srho, sgh);
          out.t_hsum[t] = hi;
          out.t_hfin[t] = hfin;
          out.p_nits[p] = nit;
          atomicMax(&out.leaf_nits[pleaf[p]], nit);
        }
      }
    }
  };
  if constexpr (BIG) {
    for (int wt = t0 + w * TILE_P; wt < t1; wt += W * TILE_P) wave16(wt);
  } else {
    if (t0 + w * TILE_P < t1) wave16(t0 + w * TILE_P);
    // a list of any wavefront too long: the group again in the large form
    if (!bad && __syncthreads_or(redo) && tid == 0) {
      tl.nc[g] = -1;
      tl.big[atomicAdd(tl.nbig, 1)] = g;
    }
  }
  };
  if constexpr (BIG) {  // the listed groups in turn
    const int nbig = *tl.nbig;
    for (int k = blockIdx.x; k < nbig; k += gridDim.x) {
      const int g = tl.big[k];
      if (k < tl.bcap) {
        group(g, k);
        __syncthreads();
      } else {  // no room for its lists
        for (int t = gt[g] + tid; t < gt[g + 1]; t += 64 * W) out.retry[act[t]] = 1;
        if (tid == 0) atomicOr(flags, DFL_TILE);
      }
    }
  } else {
    const int g = xcd_block(blockIdx.x, gridDim.x);
    if (g < ngroups) group(g, 0);
  }
}

void launch_dens_tile(phsph_ctx *c, int icall, double rfac, double lmargin, const double *hmax0,
                      const DensIterOut &out, const TileLists &tl) {
  const int ng = c->ngroups;
  // the large form: as many workgroups as the CUs hold
  const dim3 gr(xcd_grid(ng)), gb((unsigned)(c->ncu > 0 ? c->ncu : 256));
#define DT(KK, VV, GG)                                                                                             \
  hipLaunchKernelGGL((k_dens_tile<KK, VV>), GG, dim3(64 * TileCap<KK, VV>::W), 0, c->stream, c->dc, icall, rfac,   \
                     lmargin, c->act.p, ng, c->tg_t.p, c->gbox.p, c->pleaf.p, c->gcand.p, c->gncand.p,     \
                     c->goff_p, c->caps.gcand, c->nd_lo.p, c->nd_hi.p, c->nd.p, c->tp4.p, hmax0, out, tl,        \
                     c->counters.p)
  const bool w4 = c->tg_max <= 4 * TILE_P;
  if (c->p.kernel == PHSPH_KERNEL_CUBIC) {
    if (w4) DT(PHSPH_KERNEL_CUBIC, TILE_4, gr); else DT(PHSPH_KERNEL_CUBIC, TILE_5, gr);
    DT(PHSPH_KERNEL_CUBIC, TILE_BIG, gb);
  } else {
    if (w4) DT(PHSPH_KERNEL_QUINTIC, TILE_4, gr); else DT(PHSPH_KERNEL_QUINTIC, TILE_5, gr);
    DT(PHSPH_KERNEL_QUINTIC, TILE_BIG, gb);
  }
#undef DT
}

// The arrays of a context are sized for its tile groups and kept.  A thirtieth
// of the groups and 1024 have room in the large form.
template <int K>
static void tile_caps(const phsph_ctx *c, TileLists &tl) {
  const bool w4 = c->tg_max <= 4 * TILE_P;
  tl.lw = w4 ? TileCap<K, TILE_4>::W : TileCap<K, TILE_5>::W;
  tl.ncap = w4 ? TileCap<K, TILE_4>::NC : TileCap<K, TILE_5>::NC;
  tl.lc = TileCap<K, TILE_4>::LC;
  tl.bncap = TileCap<K, TILE_BIG>::NC;
  tl.blc = TileCap<K, TILE_BIG>::LC;
}
static void tile_shape(const phsph_ctx *c, TileLists &tl) {
  const size_t ng = c->ntg;
  if (c->p.kernel == PHSPH_KERNEL_CUBIC) tile_caps<PHSPH_KERNEL_CUBIC>(c, tl);
  else tile_caps<PHSPH_KERNEL_QUINTIC>(c, tl);
  tl.bcap = std::min((int)std::min(ng, 1024 + ng / 32), c->caps.tlarge);
}
// the memory of the lists of a context's tile groups
size_t tile_list_bytes(const phsph_ctx *c) {
  TileLists tl{};
  tile_shape(c, tl);
  const size_t group = sizeof(uint32_t) * tl.ncap + sizeof(uint16_t) * tl.lw * tl.lc * TILE_P,
               large = sizeof(uint32_t) * tl.bncap + sizeof(uint16_t) * TILE_BW * tl.blc * TILE_P;
  return group * c->ntg + large * tl.bcap;
}
int tile_lists(phsph_ctx *c, TileLists &tl) {
  const size_t ng = c->ntg;
  tile_shape(c, tl);
  PH_HIPCHECK(c, c->tl_cand.ensure(ng * tl.ncap));
  PH_HIPCHECK(c, c->tl_list.ensure(ng * tl.lw * tl.lc * TILE_P));
  PH_HIPCHECK(c, c->tl_nc.ensure(ng + 1));
  PH_HIPCHECK(c, c->tg_big.ensure(ng + 1));
  PH_HIPCHECK(c, c->tl_bcand.ensure((size_t)tl.bcap * tl.bncap));
  PH_HIPCHECK(c, c->tl_blist.ensure((size_t)tl.bcap * TILE_BW * tl.blc * TILE_P));
  PH_HIPCHECK(c, c->tl_bnc.ensure(tl.bcap + 1));
  tl.gt = c->tg_t.p;
  tl.cand = c->tl_cand.p;
  tl.list = c->tl_list.p;
  tl.nc = c->tl_nc.p;
  tl.big = c->tg_big.p;
  tl.nbig = c->tg_big.p + ng;
  tl.bcand = c->tl_bcand.p;
  tl.blist = c->tl_blist.p;
  tl.bnc = c->tl_bnc.p;
  return PHSPH_OK;
}
