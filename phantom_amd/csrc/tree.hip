// tree.hip -- kd-tree build on the GPU with the reference's split rule
// (maketree, kdtree.F90:117-314; construct_node :531-929;
// sort_particles_in_cell :937-1001).
//
// The reference builds depth-first with one thread per subtree; with one
// OpenMP thread its result (leaf membership, node centres, in-leaf order)
// is a pure function of the input.  This build reproduces that function:
//
//  * Every node's centre of mass is the sequential FP64 sum over the node's
//    particles in their current order, divided by (total mass * 1/m_gas)
//    (:612-675).  Nodes with at most SUB_MAX particles are built inside one
//    workgroup with exactly that sequential arithmetic on LDS-resident
//    particles.  Larger nodes (up to MID_MAX by one workgroup, above by all)
//    sum in parallel and bound the difference to the sequential sum
//    (|S_seq - S| <= 2 gamma_{n-1} sum|a_i|); if any particle lies within
//    that bound of the split plane the node is re-summed sequentially, so
//    the split is always the reference's.
//  * The partition is the reference's two-pointer swap partition.  For a
//    parallel node its permutation is computed directly: the k-th element
//    > pivot in the left part swaps with the k-th element <= pivot counted
//    from the right end of the right part, everything else stays.
//  * Children are numbered 2n, 2n+1 (Gafton & Rosswog indexing, :820-823).
#include "tile.h"

#include <algorithm>

#define SUB_MAX TREE_SUB_MAX  // particles per LDS subtree
#define SUB_BS 256
#define SUB_QMAX 192  // >= 2*floor(SUB_MAX/(MINPART+1)) nodes per level
#define MID_MAX 16384  // particles per node that one workgroup splits (k_mid)
#define MID_BS 1024
#define MAXLEVELS 64

enum { CNT_ERR = 0, CNT_FALLBACK = 1, CNT_MAXLEVEL = 2, CNT_MINLEVEL = 3, CNT_NAN = 4, CNT_NLEAF = 5, CNT_LIVE = 6,
       CNT_SEQMAX = 7, CNT_TGMAX = 8, CNT_NTG = 9, CNT_NSMALL = 10, CNT_NMID = 11, CNT_N = 12 };
// per level of the large nodes: their number and that of their chunks
enum { LEV_NBIG = 0, LEV_NCHUNK = 1, LEV_N = 2 };
enum { TERR_NODEID = 1, TERR_QUEUE = 2, TERR_COUNT = 4 };

// ------------------------------------------------------------------------
// block helpers (256 threads = 4 waves)
// ------------------------------------------------------------------------
template <int BS>
__device__ double block_sum(double v, double *sh) {
  v = wave_sum(v);
  int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) sh[w] = v;
  __syncthreads();
  double r = 0.;
  for (int k = 0; k < BS / 64; k++) r += sh[k];  // fixed order: deterministic
  __syncthreads();
  return r;
}
template <int BS>
__device__ double block_max(double v, double *sh) {
  v = wave_max(v);
  int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) sh[w] = v;
  __syncthreads();
  double r = sh[0];
  for (int k = 1; k < BS / 64; k++) r = fmax(r, sh[k]);
  __syncthreads();
  return r;
}
template <int BS>
__device__ double block_min(double v, double *sh) {
  v = wave_min(v);
  int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) sh[w] = v;
  __syncthreads();
  double r = sh[0];
  for (int k = 1; k < BS / 64; k++) r = fmin(r, sh[k]);
  __syncthreads();
  return r;
}
// exclusive scan of 0/1 flags over the block; returns exclusive prefix and
// writes the block total to *total
template <int BS>
__device__ int block_excl_scan(int b, int *shi, int *total) {
  int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  unsigned long long m = __ballot(b);
  int pre = __popcll(m & ((1ull << l) - 1ull));
  int wt = __popcll(m);
  __syncthreads();
  if (l == 0) shi[w] = wt;
  __syncthreads();
  int off = 0, tot = 0;
  for (int k = 0; k < BS / 64; k++) {
    if (k < w) off += shi[k];
    tot += shi[k];
  }
  __syncthreads();
  *total = tot;
  return off + pre;
}

// ------------------------------------------------------------------------
// root: periodic wrap, NaN check, bounds, live flags (construct_root_node)
// ------------------------------------------------------------------------
__global__ void k_root_wrap(DevConst dc, double *xyzh, int ld, int np, int32_t *live, double *bred,
                            int32_t *counters) {
  __shared__ double sh[8];
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  double mn[3] = {PH_HUGE64, PH_HUGE64, PH_HUGE64}, mx[3] = {-PH_HUGE64, -PH_HUGE64, -PH_HUGE64};
  int isl = 0;
  if (i < np) {
    double *r = xyzh + (size_t)i * ld;
    double h = r[3];
    if (h >= PH_TINY64) {
      isl = 1;
      double x = r[0], y = r[1], z = r[2];
      if (dc.periodic) {  // cross_boundary (boundary.f90:123-160)
        if (x < dc.xmin) x = xadd(x, dc.dxbound);
        else if (x > dc.xmax) x = xsub(x, dc.dxbound);
        if (y < dc.ymin) y = xadd(y, dc.dybound);
        else if (y > dc.ymax) y = xsub(y, dc.dybound);
        if (z < dc.zmin) z = xadd(z, dc.dzbound);
        else if (z > dc.zmax) z = xsub(z, dc.dzbound);
        r[0] = x; r[1] = y; r[2] = z;
      }
      if (isnan(x) || isnan(y) || isnan(z)) atomicAdd(&counters[CNT_NAN], 1);
      mn[0] = x; mn[1] = y; mn[2] = z;
      mx[0] = x; mx[1] = y; mx[2] = z;
    }
    live[i] = isl;
  }
  for (int c = 0; c < 3; c++) {
    double a = block_min<256>(mn[c], sh);
    double b = block_max<256>(mx[c], sh);
    if (threadIdx.x == 0) {
      bred[(size_t)blockIdx.x * 6 + c] = a;
      bred[(size_t)blockIdx.x * 6 + 3 + c] = b;
    }
  }
}

// final bounds: starts from particle 1 before any wrap (kdtree.F90:375-380)
__global__ void k_root_bounds(const double *bred, int nb, double x0, double y0, double z0, double *box) {
  __shared__ double sh[8];
  double mn[3] = {x0, y0, z0}, mx[3] = {x0, y0, z0};
  for (int b = threadIdx.x; b < nb; b += blockDim.x)
    for (int c = 0; c < 3; c++) {
      mn[c] = fmin(mn[c], bred[(size_t)b * 6 + c]);
      mx[c] = fmax(mx[c], bred[(size_t)b * 6 + 3 + c]);
    }
  for (int c = 0; c < 3; c++) {
    double a = block_min<256>(mn[c], sh);
    double b = block_max<256>(mx[c], sh);
    if (threadIdx.x == 0) { box[c] = a; box[3 + c] = b; }
  }
}

// stable compaction of live particles: per-block counts
__global__ void k_count_blocks(const int32_t *live, int np, int32_t *bcount) {
  __shared__ int shi[8];
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  int b = (i < np) ? live[i] : 0;
  int tot;
  block_excl_scan<256>(b, shi, &tot);
  if (threadIdx.x == 0) bcount[blockIdx.x] = tot;
}
// exclusive scan of block counts in place, total to *total: one block of
// 1024 threads, four consecutive counts per thread
__global__ void __launch_bounds__(1024) k_scan_blocks(int32_t *bcount, int nb, int32_t *total) {
  __shared__ int wsum[16];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  int carry = 0;
  for (int base = 0; base < nb; base += 4096) {
    const int i0 = base + tid * 4;
    int v[4];
    for (int k = 0; k < 4; k++) v[k] = (i0 + k < nb) ? bcount[i0 + k] : 0;
    const int t = v[0] + v[1] + v[2] + v[3];
    int incl = t;
    for (int o = 1; o < 64; o <<= 1) {
      const int u = __shfl_up(incl, o, 64);
      if (lane >= o) incl += u;
    }
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    int woff = 0, btot = 0;
    for (int k = 0; k < 16; k++) {
      const int x = wsum[k];
      if (k < w) woff += x;
      btot += x;
    }
    int run = carry + woff + incl - t;
    for (int k = 0; k < 4; k++) {
      if (i0 + k < nb) bcount[i0 + k] = run;
      run += v[k];
    }
    carry += btot;
    __syncthreads();
  }
  if (tid == 0) *total = carry;
}
// scatter live particles into the tree cache (construct_root_node :429-456)
__global__ void k_fill_cache(DevConst dc, const double *xyzh, int ld, int np, const int32_t *live,
                             const int32_t *bcount, const int8_t *iphase, double *tx, double *ty, double *tz,
                             double *th, int32_t *iparts) {
  __shared__ int shi[8];
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  int b = (i < np) ? live[i] : 0;
  int tot;
  int pre = block_excl_scan<256>(b, shi, &tot);
  if (b) {
    int pos = bcount[blockIdx.x] + pre;
    const double *r = xyzh + (size_t)i * ld;
    tx[pos] = r[0]; ty[pos] = r[1]; tz[pos] = r[2]; th[pos] = r[3];
    int active = iphase ? (iphase[i] > 0) : 1;
    iparts[pos] = (dc.ind_timesteps && !active) ? -(i + 1) : (i + 1);
  }
}

__global__ void k_fill_i32(int32_t *a, int64_t n, int32_t v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = v;
}

// ------------------------------------------------------------------------
// shared per-node finishing: write the node, decide the split
// ------------------------------------------------------------------------
__device__ __forceinline__ int pick_axis(const double *box) {
  // maxloc(xmaxi - xmini): first maximum (kdtree.F90:815)
  double e0 = xsub(box[3], box[0]), e1 = xsub(box[4], box[1]), e2 = xsub(box[5], box[2]);
  int a = 0;
  double e = e0;
  if (e1 > e) { e = e1; a = 1; }
  if (e2 > e) { a = 2; }
  return a;
}

// ------------------------------------------------------------------------
// large nodes (more than MID_MAX particles).  Every large node of a level is
// cut into chunks of BN_CH consecutive tree positions, and each pass of
// construct_node runs over all chunks of all large nodes of the level at
// once, one workgroup per chunk.  One wavefront per node combines its chunk
// results in a fixed order.  Per level: sums -> centre -> ambiguity
// test -> sequential sums (ambiguous nodes only) -> size and left count ->
// node record -> partition (count, scan, scatter, swap) -> children, which
// go to the next level's large nodes or to the list of their size.
// ------------------------------------------------------------------------
#define BN_CH 2048
#define BN_BS 256
#define BN_U (BN_CH / BN_BS)
#define BN_RED 24       // doubles per chunk in ch_red: sums/size/quads, then
#define BN_BOX 12       // from BN_BOX the two children's bounding boxes

// exclusive scan of per-thread counts over the block (block total in *total)
template <int BS>
__device__ int block_excl_scan_int(int v, int *shi, int *total) {
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  int incl = v;
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(incl, o, 64);
    if (l >= o) incl += u;
  }
  __syncthreads();
  if (l == 63) shi[w] = incl;
  __syncthreads();
  int off = 0, tot = 0;
  for (int k = 0; k < BS / 64; k++) {
    if (k < w) off += shi[k];
    tot += shi[k];
  }
  __syncthreads();
  *total = tot;
  return off + incl - v;
}

// K per-thread values reduced over the block in a fixed order (kind 0: sum,
// 1: max, 2: min); the result is valid in thread 0
template <int BS, int K>
__device__ void block_reduce(double (&v)[K], const int (&kind)[K], double *sh) {
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < K; k++) {
    double x = v[k];
    for (int o = 32; o > 0; o >>= 1) {
      const double y = __shfl_xor(x, o, 64);
      x = (kind[k] == 0) ? x + y : (kind[k] == 1) ? fmax(x, y) : fmin(x, y);
    }
    v[k] = x;
  }
  __syncthreads();
  if (l == 0)
    for (int k = 0; k < K; k++) sh[w * K + k] = v[k];
  __syncthreads();
  if (threadIdx.x == 0)
    for (int k = 0; k < K; k++) {
      double x = sh[k];
      for (int ww = 1; ww < BS / 64; ww++) {
        const double y = sh[ww * K + k];
        x = (kind[k] == 0) ? x + y : (kind[k] == 1) ? fmax(x, y) : fmin(x, y);
      }
      v[k] = x;
    }
}

__device__ __forceinline__ const double *axis_arr(int a, const double *tx, const double *ty, const double *tz) {
  return (a == 0) ? tx : (a == 1) ? ty : tz;
}

// The lists that split nodes add their children to: nodes of at most SUB_MAX
// particles (k_subtrees) and of at most MID_MAX (k_mid), each with its split
// axis, and the large nodes of the next level with their chunks.
struct NodeLists {
  int32_t *small, *smallx, *mid, *midx;
  BigNode *bn;       // next level's
  int32_t *ch_node;  // chunk -> entry of bn
  int32_t *lev;      // next level's LEV_ counts
  int bncap, maxch;
  int32_t *counters;
};

// one node to its list, by a whole wavefront
__device__ __forceinline__ void list_node(const NodeLists &L, int nnode, int lo, int hi, int axis) {
  const int lane = threadIdx.x & 63, n = hi - lo + 1;
  if (n <= MID_MAX) {
    if (lane == 0) {
      const bool sm = n <= SUB_MAX;
      const int idx = atomicAdd(&L.counters[sm ? CNT_NSMALL : CNT_NMID], 1);
      (sm ? L.small : L.mid)[idx] = nnode;
      (sm ? L.smallx : L.midx)[idx] = axis;
    }
    return;
  }
  const int nch = (n + BN_CH - 1) / BN_CH;
  int idx = 0, off = 0;
  if (lane == 0) {
    idx = atomicAdd(&L.lev[LEV_NBIG], 1);
    off = atomicAdd(&L.lev[LEV_NCHUNK], nch);
  }
  idx = __shfl(idx, 0, 64);
  off = __shfl(off, 0, 64);
  if (idx >= L.bncap || off + nch > L.maxch) {
    if (lane == 0) atomicOr(&L.counters[CNT_ERR], TERR_QUEUE);
    return;
  }
  if (lane == 0) {
    BigNode b;
    for (int k = 0; k < 3; k++) b.com[k] = 0.;
    b.tot = 0.; b.hmax = 0.; b.delta = 0.; b.pivot = 0.;
    b.lo = lo; b.hi = hi; b.nnode = nnode;
    b.iaxis = axis;
    b.chunk0 = off; b.nchunk = nch;
    b.nl = 0; b.part = 0; b.nbad = 0; b.pad_ = 0;
    L.bn[idx] = b;
  }
  for (int k = lane; k < nch; k += 64) L.ch_node[off + k] = idx;
}

// the root: its range, and its list
__global__ void k_tree_seed(const double *rootbox, int nlive, int32_t *nd_lo, int32_t *nd_hi, NodeLists L) {
  if (threadIdx.x == 0) {
    nd_lo[1] = 0;
    nd_hi[1] = nlive - 1;
  }
  list_node(L, 1, 0, nlive - 1, pick_axis(rootbox));
}

// node f of the level; false past the level's count.  A level whose nodes or
// chunks passed their capacity has raised an error and is not built.
__device__ __forceinline__ bool bn_node(const int32_t *lev, int bncap, int maxch, int f) {
  return f < lev[LEV_NBIG] && lev[LEV_NBIG] <= bncap && lev[LEV_NCHUNK] <= maxch;
}
// chunk c of the level: its node (entry of bn) and positions [p0, p1];
// false for a block past the level's chunk count
__device__ __forceinline__ bool bn_chunk(const BigNode *bn, const int32_t *ch_node, const int32_t *lev, int bncap,
                                         int maxch, int c, int &f, int &p0, int &p1) {
  if (c >= lev[LEV_NCHUNK] || lev[LEV_NBIG] > bncap || lev[LEV_NCHUNK] > maxch) return false;
  f = ch_node[c];
  p0 = bn[f].lo + (c - bn[f].chunk0) * BN_CH;
  p1 = min(bn[f].hi, p0 + BN_CH - 1);
  return true;
}

// the bound on the distance of the parallel centre of a node from the
// sequential one on the split axis (|S_seq - S| <= 2 gamma_{n-1} sum|a_i|)
__device__ __forceinline__ double centre_bound(int n, double sum_abs, double D, double centre) {
  const double uu = 1.1102230246251565e-16;
  const double nu = (double)(n - 1) * uu;
  const double gam = nu / (1. - nu);
  return 2. * (2. * gam * sum_abs / D + (2. * gam + 4. * uu) * fabs(centre)) + 1e-300;
}

// parallel sums of m*x over a chunk, their absolute values, and hmax
__global__ void __launch_bounds__(BN_BS) k_bn_sums(DevConst dc, const BigNode *bn, const int32_t *ch_node, int bncap,
                                                   int maxch, const int32_t *lev, const double *tx, const double *ty,
                                                   const double *tz, const double *th, double *ch_red) {
  __shared__ double sh[BN_BS / 64 * 7];
  const int c = blockIdx.x;
  int f, p0, p1;
  if (!bn_chunk(bn, ch_node, lev, bncap, maxch, c, f, p0, p1)) return;
  const double pm = dc.pmass;
  const double dfac = (pm > 0.) ? 1. / pm : 1.;
  const double fac = xmul(pm, dfac);
  double v[7] = {0., 0., 0., 0., 0., 0., 0.};
#pragma unroll
  for (int u = 0; u < BN_U; u++) {
    const int p = p0 + u * BN_BS + threadIdx.x;
    if (p <= p1) {
      const double vx = xmul(fac, tx[p]), vy = xmul(fac, ty[p]), vz = xmul(fac, tz[p]);
      v[0] += vx; v[1] += vy; v[2] += vz;
      v[3] += fabs(vx); v[4] += fabs(vy); v[5] += fabs(vz);
      v[6] = fmax(v[6], th[p]);
    }
  }
  const int kind[7] = {0, 0, 0, 0, 0, 0, 1};
  block_reduce<BN_BS, 7>(v, kind, sh);
  if (threadIdx.x == 0)
    for (int k = 0; k < 7; k++) ch_red[(size_t)c * BN_RED + k] = v[k];
}

// centre of mass from the parallel sums, and the bound on its distance from
// the sequential one on the split axis (|S_seq - S| <= 2 gamma_{n-1} sum|a_i|)
__global__ void k_bn_centre(DevConst dc, BigNode *bn, int bncap, int maxch, const int32_t *lev,
                            const double *ch_red) {
  const int f = blockIdx.x, lane = threadIdx.x;
  if (!bn_node(lev, bncap, maxch, f)) return;
  BigNode *b = bn + f;
  const int nchunk = b->nchunk, chunk0 = b->chunk0;
  double s[3] = {0., 0., 0.}, a[3] = {0., 0., 0.}, hm = 0.;
  for (int k = lane; k < nchunk; k += 64) {
    const double *r = ch_red + (size_t)(chunk0 + k) * BN_RED;
    s[0] += r[0]; s[1] += r[1]; s[2] += r[2];
    a[0] += r[3]; a[1] += r[4]; a[2] += r[5];
    hm = fmax(hm, r[6]);
  }
  for (int k = 0; k < 3; k++) {
    s[k] = wave_sum(s[k]);
    a[k] = wave_sum(a[k]);
  }
  hm = wave_max(hm);
  if (lane == 0) {
    const int n = b->hi - b->lo + 1;
    const double pm = dc.pmass;
    const double dfac = (pm > 0.) ? 1. / pm : 1.;
    const double tot = xmul((double)n, pm);
    const double D = xmul(tot, dfac);
    double com[3];
    for (int k = 0; k < 3; k++) com[k] = s[k] / D;
    const int ia = b->iaxis;
    const double a_ax = a[ia], c_ax = com[ia];
    for (int k = 0; k < 3; k++) b->com[k] = com[k];
    b->tot = tot;
    b->hmax = hm;
    b->delta = centre_bound(n, a_ax, D, c_ax);
    b->pivot = c_ax;
  }
}

// does any particle of the chunk lie within delta of the split plane?
__global__ void __launch_bounds__(BN_BS) k_bn_amb(const BigNode *bn, const int32_t *ch_node, int bncap, int maxch,
                                                  const int32_t *lev, const double *tx, const double *ty,
                                                  const double *tz, int32_t *ch_i) {
  const int c = blockIdx.x;
  int f, p0, p1;
  if (!bn_chunk(bn, ch_node, lev, bncap, maxch, c, f, p0, p1)) return;
  const double *tax = axis_arr(bn[f].iaxis, tx, ty, tz);
  const double c_ax = bn[f].pivot, delta = bn[f].delta;
  int amb = 0;
#pragma unroll
  for (int u = 0; u < BN_U; u++) {
    const int p = p0 + u * BN_BS + threadIdx.x;
    if (p <= p1) amb |= (fabs(tax[p] - c_ax) <= delta);
  }
  amb = __syncthreads_or(amb);
  if (threadIdx.x == 0) ch_i[(size_t)c * 4 + 0] = amb;
}

// ------------------------------------------------------------------------
// Exact sequential sums (kdtree.F90:655-665) without the sequence.  While a
// running sum s stays inside one binade [2^e, 2^(e+1)) it is a multiple of
// u = 2^(e-52), and adding a rounds a to a multiple of u whatever s is, except
// for a tie (a an odd multiple of u/2).  So the sums up to every element are
// s + u (prefix sums of rint(a/u)), exact in FP64 as long as they stay below
// 2^53 u.  A workgroup takes SEQ_ST elements at a time, stops at the first that
// ties or leaves the open binade, adds the next ones there in order, and goes
// on.  Sums that swing about zero change their binade all the time: the run
// in order grows while little is gained in between.
//
// On the lattice shock tube (1.1M particles) 1.3 ms over all levels; as chains
// of dependent FP64 additions 5.7 ms (2.8 ns each; the two nodes of level 1 3.1
// -> 0.48 ms, levels that split along y and z, whose sums swing, 0.6 -> 0.5).
// ------------------------------------------------------------------------
#define SEQ_ST 8192
#define SEQ_BS 1024
constexpr int SEQ_BUF = SEQ_ST + SEQ_ST / 8 + 32;  // doubles of LDS: rows of eight elements and a word of padding
constexpr int SEQ_SW = SEQ_BS / 64 + 2;
__device__ __forceinline__ int seq_at(int k) { return k + (k >> 3); }
__device__ __forceinline__ int exp_of(double a) { return (int)((__double_as_longlong(a) >> 52) & 0x7ff) - 1023; }
__device__ __forceinline__ double two_to(int e) { return __longlong_as_double((long long)(1023 + e) << 52); }

// a added n times to zero, in order: within a binade the same rounded
// increment every time (after a tie the sum is even, and stays so)
__device__ double seq_mass(int n, double a) {
  double s = 0.;
  if (!(a > 1e-250 && a < 1e250)) {
    for (int k = 0; k < n; k++) s = xadd(s, a);
    return s;
  }
  int k = 0;
  while (k < n) {
    s = xadd(s, a);
    k++;
    const int e = exp_of(s);
    const double S = s * two_to(52 - e), t = a * two_to(52 - e);
    if (t >= 2251799813685248.) continue;  // 2^51
    const double fl = floor(t), fr = t - fl;
    const long long il = (long long)fl, is = (long long)S;
    long long m = il + (fr > 0.5 ? 1 : 0);
    if (fr == 0.5) {
      if (is & 1) continue;
      m = il + (il & 1);
    }
    if (m == 0) break;
    const long long c = min((long long)(n - k), ((1ll << 53) - 1 - is) / m);
    s = (double)(is + c * m) * two_to(e - 52);
    k += (int)c;
  }
  return s;
}

// additions of buf[seq_at(k)], k = k0 .. k1-1, to acc in order: rows of eight,
// two rows read ahead (up to three past the last one: SEQ_BUF has room)
__device__ __forceinline__ double seq_chain(double acc, const double *buf, int k0, int k1) {
  int k = k0;
  while (k < k1 && (k & 7)) acc = xadd(acc, buf[seq_at(k++)]);
  const double *r = buf + seq_at(k);
  const int nr = (k1 - k) >> 3;
  auto read = [&](double (&d)[8], int j) {
#pragma unroll
    for (int u = 0; u < 8; u++) d[u] = r[9 * j + u];
  };
  auto add = [&](const double (&d)[8]) {
#pragma unroll
    for (int u = 0; u < 8; u++) acc = xadd(acc, d[u]);
  };
  if (nr > 0) {
    double v[8], w[8], x[8];
    read(v, 0); read(w, 1); read(x, 2);
    int j = 0;
    for (; j + 3 <= nr; j += 3) {
      add(v); read(v, j + 3);
      add(w); read(w, j + 4);
      add(x); read(x, j + 5);
    }
    if (j < nr) add(v);
    if (j + 1 < nr) add(w);
    k += 8 * nr;
  }
  for (; k < k1; k++) acc = xadd(acc, buf[seq_at(k)]);
  return acc;
}

// the running sums of fac*ta and of the mass over the particles [lo, hi], by a
// whole workgroup of SEQ_BS threads (buf: SEQ_BUF, sw: SEQ_SW doubles of LDS)
__device__ void seq_axis(double *buf, double *sw, int *si, int lo, int hi, double pm, double fac, const double *ta,
                         double &sum, double &tot) {
  constexpr int E = SEQ_ST / SEQ_BS, NW = SEQ_BS / 64;
  static_assert(E == 8, "the padding follows a thread's elements");
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int n = hi - lo + 1, k0 = tid * E;
  if (tid == 0) sw[NW] = 0.;
  if (tid == SEQ_BS - 64) sw[NW + 1] = seq_mass(n, pm);
  int run = 1024;  // length of the next run in order: the first elements double the sum again and again
  for (int base = 0; base < n; base += SEQ_ST) {
    const int cnt = min(SEQ_ST, n - base);
    __syncthreads();
    for (int k = tid; k < cnt; k += SEQ_BS) buf[seq_at(k)] = xmul(fac, ta[lo + base + k]);
    __syncthreads();
    int q = 0;
    while (q < cnt) {
      const double acc = sw[NW], A = fabs(acc);
      int first = q;
      if (A > 1e-250 && A < 1e250) {
        const int e = exp_of(A);
        const double scale = copysign(two_to(52 - e), acc), S = A * two_to(52 - e);
        double m[E], loc = 0.;
        unsigned stop = 0u;
#pragma unroll
        for (int u = 0; u < E; u++) {
          const int k = k0 + u;
          const bool use = k >= q && k < cnt;
          const double t = use ? buf[seq_at(k)] * scale : 0.;
          const double r = rint(t);
          const bool ok = fabs(t) < 1125899906842624. && fabs(t - r) != 0.5;  // 2^50
          m[u] = ok ? r : 0.;
          stop |= ok ? 0u : 1u << u;
          loc += m[u];
        }
        double v = loc;
        for (int o = 1; o < 64; o <<= 1) {
          const double y = __shfl_up(v, o, 64);
          if (lane >= o) v += y;
        }
        if (lane == 63) sw[w] = v;
        if (tid == 0) *si = cnt;
        v = __shfl_up(v, 1, 64);  // the sum of the lanes below
        if (lane == 0) v = 0.;
        __syncthreads();
        double s0 = S;
        for (int i = 0; i < w; i++) s0 += sw[i];
        s0 += v;
        double s = s0;
        int ex = cnt;
#pragma unroll
        for (int u = 0; u < E; u++) {
          const int k = k0 + u;
          s += m[u];
          const bool out = (stop >> u & 1u) || !(s > 4503599627370496. && s < 9007199254740992.);  // 2^52, 2^53
          if (out && k >= q && k < cnt) ex = min(ex, k);
        }
        if (ex < cnt) atomicMin(si, ex);
        __syncthreads();
        first = *si;
        if (first > q && first - 1 >= k0 && first - 1 < k0 + E) {
#pragma unroll
          for (int u = 0; u < E; u++)
            if (k0 + u < first) s0 += m[u];
          sw[NW] = copysign(s0 * two_to(e - 52), acc);
        }
      }
      __syncthreads();
      if (first > q) run = (first - q < 1024) ? min(4 * run, SEQ_ST) : 64;
      q = first;
      if (q < cnt) {
        const int end = min(cnt, q + run);
        if (w == 0) {
          const double a = seq_chain(sw[NW], buf, q, end);
          if (lane == 0) sw[NW] = a;
        }
        q = end;
        __syncthreads();
      }
    }
  }
  __syncthreads();
  sum = sw[NW];
  tot = sw[NW + 1];
  __syncthreads();
}

// The sequential sums of the nodes with a particle within delta of the plane.
// The split depends on those of the split axis and the mass; the centre's
// other coordinates stay the parallel sums' (the bound of k_bn_centre).
__global__ void __launch_bounds__(SEQ_BS) k_bn_seq(DevConst dc, BigNode *bn, int bncap, int maxch, const int32_t *lev,
                                                   int32_t *counters, const int32_t *ch_i, const double *tx,
                                                   const double *ty, const double *tz) {
  __shared__ double buf[SEQ_BUF];
  __shared__ double sw[SEQ_SW];
  __shared__ int si;
  const int f = blockIdx.x, tid = threadIdx.x;
  if (!bn_node(lev, bncap, maxch, f)) return;
  const int nchunk = bn[f].nchunk, chunk0 = bn[f].chunk0;
  int amb = 0;
  for (int k = tid; k < nchunk; k += SEQ_BS) amb |= ch_i[(size_t)(chunk0 + k) * 4 + 0];
  amb = __syncthreads_or(amb);
  if (!amb) return;
  const int lo = bn[f].lo, hi = bn[f].hi, iaxis = bn[f].iaxis;
  const double pm = dc.pmass;
  const double dfac = (pm > 0.) ? 1. / pm : 1.;
  double sum, tot;
  seq_axis(buf, sw, &si, lo, hi, pm, xmul(pm, dfac), axis_arr(iaxis, tx, ty, tz), sum, tot);
  if (tid == 0) {
    BigNode *b = bn + f;
    b->pivot = b->com[iaxis] = sum / xmul(tot, dfac);
    b->tot = tot;
    atomicAdd(&counters[CNT_FALLBACK], 1);
    atomicMax(&counters[CNT_SEQMAX], hi - lo + 1);
  }
}

// size (kdtree.F90:697-782) and the count of particles on the left of the
// pivot, per chunk; under self-gravity also the chunk's share of the second
// moments about the centre of mass (kdtree.F90:724-750)
__global__ void __launch_bounds__(BN_BS) k_bn_size(DevConst dc, const BigNode *bn, const int32_t *ch_node,
                                                   int bncap, int maxch, const int32_t *lev, const double *tx,
                                                   const double *ty, const double *tz, double *ch_red,
                                                   int32_t *ch_i, int quads) {
  __shared__ double sh[BN_BS / 64 * 20];
  const int c = blockIdx.x;
  int f, p0, p1;
  if (!bn_chunk(bn, ch_node, lev, bncap, maxch, c, f, p0, p1)) return;
  const double c0 = bn[f].com[0], c1 = bn[f].com[1], c2 = bn[f].com[2], pivot = bn[f].pivot;
  const double *tax = axis_arr(bn[f].iaxis, tx, ty, tz);
  const double pm = dc.pmass;
  // [8..13] bounding box of the particles on the left of the pivot (the
  // left child after a split at the pivot), [14..19] of those on the right
  double v[20] = {0., 0., 0., 0., 0., 0., 0., 0.};
  for (int k = 0; k < 3; k++) {
    v[8 + k] = PH_HUGE64; v[11 + k] = -PH_HUGE64;
    v[14 + k] = PH_HUGE64; v[17 + k] = -PH_HUGE64;
  }
#pragma unroll
  for (int u = 0; u < BN_U; u++) {
    const int p = p0 + u * BN_BS + threadIdx.x;
    if (p <= p1) {
      const double r[3] = {tx[p], ty[p], tz[p]};
      v[0] = fmax(v[0], r2_exact(xsub(r[0], c0), xsub(r[1], c1), xsub(r[2], c2)));
      const bool left = tax[p] <= pivot;
      v[1] += left ? 1. : 0.;
      const int o = left ? 8 : 14;
      for (int k = 0; k < 3; k++) {
        v[o + k] = fmin(v[o + k], r[k]);
        v[o + 3 + k] = fmax(v[o + 3 + k], r[k]);
      }
      if (quads) {
        const double dx = r[0] - c0, dy = r[1] - c1, dz = r[2] - c2;
        v[2] += pm * (dx * dx); v[3] += pm * (dx * dy); v[4] += pm * (dx * dz);
        v[5] += pm * (dy * dy); v[6] += pm * (dy * dz); v[7] += pm * (dz * dz);
      }
    }
  }
  const int kind[20] = {1, 0, 0, 0, 0, 0, 0, 0, 2, 2, 2, 1, 1, 1, 2, 2, 2, 1, 1, 1};
  block_reduce<BN_BS, 20>(v, kind, sh);
  if (threadIdx.x == 0) {
    ch_red[(size_t)c * BN_RED + 0] = v[0];
    ch_i[(size_t)c * 4 + 1] = (int)v[1];
    if (quads)
      for (int k = 0; k < 6; k++) ch_red[(size_t)c * BN_RED + 1 + k] = v[2 + k];
    for (int k = 0; k < 12; k++) ch_red[(size_t)c * BN_RED + BN_BOX + k] = v[8 + k];
  }
}

// the node record, and the split: left count or, with everything on one
// side, half and half in place (kdtree.F90:856-865)
__global__ void k_bn_node(BigNode *bn, int bncap, int maxch, const int32_t *lev, int32_t *counters,
                          const double *ch_red, const int32_t *ch_i, phsph_kdnode *nd, int32_t *leaf_flag, int level,
                          int maxlevel_indexed, int64_t nslots, double *quads) {
  const int f = blockIdx.x, lane = threadIdx.x;
  if (!bn_node(lev, bncap, maxch, f)) return;
  BigNode *b = bn + f;
  const int nchunk = b->nchunk, chunk0 = b->chunk0;
  double r2 = 0.;
  int cl = 0;
  for (int k = lane; k < nchunk; k += 64) {
    r2 = fmax(r2, ch_red[(size_t)(chunk0 + k) * BN_RED + 0]);
    cl += ch_i[(size_t)(chunk0 + k) * 4 + 1];
  }
  r2 = wave_max(r2);
  cl = wave_sum_i(cl);
  if (quads) {  // second moments: chunk shares in chunk order per lane, then across lanes
    double q[6] = {0., 0., 0., 0., 0., 0.};
    for (int k = lane; k < nchunk; k += 64)
      for (int j = 0; j < 6; j++) q[j] += ch_red[(size_t)(chunk0 + k) * BN_RED + 1 + j];
    for (int j = 0; j < 6; j++) q[j] = wave_sum(q[j]);
    if (lane == 0)
      for (int j = 0; j < 6; j++) quads[6 * (size_t)b->nnode + j] = q[j];
  }
  if (lane == 0) {
    const int nnode = b->nnode, il = 2 * nnode, ir = il + 1;
    const int n = b->hi - b->lo + 1;
    phsph_kdnode e;
    e.xcen[0] = b->com[0]; e.xcen[1] = b->com[1]; e.xcen[2] = b->com[2];
    e.size = xadd(sqrt(r2), PH_EPS64);
    e.hmax = b->hmax;
    e.mass = b->tot;
    e.leftchild = il;
    e.rightchild = ir;
    e.parent = nnode / 2;
    e.idum = 0;
    nd[nnode] = e;
    leaf_flag[nnode] = 0;
    b->nbad = 0;
    if (level >= maxlevel_indexed || (int64_t)ir >= nslots) {
      atomicOr(&counters[CNT_ERR], TERR_NODEID);
      b->nl = 0;
      b->part = 0;
    } else if (cl > 0 && cl < n) {
      b->nl = cl;
      b->part = 1;
    } else {
      b->nl = n / 2;
      b->part = 0;
    }
  }
}

// sort_particles_in_cell as a permutation: the k-th element > pivot in the
// left part [lo, lo+nl-1] swaps with the k-th element <= pivot counted from
// the right end of the right part.  Per chunk, the counts of both kinds.
__global__ void __launch_bounds__(BN_BS) k_bn_pcount(const BigNode *bn, const int32_t *ch_node, int bncap, int maxch,
                                                     const int32_t *lev, const double *tx, const double *ty,
                                                     const double *tz, int32_t *ch_i) {
  __shared__ double sh[BN_BS / 64 * 2];
  const int c = blockIdx.x;
  int f, p0, p1;
  if (!bn_chunk(bn, ch_node, lev, bncap, maxch, c, f, p0, p1)) return;
  if (!bn[f].part) return;
  const int lend = bn[f].lo + bn[f].nl - 1;
  const double pivot = bn[f].pivot;
  const double *tax = axis_arr(bn[f].iaxis, tx, ty, tz);
  double v[2] = {0., 0.};
#pragma unroll
  for (int u = 0; u < BN_U; u++) {
    const int p = p0 + u * BN_BS + threadIdx.x;
    if (p <= p1) {
      const bool le = tax[p] <= pivot;
      if (p <= lend) v[0] += le ? 0. : 1.;
      else v[1] += le ? 1. : 0.;
    }
  }
  const int kind[2] = {0, 0};
  block_reduce<BN_BS, 2>(v, kind, sh);
  if (threadIdx.x == 0) {
    ch_i[(size_t)c * 4 + 2] = (int)v[0];
    ch_i[(size_t)c * 4 + 3] = (int)v[1];
  }
}

// per node: chunk offsets of both kinds in position order
__global__ void k_bn_pscan(BigNode *bn, int bncap, int maxch, const int32_t *lev, int32_t *counters,
                           const int32_t *ch_i, int32_t *ch_off) {
  const int f = blockIdx.x, lane = threadIdx.x;
  if (!bn_node(lev, bncap, maxch, f)) return;
  BigNode *b = bn + f;
  if (!b->part) return;
  const int nchunk = b->nchunk, chunk0 = b->chunk0;
  int carry_l = 0, carry_r = 0;
  for (int base = 0; base < nchunk; base += 64) {
    const int k = base + lane;
    int vl = 0, vr = 0;
    if (k < nchunk) {
      vl = ch_i[(size_t)(chunk0 + k) * 4 + 2];
      vr = ch_i[(size_t)(chunk0 + k) * 4 + 3];
    }
    int il = vl, ir = vr;
    for (int o = 1; o < 64; o <<= 1) {
      const int ul = __shfl_up(il, o, 64), ur = __shfl_up(ir, o, 64);
      if (lane >= o) { il += ul; ir += ur; }
    }
    if (k < nchunk) {
      ch_off[(size_t)(chunk0 + k) * 2 + 0] = carry_l + il - vl;
      ch_off[(size_t)(chunk0 + k) * 2 + 1] = carry_r + ir - vr;
    }
    carry_l += __shfl(il, 63, 64);
    carry_r += __shfl(ir, 63, 64);
  }
  if (lane == 0) {
    b->nbad = min(carry_l, carry_r);
    if (carry_l != carry_r) atomicOr(&counters[CNT_ERR], TERR_COUNT);
  }
}

// ranks of the misplaced elements: the k-th left one goes to tmpA[lo+k],
// the k-th right one counted from the right end to tmpB[lo+k]
__global__ void __launch_bounds__(BN_BS) k_bn_pscatter(const BigNode *bn, const int32_t *ch_node, int bncap, int maxch,
                                                       const int32_t *lev, const double *tx,
                                                       const double *ty, const double *tz, const int32_t *ch_off,
                                                       int32_t *tmpA, int32_t *tmpB) {
  __shared__ int shi[BN_BS / 64];
  const int c = blockIdx.x;
  int f, p0, p1;
  if (!bn_chunk(bn, ch_node, lev, bncap, maxch, c, f, p0, p1)) return;
  if (!bn[f].part) return;
  const int lo = bn[f].lo, lend = lo + bn[f].nl - 1, nbad = bn[f].nbad;
  const double pivot = bn[f].pivot;
  const double *tax = axis_arr(bn[f].iaxis, tx, ty, tz);
  const int q0 = p0 + threadIdx.x * BN_U;  // BN_U consecutive positions per thread: ranks follow positions
  int fl[BN_U], fr[BN_U], nl_ = 0, nr_ = 0;
#pragma unroll
  for (int u = 0; u < BN_U; u++) {
    const int p = q0 + u;
    fl[u] = 0;
    fr[u] = 0;
    if (p <= p1) {
      const bool le = tax[p] <= pivot;
      if (p <= lend) fl[u] = le ? 0 : 1;
      else fr[u] = le ? 1 : 0;
    }
    nl_ += fl[u];
    nr_ += fr[u];
  }
  int tl, tr;
  int rl = ch_off[(size_t)c * 2 + 0] + block_excl_scan_int<BN_BS>(nl_, shi, &tl);
  int rr = ch_off[(size_t)c * 2 + 1] + block_excl_scan_int<BN_BS>(nr_, shi, &tr);
#pragma unroll
  for (int u = 0; u < BN_U; u++) {
    if (fl[u]) {
      const int k = rl++;
      if (k < nbad) tmpA[lo + k] = q0 + u;
    }
    if (fr[u]) {
      const int k = nbad - 1 - rr++;
      if (k >= 0) tmpB[lo + k] = q0 + u;
    }
  }
}

// The swaps: chunk c of a node takes pairs k0 .. k0+BN_CH-1.  A node that is
// halved in place gets the bounding boxes of both halves here instead, per
// chunk (one split at the pivot has its children's boxes from k_bn_size).
__global__ void __launch_bounds__(BN_BS) k_bn_swap(const BigNode *bn, const int32_t *ch_node, int bncap, int maxch,
                                                   const int32_t *lev, const int32_t *tmpA, const int32_t *tmpB,
                                                   double *tx, double *ty, double *tz, double *th, int32_t *iparts,
                                                   double *ch_red) {
  __shared__ double sh[BN_BS / 64 * 12];
  const int c = blockIdx.x;
  int f, p0, p1;
  if (!bn_chunk(bn, ch_node, lev, bncap, maxch, c, f, p0, p1)) return;
  const int lo = bn[f].lo, hi = bn[f].hi, nbad = bn[f].nbad, nl = bn[f].nl;
  if (bn[f].part) {
    const int k0 = p0 - lo;
#pragma unroll
    for (int u = 0; u < BN_U; u++) {
      const int k = k0 + u * BN_BS + threadIdx.x;
      if (k < nbad) {
        const int pa = tmpA[lo + k], pb = tmpB[lo + k];
        if (pa >= lo && pa <= hi && pb >= lo && pb <= hi) {
          const double t0 = tx[pa], t1 = ty[pa], t2 = tz[pa], t3 = th[pa];
          const int32_t ti = iparts[pa];
          tx[pa] = tx[pb]; ty[pa] = ty[pb]; tz[pa] = tz[pb]; th[pa] = th[pb]; iparts[pa] = iparts[pb];
          tx[pb] = t0; ty[pb] = t1; tz[pb] = t2; th[pb] = t3; iparts[pb] = ti;
        }
      }
    }
    return;
  }
  if (nl == 0) return;
  const int hA = lo + nl - 1;
  double v[12];
  for (int k = 0; k < 3; k++) {
    v[k] = PH_HUGE64; v[3 + k] = -PH_HUGE64;
    v[6 + k] = PH_HUGE64; v[9 + k] = -PH_HUGE64;
  }
#pragma unroll
  for (int u = 0; u < BN_U; u++) {
    const int p = p0 + u * BN_BS + threadIdx.x;
    if (p <= p1) {
      const double r[3] = {tx[p], ty[p], tz[p]};
      const int o = (p <= hA) ? 0 : 6;
      for (int k = 0; k < 3; k++) {
        v[o + k] = fmin(v[o + k], r[k]);
        v[o + 3 + k] = fmax(v[o + 3 + k], r[k]);
      }
    }
  }
  const int kind[12] = {2, 2, 2, 1, 1, 1, 2, 2, 2, 1, 1, 1};
  block_reduce<BN_BS, 12>(v, kind, sh);
  if (threadIdx.x == 0)
    for (int k = 0; k < 12; k++) ch_red[(size_t)c * BN_RED + BN_BOX + k] = v[k];
}

// children: ranges, split axes, lists
__global__ void k_bn_finish(const BigNode *bn, int bncap, int maxch, const int32_t *lev, const double *ch_red,
                            int32_t *nd_lo, int32_t *nd_hi, NodeLists L) {
  const int f = blockIdx.x, lane = threadIdx.x;
  if (!bn_node(lev, bncap, maxch, f)) return;
  const BigNode *b = bn + f;
  const int nchunk = b->nchunk, chunk0 = b->chunk0, nl = b->nl;
  if (nl == 0) return;
  double v[12];
  for (int k = 0; k < 3; k++) {
    v[k] = PH_HUGE64; v[3 + k] = -PH_HUGE64;
    v[6 + k] = PH_HUGE64; v[9 + k] = -PH_HUGE64;
  }
  for (int j = lane; j < nchunk; j += 64) {
    const double *r = ch_red + (size_t)(chunk0 + j) * BN_RED + BN_BOX;
    for (int k = 0; k < 3; k++) {
      v[k] = fmin(v[k], r[k]); v[3 + k] = fmax(v[3 + k], r[3 + k]);
      v[6 + k] = fmin(v[6 + k], r[6 + k]); v[9 + k] = fmax(v[9 + k], r[9 + k]);
    }
  }
  for (int k = 0; k < 3; k++) {
    v[k] = wave_min(v[k]); v[3 + k] = wave_max(v[3 + k]);
    v[6 + k] = wave_min(v[6 + k]); v[9 + k] = wave_max(v[9 + k]);
  }
  const int il = 2 * b->nnode, ir = il + 1;
  const int lA = b->lo, hA = b->lo + nl - 1, lB = b->lo + nl, hB = b->hi;
  if (lane == 0) {
    nd_lo[il] = lA; nd_hi[il] = hA; nd_lo[ir] = lB; nd_hi[ir] = hB;
  }
  list_node(L, il, lA, hA, pick_axis(v));
  list_node(L, ir, lB, hB, pick_axis(v + 6));
}

// ------------------------------------------------------------------------
// middle nodes (more than SUB_MAX and at most MID_MAX particles): one
// workgroup splits a node and its descendants down to SUB_MAX, level by
// level, with the passes of the large nodes.  The wavefronts are shared out
// over the nodes of a level, 16 for one, 8 each for two, down to one each for
// the 9 to 15 there can be.  Which particles lie on the left of the pivot is
// kept as one word per 64 particles, so the partition's counts and ranks need
// no pass over memory, and its pairs go through LDS.
//
// As launches over all chunks the levels of these nodes cost 13 launches each,
// 5 us a launch on sets that do not fill the chip: the call on 262144 particles
// 2.32 -> 1.84 ms, on 4096 1.11 -> 0.95 ms.  0.57 ms on 8.4M particles (the last
// four levels of large nodes took 1.6 ms).  Bound by latency on small sets, by
// memory where the workgroups' particles pass the L2.  MID_MAX: the range of a
// 16-bit position in the pairs is 65536; 16384 leaves a set of 262144 16
// workgroups, and above it a workgroup is no faster than the launches.
// ------------------------------------------------------------------------
#define MID_W (MID_BS / 64)
#define MID_Q 16      // nodes of a level: floor(MID_MAX / (SUB_MAX + 1)) = 15 at most
#define MID_RED 20    // doubles per wavefront: sums, or size, child boxes and second moments
#define MID_WORDS (MID_MAX / 64 + 2 * MID_Q)

template <bool QUADS>
__global__ void __launch_bounds__(MID_BS) k_mid(DevConst dc, double *tx, double *ty, double *tz, double *th,
                                                int32_t *iparts, int32_t *nd_lo, int32_t *nd_hi, phsph_kdnode *nd,
                                                int32_t *leaf_flag, int maxlevel_indexed, int64_t nslots,
                                                double *quads, NodeLists L) {
  // the stage of the sequential sums, then the pairs of the partition
  static_assert(SEQ_BUF * 8 >= MID_MAX * 2, "the pairs fit the stage");
  static_assert(SEQ_BS == MID_BS, "seq_axis is run by the whole workgroup");
  __shared__ double buf[SEQ_BUF];
  uint16_t *pairs = reinterpret_cast<uint16_t *>(buf);
  __shared__ double sw[SEQ_SW];
  __shared__ int si;
  __shared__ double red[MID_W][MID_RED];
  __shared__ int redn[MID_W];                       // particles on the left of the pivot
  __shared__ unsigned long long lew[MID_WORDS];     // bit of each particle: on the left
  __shared__ uint16_t rkl[MID_WORDS], rkr[MID_WORDS];  // misplaced ones before the word, left and right part
  // nodes of a level: id, range, split axis; then centre, pivot, mass, split
  __shared__ int qn[2][MID_Q], ql[2][MID_Q], qh[2][MID_Q], qx[2][MID_Q];
  __shared__ int qcount[2];
  __shared__ double qpiv[MID_Q], qtot[MID_Q];
  __shared__ int qamb[MID_Q], qnl[MID_Q], qnbad[MID_Q], qcx[MID_Q][2];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  if ((int)blockIdx.x >= L.counters[CNT_NMID]) return;
  const int root = L.mid[blockIdx.x];
  const int lo0 = nd_lo[root], n0 = nd_hi[root] - lo0 + 1;
  if (n0 <= SUB_MAX || n0 > MID_MAX) return;
  const double pm = dc.pmass;
  const double dfac = (pm > 0.) ? 1. / pm : 1.;
  const double fac = xmul(pm, dfac);
  if (tid == 0) {
    qn[0][0] = root; ql[0][0] = 0; qh[0][0] = n0 - 1; qx[0][0] = L.midx[blockIdx.x];
    qcount[0] = 1;
    qcount[1] = 0;
  }
  __syncthreads();
  int cur = 0, level = 31 - __clz(root);
  while (true) {
    const int nq = min(qcount[cur], MID_Q);
    if (nq == 0) break;
    const int nxt = cur ^ 1;
    int Lw = MID_W;  // wavefronts per node
    while (Lw > 1 && nq * Lw > MID_W) Lw >>= 1;
    const int t = w / Lw, wi = w % Lw, w0 = t * Lw;  // node, wavefront of the node, its first wavefront
    const bool on = t < nq;
    const int tq = on ? t : 0;
    const int a0 = ql[cur][tq], n = on ? qh[cur][tq] - a0 + 1 : 0, axis = qx[cur][tq], nnode = qn[cur][tq];
    const int nw = (n + 63) / 64;               // words of 64 particles
    const int wo = a0 / 64 + a0 / SUB_MAX;      // first word: nodes of more than SUB_MAX share none
    const int base = lo0 + a0;
    if (tid < MID_Q) qamb[tid] = 0;
    {  // sums
      double v0 = 0., v1 = 0., v2 = 0., va = 0., vh = 0.;
#pragma unroll 4
      for (int j = wi; j < nw; j += Lw) {
        const int k = 64 * j + lane;
        if (k < n) {
          const double x = xmul(fac, tx[base + k]), y = xmul(fac, ty[base + k]), z = xmul(fac, tz[base + k]);
          v0 += x; v1 += y; v2 += z;
          va += fabs(axis == 0 ? x : axis == 1 ? y : z);
          vh = fmax(vh, th[base + k]);
        }
      }
      v0 = wave_all(v0, OpAdd()); v1 = wave_all(v1, OpAdd()); v2 = wave_all(v2, OpAdd());
      va = wave_all(va, OpAdd()); vh = wave_all(vh, OpMax());
      if (lane == 0) {
        red[w][0] = v0; red[w][1] = v1; red[w][2] = v2; red[w][3] = va; red[w][4] = vh;
      }
    }
    __syncthreads();
    double c0 = 0., c1 = 0., c2 = 0., tot = 0., hmax = 0., delta = 0.;
    if (on) {
      double s0 = 0., s1 = 0., s2 = 0., sa = 0.;
      for (int i = w0; i < w0 + Lw; i++) {
        s0 += red[i][0]; s1 += red[i][1]; s2 += red[i][2]; sa += red[i][3];
        hmax = fmax(hmax, red[i][4]);
      }
      tot = xmul((double)n, pm);
      const double D = xmul(tot, dfac);
      c0 = s0 / D; c1 = s1 / D; c2 = s2 / D;
      delta = centre_bound(n, sa, D, axis == 0 ? c0 : axis == 1 ? c1 : c2);
    }
    __syncthreads();  // red is written again
    // size, left count and the children's boxes; with a particle within delta
    // of the plane once more about the sequential centre
    bool todo = on, exact = false;
    while (true) {
      const double piv = (axis == 0) ? c0 : (axis == 1) ? c1 : c2;
      if (todo) {
        double r2 = 0., bx[12], q[QUADS ? 6 : 1] = {0.};
        for (int k = 0; k < 3; k++) {
          bx[k] = bx[6 + k] = PH_HUGE64;
          bx[3 + k] = bx[9 + k] = -PH_HUGE64;
        }
        int amb = 0, cl = 0;
#pragma unroll 2
        for (int j = wi; j < nw; j += Lw) {
          const int k = 64 * j + lane;
          const bool in = k < n;
          const int p = base + min(k, n - 1);
          const double x = tx[p], y = ty[p], z = tz[p];
          const double ax = (axis == 0) ? x : (axis == 1) ? y : z;
          const bool left = in && ax <= piv;
          amb |= in && fabs(ax - piv) <= delta;
          const unsigned long long m = __ballot(left);
          if (lane == 0) lew[wo + j] = m;
          cl += __popcll(m);
          if (in) {
            r2 = fmax(r2, r2_exact(xsub(x, c0), xsub(y, c1), xsub(z, c2)));
            bx[0] = left ? fmin(bx[0], x) : bx[0];    bx[6] = left ? bx[6] : fmin(bx[6], x);
            bx[1] = left ? fmin(bx[1], y) : bx[1];    bx[7] = left ? bx[7] : fmin(bx[7], y);
            bx[2] = left ? fmin(bx[2], z) : bx[2];    bx[8] = left ? bx[8] : fmin(bx[8], z);
            bx[3] = left ? fmax(bx[3], x) : bx[3];    bx[9] = left ? bx[9] : fmax(bx[9], x);
            bx[4] = left ? fmax(bx[4], y) : bx[4];    bx[10] = left ? bx[10] : fmax(bx[10], y);
            bx[5] = left ? fmax(bx[5], z) : bx[5];    bx[11] = left ? bx[11] : fmax(bx[11], z);
            if constexpr (QUADS) {
              const double dx = x - c0, dy = y - c1, dz = z - c2;
              q[0] += pm * (dx * dx); q[1] += pm * (dx * dy); q[2] += pm * (dx * dz);
              q[3] += pm * (dy * dy); q[4] += pm * (dy * dz); q[5] += pm * (dz * dz);
            }
          }
        }
        r2 = wave_all(r2, OpMax());
#pragma unroll
        for (int k = 0; k < 3; k++) {
          bx[k] = wave_all(bx[k], OpMin()); bx[6 + k] = wave_all(bx[6 + k], OpMin());
          bx[3 + k] = wave_all(bx[3 + k], OpMax()); bx[9 + k] = wave_all(bx[9 + k], OpMax());
        }
        if constexpr (QUADS)
          for (int k = 0; k < 6; k++) q[k] = wave_all(q[k], OpAdd());
        const bool anyamb = __ballot(amb) != 0ull;
        if (lane == 0) {
          red[w][0] = r2;
          for (int k = 0; k < 12; k++) red[w][1 + k] = bx[k];
          if constexpr (QUADS)
            for (int k = 0; k < 6; k++) red[w][13 + k] = q[k];
          redn[w] = cl;
          if (!exact && anyamb) qamb[t] = 1;
        }
      }
      __syncthreads();
      // nodes that are ambiguous and not yet exact
      bool any = false;
      for (int i = 0; i < nq; i++) {
        if (qamb[i] != 1) continue;
        any = true;
        double sum, mass;
        seq_axis(buf, sw, &si, lo0 + ql[cur][i], lo0 + qh[cur][i], pm, fac, axis_arr(qx[cur][i], tx, ty, tz), sum,
                 mass);
        if (tid == 0) {
          qpiv[i] = sum / xmul(mass, dfac);
          qtot[i] = mass;
          atomicAdd(&L.counters[CNT_FALLBACK], 1);
          atomicMax(&L.counters[CNT_SEQMAX], qh[cur][i] - ql[cur][i] + 1);
        }
        __syncthreads();
      }
      if (!any) break;
      todo = on && qamb[t] == 1;
      if (todo) {
        c0 = (axis == 0) ? qpiv[t] : c0;
        c1 = (axis == 1) ? qpiv[t] : c1;
        c2 = (axis == 2) ? qpiv[t] : c2;
        tot = qtot[t];
        exact = true;
      }
      __syncthreads();
      if (tid < MID_Q && qamb[tid] == 1) qamb[tid] = 2;
      __syncthreads();
    }
    if (on && wi == 0) {  // the node's record and the split, by its first wavefront
      double r2 = 0., bx[12];
      int cl = 0;
      for (int k = 0; k < 3; k++) {
        bx[k] = bx[6 + k] = PH_HUGE64;
        bx[3 + k] = bx[9 + k] = -PH_HUGE64;
      }
      for (int i = w0; i < w0 + Lw; i++) {
        r2 = fmax(r2, red[i][0]);
        cl += redn[i];
        for (int k = 0; k < 3; k++) {
          bx[k] = fmin(bx[k], red[i][1 + k]); bx[6 + k] = fmin(bx[6 + k], red[i][7 + k]);
          bx[3 + k] = fmax(bx[3 + k], red[i][4 + k]); bx[9 + k] = fmax(bx[9 + k], red[i][10 + k]);
        }
      }
      if (QUADS && lane < 6) {
        double q = 0.;
        for (int i = w0; i < w0 + Lw; i++) q += red[i][13 + lane];
        quads[6 * (size_t)nnode + lane] = q;
      }
      const int il = 2 * nnode, ir = il + 1;
      const bool bad_id = level >= maxlevel_indexed || (int64_t)ir >= nslots;
      if (lane == 0) {
        phsph_kdnode e;
        e.xcen[0] = c0; e.xcen[1] = c1; e.xcen[2] = c2;
        e.size = xadd(sqrt(r2), PH_EPS64);
        e.hmax = hmax;
        e.mass = tot;
        e.leftchild = il;
        e.rightchild = ir;
        e.parent = nnode / 2;
        e.idum = 0;
        nd[nnode] = e;
        leaf_flag[nnode] = 0;
        if (bad_id) atomicOr(&L.counters[CNT_ERR], TERR_NODEID);
      }
      int nl = 0, nbad = 0;
      if (!bad_id && cl > 0 && cl < n) {
        nl = cl;
        int nr = 0;
        for (int b = 0; b < nw; b += 64) {
          const int j = b + lane;
          int vl = 0, vr = 0;
          if (j < nw) {
            const unsigned long long m = lew[wo + j];
            const int r = cl - 64 * j;  // particles of the word in the left part
            const unsigned long long lp = (r >= 64) ? ~0ull : (r <= 0) ? 0ull : ((1ull << r) - 1ull);
            vl = __popcll(~m & lp);
            vr = __popcll(m & ~lp);
          }
          int sl = vl, sr = vr;
          for (int o = 1; o < 64; o <<= 1) {
            const int ul = __shfl_up(sl, o, 64), ur = __shfl_up(sr, o, 64);
            if (lane >= o) { sl += ul; sr += ur; }
          }
          if (j < nw) {
            rkl[wo + j] = (uint16_t)(nbad + sl - vl);
            rkr[wo + j] = (uint16_t)(nr + sr - vr);
          }
          nbad += __shfl(sl, 63, 64);
          nr += __shfl(sr, 63, 64);
        }
        if (nbad != nr) {
          if (lane == 0) atomicOr(&L.counters[CNT_ERR], TERR_COUNT);
          nbad = 0;
        }
      } else if (!bad_id) {  // everything on one side: halves in place (kdtree.F90:856-865)
        nl = n / 2;
        for (int k = 0; k < 3; k++) {
          bx[k] = bx[6 + k] = PH_HUGE64;
          bx[3 + k] = bx[9 + k] = -PH_HUGE64;
        }
        for (int k = lane; k < n; k += 64) {
          const double r[3] = {tx[base + k], ty[base + k], tz[base + k]};
          const bool left = k < nl;
          for (int i = 0; i < 3; i++) {
            bx[i] = left ? fmin(bx[i], r[i]) : bx[i];
            bx[3 + i] = left ? fmax(bx[3 + i], r[i]) : bx[3 + i];
            bx[6 + i] = left ? bx[6 + i] : fmin(bx[6 + i], r[i]);
            bx[9 + i] = left ? bx[9 + i] : fmax(bx[9 + i], r[i]);
          }
        }
        for (int i = 0; i < 3; i++) {
          bx[i] = wave_min(bx[i]); bx[6 + i] = wave_min(bx[6 + i]);
          bx[3 + i] = wave_max(bx[3 + i]); bx[9 + i] = wave_max(bx[9 + i]);
        }
      }
      if (lane == 0) {
        qnl[t] = nl;
        qnbad[t] = nbad;
        qcx[t][0] = pick_axis(bx);
        qcx[t][1] = pick_axis(bx + 6);
      }
    }
    __syncthreads();
    const int nl = on ? qnl[t] : 0, nbad = on ? qnbad[t] : 0;
    // ranks of the misplaced ones (k_bn_pscatter): pair j is pairs[a0 + j] and
    // pairs[a0 + nbad + j], positions of this workgroup's particles
    if (nbad > 0) {
      const unsigned long long lt = lanemask_lt();
      for (int j = wi; j < nw; j += Lw) {
        const unsigned long long m = lew[wo + j];
        const int r = nl - 64 * j;
        const unsigned long long lp = (r >= 64) ? ~0ull : (r <= 0) ? 0ull : ((1ull << r) - 1ull);
        const unsigned long long ml = ~m & lp, mr = m & ~lp;
        const uint16_t pos = (uint16_t)(a0 + 64 * j + lane);
        if ((ml >> lane) & 1ull) pairs[a0 + rkl[wo + j] + __popcll(ml & lt)] = pos;
        if ((mr >> lane) & 1ull) pairs[a0 + 2 * nbad - 1 - (rkr[wo + j] + __popcll(mr & lt))] = pos;
      }
    }
    __syncthreads();
#pragma unroll 2
    for (int k = wi * 64 + lane; k < nbad; k += 64 * Lw) {
      const int pa = lo0 + pairs[a0 + k], pb = lo0 + pairs[a0 + nbad + k];
      const double t0 = tx[pa], t1 = ty[pa], t2 = tz[pa], t3 = th[pa];
      const double u0 = tx[pb], u1 = ty[pb], u2 = tz[pb], u3 = th[pb];
      const int32_t ti = iparts[pa], ui = iparts[pb];
      tx[pa] = u0; ty[pa] = u1; tz[pa] = u2; th[pa] = u3; iparts[pa] = ui;
      tx[pb] = t0; ty[pb] = t1; tz[pb] = t2; th[pb] = t3; iparts[pb] = ti;
    }
    if (nl > 0 && wi == 0) {
      const int il = 2 * nnode;
      if (lane < 2) {
        const int a = lane ? a0 + nl : a0, e = lane ? a0 + n - 1 : a0 + nl - 1, x = qcx[t][lane];
        nd_lo[il + lane] = lo0 + a;
        nd_hi[il + lane] = lo0 + e;
        if (e - a + 1 > SUB_MAX) {
          const int slot = atomicAdd(&qcount[nxt], 1);
          if (slot < MID_Q) {
            qn[nxt][slot] = il + lane; ql[nxt][slot] = a; qh[nxt][slot] = e; qx[nxt][slot] = x;
          } else {
            atomicOr(&L.counters[CNT_ERR], TERR_QUEUE);
          }
        } else {
          const int idx = atomicAdd(&L.counters[CNT_NSMALL], 1);
          L.small[idx] = il + lane;
          L.smallx[idx] = x;
        }
      }
    }
    __syncthreads();
    if (tid == 0) qcount[cur] = 0;
    cur = nxt;
    level++;
    __syncthreads();
  }
}

// ------------------------------------------------------------------------
// small nodes: one workgroup builds the whole subtree in LDS, level by
// level, with the reference's sequential arithmetic.  A node takes L lanes of
// one wavefront, L the power of two that spreads the level's nodes over the
// workgroup (64 lanes for the first four nodes, one for more than 128): maxima,
// minima and the partition run across the lanes (the partition as the
// permutation of sort_particles_in_cell, see k_bn_pcount), and the four running
// sums are four dependent chains in the lanes, one each where there are four.
// Latency-bound by the chains: 1.94 ms on 8.4M particles, 0.38 ms on the 1M
// polytrope; one thread per node of up to 64 particles took 2.82 and 0.87 (16 to
// 64 lanes of 256 busy, reads of nodes of equal size in one LDS bank), and one
// launch per level 0.70 on the polytrope, whose nodes get small at three levels.
// The rows carry one word of padding per 32 particles and start 16 banks apart,
// so that equal nodes and the four chains read distinct banks.
// ------------------------------------------------------------------------
__device__ __forceinline__ int sub_at(int k) { return k + (k >> 5); }
#define SUB_ROW (SUB_MAX + SUB_MAX / 32 + 8)

// the running sum of one node's row in position order: fac*x for the
// coordinates, the particle mass for the mass (kdtree.F90:655-665)
__device__ __forceinline__ double sub_chain(const double *row, int a0, int a1, bool ism, double pm, double fac) {
  double acc = 0.;
  for (int k = a0; k <= a1; k += 16) {
    double v[16];
#pragma unroll
    for (int u = 0; u < 16; u++) v[u] = ism ? pm : row[sub_at(min(k + u, a1))];
    if (k + 15 <= a1) {
#pragma unroll
      for (int u = 0; u < 16; u++) acc = xadd(acc, ism ? v[u] : xmul(fac, v[u]));
    } else {
#pragma unroll
      for (int u = 0; u < 16; u++) {
        const double b = xadd(acc, ism ? v[u] : xmul(fac, v[u]));
        acc = (k + u <= a1) ? b : acc;
      }
    }
  }
  return acc;
}

template <bool QUADS>
__global__ void __launch_bounds__(SUB_BS) k_subtrees(DevConst dc, const int32_t *small, const int32_t *smallx,
                                                     double *tx, double *ty, double *tz, double *th,
                                                     int32_t *iparts, int32_t *nd_lo, int32_t *nd_hi,
                                                     phsph_kdnode *nd, int32_t *leaf_flag, int maxlevel_indexed,
                                                     int64_t nslots, double *quads, int32_t *counters) {
  __shared__ double srow[4][SUB_ROW];  // x, y, z, h
  __shared__ int32_t sip[SUB_MAX];
  __shared__ int32_t sidx[SUB_MAX];  // partition pairs
  // nodes of a level: id, range, axis of the longest side of the bounding box
  __shared__ int32_t qn[2][SUB_QMAX], ql[2][SUB_QMAX], qh[2][SUB_QMAX], qx[2][SUB_QMAX];
  __shared__ int qcount[2];
  const int tid = threadIdx.x, lane = tid & 63;
  double *sx = srow[0], *sy = srow[1], *sz = srow[2], *shh = srow[3];
  const int nsmall = counters[CNT_NSMALL];
  int maxlev = 0, minlev = 1 << 30;
  // the launch has about as many workgroups as there are nodes
  for (int f = blockIdx.x; f < nsmall; f += gridDim.x) {
    const int root = small[f];
    const int lo = nd_lo[root], hi = nd_hi[root];
    const int n = hi - lo + 1;
    if (n > SUB_MAX) continue;
    for (int k = tid; k < n; k += SUB_BS) {
      const int s = sub_at(k);
      sx[s] = tx[lo + k]; sy[s] = ty[lo + k]; sz[s] = tz[lo + k]; shh[s] = th[lo + k];
      sip[k] = iparts[lo + k];
    }
    if (tid == 0) {
      qn[0][0] = root; ql[0][0] = 0; qh[0][0] = n - 1;
      qx[0][0] = smallx[f];
      qcount[0] = 1;
      qcount[1] = 0;
    }
    __syncthreads();
    const double pm = dc.pmass;
    const double dfac = (pm > 0.) ? 1. / pm : 1.;
    const double fac = xmul(pm, dfac);
    int cur = 0;
    int level = 31 - __clz(root);
    while (qcount[cur] > 0) {
      const int nq = min(qcount[cur], SUB_QMAX);
      const int nxt = cur ^ 1;
      int L = 64;
      while (L > 1 && nq * L > SUB_BS) L >>= 1;
      const int sub = lane & (L - 1), l0 = lane & ~(L - 1);  // lane within the node's lanes, their first lane
      // this node's lanes of a ballot, and those below this lane
      const unsigned long long lm = (L == 64) ? ~0ull : (((1ull << L) - 1ull) << l0);
      const unsigned long long lt = lm & lanemask_lt();
      for (int t = tid / L; t < nq; t += SUB_BS / L) {
        const int a0 = ql[cur][t], a1 = qh[cur][t], nnode = qn[cur][t];
        const int npn = a1 - a0 + 1;
        double s[4];
        if (L >= 4) {
          double acc = 0.;
          if (sub < 4) acc = sub_chain(srow[sub & 3], a0, a1, sub == 3, pm, fac);
  #pragma unroll
          for (int c = 0; c < 4; c++) s[c] = __shfl(acc, l0 + c, 64);
        } else {
  #pragma unroll
          for (int c = 0; c < 4; c++) s[c] = sub_chain(srow[c], a0, a1, c == 3, pm, fac);
        }
        const double tot = s[3], D = xmul(tot, dfac);
        const double com0 = s[0] / D, com1 = s[1] / D, com2 = s[2] / D;
        const int iaxis = qx[cur][t];
        const double pivot = (iaxis == 0) ? com0 : (iaxis == 1) ? com1 : com2;
        const double *sa = srow[iaxis];
        double hmax = 0., r2max = 0., qd[QUADS ? 6 : 1] = {0.};
        int act = 0, cl = 0;
  #pragma unroll 4
        for (int k = a0 + sub; k <= a1; k += L) {
          const int q = sub_at(k);
          const double dx = xsub(sx[q], com0), dy = xsub(sy[q], com1), dz = xsub(sz[q], com2);
          const double r2 = r2_exact(dx, dy, dz);
          if constexpr (QUADS) {
            qd[0] += pm * (dx * dx); qd[1] += pm * (dx * dy); qd[2] += pm * (dx * dz);
            qd[3] += pm * (dy * dy); qd[4] += pm * (dy * dz); qd[5] += pm * (dz * dz);
          }
          r2max = (r2 > r2max) ? r2 : r2max;
          hmax = (shh[q] > hmax) ? shh[q] : hmax;
          act |= sip[k] > 0;
          cl += sa[q] <= pivot;
        }
        for (int o = L >> 1; o > 0; o >>= 1) {
          r2max = fmax(r2max, __shfl_xor(r2max, o, 64));
          hmax = fmax(hmax, __shfl_xor(hmax, o, 64));
          act |= __shfl_xor(act, o, 64);
          cl += __shfl_xor(cl, o, 64);
          if constexpr (QUADS)
            for (int i = 0; i < 6; i++) qd[i] += __shfl_xor(qd[i], o, 64);
        }
        const bool isleaf = npn <= PH_MINPART;
        const int il = 2 * nnode, ir = il + 1;
        const bool bad_id = !isleaf && (level >= maxlevel_indexed || (int64_t)ir >= nslots);
        if (sub == 0) {
          phsph_kdnode e;
          e.xcen[0] = com0; e.xcen[1] = com1; e.xcen[2] = com2;
          e.size = xadd(sqrt(r2max), PH_EPS64);
          e.hmax = hmax;
          e.mass = tot;
          e.leftchild = isleaf ? 0 : il;
          e.rightchild = isleaf ? 0 : ir;
          e.parent = nnode / 2;
          e.idum = 0;
          nd[nnode] = e;
          if constexpr (QUADS)
            for (int i = 0; i < 6; i++) quads[6 * (size_t)nnode + i] = qd[i];
          nd_lo[nnode] = lo + a0;
          nd_hi[nnode] = lo + a1;
          leaf_flag[nnode] = isleaf ? ((dc.ind_timesteps && !act) ? -1 : 1) : 0;
          if (bad_id) atomicOr(&counters[CNT_ERR], TERR_NODEID);
          if (isleaf) {
            maxlev = max(maxlev, level);
            minlev = min(minlev, level);
          }
        }
        if (isleaf || bad_id) continue;
        int nl = npn / 2;  // everything on one side: halves in place (kdtree.F90:856-865)
        if (cl > 0 && cl < npn) {
          // the k-th element > pivot of the left part [a0, a0+cl-1] swaps
          // with the k-th element <= pivot counted from the right end
          const int lend = a0 + cl - 1;
          int nbad = 0;
          for (int base = a0; base <= lend; base += L) {
            const int k = base + sub;
            const bool b = k <= lend && !(sa[sub_at(min(k, lend))] <= pivot);
            const unsigned long long m = __ballot(b) & lm;
            if (b) sidx[a0 + nbad + __popcll(m & lt)] = k;
            nbad += __popcll(m);
          }
          int nr = 0;
          for (int base = lend + 1; base <= a1; base += L) {
            const int k = base + sub;
            const bool b = k <= a1 && sa[sub_at(min(k, a1))] <= pivot;
            const unsigned long long m = __ballot(b) & lm;
            const int j = nbad - 1 - (nr + __popcll(m & lt));
            if (b && j >= 0) sidx[a0 + nbad + j] = k;
            nr += __popcll(m);
          }
          if (nr != nbad && sub == 0) atomicOr(&counters[CNT_ERR], TERR_COUNT);
          const int npair = min(nbad, nr);
          wave_lds_sync();
          for (int j = sub; j < npair; j += L) {
            const int ia = sidx[a0 + j], ib = sidx[a0 + nbad + j];
            const int pa = sub_at(ia), pb = sub_at(ib);
            const double t0 = sx[pa], t1 = sy[pa], t2 = sz[pa], t3 = shh[pa];
            const int32_t ti = sip[ia];
            sx[pa] = sx[pb]; sy[pa] = sy[pb]; sz[pa] = sz[pb]; shh[pa] = shh[pb]; sip[ia] = sip[ib];
            sx[pb] = t0; sy[pb] = t1; sz[pb] = t2; shh[pb] = t3; sip[ib] = ti;
          }
          wave_lds_sync();
          nl = cl;
        }
        const int hA = a0 + nl - 1;
        double bA[6], bB[6];
  #pragma unroll
        for (int c = 0; c < 3; c++) {
          bA[c] = PH_HUGE64; bA[3 + c] = -PH_HUGE64;
          bB[c] = PH_HUGE64; bB[3 + c] = -PH_HUGE64;
        }
  #pragma unroll 4
        for (int k = a0 + sub; k <= a1; k += L) {
          const bool left = k <= hA;
  #pragma unroll
          for (int c = 0; c < 3; c++) {
            const double v = srow[c][sub_at(k)];
            bA[c] = left ? fmin(bA[c], v) : bA[c];
            bA[3 + c] = left ? fmax(bA[3 + c], v) : bA[3 + c];
            bB[c] = left ? bB[c] : fmin(bB[c], v);
            bB[3 + c] = left ? bB[3 + c] : fmax(bB[3 + c], v);
          }
        }
        for (int o = L >> 1; o > 0; o >>= 1) {
  #pragma unroll
          for (int c = 0; c < 3; c++) {
            bA[c] = fmin(bA[c], __shfl_xor(bA[c], o, 64));
            bA[3 + c] = fmax(bA[3 + c], __shfl_xor(bA[3 + c], o, 64));
            bB[c] = fmin(bB[c], __shfl_xor(bB[c], o, 64));
            bB[3 + c] = fmax(bB[3 + c], __shfl_xor(bB[3 + c], o, 64));
          }
        }
        if (sub == 0) {
          const int slot = atomicAdd(&qcount[nxt], 2);
          if (slot + 1 >= SUB_QMAX) {
            atomicOr(&counters[CNT_ERR], TERR_QUEUE);
          } else {
            qn[nxt][slot] = il; ql[nxt][slot] = a0; qh[nxt][slot] = hA;
            qn[nxt][slot + 1] = ir; ql[nxt][slot + 1] = hA + 1; qh[nxt][slot + 1] = a1;
            qx[nxt][slot] = pick_axis(bA);
            qx[nxt][slot + 1] = pick_axis(bB);
          }
        }
      }
      __syncthreads();
      if (tid == 0) qcount[cur] = 0;
      cur ^= 1;
      level++;
      __syncthreads();
    }
    for (int k = tid; k < n; k += SUB_BS) {
      const int s = sub_at(k);
      tx[lo + k] = sx[s]; ty[lo + k] = sy[s]; tz[lo + k] = sz[s]; th[lo + k] = shh[s];
      iparts[lo + k] = sip[k];
    }
    __syncthreads();
  }
  // block max/min of levels
  if (maxlev > 0 || minlev < (1 << 30)) {
    atomicMax(&counters[CNT_MAXLEVEL], maxlev);
    atomicMin(&counters[CNT_MINLEVEL], minlev);
  }
}

// leaves in node-id order (stable compaction over node slots)
__global__ void k_leaf_count(const int32_t *leaf_flag, int64_t ncells, int32_t *bcount) {
  __shared__ int shi[8];
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x + 1;
  int b = (i <= ncells) ? (leaf_flag[i] != 0) : 0;
  int tot;
  block_excl_scan<256>(b, shi, &tot);
  if (threadIdx.x == 0) bcount[blockIdx.x] = tot;
}
// Tile groups (tile.h): the leaf that begins its highest ancestor of at most
// gmax particles marks that node's first tree position.
__global__ void k_leaf_fill(const int32_t *leaf_flag, int64_t ncells, const int32_t *bcount, int32_t *leaves,
                            const int32_t *nd_lo, const int32_t *nd_hi, int gmax, int32_t *tflag, int32_t *tmax) {
  __shared__ int shi[8];
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x + 1;
  int b = (i <= ncells) ? (leaf_flag[i] != 0) : 0;
  int tot;
  int pre = block_excl_scan<256>(b, shi, &tot);
  int m = 0;
  if (b) {
    leaves[bcount[blockIdx.x] + pre] = (int32_t)i;
    int n = (int)i;
    while (n > 1 && nd_hi[n >> 1] - nd_lo[n >> 1] < gmax) n >>= 1;
    if (nd_lo[n] == nd_lo[i]) {
      tflag[nd_lo[n]] = 1;
      m = nd_hi[n] - nd_lo[n] + 1;
    }
  }
  for (int o = 32; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o, 64));
  if ((threadIdx.x & 63) == 0 && m > 0) atomicMax(tmax, m);
}
// first positions of the tile groups in tree order, and the end
__global__ void k_tile_fill(const int32_t *tflag, int n, const int32_t *bcount, const int32_t *ntg, int32_t *tg_lo) {
  __shared__ int shi[8];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int b = (i < n) ? tflag[i] : 0;
  int tot;
  const int pre = block_excl_scan<256>(b, shi, &tot);
  if (b) tg_lo[bcount[blockIdx.x] + pre] = i;
  if (i == 0) tg_lo[*ntg] = n;
}
__global__ void k_pleaf(const int32_t *leaves, int nleaves, const int32_t *nd_lo, const int32_t *nd_hi,
                        int32_t *pleaf) {
  int l = blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= nleaves) return;
  int c = leaves[l];
  for (int p = nd_lo[c]; p <= nd_hi[c]; p++) pleaf[p] = l;
}

// ------------------------------------------------------------------------
int tree_build(phsph_ctx *c, double *d_xyzh, int ld, int np, const int8_t *d_iphase) {
  hipStream_t s = c->stream;
  c->tree_valid = false;
  c->np = np;
  const int64_t maxp = (c->p.maxp > np) ? c->p.maxp : np;
  const int64_t ncellsmax = 2 * maxp;
  c->maxlevel_indexed = (int)(log((double)(ncellsmax + 1)) / log(2.)) - 1;
  const int64_t nidx = ((int64_t)1 << (c->maxlevel_indexed + 1));  // ids 1 .. 2^(L+1)-1
  c->nslots = nidx;
  const unsigned nb = nblocks(np, 256);
  PH_HIPCHECK(c, c->counters.ensure(CNT_N));
  PH_HIPCHECK(c, c->nd.ensure(nidx));
  PH_HIPCHECK(c, c->nd_lo.ensure(nidx));
  PH_HIPCHECK(c, c->nd_hi.ensure(nidx));
  PH_HIPCHECK(c, c->leaf_flag.ensure(nidx));
  PH_HIPCHECK(c, c->tx.ensure(np)); PH_HIPCHECK(c, c->ty.ensure(np));
  PH_HIPCHECK(c, c->tz.ensure(np)); PH_HIPCHECK(c, c->th.ensure(np));
  PH_HIPCHECK(c, c->iparts.ensure(np));
  PH_HIPCHECK(c, c->tmpi.ensure(np)); PH_HIPCHECK(c, c->tmpi2.ensure(np));
  PH_HIPCHECK(c, c->dred.ensure((size_t)nb * 6 + 16));
  // Disjoint sets of particles: the nodes of at most SUB_MAX are at most np,
  // those of at most MID_MAX np/(SUB_MAX+1), the large ones np/(MID_MAX+1)
  // per level, and their chunks at most np/BN_CH + one per node.
  const int mid_cap = np / (SUB_MAX + 1) + 1;
  const int bn_cap = np / (MID_MAX + 1) + 1;
  const int maxch = np / BN_CH + bn_cap + 1;
  PH_HIPCHECK(c, c->small_n.ensure((size_t)np + nb + 2));
  PH_HIPCHECK(c, c->small_x.ensure((size_t)np + 2));
  PH_HIPCHECK(c, c->mid_n.ensure((size_t)mid_cap * 2));
  PH_HIPCHECK(c, c->lev_cnt.ensure((size_t)(MAXLEVELS + 2) * LEV_N));
  PH_HIPCHECK(c, c->bnode.ensure((size_t)bn_cap * 2));
  PH_HIPCHECK(c, c->ch_node.ensure((size_t)maxch * 2));
  PH_HIPCHECK(c, c->ch_i.ensure((size_t)maxch * 4));
  PH_HIPCHECK(c, c->ch_off.ensure((size_t)maxch * 2));
  PH_HIPCHECK(c, c->ch_red.ensure((size_t)maxch * BN_RED));
  // under self-gravity the nodes' second moments about their centres of mass
  // (kdtree.F90:724-750) are formed here
  double *quads = nullptr;
  if (c->p.gravity) {
    PH_HIPCHECK(c, c->quads.ensure((size_t)c->nslots * 6));
    quads = c->quads.p;
  }
  int32_t *live = c->tmpi.p;
  int32_t *bcount = c->small_n.p;  // block counts of the compaction

  // the reference seeds the bounds with particle 1 before wrapping it
  double x0[3];
  PH_HIPCHECK(c, hipMemcpyAsync(x0, d_xyzh, 3 * sizeof(double), hipMemcpyDeviceToHost, s));
  int32_t hc[CNT_N] = {};
  hc[CNT_MINLEVEL] = 1 << 30;
  PH_HIPCHECK(c, dev_set(c, c->counters.p, hc, sizeof(hc)));
  PH_HIPCHECK(c, hipStreamSynchronize(s));
  {
    LaunchTimer lt(c, "tree_root");
    hipLaunchKernelGGL(k_root_wrap, dim3(nb), dim3(256), 0, s, c->dc, d_xyzh, ld, np, live, c->dred.p,
                       c->counters.p);
    hipLaunchKernelGGL(k_count_blocks, dim3(nb), dim3(256), 0, s, live, np, bcount);
    hipLaunchKernelGGL(k_scan_blocks, dim3(1), dim3(1024), 0, s, bcount, (int)nb, c->counters.p + CNT_LIVE);
    hipLaunchKernelGGL(k_fill_cache, dim3(nb), dim3(256), 0, s, c->dc, d_xyzh, ld, np, live, bcount, d_iphase,
                       c->tx.p, c->ty.p, c->tz.p, c->th.p, c->iparts.p);
  }
  PH_HIPCHECK(c, hipGetLastError());
  int32_t cnt[CNT_N];
  PH_HIPCHECK(c, hipMemcpyAsync(cnt, c->counters.p, sizeof(cnt), hipMemcpyDeviceToHost, s));
  PH_HIPCHECK(c, hipStreamSynchronize(s));
  if (cnt[CNT_NAN] > 0) PH_RET(c, PHSPH_ERR_NAN, "maketree: NaN in particle position");
  c->nlive = cnt[CNT_LIVE];
  if (c->nlive == 0) PH_RET(c, PHSPH_ERR_NODATA, "maketree: no particles or all particles dead/accreted");

  double *rootbox = c->dred.p + (size_t)nb * 6;
  hipLaunchKernelGGL(k_root_bounds, dim3(1), dim3(256), 0, s, c->dred.p, (int)nb, x0[0], x0[1], x0[2], rootbox);
  hipLaunchKernelGGL(k_fill_i32, dim3(nblocks(c->nslots, 256)), dim3(256), 0, s, c->leaf_flag.p, c->nslots, 0);
  hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(256), 0, s, c->lev_cnt.p, (int64_t)(MAXLEVELS + 2) * LEV_N, 0);
  int level = 0;
  auto lists = [&](int lv) {  // the lists of nodes whose large ones are of level lv
    NodeLists L;
    L.small = c->small_n.p; L.smallx = c->small_x.p;
    L.mid = c->mid_n.p; L.midx = c->mid_n.p + mid_cap;
    L.bn = c->bnode.p + (size_t)(lv & 1) * bn_cap;
    L.ch_node = c->ch_node.p + (size_t)(lv & 1) * maxch;
    L.lev = c->lev_cnt.p + (size_t)lv * LEV_N;
    L.bncap = bn_cap; L.maxch = maxch;
    L.counters = c->counters.p;
    return L;
  };
  hipLaunchKernelGGL(k_tree_seed, dim3(1), dim3(64), 0, s, rootbox, c->nlive, c->nd_lo.p, c->nd_hi.p, lists(0));
  const bool dbg = getenv("PHSPH_DEBUG") != nullptr;
  int nmid = (c->nlive > SUB_MAX && c->nlive <= MID_MAX) ? 1 : 0;
  if (c->nlive > MID_MAX) {
    LaunchTimer lt(c, "tree_bignodes");
    int32_t *cnt_d = c->counters.p;
    while (true) {
      const NodeLists L = lists(level), Ln = lists(level + 1);
      BigNode *bn = L.bn;
      const int32_t *chn = L.ch_node, *lev = L.lev;
      // at most 2^level large nodes, and chunks of BN_CH with one part chunk a node
      const int gn = (level < 20) ? std::min(bn_cap, 1 << level) : bn_cap;
      const int gch = std::min(maxch, c->nlive / BN_CH + gn);
      hipLaunchKernelGGL(k_bn_sums, dim3(gch), dim3(BN_BS), 0, s, c->dc, bn, chn, bn_cap, maxch, lev, c->tx.p, c->ty.p,
                         c->tz.p, c->th.p, c->ch_red.p);
      hipLaunchKernelGGL(k_bn_centre, dim3(gn), dim3(64), 0, s, c->dc, bn, bn_cap, maxch, lev, c->ch_red.p);
      hipLaunchKernelGGL(k_bn_amb, dim3(gch), dim3(BN_BS), 0, s, bn, chn, bn_cap, maxch, lev, c->tx.p, c->ty.p,
                         c->tz.p, c->ch_i.p);
      hipLaunchKernelGGL(k_bn_seq, dim3(gn), dim3(SEQ_BS), 0, s, c->dc, bn, bn_cap, maxch, lev, cnt_d, c->ch_i.p,
                         c->tx.p, c->ty.p, c->tz.p);
      hipLaunchKernelGGL(k_bn_size, dim3(gch), dim3(BN_BS), 0, s, c->dc, bn, chn, bn_cap, maxch, lev, c->tx.p, c->ty.p,
                         c->tz.p, c->ch_red.p, c->ch_i.p, quads ? 1 : 0);
      hipLaunchKernelGGL(k_bn_node, dim3(gn), dim3(64), 0, s, bn, bn_cap, maxch, lev, cnt_d, c->ch_red.p, c->ch_i.p,
                         c->nd.p, c->leaf_flag.p, level, c->maxlevel_indexed, c->nslots, quads);
      hipLaunchKernelGGL(k_bn_pcount, dim3(gch), dim3(BN_BS), 0, s, bn, chn, bn_cap, maxch, lev, c->tx.p, c->ty.p,
                         c->tz.p, c->ch_i.p);
      hipLaunchKernelGGL(k_bn_pscan, dim3(gn), dim3(64), 0, s, bn, bn_cap, maxch, lev, cnt_d, c->ch_i.p, c->ch_off.p);
      hipLaunchKernelGGL(k_bn_pscatter, dim3(gch), dim3(BN_BS), 0, s, bn, chn, bn_cap, maxch, lev, c->tx.p, c->ty.p,
                         c->tz.p, c->ch_off.p, c->tmpi.p, c->tmpi2.p);
      hipLaunchKernelGGL(k_bn_swap, dim3(gch), dim3(BN_BS), 0, s, bn, chn, bn_cap, maxch, lev, c->tmpi.p, c->tmpi2.p,
                         c->tx.p, c->ty.p, c->tz.p, c->th.p, c->iparts.p, c->ch_red.p);
      hipLaunchKernelGGL(k_bn_finish, dim3(gn), dim3(64), 0, s, bn, bn_cap, maxch, lev, c->ch_red.p, c->nd_lo.p,
                         c->nd_hi.p, Ln);
      PH_HIPCHECK(c, hipGetLastError());
      level++;
      // the largest node of a level holds at least nlive / 2^level particles:
      // while that is a large one there is a next level without asking
      if (level < 20 && ((int64_t)MID_MAX << level) < (int64_t)c->nlive) continue;
      int32_t lc[LEV_N];
      PH_HIPCHECK(c, hipMemcpyAsync(lc, Ln.lev, sizeof(lc), hipMemcpyDeviceToHost, s));
      PH_HIPCHECK(c, hipMemcpyAsync(cnt, c->counters.p, sizeof(cnt), hipMemcpyDeviceToHost, s));
      PH_HIPCHECK(c, hipStreamSynchronize(s));
      nmid = cnt[CNT_NMID];
      if (cnt[CNT_ERR] || lc[LEV_NBIG] == 0) break;
      if (level > MAXLEVELS) PH_RET(c, PHSPH_ERR_CAPACITY, "maketree: more than 64 levels");
    }
  }
  if (!cnt[CNT_ERR] && nmid > 0) {
    LaunchTimer lt(c, "tree_midnodes");
#define MID(QQ)                                                                                                     \
  hipLaunchKernelGGL((k_mid<QQ>), dim3(std::min(nmid, mid_cap)), dim3(MID_BS), 0, s, c->dc, c->tx.p, c->ty.p,         \
                     c->tz.p, c->th.p, c->iparts.p, c->nd_lo.p, c->nd_hi.p, c->nd.p, c->leaf_flag.p,                  \
                     c->maxlevel_indexed, c->nslots, quads, lists(level + 1))
    if (quads) MID(true); else MID(false);
#undef MID
  }
  if (!cnt[CNT_ERR]) {
    LaunchTimer lt(c, "tree_subtrees");
    // nodes of at most SUB_MAX particles have 512 to 1024 in an even set
    const unsigned g = (unsigned)std::min<int64_t>((int64_t)np, 64 + (int64_t)c->nlive / 384);
#define SUBT(QQ)                                                                                                    \
  hipLaunchKernelGGL((k_subtrees<QQ>), dim3(g), dim3(SUB_BS), 0, s, c->dc, c->small_n.p, c->small_x.p, c->tx.p,       \
                     c->ty.p, c->tz.p, c->th.p, c->iparts.p, c->nd_lo.p, c->nd_hi.p, c->nd.p, c->leaf_flag.p,         \
                     c->maxlevel_indexed, c->nslots, quads, c->counters.p)
    if (quads) SUBT(true); else SUBT(false);
#undef SUBT
  }
  PH_HIPCHECK(c, hipGetLastError());
  PH_HIPCHECK(c, hipMemcpyAsync(cnt, c->counters.p, sizeof(cnt), hipMemcpyDeviceToHost, s));
  PH_HIPCHECK(c, hipStreamSynchronize(s));
  if (dbg)
    fprintf(stderr, "maketree: %d levels of large nodes, %d middle nodes, %d subtrees, %d sums in order, longest %d\n",
            level, nmid, cnt[CNT_NSMALL], cnt[CNT_FALLBACK], cnt[CNT_SEQMAX]);
  if (cnt[CNT_ERR] & TERR_NODEID)
    PH_RET(c, PHSPH_ERR_CAPACITY,
           "maketree: tree deeper than maxlevel_indexed; pass a larger maxp (ncellsmax = 2*maxp)");
  if (cnt[CNT_ERR]) PH_RET(c, PHSPH_ERR_STATE, "maketree: internal queue overflow");
  c->maxlevel = cnt[CNT_MAXLEVEL];
  c->minlevel = cnt[CNT_MINLEVEL];
  c->ncells = (c->maxlevel < c->maxlevel_indexed) ? (((int64_t)1 << (c->maxlevel + 1)) - 1)
                                                  : (((int64_t)1 << (c->maxlevel_indexed + 1)) - 1);
  c->tree_fallbacks = cnt[CNT_FALLBACK];
  // leaves in node-id order
  const unsigned nbl = nblocks(c->ncells, 256);
  const unsigned nbt = nblocks(c->nlive, 256);
  PH_HIPCHECK(c, c->tmpi2.ensure((size_t)std::max(nbl, nbt) + 1));
  // Nodes of a level hold about nlive / 2^level particles: the tile limit of
  // 64 or 80 that fills wavefronts of 16 better (a mean of 60 to 76 mostly
  // passes 64, and half nodes of 30 to 38 would leave part of a third
  // wavefront idle; any other mean, or its half, stays below 64)
  double mean = (double)c->nlive;
  while (mean > 76.) mean *= 0.5;
  const int gmax = (mean > 60.) ? 80 : 64;
  // at most one group per leaf
  PH_HIPCHECK(c, c->tg_lo.ensure((size_t)c->nlive + 2));
  PH_HIPCHECK(c, c->leaves.ensure(c->nlive + 1));
  PH_HIPCHECK(c, c->pleaf.ensure(c->nlive + 1));
  {
    LaunchTimer lt(c, "tree_leaves");
    hipLaunchKernelGGL(k_fill_i32, dim3(nbt), dim3(256), 0, s, c->tmpi.p, (int64_t)c->nlive, 0);
    hipLaunchKernelGGL(k_leaf_count, dim3(nbl), dim3(256), 0, s, c->leaf_flag.p, c->ncells, c->tmpi2.p);
    hipLaunchKernelGGL(k_scan_blocks, dim3(1), dim3(1024), 0, s, c->tmpi2.p, (int)nbl,
                       c->counters.p + CNT_NLEAF);
    hipLaunchKernelGGL(k_leaf_fill, dim3(nbl), dim3(256), 0, s, c->leaf_flag.p, c->ncells, c->tmpi2.p,
                       c->leaves.p, c->nd_lo.p, c->nd_hi.p, gmax, c->tmpi.p, c->counters.p + CNT_TGMAX);
    hipLaunchKernelGGL(k_count_blocks, dim3(nbt), dim3(256), 0, s, c->tmpi.p, c->nlive, c->tmpi2.p);
    hipLaunchKernelGGL(k_scan_blocks, dim3(1), dim3(1024), 0, s, c->tmpi2.p, (int)nbt, c->counters.p + CNT_NTG);
    hipLaunchKernelGGL(k_tile_fill, dim3(nbt), dim3(256), 0, s, c->tmpi.p, c->nlive, c->tmpi2.p,
                       c->counters.p + CNT_NTG, c->tg_lo.p);
  }
  PH_HIPCHECK(c, hipMemcpyAsync(cnt, c->counters.p, sizeof(cnt), hipMemcpyDeviceToHost, s));
  PH_HIPCHECK(c, hipStreamSynchronize(s));
  c->nleaves = cnt[CNT_NLEAF];
  c->ntg = cnt[CNT_NTG];
  c->tg_max = cnt[CNT_TGMAX];
  hipLaunchKernelGGL(k_pleaf, dim3(nblocks(c->nleaves, 256)), dim3(256), 0, s, c->leaves.p, c->nleaves,
                     c->nd_lo.p, c->nd_hi.p, c->pleaf.p);
  PH_HIPCHECK(c, hipGetLastError());
  c->tree_valid = true;
  // statistics of a density call belong to the tree it ran on
  c->nact_dens = 0;
  c->trial_stale = true;
  c->nrhocalc = -1;
  c->nactualtot = -1;
  if (c->p.gravity) return grav_tree(c);
  return PHSPH_OK;
}
