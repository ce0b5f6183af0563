/*
 * deblend.hip -- multi-threshold deblending (init_deblend, parcel_out, clear_deblend;
 * the reference's src/cuda/cudadeblend.cu:508, :579, :1937).
 *
 * Semantics (cudadeblend.cu:199-483, :579-1615; cudaanalyse.cu:1686-1904):
 *   t_i = (float)(t0 * pow(fdpeak/t0, i/N)) per raw object, i = 1..N-1;
 *   level i holds the pixels of the kept level-(i-1) components with cd >= t_i, split
 *   into 8-connected components labelled by their first raster pixel; components with
 *   fewer than deb_minarea pixels are dropped; each kept component records its parent
 *   (the level-(i-1) component containing it), pixel count, and the float sum of cd over
 *   its pixels in raster order;
 *   a component is significant when fdflux - t_i*npix > fdflux_root*DEBLEND_MINCONT;
 *   A(c) = [fewer than two significant children] and A of every child;
 *   a level-0 object is kept when A(root); a deeper one when its parent has at least
 *   two significant children, it is significant, and A(c);
 *   kept objects are ordered by root, then level, then first pixel; each is preanalysed
 *   over its level pixels (FULL, cudaanalyse.cu:1686-1904), and every other pixel of the
 *   root goes to the kept object of the same root that minimises
 *   0.5*(cxx dx^2 + cyy dy^2 + cxy dx dy)/abcor (gatherup, cudadeblend.cu:1262-1360).
 *
 * Two facts about these level sets reduce the work without changing any result.
 * Let tau_i = max(t_1..t_i) and V_i = {p in the raw object : cd[p] >= tau_i}.
 *   (1) Every component of level i is a component of V_i, and every component of V_i
 *       with at least deb_minarea pixels is a kept component of level i (its ancestors
 *       are larger, hence kept).  So the kept components of level i are the components
 *       of V_i with >= deb_minarea pixels: no level needs the previous level's labels
 *       to decide membership, only a per-pixel level index m(p) = max{i : tau_i <= cd}.
 *   (2) The highest pixel of a component of V_i is a local maximum of cd over the raw
 *       object (no 8-neighbour in the object is higher), with value >= tau_i.  So a
 *       level with two or more components needs two local maxima >= tau_i: with v2 the
 *       second-highest local maximum, every level with tau_i > v2 holds at most one
 *       component.  Nodes at or below such levels have at most one child, which makes
 *       them irrelevant to A() and never kept; levels are processed only up to
 *       L* = (first i with tau_i > v2) - 1, and a raw object with a single local
 *       maximum (L* = 0) is kept as it is without any level work.
 *
 * Kernels:
 *   k_deb_thresh     one lane per (object, level): the sub-thresholds (canonical pow)
 *   k_deb_lmax<0,1>  one lane per raw pixel: local maxima (flagged per pixel); per object
 *                    their number, the highest (packed value and index, 64-bit
 *                    atomicMax), then, over the flagged pixels only, the second-highest
 *   k_deb_lsfirst    one lane per (object, level): L* from the second-highest maximum
 *   k_deb_nodecap    one lane per object: a bound on its kept nodes, scanned into the
 *                    node table's regions
 *   k_deb_classify   one lane per object: single-peak objects are finished; the rest are
 *                    binned by size into classes
 *   k_deb_tree_lds   one workgroup per object (256, 512 or 1024 lanes by class; the classes
 *                    run side by side on their own streams), all state in LDS: the
 *                    component tree as a max-tree (see deb_tree)
 *   k_deb_order      the objects too large for that, largest first
 *   k_deb_tree_glb   the same code for them, with only the parent words and level indices in
 *                    LDS
 *   k_deb_wide_*     the same passes over the pixels of the objects above 29,696 pixels, a
 *                    kernel each, all state in global memory
 *   k_deb_objlist    one wavefront per raw object: its kept nodes -> objects
 *   k_deb_pre        a row of 16 lanes, a wavefront or a workgroup per object: FULL
 *                    preanalysis over the node's level pixels (kcomp names them; lanes compute
 *                    the terms, the sums are folded in raster order: sxg_wave.h)
 *   k_deb_gather     one lane per raw pixel: gatherup of the pixels no kept node holds
 *   then the raw pixels are regrouped by object, stably (opix, objoff): every later
 *   per-object pass reads one contiguous raster-ordered range
 */
#include <algorithm>
#include <cmath>

#include "sxg_internal.h"
#include "sxg_objects.h"
#include "sxg_wave.h"

/* size classes of the raw objects with a tree (k_deb_classify), and the words of the
   per-frame counter block (DebArgs::ccount): objects per class, the largest LDS need of
   classes 0..2, pixels per class (3 and 4 together) */
#define DEB_NCLASS 5
#define DEB_CLDS DEB_NCLASS
#define DEB_CPIX (DEB_CLDS + 3)
#define DEB_NCOUNT (DEB_CPIX + 4)
/* pixels of the largest tree that one workgroup builds (class 3; above: class 4) */
#define DEB_HALF 29696
/* rounds of path shortening before the joins */
#define DEB_JUMPS 3

/* unsigned order-preserving key of a float (0 is below every non-NaN value) */
__device__ inline unsigned uord(float v) { return (unsigned)f2ord(v) ^ 0x80000000u; }
__device__ inline float uord_inv(unsigned u) { return ord2f((int)(u ^ 0x80000000u)); }

/* ---------------------------------------------------------------- thresholds ---- */
/* the base of object r: basethresh, or with per-pixel thresholds (weight map) the
   lowest threshold among the object's pixels, rawt0[r] */
__global__ void __launch_bounds__(256) k_deb_thresh(const float *__restrict__ fdpeak, int nraw,
                                                    int nthresh, float basethresh,
                                                    const float *__restrict__ rawt0, int perpix,
                                                    float *thr, const PlanDev *pd)
{
    const long k = (long)blockIdx.x * 256 + threadIdx.x;
    if (pd) {
        nraw = pd->nraw;
        basethresh = pd->dthresh;
    }
    if (k >= (long)nraw * nthresh) return;
    const int r = (int)(k / nthresh), i = (int)(k - (long)r * nthresh);
    const float b = perpix ? rawt0[r] : basethresh;
    const double t0 = (double)b, pk = (double)fdpeak[r];
    thr[k] = i == 0 ? b : (float)(t0 * sx_pow(pk / t0, (double)i / nthresh));
}


/* ------------------------------------------------------------------- levels ---- */
/* LDS bytes per pixel of k_deb_tree_lds: the sum (8), parent and count words (4 each), the
   list entry (2), the level index */
#define DEB_LDS_BYTES_PER_PIX 19
/* LDS a workgroup may use (dynamic part; the static part of deb_tree is under 3 KiB) */
#define DEB_LDS_LIMIT ((size_t)160 * 1024 - 4096)

/* LDS of k_deb_tree_lds for a tree over n pixels */
__host__ __device__ inline int deb_lds_bytes(int n)
{
    return ((n + 63) & ~63) * DEB_LDS_BYTES_PER_PIX;
}

struct DebArgs {
    const int *fpia;        /* raw pixel list (raster order within each raw object) */
    const int *rawkey;      /* raw object id of each raw-list entry */
    const int *off, *cnt, *first, *xmin, *xmax;   /* raw objects */
    const float *cd;
    const int *lab;         /* detection labels (root pixel of each detected pixel) */
    int *kcomp;             /* kcomp[g]: the kept node (of a raw object with a tree) whose
                               level pixels hold the raw pixel g, or -1 */
    long P0;
    const float *thr;       /* thr[r * nthresh + i] */
    int nthresh, debarea;
    double mincont;
    int W, H, nraw;
    int cstride;            /* entries per class in clist (nraw, or its capacity) */
    const PlanDev *pd;      /* planned run: the device counts (nraw, npix), else nullptr */
    Comp *comps;            /* output node table, region compoff[r] of each raw object */
    int *compoff;           /* node capacity of each raw object, then its region */
    int *rootnc;            /* kept nodes per raw object */
    int *rootkept;          /* kept objects per raw object */
    unsigned long long *top1;   /* highest local maximum: uord(cd) << 32 | raw-list index */
    unsigned *top2;         /* uord(cd) of the second-highest local maximum, 0 if none */
    int *nmax;              /* local maxima per raw object */
    unsigned char *lmflag;  /* per raw-list entry: 1 for a local maximum (first pass) */
    int *lstar;             /* first level above the second-highest maximum, then L* */
    int *clist;             /* objects of each size class: clist[cls * nraw + j] */
    int *ccount;            /* DEB_NCOUNT counters */
    unsigned long long *dwork;  /* [0] pixels, [1] pixel-levels of the multi-peak objects,
                                   [2] node capacity of the frame */
    /* global scratch for the objects built in global memory, by raw-list position, and a
       record for each of class 4 */
    double *g_sum;
    unsigned long long *g_par, *g_cnt;
    int *g_list;
    unsigned char *g_m;
    struct DebWide *wide;
};

/* the raw objects and their pixels: the device counts of a planned run */
__device__ inline int deb_nraw(const DebArgs &a) { return a.pd ? a.pd->nraw : a.nraw; }
__device__ inline long deb_P0(const DebArgs &a) { return a.pd ? (long)a.pd->npix : a.P0; }
/* PASS 0: local maxima (no 8-neighbour of the raw object is higher): the highest of each
   raw object and their number; PASS 1: the highest of the others */
template <int PASS> __global__ void __launch_bounds__(256) k_deb_lmax(DebArgs a)
{
    const long g = (long)blockIdx.x * 256 + threadIdx.x;
    if (g >= deb_P0(a)) return;
    /* the second pass visits the local maxima the first one flagged */
    if (PASS == 1 && !a.lmflag[g]) return;
    const int p = a.fpia[g], r = a.rawkey[g];
    const float v = a.cd[p];
    if (PASS == 0) {
        const int root = a.lab[p];
        const int W = a.W, H = a.H;
        const int y = p / W, x = p - y * W;
        /* the eight neighbours' labels and values, loaded unconditionally from positions
           clamped into the frame (all sixteen loads in flight together), then compared;
           a position outside the frame takes no part */
        int lq[8], inb[8];
        float cq[8];
#pragma unroll
        for (int n = 0; n < 8; n++) {
            const int dd = n < 4 ? n : n + 1;   /* the 3x3 neighbourhood without its centre */
            const int yy = y + dd / 3 - 1, xx = x + dd % 3 - 1;
            inb[n] = (yy >= 0) & (yy < H) & (xx >= 0) & (xx < W);
            const int q = inb[n] ? yy * W + xx : p;
            lq[n] = a.lab[q];
            cq[n] = a.cd[q];
        }
        int higher = 0;
#pragma unroll
        for (int n = 0; n < 8; n++) higher |= inb[n] & (lq[n] == root) & (cq[n] > v);
        const bool top = higher == 0;
        a.lmflag[g] = top ? 1 : 0;
        if (!top) return;
    }
    const unsigned u = uord(v);
    const unsigned long long key = ((unsigned long long)u << 32) | (unsigned)g;
    if (PASS == 0) {
        atomicMax(&a.top1[r], key);
        atomicAdd(&a.nmax[r], 1);
    } else if (a.top1[r] != key) {
        atomicMax(&a.top2[r], u);
    }
}

__global__ void __launch_bounds__(256) k_deb_prep(DebArgs a)
{
    const int r = blockIdx.x * 256 + threadIdx.x;
    if (r < DEB_NCOUNT) a.ccount[r] = 0;
    if (r < 3) a.dwork[r] = 0ull;
    if (r >= deb_nraw(a)) return;
    a.top1[r] = 0ull;
    a.top2[r] = 0u;
    a.nmax[r] = 0;
    a.lstar[r] = a.nthresh;
}

/* one lane per (raw object, level >= 1): the first level whose running-maximum
   sub-threshold tau exceeds the second-highest local maximum (tau_i > v2 iff some
   t_j > v2, j <= i; a NaN sub-threshold empties its level and ends the descent) */
__global__ void __launch_bounds__(256) k_deb_lsfirst(DebArgs a)
{
    const long k = (long)blockIdx.x * 256 + threadIdx.x;
    const int N = a.nthresh;
    if (k >= (long)deb_nraw(a) * N) return;
    const int r = (int)(k / N), i = (int)(k - (long)r * N);
    const unsigned u2 = a.top2[r];
    if (i == 0 || u2 == 0u) return;
    const float t = a.thr[k];
    if (t != t || t > uord_inv(u2)) atomicMin(&a.lstar[r], i);
}

/* kept nodes of an object, at most: they are disjoint, each with at least deb_minarea
   pixels and a local maximum (its highest pixel); one where the object is kept whole */
__host__ __device__ inline int deb_nodecap(int nmax, int n, int ls, int debarea)
{
    return ls == 0 ? 1 : max(1, min(nmax, n / debarea));
}

/* L* and the node capacity of each raw object (the total in 64 bits: one atomic per
   wavefront) */
__global__ void __launch_bounds__(256) k_deb_nodecap(DebArgs a)
{
    const int r = blockIdx.x * 256 + threadIdx.x;
    unsigned long long c = 0;
    if (r < deb_nraw(a)) {
        const int ls = a.top2[r] == 0u ? 0 : a.lstar[r] - 1;
        a.lstar[r] = ls;
        const int cap = deb_nodecap(a.nmax[r], a.cnt[r], ls, a.debarea);
        a.compoff[r] = cap;
        c = (unsigned long long)cap;
    }
    for (int d = 32; d > 0; d >>= 1) c += __shfl_xor(c, d);
    if ((threadIdx.x & 63) == 0 && c) atomicAdd(&a.dwork[2], c);
}

/* single-peak objects are kept as they are (one node); the others go to a size class (0:
   up to cap0 pixels, 256 lanes in LDS; 1: up to cap1, 512 lanes in LDS; 2: up to cap2, 1024
   lanes in LDS; 3: up to DEB_HALF, one workgroup with its sums in global memory; 4: the whole
   chip).  The counters take one atomic per workgroup and class (one per wavefront, as the
   order kernels had, took 19 us for 22,000 raw objects, 7 now). */
__global__ void __launch_bounds__(256) k_deb_classify(DebArgs a, int cap0, int cap1, int cap2)
{
    __shared__ int s_n[DEB_NCLASS], s_px[DEB_NCLASS], s_need[DEB_NCLASS], s_base[DEB_NCLASS];
    __shared__ unsigned long long s_work[2];
    const int r = blockIdx.x * 256 + threadIdx.x;
    const int lane = threadIdx.x & 63;
    if (threadIdx.x < DEB_NCLASS)
        s_n[threadIdx.x] = s_px[threadIdx.x] = s_need[threadIdx.x] = 0;
    if (threadIdx.x < 2) s_work[threadIdx.x] = 0;
    __syncthreads();
    int cls = -1, n = 0, ls = 0, need = 0;
    if (r < deb_nraw(a)) {
        n = a.cnt[r];
        ls = a.lstar[r];
        if (ls == 0) {
            a.rootnc[r] = 1;
            a.rootkept[r] = 1;
        } else {
            need = deb_lds_bytes(n);
            cls = n <= cap0 ? 0 : n <= cap1 ? 1 : n <= cap2 ? 2 : n <= DEB_HALF ? 3 : 4;
        }
    }
    unsigned long long w0 = cls >= 0 ? (unsigned long long)n : 0ull;
    unsigned long long w1 = cls >= 0 ? (unsigned long long)n * ls : 0ull;
    for (int d = 32; d > 0; d >>= 1) {
        w0 += __shfl_xor(w0, d);
        w1 += __shfl_xor(w1, d);
    }
    if (lane == 0 && w0) {
        atomicAdd(&s_work[0], w0);
        atomicAdd(&s_work[1], w1);
    }
    int slot = 0;
    for (int c = 0; c < DEB_NCLASS; c++) {
        const unsigned long long b = __ballot(cls == c);
        if (!b) continue;
        const int lead = __builtin_ctzll(b);
        int base = 0;
        if (lane == lead) base = atomicAdd(&s_n[c], __popcll(b));
        base = __shfl(base, lead);
        int mx = cls == c ? need : 0, px = cls == c ? n : 0;
        for (int d = 32; d > 0; d >>= 1) {
            mx = max(mx, __shfl_xor(mx, d));
            px += __shfl_xor(px, d);
        }
        if (lane == lead) {
            atomicMax(&s_need[c], mx);
            atomicAdd(&s_px[c], px);
        }
        if (cls == c) slot = base + __popcll(b & sxw_lanes_below(lane));
    }
    __syncthreads();
    if (threadIdx.x < DEB_NCLASS && s_n[threadIdx.x]) {
        const int c = threadIdx.x;
        s_base[c] = atomicAdd(&a.ccount[c], s_n[c]);
        if (c < 3) atomicMax(&a.ccount[DEB_CLDS + c], s_need[c]);
        atomicAdd(&a.ccount[DEB_CPIX + min(c, 3)], s_px[c]);
    }
    if (threadIdx.x >= 64 && threadIdx.x < 66 && s_work[threadIdx.x - 64])
        atomicAdd(&a.dwork[threadIdx.x - 64], s_work[threadIdx.x - 64]);
    __syncthreads();
    if (cls >= 0) a.clist[(size_t)cls * a.cstride + s_base[cls] + slot] = r;
}

/*
 * Significance test fdflux - t*npix > fdflux_root * DEBLEND_MINCONT, where fdflux is the
 * float sum of cd over the component's pixels in raster order, decided from bounds.
 * s and sabs are the exact-to-double sums of cd and |cd| (any order); the sequential
 * float sum differs from s by at most gamma_{n-1} * sabs, gamma_m = m u / (1 - m u),
 * u = 2^-24 (recursive summation, Higham, Accuracy and Stability of Numerical
 * Algorithms, 2nd ed., eq. 4.4), plus the double rounding of s itself.  The float
 * subtraction and the final comparison are bracketed the same way.  Returns 1 or 0 when
 * the bounds decide, -1 when the exact sequential sum is needed.
 */
__device__ inline double deb_sum_err(double sabs, int n)
{
    const double m = (double)(n > 1 ? n - 1 : 1) * 0x1p-24;
    if (m >= 0.5) return INFINITY;
    return sabs * (m / (1.0 - m) + (double)n * 0x1p-52) * 1.0001;
}

__device__ inline int deb_sig_bound(double s, double sabs, int n, float b, double v0lo,
                                    double v0hi)
{
    const double e = deb_sum_err(sabs, n);
    double lo = (s - e) - (double)b, hi = (s + e) - (double)b;
    lo -= fabs(lo) * 0x1p-23 + 1e-37;
    hi += fabs(hi) * 0x1p-23 + 1e-37;
    if (lo > v0hi) return 1;
    if (hi <= v0lo) return 0;
    return -1;
}

/*
 * The component tree of a raw object, found as a max-tree: one pass over the pixel pairs,
 * no pass over the pixels per level.
 *
 * With m(k) the level index of pixel k (V_i = {k : m(k) >= i}), the components of the level
 * sets nest.  Every pixel has a parent word: a pixel of the same level and component with a
 * smaller index (so that the pixels of a level's component form a union-find set, its root
 * the first of them in raster order), or, for such a root, a pixel of the next lower level
 * on which its component of V_m(root) grows into a larger one; 0 where there is none (below
 * is the whole object, level 0).  A word holds the parent's level over its complemented
 * index: of two candidates for the same pixel the larger word is the closer one, so
 * atomicMax keeps it and returns what it replaced, and joining two pixels (deb_join) is
 * lock-free (the merge of two root paths of Wilkinson et al., Concurrent computation of
 * attribute filters on shared memory parallel machines, IEEE TPAMI 30(10), 2008, by atomicMax
 * instead of under locks or phases): climb both to the roots of the lower pixel's level, hang
 * the deeper root below
 * the other, go on with the other root and the parent that was replaced (or kept).  Every
 * step keeps, for each level, the components that the pairs joined so far (and the pairs in
 * hand) make up, so at the end the parents are the tree whatever the order.
 *
 * A root of level j with parent level i stands for the nodes of levels i + 1 ... j, which
 * hold the same pixels: the same children, the same A(); the level that matters for
 * significance and for the kept object is i + 1, where it is one of its parent's children.
 * Nodes with fewer than deb_minarea pixels are no nodes (their subtrees have fewer still).
 * Node sums go up level by level (the roots sorted by level); significance is tested for
 * the children of nodes with two or more, by bounds first; then two or more significant
 * children void A() of a node and of those above it.
 *
 * Bound: latency of dependent LDS (or L2) accesses, half of it in the joins (12 us for 3,000
 * pixels in 1024 lanes, 55 us for 6,000 in a dense frame), then one barrier per level.  The
 * levels were walked one by one before, with five passes over all pixels each (13 us a level
 * for 4,370 pixels).  Measured, before and after: crowded 4096^2, classes 0, 1, 2: 276, 167,
 * 229 -> 76, 50, 46 us; dense 2048^2, class 3 (40 objects of 6,000 to 20,000 pixels) 2,617 ->
 * 472 us with par and m in LDS (1,470 with all state in global memory), 380 with the exact
 * flux of the object ahead of those of its nodes.  Objects of more
 * pixels than that LDS holds (class 4) are built by the whole chip: k_deb_wide_levels.  Lanes: class 0 with
 * 64 lanes 138 us, class 1 with 256 lanes 73 us (more pixels a lane, one after the other).
 * Left out: the pixels entering level by level from the highest (each join is short then,
 * but a level costs two barriers and 3 us of contended joins whatever its size: class 2 46
 * -> 115 us).
 */
/* WIDE: objects of 65536 pixels and more */
template <bool WIDE> struct DebWord;
template <> struct DebWord<false> { typedef unsigned T; };
template <> struct DebWord<true> { typedef unsigned long long T; };
/* words that other wavefronts of the workgroup change: from LDS, or for global memory (G)
   from the device-coherent level */
template <bool G, class V> __device__ inline V deb_ld(const V *p)
{
    if (G) return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
template <bool G, class V> __device__ inline void deb_st(V *p, V v)
{
    if (G) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
/* all accesses of the workgroup before it are done (G: those to global memory too) */
template <bool G> __device__ inline void deb_sync()
{
    if (G) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __syncthreads();
}

template <bool WIDE> struct DebTree {
    typedef typename DebWord<WIDE>::T T;
    static constexpr int SH = WIDE ? 32 : 16;       /* level bits above the index */
    static constexpr T IM = ((T)1 << SH) - 1;
    static constexpr int CB = WIDE ? 32 : 24;       /* pixel count of a node, flags above */
    static constexpr T CM = ((T)1 << CB) - 1;
    static constexpr T CH1 = (T)1 << CB, CH2 = (T)2 << CB;       /* one, two children */
    static constexpr T SON1 = (T)4 << CB, SON2 = (T)8 << CB;     /* one, two significant */
    static constexpr T SIG = (T)16 << CB, NOTA = (T)32 << CB;    /* significant; A() void */
    __device__ static int lev(T w) { return (int)(w >> SH); }
    __device__ static int idx(T w) { return (int)(~w & IM); }
    __device__ static T word(int level, int x) { return ((T)level << SH) | (~(T)x & IM); }
    /* par and m where they are kept (PG: global memory, else LDS) */
    template <bool PG> struct Par {
        T *par;
        __device__ T ld(int k) const { return deb_ld<PG>(&par[k]); }
        __device__ void st(int k, T w) const { deb_st<PG>(&par[k], w); }
        /* the root of a's level above a, halving the path on the way; pa: its parent word */
        __device__ int root(int a, int ma, T &pa) const
        {
            pa = ld(a);
            while (lev(pa) == ma) {
                const int b = idx(pa);
                const T gp = ld(b);
                if (lev(gp) == ma) atomicMax(&par[a], gp);
                a = b;
                pa = gp;
            }
            return a;
        }
        __device__ void join(int a, int ma, int b, int mb) const
        {
            while (true) {
                T pa, pb;
                a = root(a, ma, pa);
                b = root(b, mb, pb);
                if (a == b) return;
                if (ma < mb || (ma == mb && a < b)) {
                    const int t = a, tm = ma;
                    a = b;
                    ma = mb;
                    b = t;
                    mb = tm;
                    pa = pb;
                }
                /* a is the deeper one, or the later one of a level */
                if (ma > mb && lev(pa) >= mb) {
                    a = idx(pa);
                    ma = lev(pa);
                    continue;
                }
                const T w = word(mb, b), old = atomicMax(&par[a], w);
                if (old == 0 || old == w) return;
                a = b;
                ma = mb;
                b = idx(old);
                mb = lev(old);
            }
        }
    };
};

/* float sum of val(k) over k < n with sel(k), in increasing k, by one wavefront (every lane
   returns it); ends once `need` values are in.  Four 64-entry chunks are tested and read
   together, so their loads are in flight at once; a value left out adds +0, an identity. */
template <class Sel, class Val>
__device__ inline float wave_ordered_sum(int n, Sel sel, Val val, int need)
{
    const int lane = threadIdx.x & 63;
    float f = 0.0f;
    int got = 0;
    for (int base = 0; base < n && got < need; base += 4 * 64) {
        bool in[4];
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int k = base + u * 64 + lane;
            in[u] = k < n && sel(k);
        }
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = in[u] ? val(base + u * 64 + lane) : 0.0f;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const unsigned long long b = __ballot(in[u]);
            got += __popcll(b);
            if (b) f = sxw_fold64(f, v[u]);
        }
    }
    return f;
}

/*
 * The passes over the pixels of one object.  WIDE: parent words of 64 bits and level indices in
 * global memory, written by several workgroups in turn; else in LDS.  G: the other arrays in
 * global memory.  Per raw-list index of the object: sum (its cd, then the sum of a node; later
 * two int arrays), par, cnt (while the neighbours are found the pixel list, in LDS; then count
 * and flags of a node, later the order key of a kept node), list (the neighbours, then the roots
 * by level), m.
 */
template <bool WIDE, bool G, class IT> struct DebObj {
    typedef DebTree<WIDE> D;
    typedef typename D::T T;
    typename D::template Par<WIDE> par;
    double *sum;
    T *cnt;
    IT *list;
    unsigned char *m;
    const int *pl;     /* the pixels */
    int n, W, span;    /* span: list entries that may lie between a pixel and its row above */

    /* levels of the neighbours (0: none), their places, and which of them is the first
       parent: 1 W, 2 NW, 3 N, 4 NE, 0 none; same: W of the pixel's level */
    struct Nb {
        int mw, mnw, mn, mne, j0, jn, jne, first;
        bool same;
    };
    __device__ Nb around(int k, int mk, int enc, bool west) const
    {
        Nb q;
        q.j0 = k - (enc >> 3);
        q.jn = q.j0 + (enc & 1);
        q.jne = q.jn + ((enc >> 1) & 1);
        q.mw = west ? m[k - 1] & 63 : 0;
        q.mnw = (enc & 1) ? m[q.j0] & 63 : 0;
        q.mn = (enc & 2) ? m[q.jn] & 63 : 0;
        q.mne = (enc & 4) ? m[q.jne] & 63 : 0;
        q.same = q.mw == mk;
        if (q.same) q.first = 1;
        else if (q.mnw == mk) q.first = 2;
        else if (q.mn == mk) q.first = 3;
        else if (q.mne == mk) q.first = 4;
        else {
            int best = 0;
            q.first = 0;
            if (q.mw < mk && q.mw > best) best = q.mw, q.first = 1;
            if (q.mnw < mk && q.mnw > best) best = q.mnw, q.first = 2;
            if (q.mn < mk && q.mn > best) best = q.mn, q.first = 3;
            if (q.mne < mk && q.mne > best) best = q.mne, q.first = 4;
        }
        return q;
    }
    /* the neighbours of pixel k in the row above are consecutive list entries, searched for
       among those that can lie between (a row of the object's width on either side of the row's
       end): their distance and which of them are there into list, whether W is into bit 7 of
       m */
    __device__ void look(int k) const
    {
        const int mk = m[k] & 63;
        if (mk == 0) return;
        const int p = pl[k];
        const int y = p / W, x = p - y * W;
        int enc = 0, j0 = k;
        if (y > 0) {
            const int q0 = p - W - (x > 0 ? 1 : 0);
            int l = max(0, k - span), h = k;
            while (l < h) {
                const int mid = (l + h) >> 1;
                if (pl[mid] < q0) l = mid + 1;
                else h = mid;
            }
            int j = j0 = l;
            if (x > 0 && j < k && pl[j] == p - W - 1) enc |= 1, j++;
            if (j < k && pl[j] == p - W) enc |= 2, j++;
            if (x < W - 1 && j < k && pl[j] == p - W + 1) enc |= 4;
        }
        deb_st<G>(&list[k], (IT)(enc | (k - j0) << 3));
        if (x > 0 && k > 0 && pl[k - 1] == p - 1) m[k] = (unsigned char)(mk | 128);
    }
    /* first parents, one pair per pixel, without atomics: a pixel at the head of its run
       (neighbours along the row on one level, inside the wavefront's 64 entries); a head at a
       backward neighbour of its level, else at the one of the highest level below.  Every lane
       of the wavefront calls, with consecutive entries; in: it has a pixel */
    __device__ void first(int k, bool in) const
    {
        const int lane = threadIdx.x & 63;
        const int mk = in ? m[k] & 63 : 0;
        bool same = false;
        Nb q{};
        if (mk > 0) {
            q = around(k, mk, (int)deb_ld<G>(&list[k]), (m[k] & 128) != 0);
            same = q.same && lane > 0;
        }
        const unsigned long long heads = __ballot(!same);
        T w = 0;
        if (mk > 0) {
            if (same)
                w = D::word(mk, k - lane + 63 - __builtin_clzll(heads & (~0ull >> (63 - lane))));
            else if (q.first)
                w = q.first == 1 ? D::word(q.mw, k - 1) : q.first == 2 ? D::word(q.mnw, q.j0)
                    : q.first == 3 ? D::word(q.mn, q.jn) : D::word(q.mne, q.jne);
        }
        if (in) par.st(k, w);
    }
    /* chains of a level cut short: a pixel at its parent's parent (only its own thread
       changes a word here, and every value read is above it on its level) */
    __device__ void shorten(int k) const
    {
        const int mk = m[k] & 63;
        if (mk == 0) return;
        const T w = par.ld(k);
        if (D::lev(w) != mk) return;
        const T g = par.ld(D::idx(w));
        if (D::lev(g) == mk) par.st(k, g);
    }
    /* the other pairs.  One is left out where two others imply it at its level: N through W
       and NW; NW through W or N; NE through N. */
    __device__ void joins(int k) const
    {
        const int mk = m[k] & 63;
        if (mk == 0) return;
        const Nb q = around(k, mk, (int)deb_ld<G>(&list[k]), (m[k] & 128) != 0);
        const int en = min(mk, q.mn), enw = min(mk, q.mnw), ene = min(mk, q.mne);
        if (q.mw > 0 && q.first != 1) par.join(k, mk, k - 1, q.mw);
        if (en > 0 && q.first != 3 && min(q.mw, q.mnw) < en) par.join(k, mk, q.jn, q.mn);
        if (enw > 0 && q.first != 2 && q.mw < enw && q.mn < enw)
            par.join(k, mk, q.j0, q.mnw);
        if (ene > 0 && q.first != 4 && q.mn < ene) par.join(k, mk, q.jne, q.mne);
    }
    /* pixel k at the root of its level, a root at the root above it (a pixel of level 0
       belongs to the whole object only); the level of a root, else 0 */
    __device__ int settle(int k) const
    {
        const int mk = m[k] & 63;
        m[k] = (unsigned char)mk;
        if (mk == 0) return 0;
        const T w = par.ld(k);
        T pw;
        if (D::lev(w) == mk) {
            const int q = par.root(D::idx(w), mk, pw);
            par.st(k, D::word(mk, q));
            return 0;
        }
        if (w) {
            const int q = par.root(D::idx(w), D::lev(w), pw);
            par.st(k, D::word(D::lev(w), q));
        }
        return mk;
    }
    /* pixel k to the kept node that holds it (place: by node, see deb_nodes), and the last
       pixel of each kept node from the last of every run of its pixels.  Every lane of the
       wavefront calls, with consecutive entries; in: it has a pixel */
    __device__ void assign(int k, bool in, const int *slot, const int *place, int *kcomp,
                           Comp *C) const
    {
        const int lane = threadIdx.x & 63;
        int c = -1;
        const int mk = in ? m[k] : 0;
        if (mk > 0) {
            const T w = par.ld(k);
            const int s = deb_ld<G>(&slot[D::lev(w) == mk ? D::idx(w) : k]);
            if (s >= 0) c = deb_ld<G>(&place[s]);
        }
        const int next = __shfl_down(c, 1);
        if (!in) return;
        kcomp[k] = c;
        if (c >= 0 && (lane == 63 || k == n - 1 || next != c)) atomicMax(&C[c].hi, k);
    }
};

/*
 * What follows when the pixels hang on their roots, by one workgroup: the node sums, the
 * significance, A() and the kept nodes (into C, with lo = hi = the first pixel; their number,
 * 0 where there is no split).  s_lev: roots of each level, s_at: where those of a level end in
 * list (highest level first); tthr: sub-thresholds; rsum, rabs: bounds of the root's flux.
 * Leaves in sum the slot of each node, that of its kept node or -1, and from cap on the place
 * of each slot's kept node in C.
 */
template <int NT, bool WIDE, bool G, class IT>
__device__ __forceinline__ int deb_nodes(const DebArgs &a, const DebObj<WIDE, G, IT> &t,
                                         const int *const fp, int cap, int ls, const int *s_lev,
                                         const int *s_at, const float *tthr, double rsum,
                                         double rabs, Comp *C)
{
    typedef DebTree<WIDE> D;
    typedef typename D::T T;
    __shared__ T s_top;              /* flags of level 0, the whole object */
    __shared__ int s_nk, s_nopen, s_open[256];
    __shared__ float s_fr;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const auto par = t.par;
    T *const cnt = t.cnt;
    double *const sum = t.sum;
    IT *const list = t.list;
    const unsigned char *const m = t.m;
    const int n = t.n;
    if (tid == 0) {
        s_top = 0;
        s_nk = s_nopen = 0;
    }
    /* the roots of level i end at s_at[i]; those of level 1 are the last */
    const int nn = s_at[1];
    for (int i = ls; i >= 2; i--) {
        const int e = s_at[i], b = e - s_lev[i];
        if (b == e) continue;
        for (int c = b + tid; c < e; c += NT) {
            const int k = deb_ld<G>(&list[c]);
            const T w = par.ld(k);
            if (w) {
                atomicAdd(&cnt[D::idx(w)], deb_ld<G>(&cnt[k]));
                atomicAdd(&sum[D::idx(w)], deb_ld<G>(&sum[k]));
            }
        }
        deb_sync<G>();
    }
    deb_sync<G>();
    /* children */
    auto mark = [&](T w, T f1, T f2) {
        T *q = w ? &cnt[D::idx(w)] : &s_top;
        if (atomicOr(q, f1) & f1) atomicOr(q, f2);
    };
    auto flags = [&](T w) -> T { return w ? deb_ld<G>(&cnt[D::idx(w)]) : deb_ld<false>(&s_top); };
    for (int c = tid; c < nn; c += NT) {
        const int k = deb_ld<G>(&list[c]);
        if ((int)(deb_ld<G>(&cnt[k]) & D::CM) >= a.debarea) mark(par.ld(k), D::CH1, D::CH2);
    }
    deb_sync<G>();
    /* significance of the nodes that have siblings */
    const bool nonneg = rabs == rsum;
    double v0lo, v0hi;
    {
        /* value0 = (double)fdflux_root * mincont with fdflux_root in [rsum - e, rsum + e] */
        const double e = deb_sum_err(rabs, n);
        const double p = (rsum - e) * a.mincont, q = (rsum + e) * a.mincont;
        v0lo = fmin(p, q) - fabs(fmin(p, q)) * 0x1p-50 - 1e-300;
        v0hi = fmax(p, q) + fabs(fmax(p, q)) * 0x1p-50 + 1e-300;
    }
    bool exact = false;              /* the root's flux is known: v0lo = v0hi */
    auto val = [&](int k) { return a.cd[fp[k]]; };
    auto test = [&](int k, int cc, T w) {
        const double s = deb_ld<G>(&sum[k]);
        const int sig = deb_sig_bound(s, nonneg ? s : rabs, cc, tthr[D::lev(w) + 1] * (float)cc,
                                      v0lo, v0hi);
        if (sig > 0) {
            atomicOr(&cnt[k], D::SIG);
            mark(w, D::SON1, D::SON2);
        }
        return sig;
    };
    for (int c0 = 0; c0 < nn; c0 += 256) {
        const int c = c0 + tid;
        if (tid < 256 && c < nn) {
            const int k = deb_ld<G>(&list[c]);
            const int cc = (int)(deb_ld<G>(&cnt[k]) & D::CM);
            const T w = par.ld(k);
            if (cc >= a.debarea && (flags(w) & D::CH2) && test(k, cc, w) < 0)
                s_open[atomicAdd(&s_nopen, 1)] = k;
        }
        deb_sync<G>();
        const int nopen = s_nopen;
        if (nopen > 0 && !exact) {
            /* where the bounds cannot decide, first the exact sequential float sum of the whole
               object: it leaves only the node's own rounding (an object of five million pixels
               has a bound of 40 % on its flux) */
            if (wid == 0) {
                const float fr = wave_ordered_sum(n, [](int) { return true; }, val, n);
                if (lane == 0) s_fr = fr;
            }
            __syncthreads();
            v0lo = v0hi = (double)s_fr * a.mincont;
            exact = true;
            if (tid < nopen) {
                const int k = s_open[tid];
                if (test(k, (int)(deb_ld<G>(&cnt[k]) & D::CM), par.ld(k)) >= 0) s_open[tid] = -1;
            }
            deb_sync<G>();
        }
        /* then the node's, a wavefront each */
        for (int j = wid; j < nopen; j += NT / 64) {
            const int node = s_open[j];
            if (node < 0) continue;
            const int mc = m[node];
            const int cc = (int)(deb_ld<G>(&cnt[node]) & D::CM);
            const T w = par.ld(node);
            const float f = wave_ordered_sum(
                n,
                [&](int i) {
                    int at = i, l = m[i];
                    if (l < mc) return false;
                    T q = par.ld(i);
                    while (l > mc || (at != node && D::lev(q) == l)) {
                        if (!q) return false;
                        at = D::idx(q);
                        l = D::lev(q);
                        if (l < mc) return false;
                        q = par.ld(at);
                    }
                    return at == node;
                },
                val, cc);
            const float lhs = f - tthr[D::lev(w) + 1] * (float)cc;
            if (lane == 0 && (double)lhs > v0lo) {
                atomicOr(&cnt[node], D::SIG);
                mark(w, D::SON1, D::SON2);
            }
        }
        deb_sync<G>();
        if (tid == 0) s_nopen = 0;
        if (c0 + 256 < nn) deb_sync<G>();
    }
    /* A(): a node with two significant children voids its own and those above */
    int *const slot = reinterpret_cast<int *>(sum), *const kept = slot + cap;
    for (int c = tid; c < nn; c += NT) {
        const int k = deb_ld<G>(&list[c]);
        deb_st<G>(&slot[k], -1);
        if (!(deb_ld<G>(&cnt[k]) & D::SON2)) continue;
        T *q = &cnt[k];
        T w = par.ld(k);
        while (!(atomicOr(q, D::NOTA) & D::NOTA)) {
            if (q == &s_top) break;
            q = w ? &cnt[D::idx(w)] : &s_top;
            if (w) w = par.ld(D::idx(w));
        }
    }
    if (tid == 0 && (deb_ld<false>(&s_top) & D::SON2)) atomicOr(&s_top, D::NOTA);
    deb_sync<G>();
    if (!(deb_ld<false>(&s_top) & D::NOTA)) return 0;
    for (int c = tid; c < nn; c += NT) {
        const int k = deb_ld<G>(&list[c]);
        const T f = deb_ld<G>(&cnt[k]);
        if ((f & (D::SIG | D::NOTA)) == D::SIG && (flags(par.ld(k)) & D::SON2)) {
            const int j = atomicAdd(&s_nk, 1);
            deb_st<G>(&slot[k], j);
            deb_st<G>(&kept[j], k);
        }
    }
    deb_sync<G>();
    const int nk = s_nk;
    for (int j = tid; j < nk; j += NT) deb_st<G>(&cnt[j], ~(T)0);
    deb_sync<G>();
    /* each node's kept node (kept nodes never nest: one at most on its way up; a value that
       another lane has put on the way is the same), and the first pixel of each kept node: a
       root is the first pixel of its level's component */
    for (int c = tid; c < nn; c += NT) {
        const int k = deb_ld<G>(&list[c]);
        int s = deb_ld<G>(&slot[k]);
        if (s < 0) {
            for (T w = par.ld(k); w && s < 0; w = par.ld(D::idx(w)))
                s = deb_ld<G>(&slot[D::idx(w)]);
            if (s >= 0) deb_st<G>(&slot[k], s);
        }
        if (s >= 0) atomicMin(&cnt[s], (T)k);
    }
    deb_sync<G>();
    /* the kept nodes ordered by level, then first pixel */
    for (int j = tid; j < nk; j += NT) {
        const T w = par.ld(deb_ld<G>(&kept[j]));
        deb_st<G>(&cnt[j], ((T)(D::lev(w) + 1) << D::SH) | deb_ld<G>(&cnt[j]));
    }
    deb_sync<G>();
    for (int j0 = wid * 64; j0 < nk; j0 += NT) {
        const int j = j0 + lane;
        const T key = j < nk ? deb_ld<G>(&cnt[j]) : 0;
        int rank = 0;
        for (int i0 = 0; i0 < nk; i0 += 64) {
            const T other = i0 + lane < nk ? deb_ld<G>(&cnt[i0 + lane]) : ~(T)0;
            for (int u = 0; u < min(64, nk - i0); u++) {
                const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)other, u);
                const unsigned hi =
                    WIDE ? (unsigned)__builtin_amdgcn_readlane((int)((unsigned long long)other >> 32), u)
                         : 0u;
                rank += (T)((unsigned long long)hi << 32 | lo) < key;
            }
        }
        if (j < nk) {
            deb_st<G>(&kept[j], rank);
            const int lo = (int)(key & D::IM);
            C[rank] = {D::lev(key), fp[lo], lo, lo};
        }
    }
    return nk;
}

/* where the roots of level `lane` start in the list, the highest level first (lev: roots of
   each level; one wavefront) */
__device__ inline int deb_level_start(const int *lev)
{
    const int lane = threadIdx.x & 63;
    const int c = lane < 63 ? lev[63 - lane] : 0;
    int x = c;
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(x, d);
        if (lane >= d) x += o;
    }
    return __shfl(x - c, 63 - lane);
}

/* an object by one workgroup, with par and m in LDS (G: the rest in global memory) */
template <int NT, bool G, class IT>
__device__ __forceinline__ void deb_tree(const DebArgs &a, const int r, const int cap, double *sum,
                                         unsigned *parw, unsigned *cnt, IT *list,
                                         unsigned char *m)
{
    typedef DebTree<false> D;
    typedef D::T T;
    __shared__ int s_lev[SXG_MAXNTHRESH + 1], s_at[SXG_MAXNTHRESH + 1];
    __shared__ float tthr[SXG_MAXNTHRESH + 1], ttau[SXG_MAXNTHRESH + 1];
    __shared__ double s_rsum[NT / 64], s_rabs[NT / 64];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int n = a.cnt[r], off = a.off[r], ls = a.lstar[r];
    const int *const fp = a.fpia + off;
    int *const pix = reinterpret_cast<int *>(G ? parw : cnt);
    const DebObj<false, G, IT> t = {{parw}, sum, cnt, list, m, pix, n, a.W,
                                    2 * (a.xmax[r] - a.xmin[r] + 1) + 1};
    const auto &par = t.par;
    if (wid == 0) {
        /* sub-thresholds 1..L* and their running maximum tau (L* <= 63: one lane each) */
        const float v = lane < ls ? a.thr[(size_t)r * a.nthresh + lane + 1] : -INFINITY;
        float tau = v;
        for (int d = 1; d < 64; d <<= 1) {
            const float o = __shfl_up(tau, d);
            if (lane >= d) tau = fmaxf(tau, o);
        }
        if (lane < ls) {
            tthr[lane + 1] = v;
            ttau[lane + 1] = tau;
        }
        s_lev[lane] = 0;
        if (lane == 0) s_lev[64] = 0;
    }
    __syncthreads();
    /* level index m = max{i <= L* : tau_i <= cd} (tau is non-decreasing), bounds of the
       root's flux */
    double rsum = 0.0, rabs = 0.0;
    for (int k = tid; k < n; k += NT) {
        const int p = fp[k];
        const float v = a.cd[p];
        rsum += v;
        rabs += fabs(v);
        int lo = 0, hi = ls;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (ttau[mid] <= v) lo = mid;
            else hi = mid - 1;
        }
        pix[k] = p;
        deb_st<G>(&sum[k], (double)v);
        m[k] = (unsigned char)lo;
    }
    rsum = sxw_sum(rsum);
    rabs = sxw_sum(rabs);
    if (lane == 0) {
        s_rsum[wid] = rsum;
        s_rabs[wid] = rabs;
    }
    deb_sync<G>();
    rsum = rabs = 0.0;
#pragma unroll
    for (int w = 0; w < NT / 64; w++) {
        rsum += s_rsum[w];
        rabs += s_rabs[w];
    }
    for (int k = tid; k < n; k += NT) t.look(k);
    deb_sync<G>();
    for (int b0 = 0; b0 < n; b0 += NT) t.first(b0 + tid, b0 + tid < n);
    deb_sync<G>();
    for (int round = 0; round < DEB_JUMPS; round++) {
        for (int k = tid; k < n; k += NT) t.shorten(k);
        deb_sync<G>();
    }
    for (int k = tid; k < n; k += NT) t.joins(k);
    deb_sync<G>();
    for (int k = tid; k < n; k += NT) {
        deb_st<G>(&cnt[k], (T)1);
        const int l = t.settle(k);
        if (l) atomicAdd(&s_lev[l], 1);
    }
    deb_sync<G>();
    if (wid == 0) {
        const int at = deb_level_start(s_lev);
        if (lane > 0) s_at[lane] = at;
    }
    /* a pixel's count and cd to its root */
    for (int k = tid; k < n; k += NT) {
        const int mk = m[k];
        if (mk == 0) continue;
        const T w = par.ld(k);
        if (D::lev(w) == mk) {
            atomicAdd(&cnt[D::idx(w)], (T)1);
            atomicAdd(&sum[D::idx(w)], deb_ld<G>(&sum[k]));
        }
    }
    deb_sync<G>();
    for (int k = tid; k < n; k += NT) {
        const int mk = m[k];
        if (mk > 0 && D::lev(par.ld(k)) != mk)
            deb_st<G>(&list[atomicAdd(&s_at[mk], 1)], (IT)k);
    }
    deb_sync<G>();
    Comp *const C = a.comps + a.compoff[r];
    const int nk = deb_nodes<NT>(a, t, fp, cap, ls, s_lev, s_at, tthr, rsum, rabs, C);
    if (tid == 0) {
        /* without a split the raw object is kept as it is */
        if (nk == 0) C[0] = {0, fp[0], 0, n - 1};
        a.rootnc[r] = a.rootkept[r] = max(nk, 1);
    }
    if (nk == 0) return;
    /* the kept nodes are in global memory */
    deb_sync<true>();
    const int *const slot = reinterpret_cast<const int *>(sum);
    for (int b0 = 0; b0 < n; b0 += NT)
        t.assign(b0 + tid, b0 + tid < n, slot, slot + cap, a.kcomp + off, C);
}

/* CLS names the size class in the kernel's symbol only (a kernel trace then times each
   class on its own) */
template <int NT, int CLS> __global__ void __launch_bounds__(NT) k_deb_tree_lds(DebArgs a, int cls)
{
    extern __shared__ __align__(16) unsigned char smem[];
    /* a planned run's grid is the class's capacity */
    if (a.pd && (int)blockIdx.x >= a.ccount[cls]) return;
    const int r = a.clist[(size_t)cls * a.cstride + blockIdx.x];
    const int cap = (a.cnt[r] + 63) & ~63;
    double *sum = reinterpret_cast<double *>(smem);
    unsigned *par = reinterpret_cast<unsigned *>(sum + cap);
    unsigned *cnt = par + cap;
    unsigned short *list = reinterpret_cast<unsigned short *>(cnt + cap);
    unsigned char *m = reinterpret_cast<unsigned char *>(list + cap);
    deb_tree<NT, false, unsigned short>(a, r, cap, sum, par, cnt, list, m);
}

/* raw objects too large for all of it, up to DEB_HALF pixels: the parent words and level
   indices, which the dependent accesses go to, still sit in LDS (5 bytes a pixel) and the rest
   in global memory */
__global__ void __launch_bounds__(1024) k_deb_tree_glb(DebArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    if (a.pd && (int)blockIdx.x >= a.ccount[3]) return;
    const int r = a.clist[3 * (size_t)a.cstride + blockIdx.x];
    const int off = a.off[r], n = a.cnt[r];
    unsigned *par = reinterpret_cast<unsigned *>(smem);
    deb_tree<1024, true, int>(a, r, n, a.g_sum + off, par,
                              reinterpret_cast<unsigned *>(a.g_cnt + off), a.g_list + off,
                              reinterpret_cast<unsigned char *>(par + DEB_HALF));
}

/*
 * The trees of the larger raw objects, one pass a kernel: a lane for every pixel of the raw list
 * that belongs to one of them, then a workgroup per object for the nodes, then the pixels again.  The same passes as in one workgroup, with all state in global
 * memory; between kernels everything is there, and inside one the words that other workgroups
 * change go through the device-coherent level.  Bound: latency of dependent accesses, in the
 * nodes those of one CU.  In one workgroup per object the passes over the pixels were one CU's
 * too; before, a workgroup per level walked them.  Trees of one frame, in us, by levels, in one
 * workgroup, and now: 300 x 291 pixels 2,070, 4,800, 530; 512 x 512 5,860, 15,850, 3,440;
 * 1024 x 1024 24,800, 73,800, 13,300; five million pixels in a 4096^2 frame 288,000, 817,000,
 * 220,000 (of which the exact flux of the whole object, and those of the nodes that need it, are
 * nearly all).
 */
struct DebWide {
    double rsum, rabs;              /* sums of cd and |cd| */
    int lev[SXG_MAXNTHRESH], at[SXG_MAXNTHRESH];   /* roots of each level; taken places of each */
};
typedef DebObj<true, true, int> DebWideObj;

__device__ inline DebWideObj deb_wide_obj(const DebArgs &a, int r)
{
    const int off = a.off[r];
    return {{a.g_par + off}, a.g_sum + off, a.g_cnt + off, a.g_list + off, a.g_m + off,
            a.fpia + off, a.cnt[r], a.W, 2 * (a.xmax[r] - a.xmin[r] + 1) + 1};
}
/* the object of raw-list entry g, or -1 where it is none of class 4 */
__device__ inline int deb_wide_root(const DebArgs &a, long g)
{
    if (g >= deb_P0(a)) return -1;
    const int r = a.rawkey[g];
    return a.cnt[r] > DEB_HALF && a.lstar[r] > 0 ? r : -1;
}
/* whether all entries of this workgroup belong to object r (the list is grouped by object) */
__device__ inline bool deb_wide_one(const DebArgs &a, int r)
{
    const long b = (long)blockIdx.x * 256;
    return r >= 0 && b + 255 < deb_P0(a) && a.rawkey[b] == r && a.rawkey[b + 255] == r;
}

/* the record of each object, whose number is in rootnc until the nodes are done */
__global__ void __launch_bounds__(64) k_deb_wide_start(DebArgs a)
{
    const int j = blockIdx.x;
    if (a.pd && j >= a.ccount[4]) return;
    if (threadIdx.x == 0) {
        a.rootnc[a.clist[4 * (size_t)a.cstride + j]] = j;
        a.wide[j].rsum = a.wide[j].rabs = 0.0;
    }
    a.wide[j].lev[threadIdx.x] = a.wide[j].at[threadIdx.x] = 0;
}

/* level index, count and sum of each pixel, its neighbours, and the bounds of the root's flux.
   A level is the number of leading sub-thresholds at or below cd: tau_i <= cd where all up to
   i are */
__global__ void __launch_bounds__(256) k_deb_wide_levels(DebArgs a)
{
    const long g = (long)blockIdx.x * 256 + threadIdx.x;
    const int r = deb_wide_root(a, g);
    double rs = 0.0, ra = 0.0;
    if (r >= 0) {
        const DebWideObj t = deb_wide_obj(a, r);
        const int k = (int)(g - a.off[r]), ls = a.lstar[r];
        const float *const thr = a.thr + (size_t)r * a.nthresh;
        const float v = a.cd[t.pl[k]];
        rs = v;
        ra = fabs(v);
        int lo = 0;
        while (lo < ls && thr[lo + 1] <= v) lo++;
        t.sum[k] = v;
        t.cnt[k] = 1;
        t.m[k] = (unsigned char)lo;
        t.look(k);
    }
    if (deb_wide_one(a, r)) {
        rs = sxw_sum(rs);
        ra = sxw_sum(ra);
        if (threadIdx.x & 63) return;
    } else if (r < 0) {
        return;
    }
    DebWide &w = a.wide[a.rootnc[r]];
    atomicAdd(&w.rsum, rs);
    atomicAdd(&w.rabs, ra);
}

__global__ void __launch_bounds__(256) k_deb_wide_first(DebArgs a)
{
    const long g = (long)blockIdx.x * 256 + threadIdx.x;
    const int r = deb_wide_root(a, g);
    if (!__ballot(r >= 0)) return;
    const DebWideObj t = r >= 0 ? deb_wide_obj(a, r) : DebWideObj{};
    t.first(r >= 0 ? (int)(g - a.off[r]) : 0, r >= 0);
}

__global__ void __launch_bounds__(256) k_deb_wide_shorten(DebArgs a)
{
    const long g = (long)blockIdx.x * 256 + threadIdx.x;
    const int r = deb_wide_root(a, g);
    if (r < 0) return;
    const DebWideObj t = deb_wide_obj(a, r);
    for (int round = 0; round < DEB_JUMPS; round++) t.shorten((int)(g - a.off[r]));
}

__global__ void __launch_bounds__(256) k_deb_wide_join(DebArgs a)
{
    const long g = (long)blockIdx.x * 256 + threadIdx.x;
    const int r = deb_wide_root(a, g);
    if (r >= 0) deb_wide_obj(a, r).joins((int)(g - a.off[r]));
}

__global__ void __launch_bounds__(256) k_deb_wide_settle(DebArgs a)
{
    __shared__ int s_n[SXG_MAXNTHRESH];
    const long g = (long)blockIdx.x * 256 + threadIdx.x;
    const int r = deb_wide_root(a, g);
    const bool one = deb_wide_one(a, r);   /* the same in every thread */
    if (one) {
        if (threadIdx.x < SXG_MAXNTHRESH) s_n[threadIdx.x] = 0;
        __syncthreads();
    }
    if (r < 0) return;
    int *const lev = a.wide[a.rootnc[r]].lev;
    const int l = deb_wide_obj(a, r).settle((int)(g - a.off[r]));
    if (!one) {
        if (l) atomicAdd(&lev[l], 1);
        return;
    }
    if (l) atomicAdd(&s_n[l], 1);
    __syncthreads();
    if (threadIdx.x < SXG_MAXNTHRESH && s_n[threadIdx.x])
        atomicAdd(&lev[threadIdx.x], s_n[threadIdx.x]);
}

/* a pixel's count and cd to its root, together for the lanes of a wavefront that share the
   root of one (four rounds: the roots that many share come up first); the roots into the list */
__global__ void __launch_bounds__(256) k_deb_wide_sums(DebArgs a)
{
    typedef DebTree<true> D;
    __shared__ int s_n[SXG_MAXNTHRESH], s_b[SXG_MAXNTHRESH];
    const long g = (long)blockIdx.x * 256 + threadIdx.x;
    const int lane = threadIdx.x & 63;
    const int r = deb_wide_root(a, g);
    const bool one = deb_wide_one(a, r);
    if (one) {
        if (threadIdx.x < SXG_MAXNTHRESH) s_n[threadIdx.x] = 0;
        __syncthreads();
    }
    long root = -1;      /* of another pixel, by raw-list entry */
    int lev = 0, k = 0;  /* a root's level */
    double v = 0.0;
    if (r >= 0) {
        const DebWideObj t = deb_wide_obj(a, r);
        k = (int)(g - a.off[r]);
        const int mk = t.m[k];
        if (mk > 0) {
            const D::T w = t.par.ld(k);
            if (D::lev(w) == mk) {
                root = a.off[r] + D::idx(w);
                v = t.sum[k];
            } else {
                lev = mk;
            }
        }
    }
#pragma unroll 1
    for (int round = 0; round < 4; round++) {
        const unsigned long long b = __ballot(root >= 0);
        if (!b) break;
        const int lead = __builtin_ctzll(b);
        const long key = __shfl(root, lead);
        const bool mine = root == key;
        const int c = __popcll(__ballot(mine));
        const double s = sxw_sum(mine ? v : 0.0);
        if (lane == lead) {
            atomicAdd(&a.g_cnt[key], (D::T)c);
            atomicAdd(&a.g_sum[key], s);
        }
        if (mine) root = -1;
    }
    if (root >= 0) {
        atomicAdd(&a.g_cnt[root], (D::T)1);
        atomicAdd(&a.g_sum[root], v);
    }
    if (r < 0) return;
    DebWide &w = a.wide[a.rootnc[r]];
    int *const list = a.g_list + a.off[r];
    if (!one) {
        if (!lev) return;
        int at = atomicAdd(&w.at[lev], 1);
        for (int l = SXG_MAXNTHRESH - 1; l > lev; l--) at += w.lev[l];
        list[at] = k;
        return;
    }
    const int place = lev ? atomicAdd(&s_n[lev], 1) : 0;
    __syncthreads();
    if (threadIdx.x < 64) {
        const int at = deb_level_start(w.lev), c = s_n[lane];
        s_b[lane] = c ? at + atomicAdd(&w.at[lane], c) : 0;
    }
    __syncthreads();
    if (lev) list[s_b[lev] + place] = k;
}

__global__ void __launch_bounds__(1024) k_deb_wide_nodes(DebArgs a)
{
    __shared__ int s_lev[SXG_MAXNTHRESH], s_at[SXG_MAXNTHRESH];
    __shared__ float tthr[SXG_MAXNTHRESH + 1];
    const int j = blockIdx.x, tid = threadIdx.x;
    if (a.pd && j >= a.ccount[4]) return;
    const int r = a.clist[4 * (size_t)a.cstride + j];
    const DebWideObj t = deb_wide_obj(a, r);
    const DebWide &w = a.wide[j];
    const int ls = a.lstar[r];
    if (tid < 64) {
        const int at = deb_level_start(w.lev);
        s_lev[tid] = w.lev[tid];
        s_at[tid] = at + w.lev[tid];
        if (tid < ls) tthr[tid + 1] = a.thr[(size_t)r * a.nthresh + tid + 1];
    }
    __syncthreads();
    Comp *const C = a.comps + a.compoff[r];
    const int nk = deb_nodes<1024>(a, t, t.pl, t.n, ls, s_lev, s_at, tthr, w.rsum, w.rabs, C);
    if (tid == 0) {
        if (nk == 0) C[0] = {0, t.pl[0], 0, t.n - 1};
        a.rootnc[r] = a.rootkept[r] = max(nk, 1);
    }
}

__global__ void __launch_bounds__(256) k_deb_wide_assign(DebArgs a)
{
    const long g = (long)blockIdx.x * 256 + threadIdx.x;
    int r = deb_wide_root(a, g);
    if (r >= 0 && a.rootkept[r] < 2) r = -1;
    if (!__ballot(r >= 0)) return;
    const DebWideObj t = r >= 0 ? deb_wide_obj(a, r) : DebWideObj{};
    const int *const slot = reinterpret_cast<const int *>(t.sum);
    const int off = r >= 0 ? a.off[r] : 0;
    t.assign((int)(g - off), r >= 0, slot, slot + t.n, a.kcomp + off,
             r >= 0 ? a.comps + a.compoff[r] : nullptr);
}

/* the objects of class 3 into out, largest first (ties in list order), so that the longest
   trees start first; more than fullmax of them in list order (the comparisons are
   quadratic).  The results do not depend on the order.  cc (planned runs): their number on
   the device. */
__global__ void __launch_bounds__(256) k_deb_order(const int *__restrict__ clist,
                                                   const int *__restrict__ cnt, int nraw,
                                                   int nc, int *__restrict__ out, const int *cc,
                                                   int fullmax)
{
    __shared__ int sn[256];
    if (cc) nc = cc[3];
    const int *L = clist + 3 * (size_t)nraw;
    int *O = out + 3 * (size_t)nraw;
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (nc > fullmax) {
        if (j < nc) O[j] = L[j];
        return;
    }
    const int nj = j < nc ? cnt[L[j]] : 0;
    int rank = 0;
    for (int t0 = 0; t0 < nc; t0 += 256) {
        __syncthreads();
        sn[threadIdx.x] = t0 + (int)threadIdx.x < nc ? cnt[L[t0 + threadIdx.x]] : -1;
        __syncthreads();
        const int tn = min(256, nc - t0);
        for (int u = 0; u < tn; u++) {
            const int x = sn[u];
            rank += x > nj || (x == nj && t0 + u < j);
        }
    }
    if (j < nc) O[rank] = L[j];
}

/* ------------------------------------------------------------------ objects ---- */
struct ObjArgs {
    DebArgs d;
    const int *objbase;     /* first object index of each raw object */
    int *objraw, *objcomp;  /* raw object and component of each object */
    int *alloc;             /* frame-wide object index of each raw pixel */
    const float *sub;       /* background-subtracted frame */
    int *okey;              /* object index of each raw-list entry */
    ObjCols o;
    int nobj;
    const int *order;       /* objects in launch order: those of large raw objects first */
};

/* nodes whose entries lo .. hi are at least PRE_BIG take a workgroup each, at least PRE_MID a
   wavefront, the others a row of 16 lanes */
#ifndef PRE_BIG
#define PRE_BIG 512
#define PRE_MID 32
#endif

/* the objects: the device count of a planned run */
__device__ inline int obj_n(const ObjArgs &A) { return A.d.pd ? A.d.pd->nobj : A.nobj; }

/* the objects by size: order[0, nbig) the big ones, order[nbig + nmid, nobj) the small ones,
   order[cap, cap + nmid) those between; cnt: their numbers */
__global__ void __launch_bounds__(256) k_pre_order(ObjArgs A, int *cnt, int *order)
{
    const int obj = blockIdx.x * 256 + threadIdx.x;
    const int nobj = obj_n(A);
    int cls = -1;
    if (obj < nobj) {
        const Comp c = A.d.comps[A.d.compoff[A.objraw[obj]] + A.objcomp[obj]];
        const int n = c.hi - c.lo + 1;
        cls = n >= PRE_BIG ? 0 : n >= PRE_MID ? 1 : 2;
    }
    const int k = sxw_place<3>(cnt, cls);
    if (cls >= 0) order[cls == 0 ? k : cls == 1 ? A.nobj + k : nobj - 1 - k] = obj;
}

/* objects of each raw object, in component-table order (one wavefront per raw object) */
__global__ void __launch_bounds__(256) k_deb_objlist(ObjArgs A, int *zero3)
{
    /* the counters of k_pre_order start at zero (no fill launch) */
    if (blockIdx.x == 0 && threadIdx.x < 3) zero3[threadIdx.x] = 0;
    const int lane = threadIdx.x & 63;
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= deb_nraw(A.d)) return;
    const int nc = A.d.rootnc[r], base = A.objbase[r];
    /* a single local maximum: the raw object is the object */
    if (A.d.lstar[r] == 0 && lane == 0)
        A.d.comps[A.d.compoff[r]] = {0, A.d.first[r], 0, A.d.cnt[r] - 1};
    for (int c = lane; c < nc; c += 64) {
        A.objraw[base + c] = r;
        A.objcomp[base + c] = c;
    }
}


/*
 * FULL preanalysis of each kept node over its level pixels, by a row of 16 lanes, a wavefront
 * or a workgroup (SxwTeam); the node's pixels get the object index.  Bound: the sequential
 * sums of the largest nodes (7 cycles a pixel), then the latency of the loads.  A node reads
 * its own stretch of the raw object's list only.  Measured (a wavefront per node over the whole raw object before): crowded
 * 4096^2 95 -> 45 us, dense 2048^2 253 -> 74, 2048^2 with saturated stars 68 -> 24.
 */
template <SxwSize Z>
__device__ __forceinline__ void pre_object(const ObjArgs &A, const int obj, double *rows)
{
    typedef SxwTeam<Z> Team;
    const int id = Team::first();
    const DebArgs &d = A.d;
    const int r = A.objraw[obj], c = A.objcomp[obj];
    const Comp C = d.comps[d.compoff[r] + c];
    const int L = C.level;
    const int n = C.hi - C.lo + 1, off = d.off[r] + C.lo, W = d.W, H = d.H;
    const int *lv = L > 0 ? d.kcomp + off : nullptr;
    /* extent, peaks, count (reductions); the node's pixels get the object index */
    float peak = (float)-SXG_BIG, cpeak = (float)-SXG_BIG;
    int xmin = 2 * SXG_MAXPICSIZE, ymin = 2 * SXG_MAXPICSIZE, xmax = 0, ymax = 0, cnt = 0;
#pragma unroll 4
    for (int k = id; k < n; k += Team::STEP) {
        if (lv && lv[k] != c) continue;
        const int p = d.fpia[off + k];
        const int y = p / W, x = p - y * W;
        A.alloc[p] = obj;
        peak = fmaxf(peak, A.sub[p]);
        cpeak = fmaxf(cpeak, d.cd[p]);
        xmin = min(xmin, x);
        xmax = max(xmax, x);
        ymin = min(ymin, y);
        ymax = max(ymax, y);
        cnt++;
    }
    peak = Team::max(peak);
    cpeak = Team::max(cpeak);
    xmin = Team::min(xmin);
    ymin = Team::min(ymin);
    xmax = Team::max(xmax);
    ymax = Team::max(ymax);
    cnt = Team::sum(cnt);
    int flag = L > 0 ? SXG_OBJ_MERGED : 0;
    if (xmin == 0 || xmax == W - 1 || ymin == 0 || ymax == H - 1) flag |= SXG_OBJ_TRUNC;
    const double dthresh = (double)d.thr[(size_t)r * d.nthresh + L];
    const double dthresh2 = (dthresh + peak) / 2.0;
    /* one fold pass: rv, the raster-order float sum of cd, and the moments, double sums
       of float terms in raster order */
    SxwSums<6, 1, Z> sums;
    int area2 = 0, dnpix = 0;
    /* the next chunk's membership and pixel are read while this chunk is folded */
    bool nin = id < n && (!lv || lv[id] == c);
    int npix_ = id < n ? d.fpia[off + id] : 0;
    for (int base = 0; base < n; base += Team::STEP) {
        const int k = base + id;
        const bool in = nin;
        const int pc = npix_;
        if (k + Team::STEP < n) {
            nin = !lv || lv[k + Team::STEP] == c;
            npix_ = d.fpia[off + k + Team::STEP];
        } else {
            nin = false;
        }
        float val = 0.0f, cval = 0.0f, tx = 0.0f, ty = 0.0f, txx = 0.0f, tyy = 0.0f, txy = 0.0f;
        if (in) {
            const int p = pc;
            const int y = p / W - ymin, x = p - (p / W) * W - xmin;
            cval = d.cd[p];
            val = A.sub[p];
            if (val > dthresh) dnpix++;
            if (val > dthresh2) area2++;
            tx = cval * x;
            ty = cval * y;
            txx = cval * x * x;
            tyy = cval * y * y;
            txy = cval * x * y;
        }
        const double t6[6] = {val, tx, ty, txx, tyy, txy};
        const float tf[2] = {cval, 0.0f};
        sums.add(rows, t6, tf, in);
    }
    sums.end(rows);
    const float rv = sums.f[0];
    area2 = Team::sum(area2);
    dnpix = Team::sum(dnpix);
    if (id != 0) return;
    Moments m;
    sxg_moments(sums.d[1], sums.d[2], sums.d[3], sums.d[4], sums.d[5], rv, false, 0.0, 0.0, xmin,
                ymin, area2, dnpix, dthresh, dthresh2, m);
    ObjCols &o = const_cast<ObjCols &>(A.o);
    o.level[obj] = L;
    o.root[obj] = r;
    o.firstpix[obj] = C.first;
    o.flag[obj] = flag;
    o.fdnpix[obj] = cnt;
    o.dnpix[obj] = dnpix;
    o.xmin[obj] = xmin; o.xmax[obj] = xmax; o.ymin[obj] = ymin; o.ymax[obj] = ymax;
    o.fdflux[obj] = rv;
    o.fdpeak[obj] = cpeak;
    o.dpeak[obj] = peak;
    o.dflux[obj] = (float)sums.d[0];
    o.dthresh[obj] = (float)dthresh;
    sxg_store_moments(o, obj, m);
}

/* by size (k_pre_order; the grid is an upper bound, the host does not know the numbers) */
__global__ void __launch_bounds__(256) k_deb_pre(ObjArgs A)
{
    __shared__ double s_rows[std::max(4 * sxw_wrows(6, 1), sxw_brows(6, 1))];
    const int nobj = obj_n(A);
    const int nbig = A.order[2 * A.nobj], nmid = A.order[2 * A.nobj + 1];
    int b = blockIdx.x;
    if (b < nbig) {
        pre_object<SXW_GROUP>(A, A.order[b], s_rows);
        return;
    }
    b -= nbig;
    if (4 * b < nmid) {
        const int wid = threadIdx.x >> 6;
        if (4 * b + wid < nmid)
            pre_object<SXW_WAVE>(A, A.order[A.nobj + 4 * b + wid],
                                 s_rows + wid * sxw_wrows(6, 1));
        return;
    }
    b -= (nmid + 3) / 4;
    const int slot = nbig + nmid + b * 16 + (threadIdx.x >> 4);
    if (slot < nobj) pre_object<SXW_ROWS>(A, A.order[slot], s_rows);
}

/* gatherup: every unassigned pixel goes to the nearest kept object of its raw object
   in the ellipse metric (first minimum in object order); then the object of every entry */
__global__ void __launch_bounds__(256) k_deb_gather(ObjArgs A, int *objcnt, int2 *objspan, long nz)
{
    const long g = (long)blockIdx.x * 256 + threadIdx.x;
    /* the per-object pixel counts and spans of k_deb_objcount start empty (no fill launch) */
    if (g < nz) {
        objcnt[g] = 0;
        objspan[g] = {0x7fffffff, -1};
    }
    if (g >= deb_P0(A.d)) return;
    const int p = A.d.fpia[g];
    const int r = A.d.rawkey[g];
    /* k_deb_pre gave every pixel of a raw object kept whole, and every pixel of a kept
       node, its object; the rest are the pixels of split raw objects outside all kept
       nodes */
    int a;
    if (A.d.rootkept[r] >= 2 && A.d.kcomp[g] < 0) {
        const int base = A.objbase[r], nk = A.d.rootkept[r];
        const int y = p / A.d.W, x = p - y * A.d.W;
        const ObjCols &o = A.o;
        float distmin = (float)1e+31, dist, dx, dy;
        a = base;
        for (int j = base; j < base + nk; j++) {
            dx = (float)(x - o.mx[j]);
            dy = (float)(y - o.my[j]);
            dist = (float)(0.5 * (o.cxx[j] * dx * dx + o.cyy[j] * dy * dy + o.cxy[j] * dx * dy) /
                           o.abcor[j]);
            if (dist < distmin) {
                distmin = dist;
                a = j;
            }
        }
        A.alloc[p] = a;
    } else {
        a = A.alloc[p];
    }
    A.okey[g] = a;
}

/* pixels per object, and for those of split raw objects the first and last list entry of
   each; lanes with the same object (long runs: the list is grouped by raw object) add their
   count once */
__global__ void __launch_bounds__(256) k_deb_objcount(ObjArgs A, int *objcnt, int2 *objspan)
{
    const long g = (long)blockIdx.x * 256 + threadIdx.x;
    const int lane = threadIdx.x & 63;
    bool act = g < deb_P0(A.d);
    const int key = act ? A.okey[g] : -1;
    unsigned long long pending = __ballot(act);
    while (pending) {
        const int leader = __builtin_ctzll(pending);
        const int k = __shfl(key, leader);
        const unsigned long long grp = __ballot(act && key == k);
        if (lane == leader) {
            atomicAdd(&objcnt[k], __popcll(grp));
            if (A.d.rootkept[A.d.rawkey[g]] >= 2) {
                atomicMin(&objspan[k].x, (int)g);
                atomicMax(&objspan[k].y, (int)g + 63 - __builtin_clzll(grp) - leader);
            }
        }
        if (act && key == k) act = false;
        pending &= ~grp;
    }
}

/*
 * The raw pixels regrouped by object, stably (each object's pixels in the raster order
 * of its raw object's list), from the object offsets: a raw object kept as one object
 * moves as one block (k_obj_place1, a lane per pixel); each object of a split one has a
 * wavefront (k_obj_place_multi) that picks its pixels from the stretch of the list between
 * its first and last, 64 entries at a time.  Bound: latency of the longest stretch's reads.
 * One wavefront per split raw object, which placed all of its objects, took 26 us in a
 * crowded 4096^2 and 255 us in a dense 2048^2 frame (18,000 entries); now 11 and 27 us.
 */
__global__ void __launch_bounds__(256) k_obj_place1(ObjArgs A, const int *__restrict__ objoff,
                                                    int *opix)
{
    const long g = (long)blockIdx.x * 256 + threadIdx.x;
    if (g >= deb_P0(A.d)) return;
    const int r = A.d.rawkey[g];
    if (A.d.rootkept[r] != 1) return;
    opix[objoff[A.okey[g]] + (int)(g - A.d.off[r])] = A.d.fpia[g];
}

/* list chunks of 64 entries read together */
#define OP_AHEAD 4
__global__ void __launch_bounds__(256) k_obj_place_multi(ObjArgs A,
                                                         const int *__restrict__ objoff,
                                                         const int2 *__restrict__ objspan,
                                                         int *opix)
{
    const int lane = threadIdx.x & 63;
    const int obj = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (obj >= obj_n(A)) return;
    const int2 span = objspan[obj];
    if (span.y < span.x) return;       /* not part of a split raw object */
    const unsigned long long below = sxw_lanes_below(lane);
    int at = objoff[obj];
    for (int k0 = span.x; k0 <= span.y; k0 += 64 * OP_AHEAD) {
        bool in[OP_AHEAD];
        int pix[OP_AHEAD];
#pragma unroll
        for (int u = 0; u < OP_AHEAD; u++) {
            const int k = min(k0 + u * 64 + lane, span.y);
            in[u] = A.okey[k] == obj && k0 + u * 64 + lane <= span.y;
            pix[u] = A.d.fpia[k];
        }
#pragma unroll
        for (int u = 0; u < OP_AHEAD; u++) {
            const unsigned long long b = __ballot(in[u]);
            if (in[u]) opix[at + __popcll(b & below)] = pix[u];
            at += __popcll(b);
        }
    }
}

__global__ void __launch_bounds__(256) k_deb_zero(int *v, long n)
{
    const long k = (long)blockIdx.x * 256 + threadIdx.x;
    if (k < n) v[k] = 0;
}

/* planned runs: the node total against its capacity (the 64-bit node sum too: a total past
   2^31 is an overflow) and the class words of the counter block against theirs; on any
   overflow of the frame the class counts are zeroed so that no tree kernel has work */
struct DebGuardCaps {
    long long lds[3], cls[DEB_NCLASS];   /* LDS bytes of classes 0..2, objects of each class */
};

__global__ void k_deb_plan_guard(const unsigned long long *dw, PlanDev *pd, int *cc,
                                 const int *ntot, long long cap_tot, DebGuardCaps gc)
{
    if (threadIdx.x != 0) return;
    if (dw[2] > (unsigned long long)cap_tot || (long long)*ntot > cap_tot || *ntot < 0)
        pd->ovf |= 1 << PL_NTOT;
    for (int c = 0; c < 3; c++)
        if (cc[DEB_CLDS + c] < 0 || (long long)cc[DEB_CLDS + c] > gc.lds[c])
            pd->ovf |= 1 << (PL_LDS0 + c);
    for (int c = 0; c < DEB_NCLASS; c++)
        if (cc[c] < 0 || (long long)cc[c] > gc.cls[c]) pd->ovf |= 1 << (PL_C0 + c);
    if (pd->ovf) {
        pd->nfg = pd->nraw = pd->npix = pd->nobj = pd->nsurv = 0;
        for (int c = 0; c < DEB_CPIX; c++) cc[c] = 0;
    }
}

/* planned runs: the frame's deblending work into its device block */
__global__ void k_deb_plan_info(const unsigned long long *dw, const int *cc, PlanDev *pd)
{
    if (threadIdx.x != 0) return;
    pd->deb_pixels = (long long)dw[0];
    pd->deb_labels = (long long)dw[1];
    for (int c = 0; c < 4; c++) pd->class_pixels[c] = cc[DEB_CPIX + c];
}

/* --------------------------------------------------------------- host side ---- */
extern "C" void init_deblend(float basethresh, int nthresh, size_t numValidObj, size_t numValidPix)
{
    SxgState &S = sxg_state();
    if (!S.have_frame) {
        sxg_set_error("init_deblend: no frame");
        return;
    }
    if (nthresh < 1 || nthresh > SXG_MAXNTHRESH) {
        sxg_set_error("init_deblend: DEBLEND_NTHRESH must be 1..64");
        return;
    }
    if ((long)numValidObj != S.nraw || (long)numValidPix != S.npix_raw) {
        sxg_set_error("init_deblend: object/pixel counts differ from run_detection");
        return;
    }
    S.nthresh = nthresh;
    S.deb_base = basethresh;
    float *thr = sxg_take<float>("deb.thr", (size_t)(S.nraw > 0 ? S.nraw : 1) * nthresh);
    if (!thr) return;
    RawObj ro;
    if (!sxg_raw_alloc(S.nraw, ro)) return;
    const long tot = (long)S.nraw * nthresh;
    if (tot > 0) {
        sxg_kt_begin(SXG_KT_DEB_THRESH);
        hipLaunchKernelGGL(k_deb_thresh, dim3(sxg_div_up(tot, 256)), dim3(256), 0, S.stream,
                           ro.fdpeak, S.nraw, nthresh, basethresh, ro.t0,
                           (int)(S.weighted && S.wargs.rel), thr,
                           (const PlanDev *)(S.plan ? S.pdev : nullptr));
        sxg_kt_end(SXG_KT_DEB_THRESH);
    }
    SXG_HIP(hipGetLastError());
    S.deb_ready = true;
}

extern "C" int parcel_out(float basethresh, int n_thresh, int deb_minarea, size_t numValidObj,
                          size_t numValidPix, double deblend_mincont)
{
    SxgState &S = sxg_state();
    if (!S.have_frame || !S.deb_ready || n_thresh != S.nthresh) {
        sxg_set_error("parcel_out: call init_deblend first with the same DEBLEND_NTHRESH");
        return -1;
    }
    if (deb_minarea < 1) {
        sxg_set_error("parcel_out: deb_minarea must be >= 1");
        return -1;
    }
    (void)basethresh; (void)numValidObj; (void)numValidPix;
    hipStream_t st = S.stream;
    /* a planned run: S.nraw and S.npix_raw are capacities, the counts are on the device */
    const FramePlan *pl = S.plan;
    PlanDev *pd = pl ? S.pdev : nullptr;
    const int nraw = S.nraw;
    const long P0 = S.npix_raw;
    sxg_stage_begin(ST_DEBLEND);
    RawObj ro;
    if (!sxg_raw_alloc(nraw, ro)) return -1;
    const size_t nr = (size_t)(nraw > 0 ? nraw : 1);
    int *compoff = sxg_take<int>("deb.compoff", nr + 1);
    int *dtot = sxg_take<int>("deb.total", 4);
    int *rootnc = sxg_take<int>("deb.rootnc", nr);
    int *rootkept = sxg_take<int>("deb.rootkept", nr);
    int *objbase = sxg_take<int>("deb.objbase", nr);
    int *alloc = sxg_take<int>("deb.alloc", S.N);
    auto *top1 = sxg_take<unsigned long long>("deb.top1", nr);
    auto *top2 = sxg_take<unsigned>("deb.top2", nr);
    int *nmax = sxg_take<int>("deb.nmax", nr);
    int *lstar = sxg_take<int>("deb.lstar", nr);
    int *clist = sxg_take<int>("deb.clist", DEB_NCLASS * nr);
    int *ccount = sxg_take<int>("deb.ccount", DEB_NCOUNT);
    auto *dwork = sxg_take<unsigned long long>("deb.dwork", 3);
    int *kcomp = sxg_take<int>("deb.kcomp", (size_t)(P0 > 0 ? P0 : 1));
    auto *lmflag = sxg_take<unsigned char>("deb.lmflag", (size_t)(P0 > 0 ? P0 : 1));
    if (!compoff || !dtot || !rootnc || !rootkept || !objbase || !alloc || !top1 || !top2 ||
        !nmax || !lstar || !clist || !ccount || !dwork || !kcomp || !lmflag)
        return -1;
    DebArgs a{};
    a.fpia = S.fpia; a.rawkey = S.fpia_keys; a.off = ro.off; a.cnt = ro.count; a.first = ro.first;
    a.xmin = ro.xmin; a.xmax = ro.xmax;
    a.cd = S.cd.as<float>(); a.lab = S.aux.as<int>();   /* the detection labels */
    a.kcomp = kcomp; a.P0 = P0; a.thr = sxg_take<float>("deb.thr", nr * n_thresh);
    a.nthresh = n_thresh; a.debarea = deb_minarea; a.mincont = deblend_mincont;
    a.W = S.W; a.H = S.H; a.nraw = nraw; a.compoff = compoff;
    a.cstride = nraw; a.pd = pd;
    a.rootnc = rootnc; a.rootkept = rootkept;
    a.top1 = top1; a.top2 = top2; a.nmax = nmax; a.lstar = lstar; a.clist = clist;
    a.lmflag = lmflag;
    a.ccount = ccount; a.dwork = dwork;
    S.deb_pixels = S.deb_labels = 0;
    for (int c = 0; c < 4; c++) S.deb_class_pixels[c] = 0;
    int nobj = 0;
    if (nraw > 0) {
        const int cap0 = (int)sxg_option(SXG_OPT_DEB_LDS_TINY);
        const int cap1 = (int)sxg_option(SXG_OPT_DEB_LDS_SMALL);
        const int cap2 = (int)sxg_option(SXG_OPT_DEB_LDS_LARGE);
        const int gr = sxg_div_up(nraw, 256);
        sxg_kt_begin(SXG_KT_DEB_LMAX);
        hipLaunchKernelGGL(k_deb_prep, dim3(sxg_div_up(nraw > 8 ? nraw : 8, 256)), dim3(256), 0,
                           st, a);
        hipLaunchKernelGGL(k_deb_lmax<0>, dim3(sxg_div_up(P0, 256)), dim3(256), 0, st, a);
        hipLaunchKernelGGL(k_deb_lmax<1>, dim3(sxg_div_up(P0, 256)), dim3(256), 0, st, a);
        hipLaunchKernelGGL(k_deb_lsfirst, dim3(sxg_div_up((long)nraw * n_thresh, 256)), dim3(256),
                           0, st, a);
        hipLaunchKernelGGL(k_deb_nodecap, dim3(gr), dim3(256), 0, st, a);
        sxg_scan_excl(compoff, compoff, nraw, dtot, st, pd ? &pd->nraw : nullptr);
        hipLaunchKernelGGL(k_deb_classify, dim3(gr), dim3(256), 0, st, a, cap0, cap1, cap2);
        sxg_kt_end(SXG_KT_DEB_LMAX);
        int cc[DEB_NCOUNT] = {};
        int ntot = 0;
        unsigned long long dw[3] = {0, 0, 0};
        if (pl) {
            /* the capacities stand for the counts; the guards check the device counts
               against them (the node total first, then every class) */
            ntot = (int)pl->cap[PL_NTOT];
            for (int c = 0; c < DEB_NCLASS; c++) cc[c] = (int)pl->cap[PL_C0 + c];
            /* the class's LDS: what its largest object may need, or less when the plan asks
               less */
            const int caps[3] = {cap0, cap1, cap2};
            DebGuardCaps gc;
            for (int c = 0; c < 3; c++)
                gc.lds[c] = cc[DEB_CLDS + c] =
                    (int)std::min<int64_t>(pl->cap[PL_LDS0 + c], deb_lds_bytes(caps[c]));
            for (int c = 0; c < DEB_NCLASS; c++) gc.cls[c] = cc[c];
            hipLaunchKernelGGL(k_deb_plan_guard, dim3(1), dim3(64), 0, st, dwork, pd, ccount,
                               dtot, (long long)pl->cap[PL_NTOT], gc);
        } else {
            if (!sxg_read_back({{ccount, cc, DEB_NCOUNT}, {dtot, &ntot, 1}, {dwork, dw, 6}}))
                return -1;
            if (dw[2] > (unsigned long long)0x7fffffff) {
                sxg_set_error("parcel_out: deblending trees exceed 2^31 nodes in one frame");
                return -1;
            }
            S.deb_pixels = (int64_t)dw[0];
            for (int c = 0; c < 4; c++) S.deb_class_pixels[c] = cc[DEB_CPIX + c];
            S.deb_labels = (int64_t)dw[1];
            S.seen.cap[PL_NTOT] = ntot;
            for (int c = 0; c < DEB_NCLASS; c++) S.seen.cap[PL_C0 + c] = cc[c];
            for (int c = 0; c < 3; c++) S.seen.cap[PL_LDS0 + c] = cc[DEB_CLDS + c];
        }
        a.comps = sxg_take<Comp>("deb.comps", (size_t)ntot + 1);
        if (!a.comps) return -1;
        sxg_kt_begin(SXG_KT_DEB_LEVELS);
        /* one launch per class (LDS: the words of its largest object's pixels), side by side:
           each kernel lasts as long as its slowest tree.  What they read was written on the
           context's stream ahead of the kernel that sent the counts, and the host has seen the
           number that this kernel stores last, so a launch on a side stream comes after it. */
        int nside = 0;
        const bool use_side = !S.single_stream && !pl && sxg_option(SXG_OPT_SIDE_STREAMS) != 0;
        static_assert(SXG_NSIDE >= DEB_NCLASS - 1, "a side stream for each class but the first");
        /* the dynamic-LDS limit is an attribute of the function, shared by every context:
           it is raised once, to the most any class asks for (DEB_LDS_LIMIT), never per
           launch (batch workers launch these kernels from several host threads) */
        static const bool lds_attr = [] {
            return hipFuncSetAttribute(reinterpret_cast<const void *>(&k_deb_tree_glb),
                                       hipFuncAttributeMaxDynamicSharedMemorySize,
                                       5 * DEB_HALF) == hipSuccess &&
                   hipFuncSetAttribute(reinterpret_cast<const void *>(&k_deb_tree_lds<1024, 2>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)DEB_LDS_LIMIT) == hipSuccess &&
                   hipFuncSetAttribute(reinterpret_cast<const void *>(&k_deb_tree_lds<512, 1>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)DEB_LDS_LIMIT) == hipSuccess &&
                   hipFuncSetAttribute(reinterpret_cast<const void *>(&k_deb_tree_lds<256, 0>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)DEB_LDS_LIMIT) == hipSuccess;
        }();
        if (!lds_attr) {
            sxg_set_error("parcel_out: cannot raise the LDS limit of the deblending kernels");
            return -1;
        }
        auto launch_lds = [&](const void *fn, int cls, int nt) -> bool {
            const size_t lds = (size_t)cc[DEB_CLDS + cls];
            if (lds > DEB_LDS_LIMIT) {
                sxg_set_error("parcel_out: LDS request above the limit (internal error)");
                return false;
            }
            void *args[] = {&a, &cls};
            const bool side = cls != 0 && use_side;
            hipStream_t ks = side ? S.side[nside] : st;
            /* each class kernel is timed on the stream it runs on */
            sxg_kt_begin_on(SXG_KT_DEB_TREE0 + cls, ks);
            SXG_HIP_RET(hipLaunchKernel(fn, dim3(cc[cls]), dim3(nt), args, lds, ks), false);
            sxg_kt_end_on(SXG_KT_DEB_TREE0 + cls, ks);
            if (side) SXG_HIP_RET(hipEventRecord(S.side_ev[nside++], ks), false);
            return true;
        };
        if (cc[3] > 0 || cc[4] > 0) {
            a.g_sum = sxg_take<double>("deb.g_sum", (size_t)P0);
            a.g_cnt = sxg_take<unsigned long long>("deb.g_cnt", (size_t)P0);
            a.g_list = sxg_take<int>("deb.g_list", (size_t)P0);
            if (!a.g_sum || !a.g_cnt || !a.g_list) return -1;
        }
        if (cc[4] > 0) {
            a.g_par = sxg_take<unsigned long long>("deb.g_par", (size_t)P0);
            a.g_m = sxg_take<unsigned char>("deb.g_m", (size_t)P0);
            a.wide = sxg_take<DebWide>("deb.wide", (size_t)cc[4]);
            if (!a.g_par || !a.g_m || !a.wide) return -1;
            hipStream_t ks = use_side ? S.side[nside] : st;
            const dim3 gp(sxg_div_up(P0, 256)), gw(cc[4]);
            sxg_kt_begin_on(SXG_KT_DEB_LVPAR, ks);
            hipLaunchKernelGGL(k_deb_wide_start, gw, dim3(64), 0, ks, a);
            hipLaunchKernelGGL(k_deb_wide_levels, gp, dim3(256), 0, ks, a);
            hipLaunchKernelGGL(k_deb_wide_first, gp, dim3(256), 0, ks, a);
            hipLaunchKernelGGL(k_deb_wide_shorten, gp, dim3(256), 0, ks, a);
            hipLaunchKernelGGL(k_deb_wide_join, gp, dim3(256), 0, ks, a);
            hipLaunchKernelGGL(k_deb_wide_settle, gp, dim3(256), 0, ks, a);
            hipLaunchKernelGGL(k_deb_wide_sums, gp, dim3(256), 0, ks, a);
            hipLaunchKernelGGL(k_deb_wide_nodes, gw, dim3(1024), 0, ks, a);
            hipLaunchKernelGGL(k_deb_wide_assign, gp, dim3(256), 0, ks, a);
            sxg_kt_end_on(SXG_KT_DEB_LVPAR, ks);
            if (use_side) SXG_HIP_RET(hipEventRecord(S.side_ev[nside++], ks), -1);
        }
        if (cc[3] > 0) {
            /* class 3 largest first */
            int *clist3 = sxg_take<int>("deb.clist3", 4 * nr);
            if (!clist3) return -1;
            DebArgs a3 = a;
            a3.clist = clist3;
            hipStream_t ks = use_side ? S.side[nside] : st;
            hipLaunchKernelGGL(k_deb_order, dim3(sxg_div_up(cc[3], 256)), dim3(256), 0, ks,
                               (const int *)a.clist, (const int *)a.cnt, nraw, cc[3], clist3,
                               (const int *)(pl ? ccount : nullptr),
                               (int)std::min<long>(sxg_option(SXG_OPT_DEB_ORDER_FULL),
                                                   0x7fffffffL));
            sxg_kt_begin_on(SXG_KT_DEB_TREE_GLB, ks);
            hipLaunchKernelGGL(k_deb_tree_glb, dim3(cc[3]), dim3(1024), 5 * DEB_HALF, ks, a3);
            sxg_kt_end_on(SXG_KT_DEB_TREE_GLB, ks);
            if (use_side) SXG_HIP_RET(hipEventRecord(S.side_ev[nside++], ks), -1);
        }
        if (cc[2] > 0 &&
            !launch_lds(reinterpret_cast<const void *>(&k_deb_tree_lds<1024, 2>), 2, 1024))
            return -1;
        if (cc[1] > 0 &&
            !launch_lds(reinterpret_cast<const void *>(&k_deb_tree_lds<512, 1>), 1, 512))
            return -1;
        if (cc[0] > 0 &&
            !launch_lds(reinterpret_cast<const void *>(&k_deb_tree_lds<256, 0>), 0, 256))
            return -1;
        for (int j = 0; j < nside; j++) SXG_HIP_RET(hipStreamWaitEvent(st, S.side_ev[j], 0), -1);
        sxg_kt_end(SXG_KT_DEB_LEVELS);
        SXG_HIP_RET(hipGetLastError(), -1);
        if (pl) {
            sxg_scan_excl(rootkept, objbase, nraw, &pd->nobj, st, &pd->nraw);
            nobj = (int)pl->cap[PL_NOBJ];
            sxg_plan_guard(&pd->nobj, nobj, PL_NOBJ);
            /* the frame's deblending work, for its record */
            hipLaunchKernelGGL(k_deb_plan_info, dim3(1), dim3(64), 0, st,
                               (const unsigned long long *)dwork, (const int *)ccount, pd);
        } else {
            sxg_scan_excl(rootkept, objbase, nraw, dtot, st);
            if (!sxg_read_back({{dtot, &nobj, 1}})) return -1;
            S.seen.cap[PL_NOBJ] = nobj;
        }
    } else if (pl) {
        hipLaunchKernelGGL(k_deb_zero, dim3(1), dim3(256), 0, st, &pd->nobj, 1L);
    } else {
        for (int k = PL_NTOT; k <= PL_NOBJ; k++) S.seen.cap[k] = 0;
    }
    S.nobj = nobj;
    S.ranked = S.counted = false;
    S.opix = nullptr;
    S.objoff = nullptr;
    ObjCols oc;
    if (!sxg_obj_alloc(nobj, oc)) return -1;
    if (nraw > 0 && nobj > 0) {
        ObjArgs A{};
        A.d = a; A.objbase = objbase; A.alloc = alloc; A.sub = S.img.as<float>(); A.o = oc;
        A.nobj = nobj;
        A.objraw = sxg_take<int>("obj.raw", nobj);
        A.objcomp = sxg_take<int>("obj.comp", nobj);
        int *okey = sxg_take<int>("opix.key", P0), *opix = sxg_take<int>("opix.pix", P0);
        int2 *objspan = sxg_take<int2>("obj.pixspan", (size_t)nobj + 1);
        int *objcnt = sxg_take<int>("obj.pixcount", (size_t)nobj + 1);
        int *objoff = sxg_take<int>("obj.pixoff", (size_t)nobj + 1);
        if (!A.objraw || !A.objcomp || !okey || !opix || !objspan || !objcnt || !objoff) return -1;
        A.okey = okey;
        const int gp = sxg_div_up(P0, 256);
        sxg_kt_begin(SXG_KT_DEB_OBJECTS);
        int *order = sxg_take<int>("pre.order", 2 * (size_t)nobj + 3);
        if (!order) return -1;
        hipLaunchKernelGGL(k_deb_objlist, dim3(sxg_div_up(nraw, 4)), dim3(256), 0, st, A,
                           order + 2 * (size_t)nobj);
        hipLaunchKernelGGL(k_pre_order, dim3(sxg_div_up(nobj, 256)), dim3(256), 0, st, A,
                           order + 2 * (size_t)nobj, order);
        A.order = order;
        /* workgroups: one an object at the most; fewer where the counts are exact: an object
           that is a whole raw object has the length of its pixels (the pixels bound how many
           are long), and a raw object with s > 1 kept nodes adds s - 1 <= 2 (nobj - nraw) in
           all to the objects, so at most 2 (nobj - nraw) are parts */
        const long parts = pl ? nobj : 2 * ((long)nobj - nraw);
        const long bigs = std::min<long>(nobj, P0 / PRE_BIG + parts);
        const long mids = std::min<long>(nobj, P0 / PRE_MID + parts);
        const int grid = (int)std::min<long>(nobj + 2, bigs + mids / 4 + nobj / 16 + 3);
        hipLaunchKernelGGL(k_deb_pre, dim3(grid), dim3(256), 0, st, A);
        /* planned: the counts past the device's nobj stay zero, so the scan over the
           capacity puts the total at objoff[nobj] as well; the gather kernel clears them */
        const long nz = pl ? (long)nobj + 1 : (long)nobj;
        hipLaunchKernelGGL(k_deb_gather, dim3(sxg_div_up(std::max<long>(P0, nz), 256)), dim3(256),
                           0, st, A, objcnt, objspan, nz);
        sxg_kt_end(SXG_KT_DEB_OBJECTS);
        /* raw pixels regrouped by object (stable: raster order inside each object) */
        sxg_kt_begin(SXG_KT_OBJ_SORT);
        hipLaunchKernelGGL(k_deb_objcount, dim3(gp), dim3(256), 0, st, A, objcnt, objspan);
        if (pl)
            sxg_scan_excl(objcnt, objoff, nobj + 1, nullptr, st);
        else
            sxg_scan_excl(objcnt, objoff, nobj, objoff + nobj, st);
        hipLaunchKernelGGL(k_obj_place1, dim3(gp), dim3(256), 0, st, A, (const int *)objoff, opix);
        hipLaunchKernelGGL(k_obj_place_multi, dim3(sxg_div_up(nobj, 4)), dim3(256), 0, st, A,
                           (const int *)objoff, (const int2 *)objspan, opix);
        sxg_kt_end(SXG_KT_OBJ_SORT);
        S.opix = opix;
        S.objoff = objoff;
    }
    sxg_stage_end(ST_DEBLEND);
    /* the object count was read above; the kernels queued since need no wait here (the
       next entry points run on the same stream, the getters wait for it) */
    SXG_HIP_RET(hipGetLastError(), -1);
    if (!sxg_stage_wait()) return -1;
    return nobj;
}

extern "C" void clear_deblend(int nthresh)
{
    (void)nthresh;
    sxg_state().deb_ready = false;
}
