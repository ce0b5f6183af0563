/*
 * sxg_wave.h -- 64-lane wavefront helpers shared by the per-object kernels.
 *
 * The reference accumulates every per-object sum in one sequential loop over the
 * object's pixels in raster order.  A wavefront reproduces those sums bit for bit by
 * letting each lane compute the terms of one pixel (in parallel) and then adding the
 * terms of the member lanes in lane order (the raster order of a chunk of 64 list
 * entries) with readlane: the additions are the only sequential part.
 */
#pragma once
#include <hip/hip_runtime.h>

__device__ inline unsigned long long sxw_lanes_below(int lane)
{
    return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

/* a place from counter[cls] for every thread of the workgroup (256 threads, all of which
   call; cls: 0 .. NC - 1, or -1 for none), one atomic for the workgroup and class: one for each
   wavefront and class, in turn, took the order kernels 13 us for 24,000 objects, 4 now */
template <int NC> __device__ inline int sxw_place(int *counter, int cls)
{
    __shared__ int s_at[NC][4];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    int before = 0;
#pragma unroll
    for (int c = 0; c < NC; c++) {
        const unsigned long long b = __ballot(cls == c);
        if (lane == 0) s_at[c][wid] = __popcll(b);
        if (cls == c) before = __popcll(b & sxw_lanes_below(lane));
    }
    __syncthreads();
    if (threadIdx.x < NC) {
        int *const a = s_at[threadIdx.x];
        const int n0 = a[0], n1 = a[1], n2 = a[2], n = n0 + n1 + n2 + a[3];
        const int base = n ? atomicAdd(&counter[threadIdx.x], n) : 0;
        a[0] = base;
        a[1] = base + n0;
        a[2] = base + n0 + n1;
        a[3] = base + n0 + n1 + n2;
    }
    __syncthreads();
    return cls >= 0 ? s_at[cls][wid] + before : 0;
}

/* value of v in lane j (j uniform across the wavefront) */
__device__ inline float sxw_rl(float v, int j)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), j));
}
__device__ inline double sxw_rl(double v, int j)
{
    const long long u = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)u, j);
    const int hi = __builtin_amdgcn_readlane((int)(u >> 32), j);
    return __hiloint2double(hi, lo);
}

template <int N> struct SxwInt { static constexpr int value = N; };
template <class Op> __device__ inline float sxw_dpp_allf(float v, Op op);
struct SxwMaxF { __device__ float operator()(float a, float b) const { return fmaxf(a, b); } };
struct SxwMinF { __device__ float operator()(float a, float b) const { return fminf(a, b); } };
/* float extrema over the full wavefront (every lane active), without LDS */
__device__ inline float sxw_max(float v) { return sxw_dpp_allf(v, SxwMaxF{}); }
__device__ inline float sxw_minf(float v) { return sxw_dpp_allf(v, SxwMinF{}); }
template <class Op> __device__ inline int sxw_dpp_all(int v, Op op);
struct SxwMax { __device__ int operator()(int a, int b) const { return max(a, b); } };
struct SxwMin { __device__ int operator()(int a, int b) const { return min(a, b); } };
struct SxwAdd { __device__ int operator()(int a, int b) const { return a + b; } };
/* int reductions over the full wavefront (every lane active), without LDS */
__device__ inline int sxw_max(int v) { return sxw_dpp_all(v, SxwMax{}); }
__device__ inline int sxw_min(int v) { return sxw_dpp_all(v, SxwMin{}); }
__device__ inline int sxw_sum(int v) { return sxw_dpp_all(v, SxwAdd{}); }
__device__ inline double sxw_sum(double v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

/* op over the 64 lanes of an int, the result in every lane, without LDS: DPP moves
   inside each row of 16 lanes (quad permutations for the partners at distance 1 and 2,
   then the half-row and row mirrors, each of which pairs a lane with one of the group it
   has not seen yet) and one readlane per row.  Every lane of the wavefront must be
   active (the readlanes take rows 0..3 from lanes 0, 16, 32 and 48). */
template <class Op> __device__ inline int sxw_dpp_all(int v, Op op)
{
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0xB1, 0xF, 0xF, false));    /* 1,0,3,2 */
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x4E, 0xF, 0xF, false));    /* 2,3,0,1 */
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x141, 0xF, 0xF, false));   /* half mirror */
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x140, 0xF, 0xF, false));   /* mirror */
    const int a = __builtin_amdgcn_readlane(v, 0), b = __builtin_amdgcn_readlane(v, 16);
    const int c = __builtin_amdgcn_readlane(v, 32), d = __builtin_amdgcn_readlane(v, 48);
    return op(op(a, b), op(c, d));
}
template <class Op> __device__ inline float sxw_dpp_allf(float v, Op op)
{
    auto mv = [](float x, int ctrl) {
        const int i = __float_as_int(x);
        int r;
        switch (ctrl) {
        case 0: r = __builtin_amdgcn_update_dpp(i, i, 0xB1, 0xF, 0xF, false); break;
        case 1: r = __builtin_amdgcn_update_dpp(i, i, 0x4E, 0xF, 0xF, false); break;
        case 2: r = __builtin_amdgcn_update_dpp(i, i, 0x141, 0xF, 0xF, false); break;
        default: r = __builtin_amdgcn_update_dpp(i, i, 0x140, 0xF, 0xF, false); break;
        }
        return __int_as_float(r);
    };
    v = op(v, mv(v, 0));
    v = op(v, mv(v, 1));
    v = op(v, mv(v, 2));
    v = op(v, mv(v, 3));
    const float a = sxw_rl(v, 0), b = sxw_rl(v, 16), c = sxw_rl(v, 32), d = sxw_rl(v, 48);
    return op(op(a, b), op(c, d));
}

/*
 * S + x_0 + x_1 + ... + x_15 in that order, x_j the value of lane j of the row of 16 lanes
 * (S: the same in every lane of a row, and the result too; each row its own sum).  One
 * v_fmac_f64 with a row broadcast per value: fma(x, 1, S) rounds once, as S + x does.  A
 * dependent chain of them issues every 4.3 cycles, against 10 to 15 for adds fed from LDS
 * reads (a read costs its wavefront 12 cycles) and 13 for readlanes (2.4 GHz, one
 * wavefront).  Every lane must be active; s_nop: a VALU result needs two wait states before
 * a DPP read.
 */
#define SXW_RF(n) "v_fmac_f64_dpp %0, %1, %2 row_newbcast:" #n " row_mask:0xf bank_mask:0xf\n"
__device__ inline double sxw_row_fold(double S, double x)
{
    const double one = 1.0;
    asm("s_nop 1\n" SXW_RF(0) SXW_RF(1) SXW_RF(2) SXW_RF(3) SXW_RF(4) SXW_RF(5) SXW_RF(6)
        SXW_RF(7) SXW_RF(8) SXW_RF(9) SXW_RF(10) SXW_RF(11) SXW_RF(12) SXW_RF(13) SXW_RF(14)
        SXW_RF(15)
        : "+v"(S)
        : "v"(x), "v"(one));
    return S;
}

/* the same for floats */
#define SXW_RA(n) "v_add_f32_dpp %0, %1, %0 row_newbcast:" #n " row_mask:0xf bank_mask:0xf\n"
__device__ inline float sxw_row_fold(float S, float x)
{
    asm("s_nop 1\n" SXW_RA(0) SXW_RA(1) SXW_RA(2) SXW_RA(3) SXW_RA(4) SXW_RA(5) SXW_RA(6)
        SXW_RA(7) SXW_RA(8) SXW_RA(9) SXW_RA(10) SXW_RA(11) SXW_RA(12) SXW_RA(13) SXW_RA(14)
        SXW_RA(15)
        : "+v"(S)
        : "v"(x));
    return S;
}

/* S + the values of all 64 lanes in lane order, the same in every lane */
__device__ inline float sxw_fold64(float S, float x)
{
    S = sxw_rl(sxw_row_fold(S, x), 0);
    S = sxw_rl(sxw_row_fold(S, x), 16);
    S = sxw_rl(sxw_row_fold(S, x), 32);
    return sxw_rl(sxw_row_fold(S, x), 48);
}

/* keep the five largest values seen by this lane, t[0] >= ... >= t[4] (-inf = empty) */
struct SxwTop5 {
    float t[5];
    __device__ void init()
    {
#pragma unroll
        for (int i = 0; i < 5; i++) t[i] = -INFINITY;
    }
    __device__ void add(float v)
    {
#pragma unroll
        for (int i = 0; i < 5; i++) {
            const float hi = fmaxf(t[i], v), lo = fminf(t[i], v);
            t[i] = hi;
            v = lo;
        }
    }
    /* the five largest values over the wavefront, in descending order (-inf: none) */
    __device__ void five(float (&r)[5])
    {
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int round = 0; round < 5; round++) {
            const float m = sxw_max(t[0]);
            const unsigned long long b = __ballot(t[0] == m);
            if (lane == __builtin_ctzll(b)) {
#pragma unroll
                for (int i = 0; i < 4; i++) t[i] = t[i + 1];
                t[4] = -INFINITY;
            }
            r[round] = m;
        }
    }
    /* the same over the row of 16 lanes */
    __device__ void row_five(float (&r)[5]);
};

/*
 * Transposed ordered folds.  The NS terms of each member lane of a chunk are written to
 * LDS compacted in lane order (row s holds the terms of sum s); then lane s adds row s
 * in order into its own accumulator.  NS sums advance together at one LDS read and one
 * add per member, and each sum is still the sequential sum in raster order.
 * rows points to this wavefront's scratch of NS rows of SXW_ROW elements.
 */
#define SXW_ROW 66   /* row stride: rows start on different LDS banks */

template <int NS, class T>
__device__ inline void sxw_fold(T *rows, const T (&t)[NS], bool member, T &acc)
{
    const int lane = threadIdx.x & 63;
    const unsigned long long b = __ballot(member);
    const int cnt = __popcll(b);
    if (member) {
        const int pos = __popcll(b & sxw_lanes_below(lane));
#pragma unroll
        for (int s = 0; s < NS; s++) rows[s * SXW_ROW + pos] = t[s];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (lane < NS) {
        const T *row = rows + lane * SXW_ROW;
        T a = acc;
#pragma unroll 16
        for (int j = 0; j < cnt; j++) a += row[j];
        acc = a;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

/*
 * The same with ND double sums and NF float sums advancing together: lane s < ND adds
 * double row s, lane ND + s adds float row s.  Every chain lane performs one double and
 * one float add per member (the add it does not own reads a valid row and is ignored),
 * so the chains of both types interleave in one instruction stream.  drows: ND rows,
 * frows: NF rows (at least one row each).
 */
template <int ND, int NF>
__device__ inline void sxw_fold2(double *drows, float *frows, const double (&td)[ND],
                                 const float (&tf)[NF], bool member, double &dacc, float &facc)
{
    static_assert(ND + NF <= 64, "one lane per sum");
    const int lane = threadIdx.x & 63;
    const unsigned long long b = __ballot(member);
    const int cnt = __popcll(b);
    if (member) {
        const int pos = __popcll(b & sxw_lanes_below(lane));
#pragma unroll
        for (int s = 0; s < ND; s++) drows[s * SXW_ROW + pos] = td[s];
#pragma unroll
        for (int s = 0; s < NF; s++) frows[s * SXW_ROW + pos] = tf[s];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (lane < ND + NF) {
        const double *dr = drows + (lane < ND ? lane : 0) * SXW_ROW;
        const float *fr = frows + (lane >= ND ? lane - ND : 0) * SXW_ROW;
        double da = dacc;
        float fa = facc;
#pragma unroll 16
        for (int j = 0; j < cnt; j++) {
            da += dr[j];
            fa += fr[j];
        }
        dacc = da;
        facc = fa;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

/*
 * The same for up to four double sums, a row of 16 lanes for each (sxw_row_fold): 4.3 cycles
 * a member for all of them where the reads and adds above take 13.  The members' terms go to
 * LDS compacted, padded with +0 to a multiple of 16 (an identity: a sum that starts at +0 is
 * never -0).  acc: the row's sum in each of its lanes.
 */
#define SXW_WROW 80   /* row stride: two rows of lanes on all banks */
template <int ND>
__device__ inline void sxw_wfold(double *rows, const double (&t)[ND], bool member, double &acc)
{
    static_assert(ND <= 4, "a row of lanes for each sum");
    const int lane = threadIdx.x & 63;
    const unsigned long long b = __ballot(member);
    const int cnt = __popcll(b), n16 = (cnt + 15) >> 4;
    const int pos = __popcll(b & sxw_lanes_below(lane));
    const bool pad = lane >= cnt && lane < 16 * n16;
#pragma unroll
    for (int s = 0; s < ND; s++) {
        if (member) rows[s * SXW_WROW + pos] = t[s];
        if (pad) rows[s * SXW_WROW + lane] = 0.0;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const double *p = rows + min(lane >> 4, ND - 1) * SXW_WROW + (lane & 15);
    double x[4];
#pragma unroll
    for (int c = 0; c < 4; c++) x[c] = p[16 * c];
#pragma unroll
    for (int c = 0; c < 4; c++)
        if (c < n16) acc = sxw_row_fold(acc, x[c]);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

/*
 * The same over a workgroup of four wavefronts, for the objects whose sums are the longest:
 * 256 pixels a step, one per thread.  All four compute terms, then each adds three of the
 * sums, a row of 16 lanes each (sxw_row_fold), so the longest chain is 256 adds of 4.3
 * cycles for 256 pixels instead of 16 to 33 cycles a pixel (LDS reads and adds of one
 * wavefront).  A pixel left out adds +0, an identity (a sum that starts at +0 is never -0).
 * ND double sums (up to 9, or 12 without float sums: wavefront w has 3w .. 3w + 2), NF float
 * sums (up to 4, wavefront 3).  rows: sxw_brows(ND, NF) doubles.  All 256 threads call it.
 */
#define SXW_BROW 272   /* row stride in elements: two rows of lanes on all banks */
constexpr int sxw_brows(int nd, int nf) { return nd * SXW_BROW + (nf * SXW_BROW + 1) / 2; }

template <int ND, int NF>
__device__ inline void sxw_bfold(double *rows, const double (&td)[ND], const float (&tf)[NF + 1],
                                 bool member, double &dacc, float &facc)
{
    static_assert(ND <= (NF ? 9 : 12) && NF <= 4, "three sums a wavefront");
    const int tid = threadIdx.x, wid = tid >> 6, row = (tid >> 4) & 3, l16 = tid & 15;
    float *frows = reinterpret_cast<float *>(rows + ND * SXW_BROW);
#pragma unroll
    for (int s = 0; s < ND; s++) rows[s * SXW_BROW + tid] = member ? td[s] : 0.0;
#pragma unroll
    for (int s = 0; s < NF; s++) frows[s * SXW_BROW + tid] = member ? tf[s] : 0.0f;
    __syncthreads();
    if (NF && wid == 3) {
        const float *p = frows + min(row, NF > 0 ? NF - 1 : 0) * SXW_BROW + l16;
#pragma unroll
        for (int c = 0; c < 16; c++) facc = sxw_row_fold(facc, p[16 * c]);
    } else if (3 * wid < ND) {
        const double *p = rows + min(3 * wid + row, ND - 1) * SXW_BROW + l16;
#pragma unroll
        for (int c = 0; c < 16; c++) dacc = sxw_row_fold(dacc, p[16 * c]);
    }
    __syncthreads();
}

/* the sums of sxw_bfold, to every thread */
template <int ND, int NF>
__device__ inline void sxw_bfold_end(double *rows, double dacc, float facc, double (&d)[ND],
                                     float (&f)[NF + 1])
{
    const int tid = threadIdx.x, wid = tid >> 6, row = (tid >> 4) & 3, l16 = tid & 15;
    float *frows = reinterpret_cast<float *>(rows + ND);
    if (l16 == 0 && row < 3 && 3 * wid + row < ND) rows[3 * wid + row] = dacc;
    if (NF && l16 == 0 && wid == 3 && row < NF) frows[row] = facc;
    __syncthreads();
#pragma unroll
    for (int s = 0; s < ND; s++) d[s] = rows[s];
#pragma unroll
    for (int s = 0; s < NF; s++) f[s] = frows[s];
    __syncthreads();
}

/* value of v in lane J of the row of 16 */
template <int J> __device__ inline float sxw_row_bcast(float v)
{
    const int i = __float_as_int(v);
    return __int_as_float(__builtin_amdgcn_update_dpp(i, i, 0x150 + J, 0xF, 0xF, false));
}
/* op over the 16 lanes of a row, the result in every lane of it */
template <class V, class Op> __device__ inline V sxw_row_all(V v, Op op)
{
    static_assert(sizeof(V) == 4, "one register");
    auto mv = [](V x, auto ctrl) {
        const int i = __builtin_bit_cast(int, x);
        return __builtin_bit_cast(
            V, __builtin_amdgcn_update_dpp(i, i, decltype(ctrl)::value, 0xF, 0xF, false));
    };
    v = op(v, mv(v, SxwInt<0xB1>{}));
    v = op(v, mv(v, SxwInt<0x4E>{}));
    v = op(v, mv(v, SxwInt<0x141>{}));
    return op(v, mv(v, SxwInt<0x140>{}));
}

__device__ inline void SxwTop5::row_five(float (&r)[5])
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int round = 0; round < 5; round++) {
        const float m = sxw_row_all(t[0], SxwMaxF{});
        const unsigned b = (unsigned)(__ballot(t[0] == m) >> (lane & 48)) & 0xffffu;
        if ((lane & 15) == __builtin_ctz(b)) {
#pragma unroll
            for (int i = 0; i < 4; i++) t[i] = t[i + 1];
            t[4] = -INFINITY;
        }
        r[round] = m;
    }
}

/*
 * One object by a row of 16 lanes (SXW_ROWS: the many small ones; four share a wavefront,
 * and with it every instruction of the per-object arithmetic), by a wavefront (SXW_WAVE) or
 * by a workgroup of four (SXW_GROUP): the pixel index a thread starts at, the step, and
 * reductions over all of its threads.  Rows may be in different places of the program; the
 * lanes of a row are not.
 */
enum SxwSize { SXW_ROWS, SXW_WAVE, SXW_GROUP };

template <SxwSize Z> struct SxwTeam {
    static constexpr int STEP = Z == SXW_GROUP ? 256 : Z == SXW_WAVE ? 64 : 16;
    __device__ static int first() { return threadIdx.x & (STEP - 1); }
    template <class V, class Op> __device__ static V all(V v, Op op)
    {
        v = sxw_row_all(v, op);
        if constexpr (Z == SXW_WAVE) {
            const int i = __builtin_bit_cast(int, v);
            auto rl = [&](int j) {
                return __builtin_bit_cast(V, __builtin_amdgcn_readlane(i, j));
            };
            v = op(op(rl(0), rl(16)), op(rl(32), rl(48)));
        }
        if constexpr (Z == SXW_GROUP) {
            __shared__ V s[16];
            if ((threadIdx.x & 15) == 0) s[threadIdx.x >> 4] = v;
            __syncthreads();
            v = sxw_row_all(s[threadIdx.x & 15], op);
            __syncthreads();
        }
        return v;
    }
    __device__ static float max(float v) { return all(v, SxwMaxF{}); }
    __device__ static float min(float v) { return all(v, SxwMinF{}); }
    __device__ static int max(int v) { return all(v, SxwMax{}); }
    __device__ static int min(int v) { return all(v, SxwMin{}); }
    __device__ static int sum(int v) { return all(v, SxwAdd{}); }
    /* the fifth largest value (needs at least five) */
    __device__ static float fifth(SxwTop5 &t)
    {
        float r[5];
        if constexpr (Z == SXW_WAVE) {
            t.five(r);
            return r[4];
        }
        t.row_five(r);
        if constexpr (Z == SXW_GROUP) {
            __shared__ float s[16][5];
            if ((threadIdx.x & 15) == 0)
                for (int i = 0; i < 5; i++) s[threadIdx.x >> 4][i] = r[i];
            __syncthreads();
            for (int i = 0; i < 5; i++) t.t[i] = s[threadIdx.x & 15][i];
            __syncthreads();
            t.row_five(r);
        }
        return r[4];
    }
};

/* the ordered sums of an object: ND double and NF float ones; rows: LDS, for a workgroup
   sxw_brows(ND, NF) doubles, for a wavefront its own sxw_wrows(ND, NF), none for a row */
constexpr int sxw_wrows(int nd, int nf)
{
    return nf == 0 && nd <= 4 ? nd * SXW_WROW : nd * SXW_ROW + (nf * SXW_ROW + 1) / 2;
}
template <int ND, int NF, SxwSize Z> struct SxwSums {
    double d[ND];
    float f[NF + 1];
    __device__ SxwSums()
    {
#pragma unroll
        for (int s = 0; s < ND; s++) d[s] = 0.0;
#pragma unroll
        for (int s = 0; s <= NF; s++) f[s] = 0.0f;
    }
    __device__ void add(double *rows, const double (&td)[ND], const float (&tf)[NF + 1],
                        bool member)
    {
        if constexpr (Z == SXW_GROUP) {
            sxw_bfold<ND, NF>(rows, td, tf, member, d[0], f[0]);
        } else if constexpr (Z == SXW_WAVE && NF > 0) {
            float t[NF];
#pragma unroll
            for (int s = 0; s < NF; s++) t[s] = tf[s];
            sxw_fold2<ND, NF>(rows, reinterpret_cast<float *>(rows + ND * SXW_ROW), td, t, member,
                              d[0], f[0]);
        } else if constexpr (Z == SXW_WAVE && ND <= 4) {
            sxw_wfold<ND>(rows, td, member, d[0]);
        } else if constexpr (Z == SXW_WAVE) {
            sxw_fold<ND, double>(rows, td, member, d[0]);
        } else {
#pragma unroll
            for (int s = 0; s < ND; s++) d[s] = sxw_row_fold(d[s], member ? td[s] : 0.0);
#pragma unroll
            for (int s = 0; s < NF; s++) f[s] = sxw_row_fold(f[s], member ? tf[s] : 0.0f);
        }
    }
    __device__ void end(double *rows)
    {
        if constexpr (Z == SXW_GROUP) {
            sxw_bfold_end<ND, NF>(rows, d[0], f[0], d, f);
        } else if constexpr (Z == SXW_WAVE) {
            const double a = d[0];
            const float b = f[0];
#pragma unroll
            for (int s = 0; s < ND; s++) d[s] = sxw_rl(a, NF == 0 && ND <= 4 ? 16 * s : s);
#pragma unroll
            for (int s = 0; s < NF; s++) f[s] = sxw_rl(b, ND + s);
        }
    }
};

/*
 * The output offset of this workgroup (256 threads) of a two-launch compaction: the sum of the
 * counts of the workgroups before it, which every workgroup adds up itself (a launch of one
 * workgroup for the scan took longer, with its gap, than these reads), or, of more than
 * SXG_BLOCK_SUMS workgroups, the sums as a launch between the two has scanned them.  The last
 * workgroup stores the total.
 */
#define SXG_BLOCK_SUMS 4096
template <bool SCANNED> __device__ inline int sxg_block_offset(const int *bsum, int *total)
{
    if (SCANNED) return bsum[blockIdx.x];
    __shared__ int s_part[4];
    const int b = blockIdx.x;
    int s = 0;
    for (int j = threadIdx.x; j < b; j += 256) s += bsum[j];
    s = sxw_sum(s);
    if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = s;
    __syncthreads();
    s = s_part[0] + s_part[1] + s_part[2] + s_part[3];
    if (b == (int)gridDim.x - 1 && threadIdx.x == 0) *total = s + bsum[b];
    return s;
}

/*
 * Two-launch stable compaction of the indices 0 .. n - 1 that src keeps: src.read(k) is what
 * decides, src.take(k, that) the kept value (>= 0) or -1, src.put(place, k, value) stores it.
 * ITEMS indices a thread, 256 apart, so that loads and stores are coalesced; every first load
 * is issued before one is used (crowded 4096 x 4096 frame: 14 us a count of 10^6 where each
 * was waited for).
 */
template <class Src, int ITEMS>
__device__ inline void sxg_pick_values(const Src &src, long base, int n, int (&v)[ITEMS])
{
#pragma unroll
    for (int i = 0; i < ITEMS; i++) {
        const long k = base + 256 * i;
        v[i] = src.read(k < n ? (int)k : n - 1);
    }
#pragma unroll
    for (int i = 0; i < ITEMS; i++) {
        const long k = base + 256 * i;
        const int t = src.take(k < n ? (int)k : n - 1, v[i]);
        v[i] = k < n ? t : -1;
    }
}

template <class Src, int ITEMS>
__global__ void __launch_bounds__(256) k_pick_count(Src src, int n, int *bsum, const int *nd)
{
    __shared__ int s_part[4];
    if (nd) n = min(*nd, n);
    const long base = (long)blockIdx.x * (256 * ITEMS) + threadIdx.x;
    int c = 0;
    if (n > 0) {
        int v[ITEMS];
        sxg_pick_values(src, base, n, v);
#pragma unroll
        for (int i = 0; i < ITEMS; i++) c += __popcll(__ballot(v[i] >= 0));
    }
    if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) bsum[blockIdx.x] = s_part[0] + s_part[1] + s_part[2] + s_part[3];
}

template <class Src, int ITEMS, bool SCANNED>
__global__ void __launch_bounds__(256) k_pick_write(Src src, int n, const int *bsum, int *total,
                                                    const int *nd)
{
    __shared__ int s_at[64];   /* by item and wavefront: kept ones before it in the workgroup */
    if (nd) n = min(*nd, n);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const long base = (long)blockIdx.x * (256 * ITEMS) + threadIdx.x;
    int v[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; i++) v[i] = -1;
    if (n > 0) sxg_pick_values(src, base, n, v);
#pragma unroll
    for (int i = 0; i < ITEMS; i++) {
        const int c = __popcll(__ballot(v[i] >= 0));
        if (lane == 0) s_at[4 * i + wid] = c;
    }
    const int first = sxg_block_offset<SCANNED>(bsum, total);
    __syncthreads();
    if (wid == 0) {
        const int own = lane < 4 * ITEMS ? s_at[lane] : 0;
        int x = own;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(x, d);
            if (lane >= d) x += o;
        }
        s_at[lane] = first + x - own;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; i++) {
        const unsigned long long b = __ballot(v[i] >= 0);
        if (v[i] >= 0)
            src.put(s_at[4 * i + wid] + __popcll(b & sxw_lanes_below(lane)),
                    (int)(base + 256 * i), v[i]);
    }
}

int *sxg_block_sums(int nb);   /* device: nb ints */
void sxg_scan_blocks(int *bsum, int nb, int *total, hipStream_t s);
void sxg_set_int(int *p, int v, hipStream_t s);

/* With nd (planned runs) n is a capacity and the number of indices is *nd (<= n).  Up to
   2^18 indices 1024 a workgroup, so that small frames have more than a few of them, else
   4096: the sums that every workgroup adds up grow with their number. */
template <class Src>
bool sxg_pick(const Src &src, int n, int *count, hipStream_t s, const int *nd)
{
    if (n <= 0) {
        sxg_set_int(count, 0, s);
        return true;
    }
    const bool small = n <= 1 << 18;
    const int nb = (int)(((long)n + (small ? 1023 : 4095)) / (small ? 1024 : 4096));
    int *bsum = sxg_block_sums(nb);
    if (!bsum) return false;
    if (small) {
        hipLaunchKernelGGL((k_pick_count<Src, 4>), dim3(nb), dim3(256), 0, s, src, n, bsum, nd);
        hipLaunchKernelGGL((k_pick_write<Src, 4, false>), dim3(nb), dim3(256), 0, s, src, n, bsum,
                           count, nd);
        return true;
    }
    hipLaunchKernelGGL((k_pick_count<Src, 16>), dim3(nb), dim3(256), 0, s, src, n, bsum, nd);
    if (nb > SXG_BLOCK_SUMS) {
        sxg_scan_blocks(bsum, nb, count, s);
        hipLaunchKernelGGL((k_pick_write<Src, 16, true>), dim3(nb), dim3(256), 0, s, src, n, bsum,
                           count, nd);
    } else {
        hipLaunchKernelGGL((k_pick_write<Src, 16, false>), dim3(nb), dim3(256), 0, s, src, n,
                           bsum, count, nd);
    }
    return true;
}
