/*
 * kernels_class.hip - row classes: operators whose rows take few distinct
 * forms are read as one byte per row.
 *
 * A row's form is its list of (column - row, value) pairs in storage order.
 * A constant-coefficient stencil has one form per combination of missing
 * neighbours (27 for the 3D 7-point stencil, 9 for the 2D 5-point one), and
 * where the aggregates repeat, so have its Galerkin coarse levels. An
 * operator of at most CLS_MAX forms of at most CLS_ROW entries keeps, beside
 * its CSR arrays, the class of each row (one byte) and the forms (a few KB);
 * the row kernels stage the forms in LDS and stream the codes, so a sweep
 * moves 25 bytes per row (x, f, the result and the code) instead of 89 (the
 * 7-point stencil with one mask byte per row) or 132 (int32 columns). The
 * products, their order and the divisors are those of the CSR row, so every
 * result has the same bits.
 *
 * Where the forms differ only in which entries they have (constant
 * coefficients, missing neighbours eliminated: one value per offset, at most
 * CLS_ROW offsets) the byte is the mask of the entries present, and offsets
 * and values are kernel arguments: no table, no barrier, and the gathers
 * do not wait for the byte.
 *
 * Measured on level 0 of 3D Poisson 160^3 (4.1 M rows) and 2D 2048^2, FP64:
 * product 56.7 and 57.7 us with the one-byte mask and streamed values, 24.0
 * and 20.0 us from the table of forms, 13.5 and 12.1 us as a constant
 * stencil; the L1 sweep 63.3 -> 18.1 us (5.7 TB/s of its 102 MB; FP32
 * 30.9 -> 12.8 us). The FP64 sweep is bound by the vectors' traffic through L2
 * and the last-level cache. The FP32 one is not (53 MB, 4.1 TB/s): half of the
 * bytes, but as many instructions (5.1 M vector instructions a launch against
 * 5.3, the same loads), which take 40 % of its cycles to issue, and its waves
 * wait on them and on latency.
 */
#include "kernels_common.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <utility>

namespace bcmg {

namespace {

constexpr int CLS_SLOTS = 1024;   /* hash slots while the forms are collected */
/* a block of 256 rows with more forms than this raises the overflow flag by
   itself: an operator without repeated rows is told by its first blocks */
constexpr int CLS_BLOCK_MAX = 128;
constexpr unsigned long long HASH_EMPTY = 0ull;

/* the finalizer of splitmix64 (Steele, Lea and Flood, 2014) */
__device__ __forceinline__ unsigned long long mix64(unsigned long long z)
{
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

/* hash of row r's form (never HASH_EMPTY) */
__device__ __forceinline__ unsigned long long row_hash(int r, const int *__restrict__ rp,
                                                       const int *__restrict__ ci,
                                                       const double *__restrict__ av)
{
    const int e0 = rp[r], e1 = rp[r + 1];
    unsigned long long h = 0x9E3779B97F4A7C15ull * (unsigned)(e1 - e0 + 1);
    for (int e = e0; e < e1; e++) {
        h = mix64(h ^ (unsigned)(ci[e] - r));
        h = mix64(h + (unsigned long long)__double_as_longlong(av[e]));
    }
    return h | 1ull;
}

/* what the host reads of one operator's analysis, in one copy: the tables of up
   to HEAD_CLS classes (entry k of class c at [k ncls + c]) and the offsets */
constexpr int HEAD_CLS = 64;
struct ClassHead {
    int count, over, ncls, band, row, pad; /* row: the longest */
    double tv[CLS_ROW * HEAD_CLS];
    int idx[(CLS_ROW + 1) * HEAD_CLS];
    int offs[OFFSET_INTS];
};
static_assert(sizeof(ClassHead) % sizeof(double) == 0, "heads follow each other in the staging");

/* work area of one operator's analysis (device) */
struct ClassWork {
    ClassHead h;
    unsigned long long hash[CLS_SLOTS];
    int rep[CLS_SLOTS];       /* smallest row with that hash */
    int cls[CLS_SLOTS];       /* class of the slot, once numbered */
    /* the tables, entry k of class c at [k ncls + c]: lengths, then offsets;
       values, then the diagonals and the sums of magnitudes (the smoother
       divisors) */
    int idx[(CLS_ROW + 1) * CLS_MAX];
    double tv[(CLS_ROW + 2) * CLS_MAX];
};

__global__ __launch_bounds__(BS) void k_class_clear(ClassWork *w)
{
    for (int q = threadIdx.x; q < CLS_SLOTS; q += BS) {
        w->hash[q] = HASH_EMPTY;
        w->rep[q] = 0x7fffffff;
        w->cls[q] = -1;
    }
    if (threadIdx.x == 0) w->h.count = w->h.over = w->h.ncls = w->h.band = w->h.row = 0;
    if (threadIdx.x < OFFSET_INTS) w->h.offs[threadIdx.x] = threadIdx.x ? PAT_EMPTY : 0;
}

/* step 1: the largest |column - row| (columns ascend in a row), and the
   distinct row hashes of a 256-row block (an LDS table), which go into the
   operator's table with the smallest row that has them; a row of more than
   CLS_ROW entries, more than CLS_BLOCK_MAX hashes in a block or CLS_MAX in all
   raises `over`, which later blocks read first */
__global__ __launch_bounds__(BS) void k_class_collect(int n, const int *__restrict__ rp,
                                                      const int *__restrict__ ci,
                                                      const double *__restrict__ av,
                                                      ClassWork *w)
{
    constexpr int LS = 2 * BS;
    __shared__ unsigned long long lh[LS];
    __shared__ int lr[LS];
    __shared__ int far[BS / 64];
    __shared__ int lcount, skip;
    const int t = threadIdx.x;
    for (int q = t; q < LS; q += BS) {
        lh[q] = HASH_EMPTY;
        lr[q] = 0x7fffffff;
    }
    if (t == 0) {
        lcount = 0;
        skip = __hip_atomic_load(&w->h.over, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const int r = blockIdx.x * BS + t;
    int o = 0, len = 0;
    if (r < n) {
        const int e0 = rp[r], e1 = rp[r + 1];
        len = e1 - e0;
        if (len > 0) o = max(r - ci[e0], ci[e1 - 1] - r);
    }
#pragma unroll
    for (int q = 32; q > 0; q >>= 1) o = max(o, __shfl_xor(o, q, 64));
    if ((t & 63) == 0) far[t >> 6] = o;
    const bool lng = __syncthreads_or(len > CLS_ROW);
    if (t == 0) {
        for (int q = 1; q < BS / 64; q++) o = max(o, far[q]);
        if (o > __hip_atomic_load(&w->h.band, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMax(&w->h.band, o);
        if (lng) atomicOr(&w->h.over, 1);
    }
    if (skip || lng) return;
    if (r < n) {
        const unsigned long long h = row_hash(r, rp, ci, av);
        /* LS >= 2 BS slots for at most BS hashes: the probe ends */
        int s = (int)(h >> 40) & (LS - 1);
        for (;;) {
            const unsigned long long prev = atomicCAS(&lh[s], HASH_EMPTY, h);
            if (prev == HASH_EMPTY) atomicAdd(&lcount, 1);
            if (prev == HASH_EMPTY || prev == h) break;
            s = (s + 1) & (LS - 1);
        }
        atomicMin(&lr[s], r);
    }
    __syncthreads();
    if (lcount > CLS_BLOCK_MAX) {
        if (t == 0) atomicOr(&w->h.over, 1);
        return;
    }
    for (int q = t; q < LS; q += BS) {
        const unsigned long long h = lh[q];
        if (h == HASH_EMPTY) continue;
        int s = (int)(h >> 20) & (CLS_SLOTS - 1);
        for (int probe = 0;; probe++) {
            if (probe == CLS_SLOTS) {
                atomicOr(&w->h.over, 1);
                break;
            }
            unsigned long long v =
                __hip_atomic_load(&w->hash[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (v == HASH_EMPTY) {
                v = atomicCAS(&w->hash[s], HASH_EMPTY, h);
                if (v == HASH_EMPTY) {
                    if (atomicAdd(&w->h.count, 1) >= CLS_MAX) atomicOr(&w->h.over, 1);
                    v = h;
                }
            }
            if (v == h) {
                if (__hip_atomic_load(&w->rep[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >
                    lr[q])
                    atomicMin(&w->rep[s], lr[q]);
                break;
            }
            s = (s + 1) & (CLS_SLOTS - 1);
        }
    }
}

/* step 2 (one block): number the forms by their smallest row and write the
   tables (the divisors as k_diag and k_abs_rowsum form them) */
__global__ __launch_bounds__(CLS_MAX) void k_class_tables(const int *__restrict__ rp,
                                                          const int *__restrict__ ci,
                                                          const double *__restrict__ av,
                                                          ClassWork *w)
{
    __shared__ int slot[CLS_MAX], rep[CLS_MAX];
    __shared__ int m, longest;
    const int t = threadIdx.x;
    if (t == 0) m = longest = 0;
    __syncthreads();
    if (w->h.over) return;
    for (int q = t; q < CLS_SLOTS; q += CLS_MAX)
        if (w->hash[q] != HASH_EMPTY) {
            const int at = atomicAdd(&m, 1); /* at most CLS_MAX: over is clear */
            slot[at] = q;
            rep[at] = w->rep[q];
        }
    __syncthreads();
    const int nc = m;
    const int r = t < nc ? rep[t] : 0;
    const int e0 = rp[r], len = rp[r + 1] - e0;
    if (t < nc) atomicMax(&longest, len);
    __syncthreads();
    const int crow = longest; /* at most CLS_ROW: over is clear */
    if (t == 0) {
        w->h.ncls = nc;
        w->h.row = crow;
    }
    if (t >= nc) return;
    int c = 0;
    for (int q = 0; q < nc; q++) c += rep[q] < rep[t] ? 1 : 0;
    w->cls[slot[t]] = c;
    int *const idx = w->idx;
    double *const tv = w->tv;
    const bool head = nc <= HEAD_CLS;
    idx[c] = len;
    if (head) w->h.idx[c] = len;
    double d = 0.0, s = 0.0;
    for (int k = 0; k < crow; k++) {
        const bool in = k < len;
        const double v = in ? av[e0 + k] : 0.0;
        const int o = in ? ci[e0 + k] - r : 0;
        idx[(k + 1) * nc + c] = o;
        tv[k * nc + c] = v;
        if (head) {
            w->h.idx[(k + 1) * nc + c] = o;
            w->h.tv[k * nc + c] = v;
        }
        if (in) {
            if (o == 0) d = v;
            s += fabs(v);
        }
    }
    tv[crow * nc + c] = d;
    tv[(crow + 1) * nc + c] = s;
}

/* step 3: each row's class, its form compared entry by entry with the
   table's (a hash collision raises `over`); rows that pad the last block
   get class 0 */
__global__ __launch_bounds__(BS) void k_class_codes(int n, const int *__restrict__ rp,
                                                    const int *__restrict__ ci,
                                                    const double *__restrict__ av,
                                                    ClassWork *w,
                                                    unsigned char *__restrict__ code)
{
    /* raised by step 1, when the table may lack hashes, or here: no classes */
    if (__hip_atomic_load(&w->h.over, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
    const int *const idx = w->idx;
    const double *const tv = w->tv;
    const int r = blockIdx.x * BS + threadIdx.x;
    if (r >= n) {
        code[r] = 0;
        return;
    }
    const int nc = w->h.ncls;
    const unsigned long long h = row_hash(r, rp, ci, av);
    int s = (int)(h >> 20) & (CLS_SLOTS - 1);
    int probe = 0;
    for (; probe < CLS_SLOTS && w->hash[s] != h; probe++) s = (s + 1) & (CLS_SLOTS - 1);
    const int c = probe < CLS_SLOTS ? w->cls[s] : 0;
    const int e0 = rp[r], len = rp[r + 1] - e0;
    bool same = probe < CLS_SLOTS && idx[c] == len;
    for (int k = 0; same && k < len; k++)
        same = idx[(k + 1) * nc + c] == ci[e0 + k] - r &&
               __double_as_longlong(tv[k * nc + c]) == __double_as_longlong(av[e0 + k]);
    if (!same) atomicOr(&w->h.over, 1);
    code[r] = (unsigned char)c;
}

/* the forms in FP32, or rounded to bfloat16 and widened; the divisors in FP32 */
__global__ __launch_bounds__(BS) void k_class_lowp(int nv, int nall, const double *__restrict__ a,
                                                   float *__restrict__ b, int bf16)
{
    const int i = blockIdx.x * BS + threadIdx.x;
    if (i >= nall) return;
    const float v = (float)a[i];
    b[i] = (bf16 && i < nv) ? bf16_round(v) : v;
}

/* ---------------------------------------------------------- row kernels */

/* the forms of an operator as the kernels take them */
template <typename VT>
struct ClassRef {
    const unsigned char *code;
    const int *idx;
    const VT *tv;
    int nc;      /* classes */
    int crow;    /* longest row */
};

/* LDS: the values and one divisor row, then lengths and offsets */
template <typename VT>
inline size_t class_lds_bytes(int nc, int crow)
{
    return (size_t)nc * ((crow + 1) * sizeof(VT) + (crow + 1) * sizeof(int));
}

/* The forms into LDS: values [k nc + c] (k < crow), the divisor row at
   k = crow (table row `drow`; not copied when negative), lengths and offsets
   behind them. */
template <typename VT>
__device__ __forceinline__ void class_stage(const ClassRef<VT> &C, int drow, VT *&lv, int *&li)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_class[];
    lv = reinterpret_cast<VT *>(smem_class);
    li = reinterpret_cast<int *>(lv + (size_t)(C.crow + 1) * C.nc);
    const int nv = C.crow * C.nc;
#pragma unroll 1
    for (int q = threadIdx.x; q < nv + C.nc; q += BS) {
        li[q] = C.idx[q];
        if (q < nv)
            lv[q] = C.tv[q];
        else if (drow >= 0)
            lv[q] = C.tv[(size_t)drow * C.nc + (q - nv)];
    }
}

/* Row r's sum from its form: all gathers go out at once (an absent entry
   gathers the row's own element and adds nothing), the products are rounded
   and added left to right from 0 in storage order (staged_row_sum's bits). */
template <typename VT, int CR, typename XT = VT>
__device__ __forceinline__ VT class_row_sum(int c, int nc, int crow, const VT *lv, const int *li,
                                            const XT *__restrict__ x, int r)
{
    const int len = li[c];
    VT g[CR], v[CR];
    int j[CR];
#pragma unroll
    for (int k = 0; k < CR; k++) {
        j[k] = r;
        v[k] = 0;
        if (k < crow) {
            const int o = li[(k + 1) * nc + c];
            v[k] = lv[k * nc + c];
            j[k] = r + o;   /* the table holds offset 0 past the row's length */
        }
    }
#pragma unroll
    for (int k = 0; k < CR; k++) g[k] = (VT)x[j[k]];
    VT t = 0;
#pragma unroll
    for (int k = 0; k < CR; k++) t = k < len ? t + v[k] * g[k] : t;
    return t;
}

template <typename VT, int OP, int CR, int RPT, bool DTAB>
__global__ __launch_bounds__(BS) void k_rows_class(int n, ClassRef<VT> C, int drow,
                                                   const VT *__restrict__ x,
                                                   const VT *__restrict__ f,
                                                   const VT *__restrict__ d, VT *__restrict__ y)
{
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = b * (BS * RPT) + threadIdx.x;
    int c[RPT];
    VT fr[RPT], xr[RPT], dr[RPT];
#pragma unroll
    for (int q = 0; q < RPT; q++) {
        const int r = r0 + q * BS;
        c[q] = 0;
        fr[q] = xr[q] = 0;
        dr[q] = 1;
        if (r < n) {
            c[q] = C.code[r];
            if (OP != OP_SPMV) fr[q] = f[r];
            if (OP == OP_JACOBI) xr[q] = x[r];
            if (OP == OP_JACOBI && !DTAB) dr[q] = d[r];
        }
    }
    VT *lv;
    int *li;
    class_stage<VT>(C, DTAB ? drow : -1, lv, li);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < RPT; q++) {
        const int r = r0 + q * BS;
        if (r >= n) return;
        const VT t = class_row_sum<VT, CR>(c[q], C.nc, C.crow, lv, li, x, r);
        if (DTAB) dr[q] = lv[C.crow * C.nc + c[q]];
        if (OP == OP_SPMV)
            y[r] = t;
        else if (OP == OP_RESID)
            y[r] = fr[q] - t;
        else
            y[r] = (fr[q] - t) / dr[q] + xr[q];
    }
}

/* ------------------------------------------------------ constant stencils */

/* Row r's entries g[k] summed under mask m (products rounded, added left to
   right from 0), with DL1 also the row's sum of magnitudes as k_abs_rowsum
   forms it. */
template <typename VT, int K, bool DL1>
__device__ __forceinline__ void stencil_sum(unsigned m, const StencilRef<VT> &S, const VT (&g)[K],
                                            VT &t, VT &dl)
{
    t = 0;
    double a = 0.0;
#pragma unroll
    for (int k = 0; k < K; k++)
        if ((m >> k) & 1u) {
            t = t + S.v[k] * g[k];
            if (DL1) a += S.a[k];
        }
    dl = (VT)a;
}

/* The gathers of W consecutive rows from r (W VT values are 16 bytes, or
   W = 1). INNER: every r + off + W - 1 lies in [0, n), so the loads are
   unconditional 16-byte ones (any alignment of VT); else each element is
   loaded where its index is in range and its mask bit set. */
template <typename VT, int K, int W, bool INNER, typename XT = VT>
__device__ __forceinline__ void stencil_gather(const StencilRef<VT> &S, const XT *__restrict__ x,
                                               int r, int n, const unsigned (&m)[W],
                                               VT (&g)[W][K])
{
    if constexpr (INNER) {
        typedef VT vec __attribute__((ext_vector_type(W == 1 ? 2 : W)));
        typedef vec uvec __attribute__((aligned(sizeof(VT))));
#pragma unroll
        for (int k = 0; k < K; k++) {
            if constexpr (W == 1) {
                g[0][k] = (VT)x[r + S.off[k]];
            } else {
                static_assert(std::is_same<XT, VT>::value, "wide gathers read x's own type");
                const vec q = *reinterpret_cast<const uvec *>(x + r + S.off[k]);
#pragma unroll
                for (int w = 0; w < W; w++) g[w][k] = q[w];
            }
        }
    } else {
#pragma unroll
        for (int w = 0; w < W; w++)
#pragma unroll
            for (int k = 0; k < K; k++) {
                g[w][k] = 0;
                if (r + w < n && ((m[w] >> k) & 1u)) g[w][k] = (VT)x[r + w + S.off[k]];
            }
    }
}

/* Row operations on a constant stencil, W rows per thread. A block whose
   gathers stay inside the vector whatever the masks issues every load at
   once; the first and last blocks load under the masks. */
template <typename VT, int OP, int K, int W, int DIV>
__global__ __launch_bounds__(BS) void k_rows_stencil(int n, StencilRef<VT> S,
                                                     const VT *__restrict__ x,
                                                     const VT *__restrict__ f,
                                                     const VT *__restrict__ d, VT *__restrict__ y)
{
    typedef VT vec __attribute__((ext_vector_type(W == 1 ? 2 : W)));
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = b * (BS * W);
    const int r = r0 + threadIdx.x * W;
    const bool inner = S.inner.holds(r0, BS * W);
    unsigned m[W];
    VT g[W][K], fr[W], xr[W], dr[W];
#pragma unroll
    for (int w = 0; w < W; w++) {
        fr[w] = xr[w] = 0;
        dr[w] = 1;
    }
    if (inner) {
        if constexpr (W == 1) {
            m[0] = S.mask[r];
            stencil_gather<VT, K, W, true>(S, x, r, n, m, g);
            if (OP != OP_SPMV) fr[0] = f[r];
            if (OP == OP_JACOBI) xr[0] = x[r];
            if (OP == OP_JACOBI && DIV == DIV_ARRAY) dr[0] = d[r];
        } else {
            const unsigned mm = W == 2 ? *reinterpret_cast<const unsigned short *>(S.mask + r)
                                       : *reinterpret_cast<const unsigned *>(S.mask + r);
            stencil_gather<VT, K, W, true>(S, x, r, n, m, g);
            vec vf, vx, vd;
            if (OP != OP_SPMV) vf = *reinterpret_cast<const vec *>(f + r);
            if (OP == OP_JACOBI) vx = *reinterpret_cast<const vec *>(x + r);
            if (OP == OP_JACOBI && DIV == DIV_ARRAY) vd = *reinterpret_cast<const vec *>(d + r);
#pragma unroll
            for (int w = 0; w < W; w++) {
                m[w] = (mm >> (8 * w)) & 0xFFu;
                if (OP != OP_SPMV) fr[w] = vf[w];
                if (OP == OP_JACOBI) xr[w] = vx[w];
                if (OP == OP_JACOBI && DIV == DIV_ARRAY) dr[w] = vd[w];
            }
        }
    } else {
#pragma unroll
        for (int w = 0; w < W; w++) {
            m[w] = 0;
            if (r + w < n) {
                m[w] = S.mask[r + w];
                if (OP != OP_SPMV) fr[w] = f[r + w];
                if (OP == OP_JACOBI) xr[w] = x[r + w];
                if (OP == OP_JACOBI && DIV == DIV_ARRAY) dr[w] = d[r + w];
            }
        }
        stencil_gather<VT, K, W, false>(S, x, r, n, m, g);
    }
    VT o[W];
#pragma unroll
    for (int w = 0; w < W; w++) {
        VT t, dl;
        stencil_sum<VT, K, OP == OP_JACOBI && DIV == DIV_L1>(m[w], S, g[w], t, dl);
        if (OP == OP_SPMV)
            o[w] = t;
        else if (OP == OP_RESID)
            o[w] = fr[w] - t;
        else
            o[w] = (fr[w] - t) / (DIV == DIV_L1 ? dl : DIV == DIV_DIAG ? S.diag : dr[w]) + xr[w];
    }
    if (W > 1 && inner) {
        vec v;
#pragma unroll
        for (int w = 0; w < W; w++) v[w] = o[w];
        *reinterpret_cast<vec *>(y + r) = v;
    } else {
#pragma unroll
        for (int w = 0; w < W; w++)
            if (r + w < n) y[r + w] = o[w];
    }
}

/* k_spmv_dots on a constant stencil (the same 256-row blocks and trees) */
template <int K, int KO, typename ZT>
__global__ __launch_bounds__(BS) void k_spmv_dots_stencil(int n, StencilRef<double> S,
                                                          const ZT *__restrict__ z,
                                                          double *__restrict__ t,
                                                          const double *__restrict__ rv,
                                                          const double *__restrict__ to,
                                                          double *__restrict__ part)
{
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = b * BS;
    const int r = r0 + threadIdx.x;
    double sdot[K];
#pragma unroll
    for (int k = 0; k < K; k++) sdot[k] = 0.0;
    auto row = [&](auto inner) {
        const unsigned m[1] = {S.mask[r]};
        double g[1][KO];
        const double zr = (double)z[r], rr = rv[r];
        const double tor = K > 2 ? to[r] : 0.0;
        stencil_gather<double, KO, 1, decltype(inner)::value, ZT>(S, z, r, n, m, g);
        double tr, unused;
        stencil_sum<double, KO, false>(m[0], S, g[0], tr, unused);
        t[r] = tr;
        sdot[0] = rr * zr;
        sdot[1] = tr * zr;
        if (K > 2) sdot[K - 1] = tor * zr;
    };
    if (S.inner.holds(r0, BS))
        row(std::true_type{});
    else if (r < n)
        row(std::false_type{});
    block_reduce_store<K>(sdot, part + (size_t)b * K);
}

/* one sweep from zero on a constant stencil */
template <typename VT, int DIV>
__global__ __launch_bounds__(BS) void k_jz_stencil(int n, StencilRef<VT> S,
                                                   const VT *__restrict__ f, VT *__restrict__ y)
{
    const int i = blockIdx.x * BS + threadIdx.x;
    if (i >= n) return;
    VT t, dl, g[CLS_ROW];
#pragma unroll
    for (int k = 0; k < CLS_ROW; k++) g[k] = 0;
    stencil_sum<VT, CLS_ROW, DIV == DIV_L1>(DIV == DIV_L1 ? S.mask[i] : 0u, S, g, t, dl);
    y[i] = f[i] / (DIV == DIV_L1 ? dl : S.diag);
}

/* rows a slab workgroup of 1024 threads holds (four a thread: 64 KB of LDS in
   FP64), and its own rows' least number where there are more workgroups than
   CUs (the others are recomputed) */
constexpr int SLAB_ROWS = 4096;
/* the same with the rows in registers: one a thread (with four a thread, 128
   VGPRs, four sweeps took 15-20 us, no less than four launches) */
constexpr int SLAB_ROWS_REG = 1024;
constexpr int SLAB_CUS = 256;
constexpr int SLAB_MIN_SHARE = 1640;

/* Several Jacobi/L1 sweeps of a constant stencil in one launch. A workgroup
   owns rows [a, a + m) and keeps them and the rows within steps * B of them
   (B the largest |offset|) in LDS: sweep t recomputes the rows within
   (steps - t) B of its own, so no workgroup waits for another and x, f and
   the masks are read and the result written once for all sweeps. Row sums,
   divisors and the update are k_rows_stencil's, so the result has the bits
   of separate sweeps. A level whose rows all fit one workgroup has no
   redundant rows and takes any number of sweeps.
   zero: x is known to be zero, the first sweep f / d is made while loading
   (MODE 0 and 2; `steps` counts the sweeps after it). MODE 1: x starts as
   x + P x_c (k_prolong's fma; x = 0 when zero). MODE 2 (one workgroup):
   after the sweeps the residual rows are restricted into fu.fc as the
   residual and SpMV kernels do. */
template <typename VT, int K, int RPT, int MODE, int DIV>
__global__ __launch_bounds__(1024) void k_stencil_slab(int n, StencilRef<VT> S, int m, int B,
                                                       int steps, int zero,
                                                       const VT *__restrict__ f,
                                                       const VT *__restrict__ xin,
                                                       VT *__restrict__ xout, BlockFuse<VT> fu)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_slab[];
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int a = b * m, e = min(a + m, n);
    const int reach = steps * B;
    const int lo = max(0, a - reach), hi = min(n, e + reach);
    /* gathers of absent entries are not made, those of present ones stay in
       [lo, hi): no pad is needed around the rows */
    VT *cur = reinterpret_cast<VT *>(smem_slab);
    VT *nxt = cur + (m + 2 * reach);
    unsigned mk[RPT];
    VT fr[RPT], dr[RPT];
#pragma unroll
    for (int q = 0; q < RPT; q++) {
        const int i = lo + (int)threadIdx.x + 1024 * q;
        mk[q] = 0;
        fr[q] = 0;
        dr[q] = 1;
        if (i < hi) {
            mk[q] = S.mask[i];
            fr[q] = f[i];
            VT x0 = 0;
            if (MODE == 1)
                x0 = fma(fu.p[i], fu.xc[fu.agg[i]], zero ? VT(0) : xin[i]);
            else if (!zero)
                x0 = xin[i];
            VT t, dl, g[K];
#pragma unroll
            for (int k = 0; k < K; k++) g[k] = 0;
            stencil_sum<VT, K, DIV == DIV_L1>(DIV == DIV_L1 ? mk[q] : 0u, S, g, t, dl);
            dr[q] = DIV == DIV_L1 ? dl : S.diag;
            cur[i - lo] = MODE != 1 && zero ? fr[q] / dr[q] : x0;
        }
    }
    __syncthreads();
    for (int t = 1; t <= steps; t++) {
        const int wl = max(0, a - (steps - t) * B), wh = min(n, e + (steps - t) * B);
#pragma unroll
        for (int q = 0; q < RPT; q++) {
            const int i = lo + (int)threadIdx.x + 1024 * q;
            if (i >= wl && i < wh) {
                VT sum = 0;
                const VT *c = cur + (i - lo);
#pragma unroll
                for (int k = 0; k < K; k++)
                    if ((mk[q] >> k) & 1u) sum = sum + S.v[k] * c[S.off[k]];
                nxt[i - lo] = (fr[q] - sum) / dr[q] + c[0];
            }
        }
        __syncthreads();
        VT *const sw = cur;
        cur = nxt;
        nxt = sw;
    }
#pragma unroll
    for (int q = 0; q < RPT; q++) {
        const int i = lo + (int)threadIdx.x + 1024 * q;
        if (i >= a && i < e) xout[i] = cur[i - lo];
    }
    if constexpr (MODE == 2) {
#pragma unroll
        for (int q = 0; q < RPT; q++) {
            const int i = (int)threadIdx.x + 1024 * q;
            if (i < n) {
                VT sum = 0;
#pragma unroll
                for (int k = 0; k < K; k++)
                    if ((mk[q] >> k) & 1u) sum = sum + S.v[k] * cur[i + S.off[k]];
                nxt[i] = fr[q] - sum;
            }
        }
        __syncthreads();
        for (int I = threadIdx.x; I < fu.nc; I += 1024) {
            VT t = 0;
            const int e1 = fu.rrp[I + 1];
            for (int j = fu.rrp[I]; j < e1; j++) t = t + fu.rv[j] * nxt[fu.rci[j]];
            fu.fc[I] = t;
        }
    }
}

/* k_stencil_slab for any rows of at most CLS_ROW entries: the row of a thread
   stays in registers (columns as LDS positions) and the divisor comes from
   its array. Row sums in storage order from 0. */
template <typename MT, typename VT, int MODE>
__global__ __launch_bounds__(1024) void k_rows_slab(int n, const int *__restrict__ rp,
                                                    const int *__restrict__ ci,
                                                    const MT *__restrict__ av,
                                                    const VT *__restrict__ d, int m, int B,
                                                    int steps, int zero,
                                                    const VT *__restrict__ f,
                                                    const VT *__restrict__ xin,
                                                    VT *__restrict__ xout, BlockFuse<VT> fu)
{
    __shared__ VT xs[2][SLAB_ROWS_REG];
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int a = b * m, e = min(a + m, n);
    const int reach = steps * B;
    const int lo = max(0, a - reach), hi = min(n, e + reach); /* at most SLAB_ROWS_REG rows */
    const int t = threadIdx.x, i = lo + t;
    VT *cur = xs[0], *nxt = xs[1];
    VT v[CLS_ROW], fr = 0, dr = 1;
    int c[CLS_ROW], len = 0;
    if (i < hi) {
        const int j0 = rp[i];
        len = rp[i + 1] - j0;
        fr = f[i];
        dr = d[i];
        VT x0 = 0;
        if (MODE == 1)
            x0 = fma(fu.p[i], fu.xc[fu.agg[i]], zero ? VT(0) : xin[i]);
        else if (!zero)
            x0 = xin[i];
#pragma unroll
        for (int k = 0; k < CLS_ROW; k++) {
            v[k] = k < len ? mval<VT>(av[j0 + k]) : VT(0);
            c[k] = k < len ? ci[j0 + k] - lo : 0;
        }
        cur[t] = MODE != 1 && zero ? fr / dr : x0;
    }
    __syncthreads();
    for (int s = 1; s <= steps; s++) {
        /* a row of the window has all its columns in [lo, hi) */
        if (i >= a - (steps - s) * B && i < e + (steps - s) * B && i < hi) {
            VT sum = 0;
#pragma unroll
            for (int k = 0; k < CLS_ROW; k++)
                if (k < len) sum = sum + v[k] * cur[c[k]];
            nxt[t] = (fr - sum) / dr + cur[t];
        }
        __syncthreads();
        VT *const sw = cur;
        cur = nxt;
        nxt = sw;
    }
    if (i >= a && i < e) xout[i] = cur[t];
}

/* class codes -> entry masks */
struct MaskTable {
    unsigned char m[CLS_MAX];
};
__global__ __launch_bounds__(BS) void k_class_masks(int n, MaskTable T,
                                                    unsigned char *__restrict__ code)
{
    const int r = blockIdx.x * BS + threadIdx.x;
    if (r < n) code[r] = T.m[code[r]];
}

/* one sweep from zero, y = f / d with d from the row's class */
template <typename VT>
__global__ __launch_bounds__(BS) void k_jz_class(int n, ClassRef<VT> C, int drow,
                                                 const VT *__restrict__ f, VT *__restrict__ y)
{
    const int i = blockIdx.x * BS + threadIdx.x;
    if (i < n) y[i] = f[i] / C.tv[(size_t)drow * C.nc + C.code[i]];
}

/* k_spmv_dots on row classes: t = A z, per 256-row block the partial sums
   of r.z, t.z and (K = 3) to.z over the same rows in the same tree */
template <int K, int CR, typename ZT>
__global__ __launch_bounds__(BS) void k_spmv_dots_class(int n, ClassRef<double> C,
                                                        const ZT *__restrict__ z,
                                                        double *__restrict__ t,
                                                        const double *__restrict__ rv,
                                                        const double *__restrict__ to,
                                                        double *__restrict__ part)
{
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int r = b * BS + threadIdx.x;
    double sdot[K];
#pragma unroll
    for (int k = 0; k < K; k++) sdot[k] = 0.0;
    double *lv;
    int *li;
    class_stage<double>(C, -1, lv, li);
    __syncthreads();
    if (r < n) {
        const int c = C.code[r];
        const double zr = (double)z[r], rr = rv[r];
        const double tor = K > 2 ? to[r] : 0.0;
        const double tr = class_row_sum<double, CR, ZT>(c, C.nc, C.crow, lv, li, z, r);
        t[r] = tr;
        sdot[0] = rr * zr;
        sdot[1] = tr * zr;
        if (K > 2) sdot[K - 1] = tor * zr;
    }
    block_reduce_store<K>(sdot, part + (size_t)b * K);
}

template <typename VT>
ClassRef<VT> class_ref(const DevCsr &A, MatType mt);
template <>
ClassRef<double> class_ref<double>(const DevCsr &A, MatType)
{
    return {A.cls.code.get(), A.cls.idx.get(), A.cls.v64.get(), A.cls.n, A.cls.row};
}
template <>
ClassRef<float> class_ref<float>(const DevCsr &A, MatType mt)
{
    return {A.cls.code.get(), A.cls.idx.get(),
            mt == MT_BF16 ? A.cls.v16.get() : A.cls.v32.get(), A.cls.n, A.cls.row};
}

/* rows per thread: the block stages the forms (nc (crow + 1) (4 + value)
   bytes) for BS * RPT rows. Product with 1 / 2 / 4 rows: 27.2 / 24.0 / 23.3 us
   at 4.1 M rows, 8.2 / 7.7 / 7.9 at 1 M, 3.4 / 3.9 / 5.2 at 262 144 (too few
   blocks); sweeps 30.9 / 29.4 / 30.7 at 4.1 M */
constexpr int CLS_RPT_BIG = 2;
constexpr int CLS_BIG = 1 << 19;

template <typename VT, int OP, int CR, int RPT>
void rows_class_rpt(hipStream_t s, const DevCsr &A, const ClassRef<VT> &C, int drow, const VT *x,
                    const VT *f, const VT *d, VT *y)
{
    const int nb = (A.n + BS * RPT - 1) / (BS * RPT);
    const size_t lds = class_lds_bytes<VT>(C.nc, C.crow);
    if (OP == OP_JACOBI && drow >= 0)
        k_rows_class<VT, OP, CR, RPT, true><<<nb, BS, lds, s>>>(A.n, C, drow, x, f, d, y);
    else
        k_rows_class<VT, OP, CR, RPT, false><<<nb, BS, lds, s>>>(A.n, C, -1, x, f, d, y);
}

template <typename VT, int OP, int CR>
void rows_class_cr(hipStream_t s, const DevCsr &A, const ClassRef<VT> &C, int drow, const VT *x,
                   const VT *f, const VT *d, VT *y)
{
    if (A.n >= CLS_BIG)
        rows_class_rpt<VT, OP, CR, CLS_RPT_BIG>(s, A, C, drow, x, f, d, y);
    else
        rows_class_rpt<VT, OP, CR, 1>(s, A, C, drow, x, f, d, y);
}

template <typename VT, int OP>
void rows_class_op(hipStream_t s, const DevCsr &A, const ClassRef<VT> &C, int drow, const VT *x,
                   const VT *f, const VT *d, VT *y)
{
    if (C.crow <= 5)
        rows_class_cr<VT, OP, 5>(s, A, C, drow, x, f, d, y);
    else if (C.crow <= 7)
        rows_class_cr<VT, OP, 7>(s, A, C, drow, x, f, d, y);
    else
        rows_class_cr<VT, OP, CLS_ROW>(s, A, C, drow, x, f, d, y);
}

/* rows from which a thread takes two rows (FP64: 16-byte loads): product
   with 1 / 2 rows 19.4 / 13.5 us at 4.1 M rows, 6.4 / 5.0 at 1 M; at 262 144
   rows 2.88 / 2.99, where the launch is bound by latency and more threads
   are better. FP32 with 4 rows was slower than with 2 (whole 160^3 FP32
   solve 20.6 against 19.3 ms) */
constexpr int STC_WIDE = 1 << 19;
template <typename VT, int OP, int K, int W, int DIV>
void rows_stencil_w(hipStream_t s, const DevCsr &A, const StencilRef<VT> &S, const VT *x,
                    const VT *f, const VT *d, VT *y)
{
    const int nb = (A.n + BS * W - 1) / (BS * W);
    k_rows_stencil<VT, OP, K, W, DIV><<<nb, BS, 0, s>>>(A.n, S, x, f, d, y);
}

template <typename VT, int OP, int K, int DIV>
void rows_stencil_k(hipStream_t s, const DevCsr &A, const StencilRef<VT> &S, const VT *x,
                    const VT *f, const VT *d, VT *y)
{
    /* the wide form's loads and stores of f, d and y are 16-byte aligned */
    const uintptr_t al = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y) |
                         (OP != OP_SPMV ? reinterpret_cast<uintptr_t>(f) : 0) |
                         (OP == OP_JACOBI && DIV == DIV_ARRAY ? reinterpret_cast<uintptr_t>(d) : 0);
    if (A.n >= STC_WIDE && (al & 15) == 0)
        rows_stencil_w<VT, OP, K, 2, DIV>(s, A, S, x, f, d, y);
    else
        rows_stencil_w<VT, OP, K, 1, DIV>(s, A, S, x, f, d, y);
}

template <typename VT, int OP, int DIV>
void rows_stencil_op(hipStream_t s, const DevCsr &A, const StencilRef<VT> &S, const VT *x,
                     const VT *f, const VT *d, VT *y)
{
    const int k = A.cls.k;
    if (k <= 5)
        rows_stencil_k<VT, OP, 5, DIV>(s, A, S, x, f, d, y);
    else if (k <= 7)
        rows_stencil_k<VT, OP, 7, DIV>(s, A, S, x, f, d, y);
    else
        rows_stencil_k<VT, OP, CLS_ROW, DIV>(s, A, S, x, f, d, y);
}

template <typename VT, int K, int RPT, int MODE>
void slab_div(hipStream_t s, int n, const StencilRef<VT> &S, int m, int B, int steps, int zero,
              DivSource div, const VT *f, const VT *xin, VT *xout, const BlockFuse<VT> &fu)
{
    const int nb = (n + m - 1) / m;
    const size_t lds = 2 * (size_t)(m + 2 * steps * B) * sizeof(VT);
    if (div == DIV_L1)
        k_stencil_slab<VT, K, RPT, MODE, DIV_L1>
            <<<nb, 1024, lds, s>>>(n, S, m, B, steps, zero, f, xin, xout, fu);
    else
        k_stencil_slab<VT, K, RPT, MODE, DIV_DIAG>
            <<<nb, 1024, lds, s>>>(n, S, m, B, steps, zero, f, xin, xout, fu);
    BCMG_CHECK_LAUNCH();
}

template <typename VT, int K, int MODE>
void slab_rpt(hipStream_t s, int n, const StencilRef<VT> &S, int m, int B, int steps, int zero,
              DivSource div, const VT *f, const VT *xin, VT *xout, const BlockFuse<VT> &fu)
{
    const int ext = std::min(n, m + 2 * steps * B);
    if (ext <= 1024)
        slab_div<VT, K, 1, MODE>(s, n, S, m, B, steps, zero, div, f, xin, xout, fu);
    else if (ext <= 2048)
        slab_div<VT, K, 2, MODE>(s, n, S, m, B, steps, zero, div, f, xin, xout, fu);
    else if (ext <= 4096)
        slab_div<VT, K, 4, MODE>(s, n, S, m, B, steps, zero, div, f, xin, xout, fu);
    else
        throw Error(BCMG_EINVAL, "stencil slab: too many rows");
}

template <typename MT, typename VT>
void rows_slab(hipStream_t s, const DevCsr &A, const MT *av, int m, int B, int steps, int zero,
               const VT *d, const VT *f, const VT *xin, VT *xout, const BlockFuse<VT> &fu)
{
    const int n = A.n, nb = (n + m - 1) / m;
    const int ext = std::min(n, m + 2 * steps * B);
    const size_t lds = 2 * (size_t)(m + 2 * steps * B) * sizeof(VT);
    auto go = [&](auto kern) {
        kern<<<nb, 1024, lds, s>>>(n, A.row.get(), A.col.get(), av, d, m, B, steps, zero, f, xin,
                                   xout, fu);
    };
    const bool pro = fu.agg != nullptr;
    if (ext > SLAB_ROWS_REG || fu.fc) throw Error(BCMG_EINVAL, "slab sweeps: too many rows");
    if (pro)
        go(k_rows_slab<MT, VT, 1>);
    else
        go(k_rows_slab<MT, VT, 0>);
    BCMG_CHECK_LAUNCH();
}

template <typename VT, int MODE>
void slab_k(hipStream_t s, const DevCsr &A, const StencilRef<VT> &S, int m, int B, int steps,
            int zero, DivSource div, const VT *f, const VT *xin, VT *xout,
            const BlockFuse<VT> &fu)
{
    const int k = A.cls.k;
    if (k <= 5)
        slab_rpt<VT, 5, MODE>(s, A.n, S, m, B, steps, zero, div, f, xin, xout, fu);
    else if (k <= 7)
        slab_rpt<VT, 7, MODE>(s, A.n, S, m, B, steps, zero, div, f, xin, xout, fu);
    else
        slab_rpt<VT, CLS_ROW, MODE>(s, A.n, S, m, B, steps, zero, div, f, xin, xout, fu);
}

/* the divisor's table row, or -1 for the caller's array */
int div_row(const DevCsr &A, DivSource div)
{
    return div == DIV_DIAG ? A.cls.row : div == DIV_L1 ? A.cls.row + 1 : -1;
}

} // namespace

namespace {

/* Whether the forms (host copies of the tables) are one stencil with entries
   left out: at most CLS_ROW offsets in all, each with one value (the same
   bits). Then R.k, R.off and R.val hold it and T the mask of each class. */
bool constant_stencil(RowClasses &R, const int *idx, const double *val, MaskTable &T)
{
    std::vector<std::pair<int, double>> ov;
    for (int c = 0; c < R.n; c++)
        for (int k = 0; k < idx[c]; k++) {
            const int o = idx[(k + 1) * R.n + c];
            const double v = val[k * R.n + c];
            auto it = std::find_if(ov.begin(), ov.end(),
                                   [&](const std::pair<int, double> &p) { return p.first == o; });
            if (it == ov.end()) {
                if (ov.size() == CLS_ROW) return false;
                ov.emplace_back(o, v);
            } else if (std::memcmp(&it->second, &v, sizeof(v)) != 0) {
                return false;
            }
        }
    std::sort(ov.begin(), ov.end(), [](const std::pair<int, double> &a,
                                       const std::pair<int, double> &b) { return a.first < b.first; });
    R.k = (int)ov.size();
    for (int k = 0; k < R.k; k++) {
        R.off[k] = ov[k].first;
        R.val[k] = ov[k].second;
    }
    for (int c = 0; c < CLS_MAX; c++) {
        unsigned m = 0;
        for (int k = 0; c < R.n && k < idx[c]; k++)
            for (int q = 0; q < R.k; q++)
                if (R.off[q] == idx[(k + 1) * R.n + c]) m |= 1u << q;
        T.m[c] = (unsigned char)m;
    }
    return true;
}

} // namespace

/* smaller operators are not analysed: their sweeps take a few microseconds
   in one workgroup (relax_block_ok) as they are */
constexpr int CLS_MIN_ROWS = 512;

namespace {

/* whether A is analysed: its rows may all have CLS_ROW entries or fewer */
bool class_candidate(const DevCsr &A)
{
    return A.n == A.m && A.n >= CLS_MIN_ROWS && !A.cls.analysed &&
           A.nnz <= (long long)CLS_ROW * A.n;
}

/* A's analysis into w and its codes, queued; w->h tells the outcome. offsets:
   where A has no classes, also its distinct column offsets. */
void launch_class_scan(Ctx &c, DevCsr &A, ClassWork *w, bool offsets)
{
    A.cls.analysed = true;
    const int nblk = (A.n + BS - 1) / BS;
    const int *rp = A.row.get(), *ci = A.col.get();
    const double *av = A.val.get();
    A.cls.code.alloc((size_t)nblk * BS);
    k_class_clear<<<1, BS, 0, c.stream>>>(w);
    k_class_collect<<<nblk, BS, 0, c.stream>>>(A.n, rp, ci, av, w);
    k_class_tables<<<1, CLS_MAX, 0, c.stream>>>(rp, ci, av, w);
    k_class_codes<<<nblk, BS, 0, c.stream>>>(A.n, rp, ci, av, w, A.cls.code.get());
    BCMG_CHECK_LAUNCH();
    if (offsets) launch_offsets(c.stream, A, w->h.offs, &w->h.over);
}

/* what the analysis found, from the host copy of its head */
void take_classes(Ctx &c, DevCsr &A, ClassWork *w, const ClassHead &h)
{
    RowClasses &R = A.cls;
    A.band = h.band;
    if (h.over) {
        R.code.release();
        return;
    }
    R.n = h.ncls;
    R.row = h.row;
    const size_t ni = (size_t)(R.row + 1) * R.n, nv = (size_t)R.row * R.n;
    const int *idx = h.idx;
    const double *val = h.tv;
    std::vector<int> li;
    std::vector<double> lv;
    if (R.n > HEAD_CLS) {
        li.resize(ni);
        lv.resize(nv);
        BCMG_HIP(hipMemcpyAsync(li.data(), w->idx, ni * sizeof(int), hipMemcpyDeviceToHost,
                                c.stream));
        BCMG_HIP(hipMemcpyAsync(lv.data(), w->tv, nv * sizeof(double), hipMemcpyDeviceToHost,
                                c.stream));
        BCMG_HIP(hipStreamSynchronize(c.stream));
        idx = li.data();
        val = lv.data();
    }
    std::vector<int> off(idx + R.n, idx + ni);
    for (int k = 0; k < R.row; k++)
        for (int q = 0; q < R.n; q++)
            if (k >= idx[q]) off[(size_t)k * R.n + q] = 0; /* no entry; a diagonal there is */
    std::sort(off.begin(), off.end());
    off.erase(std::unique(off.begin(), off.end()), off.end());
    A.noff = std::min((int)off.size(), PAT_MAX + 1);
    A.off_lo = off.front();
    A.off_hi = off.back();
    MaskTable T;
    if (constant_stencil(R, idx, val, T)) {
        k_class_masks<<<(A.n + BS - 1) / BS, BS, 0, c.stream>>>(A.n, T, R.code.get());
        BCMG_CHECK_LAUNCH();
        return;
    }
    R.idx.alloc(ni);
    R.v64.alloc(nv + 2 * (size_t)R.n);
    BCMG_HIP(hipMemcpyAsync(R.idx.get(), w->idx, ni * sizeof(int), hipMemcpyDeviceToDevice,
                            c.stream));
    BCMG_HIP(hipMemcpyAsync(R.v64.get(), w->tv, (nv + 2 * (size_t)R.n) * sizeof(double),
                            hipMemcpyDeviceToDevice, c.stream));
}

constexpr size_t HEAD_INTS = sizeof(ClassHead) / sizeof(int);

} // namespace

void make_classes(Ctx &c, const std::vector<DevCsr *> &mats)
{
    std::vector<DevCsr *> cand;
    for (DevCsr *A : mats)
        if (class_candidate(*A) && A->maxrow > 0 && A->maxrow <= CLS_ROW) cand.push_back(A);
    if (cand.empty()) return;
    DBuf<ClassWork> work(cand.size());
    for (size_t k = 0; k < cand.size(); k++)
        launch_class_scan(c, *cand[k], work.get() + k, false);
    /* one round trip for as many operators as the pinned staging holds */
    constexpr size_t HEADS = Ctx::H_INTS / HEAD_INTS;
    static_assert(HEADS >= 1, "the staging holds a head");
    for (size_t b = 0; b < cand.size(); b += HEADS) {
        const size_t e = std::min(cand.size(), b + HEADS);
        for (size_t k = b; k < e; k++)
            BCMG_HIP(hipMemcpyAsync(c.h_ints + HEAD_INTS * (k - b), &work.get()[k].h,
                                    sizeof(ClassHead), hipMemcpyDeviceToHost, c.stream));
        BCMG_HIP(hipStreamSynchronize(c.stream));
        for (size_t k = b; k < e; k++) {
            ClassHead h;
            std::memcpy(&h, c.h_ints + HEAD_INTS * (k - b), sizeof(h));
            take_classes(c, *cand[k], work.get() + k, h);
        }
    }
}

/* An upload's analysis: the tile sizes, the classes and (where there are none)
   the offsets come back in one round trip; a symmetric stencil takes a second.
   A 32^3 Poisson upload 0.277 -> 0.250 ms, 32^3 log-normal 0.306 -> 0.264 (both
   0.213 without any analysis). */
void analyze_rows(Ctx &c, DevCsr &A)
{
    launch_block_nnz(c, A);
    DBuf<ClassWork> work;
    const bool scan = class_candidate(A);
    /* behind what resolve_tiles stages */
    constexpr size_t AT = 256;
    static_assert(AT + HEAD_INTS <= Ctx::H_INTS, "the staging holds a head");
    const bool offsets = scan && sym_candidate(A);
    if (scan) {
        work.alloc(1);
        launch_class_scan(c, A, work.get(), offsets);
        BCMG_HIP(hipMemcpyAsync(c.h_ints + AT, &work.get()->h, sizeof(ClassHead),
                                hipMemcpyDeviceToHost, c.stream));
    }
    resolve_tiles(c, {&A});
    if (scan) {
        ClassHead h;
        std::memcpy(&h, c.h_ints + AT, sizeof(h));
        take_classes(c, A, work.get(), h);
        if (A.maxrow > CLS_ROW) A.band = -1;
        std::vector<int> off;
        if (offsets && A.cls.n == 0 && offsets_found(h.offs, off)) make_sym(c, A, off);
    }
    make_narrow(c, {&A});
}

void RowClasses::make_lowp(hipStream_t s, bool bf16)
{
    if (n == 0 || k > 0) return; /* a constant stencil's values are kernel arguments */
    DBuf<float> &o = bf16 ? v16 : v32;
    const int nv = row * n, nall = (row + 2) * n;
    if (!o.get()) o.alloc(nall);
    k_class_lowp<<<blocks_for(nall), BS, 0, s>>>(nv, nall, v64.get(), o.get(), bf16 ? 1 : 0);
    BCMG_CHECK_LAUNCH();
}

template <typename VT>
bool class_ok(const DevCsr &A, MatType mt)
{
    if (!A.use_classes()) return false;
    if constexpr (std::is_same<VT, double>::value)
        return mt == MT_F64;
    else if (A.cls.k > 0)
        return mt != MT_F64;
    else
        return mt == MT_F32 ? A.cls.v32.get() != nullptr
                            : mt == MT_BF16 && A.cls.v16.get() != nullptr;
}

template <typename VT>
void launch_rows_class(hipStream_t s, const DevCsr &A, MatType mt, RowOp op, const VT *x,
                       const VT *f, const VT *d, VT *y, DivSource div)
{
    if (A.cls.k > 0) {
        const StencilRef<VT> S = stencil_ref<VT>(A, mt);
        if (op == OP_SPMV)
            rows_stencil_op<VT, OP_SPMV, DIV_ARRAY>(s, A, S, x, f, d, y);
        else if (op == OP_RESID)
            rows_stencil_op<VT, OP_RESID, DIV_ARRAY>(s, A, S, x, f, d, y);
        else if (div == DIV_ARRAY)
            rows_stencil_op<VT, OP_JACOBI, DIV_ARRAY>(s, A, S, x, f, d, y);
        else if (div == DIV_DIAG)
            rows_stencil_op<VT, OP_JACOBI, DIV_DIAG>(s, A, S, x, f, d, y);
        else
            rows_stencil_op<VT, OP_JACOBI, DIV_L1>(s, A, S, x, f, d, y);
        BCMG_CHECK_LAUNCH();
        return;
    }
    const ClassRef<VT> C = class_ref<VT>(A, mt);
    const int drow = div_row(A, div);
    if (op == OP_SPMV)
        rows_class_op<VT, OP_SPMV>(s, A, C, drow, x, f, d, y);
    else if (op == OP_RESID)
        rows_class_op<VT, OP_RESID>(s, A, C, drow, x, f, d, y);
    else
        rows_class_op<VT, OP_JACOBI>(s, A, C, drow, x, f, d, y);
    BCMG_CHECK_LAUNCH();
}

/* whether the slab kernels take A: as a constant stencil, or its rows */
template <typename VT>
static bool slab_stencil(const DevCsr &A, MatType mt)
{
    return class_ok<VT>(A, mt) && A.cls.k > 0;
}

/* Rows of its own that a workgroup takes for `steps` neighbour-reading
   sweeps (0: they do not fit; n: one workgroup), and the launch's time as
   measured (us): 25 bytes a row at 6 TB/s and, for each 256 workgroups, which
   run at a time, 3.0 + 0.4 per sweep and row of a thread on a constant
   stencil, 4.0 + 0.6 per sweep with the rows in registers. */
template <typename VT>
static int slab_fit(const DevCsr &A, bool st, int steps, double *us)
{
    const int n = A.n;
    const long long halo = 2ll * A.band * steps;
    const int per_cu = ((n + SLAB_CUS - 1) / SLAB_CUS + 63) / 64 * 64;
    int ext = 0;
    for (int e = 1024; !ext && e <= (st ? SLAB_ROWS : SLAB_ROWS_REG); e *= 2)
        if (per_cu + halo <= e || (st && n <= e)) ext = e;
    if (!ext && st && SLAB_ROWS - halo >= SLAB_MIN_SHARE) ext = SLAB_ROWS;
    if (!ext) return 0;
    const int m = st && n <= ext ? n : (int)(ext - halo);
    const int rounds = ((n + m - 1) / m + SLAB_CUS - 1) / SLAB_CUS;
    const double per = st ? 0.4 * (ext / 1024) : 0.6;
    *us = 2.0 + n * (25.0 / 6.0e6) + rounds * ((st ? 1.0 : 2.0) + steps * per);
    return m < n ? m : n;
}

/* The next of `sweeps` sweeps that go into one slab launch: the split into
   equal launches that takes least, if it takes less than a launch a sweep
   (3 us and 25 bytes a row at 6 TB/s). */
template <typename VT>
int slab_plan(const DevCsr &A, MatType mt, int sweeps, bool zero, int *m)
{
    *m = 0;
    const bool st = slab_stencil<VT>(A, mt);
    if (sweeps < 1 || A.band < 0 || A.maxrow <= 0 || A.maxrow > CLS_ROW) return 0;
    double best = sweeps * (3.0 + A.n * (25.0 / 6.0e6));
    int take = 0;
    for (int parts = 1; parts <= 8 && parts <= sweeps; parts++) {
        const int t = (sweeps + parts - 1) / parts;
        double us = 0.0;
        const int mm = slab_fit<VT>(A, st, t - (zero ? 1 : 0), &us);
        if (t < 2 && mm < A.n) continue;
        if (mm > 0 && parts * us < best) {
            best = parts * us;
            take = t;
            *m = mm;
        }
    }
    return take;
}

template <typename VT>
bool slab_one(const DevCsr &A, MatType mt)
{
    return slab_stencil<VT>(A, mt) && A.n <= SLAB_ROWS && A.band >= 0;
}

template <typename VT>
void launch_slab(hipStream_t s, const DevCsr &A, MatType mt, int m, int steps, bool zero,
                 DivSource div, const VT *d, const VT *f, const VT *xin, VT *xout,
                 const BlockFuse<VT> &fu)
{
    const bool one = m >= A.n, st = slab_stencil<VT>(A, mt);
    if (m <= 0 || A.band < 0 || (st && div == DIV_ARRAY) || (one && A.n > SLAB_ROWS))
        throw Error(BCMG_EINVAL, "slab sweeps: not an operator of that kind");
    const int B = one ? 0 : A.band;
    if (!one && (fu.fc || ((!zero || fu.agg) && xin == xout)))
        throw Error(BCMG_EINVAL, "slab sweeps: in place or restricting over several workgroups");
    const int z = zero ? 1 : 0;
    if (one) m = A.n;
    if (!st) {
        if constexpr (std::is_same<VT, double>::value) {
            rows_slab(s, A, A.val.get(), m, B, steps, z, d, f, xin, xout, fu);
        } else {
            if (mt == MT_F32)
                rows_slab(s, A, A.val32.get(), m, B, steps, z, d, f, xin, xout, fu);
            else if (mt == MT_BF16)
                rows_slab(s, A, A.val16.get(), m, B, steps, z, d, f, xin, xout, fu);
            else
                rows_slab(s, A, A.val.get(), m, B, steps, z, d, f, xin, xout, fu);
        }
        return;
    }
    const StencilRef<VT> S = stencil_ref<VT>(A, mt);
    if (fu.agg)
        slab_k<VT, 1>(s, A, S, m, B, steps, z, div, f, xin, xout, fu);
    else if (fu.fc)
        slab_k<VT, 2>(s, A, S, m, B, steps, z, div, f, xin, xout, fu);
    else
        slab_k<VT, 0>(s, A, S, m, B, steps, z, div, f, xin, xout, fu);
}

template <typename VT>
void launch_jacobi_zero_class(hipStream_t s, const DevCsr &A, MatType mt, const VT *f, VT *y,
                              DivSource div)
{
    if (A.cls.k > 0) {
        const StencilRef<VT> S = stencil_ref<VT>(A, mt);
        if (div == DIV_L1)
            k_jz_stencil<VT, DIV_L1><<<blocks_for(A.n), BS, 0, s>>>(A.n, S, f, y);
        else
            k_jz_stencil<VT, DIV_DIAG><<<blocks_for(A.n), BS, 0, s>>>(A.n, S, f, y);
        BCMG_CHECK_LAUNCH();
        return;
    }
    k_jz_class<VT><<<blocks_for(A.n), BS, 0, s>>>(A.n, class_ref<VT>(A, mt), div_row(A, div), f,
                                                  y);
    BCMG_CHECK_LAUNCH();
}

template <int K, typename ZT>
static void spmv_dots_class_k(hipStream_t s, const DevCsr &A, const ZT *z, double *t,
                              const double *r, const double *to, double *part)
{
    const int nb = (A.n + BS - 1) / BS;
    if (A.cls.k > 0) {
        const StencilRef<double> S = stencil_ref<double>(A, MT_F64);
        if (A.cls.k <= 5)
            k_spmv_dots_stencil<K, 5, ZT><<<nb, BS, 0, s>>>(A.n, S, z, t, r, to, part);
        else if (A.cls.k <= 7)
            k_spmv_dots_stencil<K, 7, ZT><<<nb, BS, 0, s>>>(A.n, S, z, t, r, to, part);
        else
            k_spmv_dots_stencil<K, CLS_ROW, ZT><<<nb, BS, 0, s>>>(A.n, S, z, t, r, to, part);
        return;
    }
    const ClassRef<double> C = class_ref<double>(A, MT_F64);
    const size_t lds = class_lds_bytes<double>(C.nc, C.crow);
    if (C.crow <= 5)
        k_spmv_dots_class<K, 5, ZT><<<nb, BS, lds, s>>>(A.n, C, z, t, r, to, part);
    else if (C.crow <= 7)
        k_spmv_dots_class<K, 7, ZT><<<nb, BS, lds, s>>>(A.n, C, z, t, r, to, part);
    else
        k_spmv_dots_class<K, CLS_ROW, ZT><<<nb, BS, lds, s>>>(A.n, C, z, t, r, to, part);
}

template <typename ZT>
void launch_spmv_dots_class(hipStream_t s, const DevCsr &A, int k, const ZT *z, double *t,
                            const double *r, const double *to, double *part)
{
    if (k == 2)
        spmv_dots_class_k<2>(s, A, z, t, r, to, part);
    else
        spmv_dots_class_k<3>(s, A, z, t, r, to, part);
    BCMG_CHECK_LAUNCH();
}
template void launch_spmv_dots_class<double>(hipStream_t, const DevCsr &, int, const double *,
                                             double *, const double *, const double *, double *);
template void launch_spmv_dots_class<float>(hipStream_t, const DevCsr &, int, const float *,
                                            double *, const double *, const double *, double *);

#define BCMG_INSTANTIATE_CLASS(VT)                                                            \
    template bool class_ok<VT>(const DevCsr &, MatType);                                      \
    template void launch_rows_class<VT>(hipStream_t, const DevCsr &, MatType, RowOp,          \
                                        const VT *, const VT *, const VT *, VT *, DivSource); \
    template int slab_plan<VT>(const DevCsr &, MatType, int, bool, int *);                    \
    template bool slab_one<VT>(const DevCsr &, MatType);                                      \
    template void launch_slab<VT>(hipStream_t, const DevCsr &, MatType, int, int, bool,       \
                                  DivSource, const VT *, const VT *, const VT *, VT *,        \
                                  const BlockFuse<VT> &);                                     \
    template void launch_jacobi_zero_class<VT>(hipStream_t, const DevCsr &, MatType,          \
                                               const VT *, VT *, DivSource);
BCMG_INSTANTIATE_CLASS(double)
BCMG_INSTANTIATE_CLASS(float)
#undef BCMG_INSTANTIATE_CLASS

} // namespace bcmg
