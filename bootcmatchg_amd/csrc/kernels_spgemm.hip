/*
 * kernels_spgemm.hip - the sparse products of smoothed aggregation on gfx950
 * (src/AMG/matchingAggregation.cu:353-390): the smoother S = I - omega D^-1 A,
 * the general product C = L R and the general transpose.
 *
 * C = L R is computed row by row in one fixed summation order: every entry
 * C(i,j) is 0 + the products L(i,e) R(e,j), taken over L's row i in storage
 * order and, within it, over R's row e in storage order (the reference's hash
 * SpGEMM adds with shared-memory atomics in arrival order, so it fixes no
 * order). With right rows of distinct columns, four or more on average, a row
 * of up to SG_CAP products is summed in an LDS hash table (k_sg_hash), and so
 * is a longer one that no form below suits better and whose columns fit. Else a
 * row's products are expanded into LDS under a 64-bit key (row, column,
 * position), bitonic-sorted, and each run of one (row, column) is summed by
 * one lane in position order:
 *   - rows with at most SG_CAP products are packed into workgroups by a
 *     prefix sum of (products + 1): a workgroup owns the rows whose prefix
 *     starts in its SG_CAP-slot range, and since such a row ends within the
 *     next SG_CAP slots, 2 SG_CAP keys hold all of them;
 *   - a longer row is taken by a workgroup SG_CH products at a time: each
 *     chunk's column runs continue their columns' sums in a dense accumulator
 *     of the workgroup (one FP64 value and one row stamp per column of C), and
 *     the touched columns are put in order at the end of the row; when the
 *     right rows are long (SG_SERIAL_MIN products per left entry or more) and
 *     hold distinct columns, no sort is needed: the left entries are taken
 *     one at a time, each adding its products column-parallel;
 *   - with SG_LDS_COLS columns or fewer the accumulators are in LDS and a
 *     wavefront owns a column tile (k_sg_wave).
 * The pattern is symbolic (a cancelled entry stays), columns ascending. The
 * file is compiled with -ffp-contract=off: products and sums are rounded
 * separately, as in the serial restatement.
 */
#include "bcmg_internal.h"
#include "kernels_common.h"

#include <algorithm>
#include <climits>
#include <cstring>
#include <vector>

namespace bcmg {

namespace {

constexpr int SG_CAP = 1024;          /* products of a packed row, at most */
constexpr int SG_KEYS = 2 * SG_CAP;   /* keys of a packed workgroup */
constexpr int SG_CH = 2048;           /* products per chunk of a long row */
constexpr int SG_SORT = 2 * SG_CH;    /* touched columns sorted in LDS, at most */
constexpr long long SG_DENSE_BYTES = 2ll << 30; /* dense accumulators, all workgroups */
constexpr int SG_DENSE_BLOCKS = 1024;
constexpr int SG_SERIAL_MIN = 64;     /* products per left entry for the serial mode */
constexpr int SG_TILES = 16;          /* wavefronts (column tiles) of a row, at most */
constexpr int SG_TILE = 1024;         /* columns of a tile, about */
constexpr int SG_LDS_COLS = SG_TILES * SG_TILE; /* columns of C, at most, for LDS accumulators */
constexpr int SG_AHEAD = 8;           /* loads of 64 right entries in flight */
constexpr int SGM_ROWS = 16;          /* rows of a dense tile */
constexpr int SGM_AHEAD = 2;          /* right rows loaded at once */
constexpr long long SGM_ELEMS = 1ll << 25; /* of a dense operand, at most (256 MiB) */
constexpr double SGM_FILL = 12.0;
constexpr long long SG_UNTOUCHED = LLONG_MIN;   /* the bits of -0.0 */
constexpr int WAVE_RANK = 256;        /* transpose rows ranked by one wavefront */
constexpr int RANK_CHUNK = 4096;      /* columns per LDS load when ranking */
constexpr int RANK_BITS = 32 * RANK_CHUNK; /* columns ranked by a bit each */
constexpr unsigned long long SG_NONE = ~0ull;
constexpr int POS_BITS = 11;          /* position field: < 2048 */
constexpr int ROW_SHIFT = 42;         /* row field above 31 column bits */
constexpr long long SG_PER_PASS = 1ll << 28; /* slots + weights per batch of rows */


/* first index t in [0, n) with a[t] >= x (n if none) */
__device__ inline int lower_bound_i(const int *a, int n, int x)
{
    int lo = 0, hi = n;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (a[mid] < x)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

/* exclusive prefix sum of v over the workgroup; *tot = the sum of all */
__device__ inline int block_scan_excl(int v, int *sh, int *tot)
{
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    int x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) sh[wv] = x;
    __syncthreads();
    int pre = 0, all = 0;
#pragma unroll
    for (int w = 0; w < BS / 64; w++) {
        const int t = sh[w];
        if (w < wv) pre += t;
        all += t;
    }
    __syncthreads();
    *tot = all;
    return pre + x - v;
}

/* ascending bitonic sort of key[0, N), N a power of two */
template <typename K>
__device__ inline void bitonic_sort(K *key, int N)
{
    for (int k = 2; k <= N; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int t = threadIdx.x; t < (N >> 1); t += BS) {
                const int i = ((t & ~(j - 1)) << 1) | (t & (j - 1));
                const int l = i + j;
                const K a = key[i], b = key[l];
                const bool up = (i & k) == 0;
                if ((a > b) == up) {
                    key[i] = b;
                    key[l] = a;
                }
            }
            __syncthreads();
        }
}

__device__ inline int pow2_at_least(int v)
{
    int N = 2;
    while (N < v) N <<= 1;
    return N;
}

/* per row: products u, output slots sl = min(products, columns of C) (a
   row has at most that many entries), packing weight ws, the long-row
   list and how many of it have fewer than smin products per left entry; the
   total of slots plus weights (what a batch of rows is bounded by); *big = 1
   if a row has 2^30 products or more. G lanes a row, per_block (a multiple of
   BS / G, at most 256) rows a workgroup with one atomic a counter: an atomic
   per wavefront of one row each took 791 us at 65 536 rows. */
template <int G>
__global__ __launch_bounds__(BS) void k_sg_count(int n, int per_block, const int *__restrict__ Lrp,
                                                 const int *__restrict__ Lci,
                                                 const int *__restrict__ Rrp, long long m,
                                                 int *__restrict__ u, int *__restrict__ sl,
                                                 int *__restrict__ ws, int *__restrict__ cnt,
                                                 int *__restrict__ large,
                                                 int *__restrict__ nlarge,
                                                 unsigned long long *__restrict__ total,
                                                 int *__restrict__ big, int smin)
{
    __shared__ int list[256], nlist, nfew, at;
    __shared__ unsigned long long part[BS / 64];
    const int lane = threadIdx.x & (G - 1);
    if (threadIdx.x == 0) nlist = nfew = 0;
    __syncthreads();
    unsigned long long t = 0;   /* the batch cost of the rows: slots plus packing weights */
    const int i1 = min(n, (int)(blockIdx.x + 1) * per_block);
    for (int i = blockIdx.x * per_block + threadIdx.x / G; i < i1; i += BS / G) {
        const int b = Lrp[i + 1], a = Lrp[i];
        long long s = 0;
        for (int e = a + lane; e < b; e += G) {
            const int k = Lci[e];
            s += Rrp[k + 1] - Rrp[k];
        }
#pragma unroll
        for (int o = G / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
        if (lane != 0) continue;
        if (s >= (1ll << 30)) atomicOr(big, 1);
        u[i] = (int)(s < (1ll << 30) ? s : (1ll << 30));
        const long long slots = s < m ? s : m;
        sl[i] = (int)slots;
        cnt[i] = 0;
        t += (unsigned long long)slots;
        if (s <= SG_CAP) {
            ws[i] = (int)s + 1;
            t += s + 1;
        } else {
            ws[i] = 0;
            list[atomicAdd(&nlist, 1)] = i;
            if (s < (long long)smin * (b - a)) atomicAdd(&nfew, 1);
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = t;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < BS / 64; w++) t += part[w];
        if (t) atomicAdd(total, t);
        if (nlist) at = atomicAdd(nlarge, nlist);
        if (nfew) atomicAdd(nlarge + 2, nfew);
    }
    __syncthreads();
    if ((int)threadIdx.x < nlist) large[at + threadIdx.x] = list[threadIdx.x];
}

/* the packed rows of one workgroup (see the file comment) */
__global__ __launch_bounds__(BS) void k_sg_small(int n, const int *__restrict__ Lrp,
                                                 const int *__restrict__ Lci,
                                                 const double *__restrict__ Lv,
                                                 const int *__restrict__ Rrp,
                                                 const int *__restrict__ Rci,
                                                 const double *__restrict__ Rv,
                                                 const int *__restrict__ ws,
                                                 const int *__restrict__ soff,
                                                 const int *__restrict__ uoff,
                                                 int *__restrict__ tcol, double *__restrict__ tval,
                                                 int *__restrict__ cnt)
{
    __shared__ unsigned long long key[SG_KEYS];
    __shared__ double val[SG_KEYS];
    __shared__ int rowid[SG_CAP], rowfirst[SG_CAP];
    __shared__ int sh[BS / 64];
    __shared__ int rng[3];
    const int lo = blockIdx.x * SG_CAP;
    if (threadIdx.x == 0) {
        const int r0 = lower_bound_i(soff, n, lo);
        const int r1 = lower_bound_i(soff, n, lo + SG_CAP);
        rng[0] = r0;
        rng[1] = r1;
        rng[2] = soff[r1] - lo;        /* slots used, <= 2 SG_CAP */
    }
    for (int t = threadIdx.x; t < SG_KEYS; t += BS) key[t] = SG_NONE;
    __syncthreads();
    const int r0 = rng[0], r1 = rng[1];
    const int N = pow2_at_least(rng[2]);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int r = r0 + wv; r < r1; r += BS / 64) {
        if (ws[r] == 0) continue;      /* a long row: a workgroup of its own */
        const int base = soff[r] - lo;
        if (lane == 0) rowid[base] = r;
        int off = base;
        const int e1 = Lrp[r + 1];
        for (int e0 = Lrp[r]; e0 < e1; e0 += 64) {
            const int e = e0 + lane;
            int len = 0, f0 = 0;
            double lv = 0.0;
            if (e < e1) {
                const int k = Lci[e];
                f0 = Rrp[k];
                len = Rrp[k + 1] - f0;
                lv = Lv[e];
            }
            int x = len;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int y = __shfl_up(x, o, 64);
                if (lane >= o) x += y;
            }
            /* the window's products spread over the lanes: product q belongs
               to the first entry whose inclusive prefix exceeds q */
            const int total = __shfl(x, 63, 64);
            for (int q0 = 0; q0 < total; q0 += 64) {
                const int q = q0 + lane;
                int lo = 0, hi = 63;
#pragma unroll
                for (int st = 0; st < 6; st++) {
                    const int mid = (lo + hi) >> 1;
                    const int v = __shfl(x, mid, 64);
                    if (v <= q)
                        lo = mid + 1;
                    else
                        hi = mid;
                }
                const int xe = __shfl(x, lo, 64), le = __shfl(len, lo, 64);
                const int fe = __shfl(f0, lo, 64);
                const double ve = __shfl(lv, lo, 64);
                if (q < total) {
                    const int f = fe + (q - (xe - le));
                    const int pos = off + q;
                    key[pos] = ((unsigned long long)base << ROW_SHIFT) |
                               ((unsigned long long)Rci[f] << POS_BITS) | (unsigned)pos;
                    val[pos] = ve * Rv[f];
                }
            }
            off += total;
        }
    }
    __syncthreads();
    bitonic_sort(key, N);
    constexpr int PT = SG_KEYS / BS;
    const int t0 = threadIdx.x * PT;
    int nh = 0;
#pragma unroll
    for (int q = 0; q < PT; q++) {
        const int t = t0 + q;
        if (t < N) {
            const unsigned long long k = key[t];
            if (k != SG_NONE && (t == 0 || (key[t - 1] >> POS_BITS) != (k >> POS_BITS))) nh++;
        }
    }
    int tot;
    const int uid0 = block_scan_excl(nh, sh, &tot);
    int uid = uid0;
#pragma unroll
    for (int q = 0; q < PT; q++) {
        const int t = t0 + q;
        if (t < N) {
            const unsigned long long k = key[t];
            if (k != SG_NONE && (t == 0 || (key[t - 1] >> POS_BITS) != (k >> POS_BITS))) {
                if (t == 0 || (key[t - 1] >> ROW_SHIFT) != (k >> ROW_SHIFT))
                    rowfirst[k >> ROW_SHIFT] = uid;
                uid++;
            }
        }
    }
    __syncthreads();
    uid = uid0;
    for (int q = 0; q < PT; q++) {
        const int t = t0 + q;
        if (t >= N) break;
        const unsigned long long k = key[t];
        if (k == SG_NONE || (t > 0 && (key[t - 1] >> POS_BITS) == (k >> POS_BITS))) continue;
        const unsigned long long g = k >> POS_BITS;
        double s = 0.0;
        int t2 = t;
        for (; t2 < N && (key[t2] >> POS_BITS) == g; t2++)
            s = s + val[key[t2] & ((1u << POS_BITS) - 1)];
        const int base = (int)(k >> ROW_SHIFT);
        const int r = rowid[base];
        const int idx = uid - rowfirst[base];
        const int o = uoff[r] + idx;
        tcol[o] = (int)(g & 0x7fffffffull);
        tval[o] = s;
        if (t2 >= N || (key[t2] >> ROW_SHIFT) != (unsigned long long)base) cnt[r] = idx + 1;
        uid++;
    }
}

/* Long rows, one workgroup each in turn (a grid-stride loop over the list):
   the row's products SG_CH at a time, sorted by (column, position); each
   column run continues its column's sum in the workgroup's dense
   accumulator (acc, valid where stamp holds the row's id, so nothing is
   cleared between rows) in position order. The touched columns are listed
   as they appear, then put in ascending order: a sort in LDS up to SG_SORT
   of them, else a scan of the stamps over the touched column range. Row ids
   in the stamps are global (row_base + r): batches share the accumulators. */
__global__ __launch_bounds__(BS) void k_sg_dense(int nlarge, const int *__restrict__ large,
                                                 const int *__restrict__ Lrp,
                                                 const int *__restrict__ Lci,
                                                 const double *__restrict__ Lv,
                                                 const int *__restrict__ Rrp,
                                                 const int *__restrict__ Rci,
                                                 const double *__restrict__ Rv,
                                                 const int *__restrict__ u,
                                                 const int *__restrict__ uoff,
                                                 int *__restrict__ tcol, double *__restrict__ tval,
                                                 double *acc_all, int *stamp_all, long long m,
                                                 int row_base, int serial_min, int skip_serial,
                                                 int only_left, int *__restrict__ cnt)
{
    __shared__ unsigned long long key[SG_CH];   /* also the sort buffer of SG_SORT ints */
    __shared__ double val[SG_CH];
    __shared__ int sh[BS / 64];
    __shared__ int ws0[BS + 1], wf0[BS];        /* a window of left entries */
    __shared__ double wlv[BS];
    __shared__ int ntouch, cmin, cmax;
    double *const acc = acc_all + (long long)blockIdx.x * m;
    int *const stamp = stamp_all + (long long)blockIdx.x * m;
    int *const skey = reinterpret_cast<int *>(key);
    for (int q = blockIdx.x; q < nlarge; q += gridDim.x) {
        const int r = large[q];
        const int id = row_base + r;
        const int U = u[r];
        const int e_end = Lrp[r + 1];
        int ew0 = Lrp[r], pb0 = 0;   /* first window some later chunk needs */
        const bool serial = serial_min > 0 && (long long)U >= (long long)serial_min * (e_end - ew0);
        if (serial && skip_serial) continue;   /* k_sg_wave takes it */
        if (only_left && cnt[r] != -1) continue;   /* k_sg_hash took it */
        int *const ocol = tcol + uoff[r];
        double *const oval = tval + uoff[r];
        if (threadIdx.x == 0) {
            ntouch = 0;
            cmin = INT_MAX;
            cmax = -1;
        }
        /* long right rows (distinct columns): one left entry at a time, its
           products added column-parallel - the same order per column */
        for (int e0 = ew0; serial && e0 < e_end; e0 += BS) {
            const int e = e0 + threadIdx.x;
            if (e < e_end) {
                const int k = Lci[e];
                wf0[threadIdx.x] = Rrp[k];
                ws0[threadIdx.x] = Rrp[k + 1];
                wlv[threadIdx.x] = Lv[e];
            }
            __syncthreads();
            const int ne = min(BS, e_end - e0);
            /* the lane's first product of the next entry is loaded before
               the current entry's accumulation, so its latency overlaps */
            int pf = wf0[0] + threadIdx.x;
            bool have = pf < ws0[0];
            int pc = have ? Rci[pf] : 0;
            double pv = have ? Rv[pf] : 0.0;
            for (int t = 0; t < ne; t++) {
                const int f1 = ws0[t];
                const double lv = wlv[t];
                const int nf = t + 1 < ne ? wf0[t + 1] + threadIdx.x : 0;
                const bool nhave = t + 1 < ne && nf < ws0[t + 1];
                const int nc = nhave ? Rci[nf] : 0;
                const double nv = nhave ? Rv[nf] : 0.0;
                for (int f = pf; have && f < f1; f += BS) {
                    const int col = f == pf ? pc : Rci[f];
                    const double prod = lv * (f == pf ? pv : Rv[f]);
                    const bool first = stamp[col] != id;
                    acc[col] = (first ? 0.0 : acc[col]) + prod;
                    if (first) {
                        stamp[col] = id;
                        ocol[atomicAdd(&ntouch, 1)] = col;
                        atomicMin(&cmin, col);
                        atomicMax(&cmax, col);
                    }
                }
                __threadfence_block();
                __syncthreads();
                pf = nf;
                have = nhave;
                pc = nc;
                pv = nv;
            }
        }
        for (int c0 = 0; !serial && c0 < U; c0 += SG_CH) {
            const int c1 = min(c0 + SG_CH, U);
            for (int t = threadIdx.x; t < SG_CH; t += BS) key[t] = SG_NONE;
            __syncthreads();
            int ew = ew0, pb = pb0;
            while (ew < e_end && pb < c1) {
                const int e = ew + threadIdx.x;
                int len = 0, f0 = 0;
                double lv = 0.0;
                if (e < e_end) {
                    const int k = Lci[e];
                    f0 = Rrp[k];
                    len = Rrp[k + 1] - f0;
                    lv = Lv[e];
                }
                int tot;
                const int s0 = pb + block_scan_excl(len, sh, &tot);
                ws0[threadIdx.x + 1] = s0 + len;
                wf0[threadIdx.x] = f0 - s0;
                wlv[threadIdx.x] = lv;
                if (threadIdx.x == 0) ws0[0] = pb;
                __syncthreads();
                /* the window's products in the chunk, spread over the lanes:
                   position p belongs to entry t with ws0[t] <= p < ws0[t + 1] */
                const int lo = max(pb, c0), hi = min(pb + tot, c1);
                for (int p = lo + threadIdx.x; p < hi; p += BS) {
                    int a = 0, b = BS;
                    while (b - a > 1) {
                        const int mid = (a + b) >> 1;
                        if (ws0[mid] <= p)
                            a = mid;
                        else
                            b = mid;
                    }
                    const int f = wf0[a] + p;
                    const int pos = p - c0;
                    key[pos] = ((unsigned long long)Rci[f] << POS_BITS) | (unsigned)pos;
                    val[pos] = wlv[a] * Rv[f];
                }
                __syncthreads();
                if (pb + tot <= c1) {
                    ew0 = ew + BS;
                    pb0 = pb + tot;
                }
                ew += BS;
                pb += tot;
            }
            __syncthreads();
            const int N = pow2_at_least(c1 - c0);
            bitonic_sort(key, N);
            for (int t = threadIdx.x; t < N; t += BS) {
                const unsigned long long k = key[t];
                if (k == SG_NONE || (t > 0 && (key[t - 1] >> POS_BITS) == (k >> POS_BITS)))
                    continue;
                const int col = (int)(k >> POS_BITS);
                const bool first = stamp[col] != id;
                double s = first ? 0.0 : acc[col];
                for (int t2 = t; t2 < N && (key[t2] >> POS_BITS) == (k >> POS_BITS); t2++)
                    s = s + val[key[t2] & ((1u << POS_BITS) - 1)];
                acc[col] = s;
                if (first) {
                    stamp[col] = id;
                    ocol[atomicAdd(&ntouch, 1)] = col;
                    atomicMin(&cmin, col);
                    atomicMax(&cmax, col);
                }
            }
            __threadfence_block();
            __syncthreads();
        }
        const int k = ntouch;
        if (k <= SG_SORT) {
            const int N = pow2_at_least(k);
            for (int t = threadIdx.x; t < N; t += BS) skey[t] = t < k ? ocol[t] : INT_MAX;
            __syncthreads();
            bitonic_sort(skey, N);
            for (int t = threadIdx.x; t < k; t += BS) {
                const int c = skey[t];
                ocol[t] = c;
                oval[t] = acc[c];
            }
        } else {
            const int j0 = cmin, j1 = cmax;
            int base = 0;
            for (int jb = j0; jb <= j1; jb += BS) {
                const int j = jb + threadIdx.x;
                const int fl = (j <= j1 && stamp[j] == id) ? 1 : 0;
                int tot;
                const int pos = base + block_scan_excl(fl, sh, &tot);
                if (fl) {
                    ocol[pos] = j;
                    oval[pos] = acc[j];
                }
                base += tot;
            }
        }
        if (threadIdx.x == 0) cnt[r] = k;
        __threadfence_block();
        __syncthreads();
    }
}

/* Rows with lo < products <= hi when R's rows hold distinct columns: a
   wavefront a row, its columns in an LDS hash table of H slots with their
   sums. The left entries are taken in order, 64 lanes on a right row; its
   columns are distinct, so an LDS add instruction meets no slot twice and each
   sum is taken in the stated order (k_sg_wave's argument). The table's entries
   then go to their ranks among the columns. A row with more than H columns
   (lo >= H only) is left: its count becomes -1 and *left 1. smin > 0: only
   rows below smin products per left entry. 64^3 smoothed, R A and T P of
   level 0 (25 M products): 2.1 ms sorted, 0.6 so; R A of level 1 (51 M, 65 536
   columns): 2.8 ms on dense accumulators, 0.7 so. LDS latency bounds it. */
template <int H>
__global__ __launch_bounds__(BS) void k_sg_hash(int n, int lo, int hi, int smin,
                                                const int *__restrict__ Lrp,
                                                const int *__restrict__ Lci,
                                                const double *__restrict__ Lv,
                                                const int *__restrict__ Rrp,
                                                const int *__restrict__ Rci,
                                                const double *__restrict__ Rv,
                                                const int *__restrict__ u,
                                                const int *__restrict__ uoff,
                                                int *__restrict__ tcol, double *__restrict__ tval,
                                                int *__restrict__ cnt, int *__restrict__ left)
{
    constexpr int Q = H / 64, SHIFT = 32 - __builtin_ctz(H);
    __shared__ double vals[BS / 64][H];
    __shared__ int keys[BS / 64][H];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int r = xcd_block(blockIdx.x, gridDim.x) * (BS / 64) + wv;
    if (r >= n) return;
    const int U = u[r], eb = Lrp[r], ee = Lrp[r + 1];
    if (U <= lo || U > hi) return;
    if (smin > 0 && (long long)U >= (long long)smin * (ee - eb)) return;
    int *const key = keys[wv];
    double *const val = vals[wv];
#pragma unroll
    for (int q = 0; q < Q; q++) {
        key[q * 64 + lane] = -1;
        val[q * 64 + lane] = 0.0;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    bool full = false;
    for (int e0 = eb; e0 < ee && !full; e0 += 64) {
        const int e = e0 + lane;
        int s0 = 0, s1 = 0;
        double lv = 0.0;
        if (e < ee) {
            const int k = Lci[e];
            s0 = Rrp[k];
            s1 = Rrp[k + 1];
            lv = Lv[e];
        }
        unsigned long long todo = __ballot(s1 > s0);
        int f = 0, f1 = 0;
        double l = 0.0;
        while ((todo || f < f1) && !full) {
            int cc[SG_AHEAD];
            double vv[SG_AHEAD], ll[SG_AHEAD];
#pragma unroll
            for (int d = 0; d < SG_AHEAD; d++) {
                if (f >= f1 && todo) {
                    const int t = __builtin_ctzll(todo);
                    todo &= todo - 1;
                    f = __builtin_amdgcn_readlane(s0, t);
                    f1 = __builtin_amdgcn_readlane(s1, t);
                    l = lane_double(lv, t);
                }
                const int p = f + lane;
                const int pc = min(p, f1 - 1);
                const int col = Rci[pc];
                cc[d] = p < f1 ? col : -1;
                vv[d] = Rv[pc];
                ll[d] = l;
                f += 64;
            }
#pragma unroll
            for (int d = 0; d < SG_AHEAD; d++) {
                const int c = cc[d];
                if (c < 0) continue;
                /* Knuth's multiplicative hash */
                int h = (int)(((unsigned)c * 2654435761u) >> SHIFT);
                int tries = 0;
                for (; tries < H; tries++) {
                    int k = __hip_atomic_load(&key[h], __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_WORKGROUP);
                    if (k == -1) k = atomicCAS(&key[h], -1, c);
                    if (k == -1 || k == c) break;
                    h = (h + 1) & (H - 1);
                }
                if (tries < H)
                    __hip_atomic_fetch_add(&val[h], ll[d] * vv[d], __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_WORKGROUP);
                else
                    full = true;
            }
            full = __ballot(full) != 0;
        }
    }
    if (full) {
        if (lane == 0) {
            cnt[r] = -1;
            *left = 1;
        }
        return;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    /* to the front of the table (a step writes at or before what it read) */
    int k = 0;
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int c = key[q * 64 + lane];
        const double v = val[q * 64 + lane];
        const unsigned long long b = __ballot(c >= 0);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        if (c >= 0) {
            const int at = k + __popcll(b & ((1ull << lane) - 1));
            key[at] = c;
            val[at] = v;
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        k += __popcll(b);
    }
    int mine[Q], rank[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) {
        mine[q] = q * 64 + lane < k ? key[q * 64 + lane] : INT_MAX;
        rank[q] = 0;
    }
#pragma unroll
    for (int g = 0; g < Q; g++) {
        if (g * 64 >= k) break;
        const int ng = min(64, k - g * 64);
        for (int t = 0; t < ng; t++) {
            const int d = __builtin_amdgcn_readlane(mine[g], t);
#pragma unroll
            for (int q = 0; q < Q; q++)
                if (q * 64 < k) rank[q] += d < mine[q] ? 1 : 0;
        }
    }
    const int o = uoff[r];
#pragma unroll
    for (int q = 0; q < Q; q++)
        if (q * 64 + lane < k) {
            tcol[o + rank[q]] = mine[q];
            tval[o + rank[q]] = val[q * 64 + lane];
        }
    if (lane == 0) cnt[r] = k;
}

/* where R's rows cross the column tiles [t W, (t + 1) W): seg[row][t] is the
   first entry of tile t, seg[row][nt] the row's end (a wavefront a row,
   columns strictly ascending) */
__global__ __launch_bounds__(BS) void k_sg_seg(int n, const int *__restrict__ rp,
                                               const int *__restrict__ ci, int W, int nt,
                                               int *__restrict__ seg)
{
    const int lane = threadIdx.x & 63;
    for (long long row = group_row(blockIdx.x, threadIdx.x, 64); row < n;
         row += row_step(gridDim.x, 64)) {
        int *const o = seg + row * (nt + 1);
        const int a = rp[row], b = rp[row + 1];
        for (int f = a + lane; f < b; f += 64) {
            const int t0 = f > a ? ci[f - 1] / W + 1 : 0, t1 = ci[f] / W;
            for (int t = t0; t <= t1; t++) o[t] = f;
        }
        const int last = b > a ? ci[b - 1] / W + 1 : 0;
        for (int t = last + lane; t <= nt; t += 64) o[t] = b;
    }
}

/* Long rows when C's columns fit LDS: a workgroup a row, a wavefront a column
   tile of it with W accumulators in LDS. A wavefront walks the left entries
   in order and adds the products of each one's segment of the right row, 64
   lanes at a time: a right row's columns are distinct, so one LDS add
   instruction never meets a column twice, and one wavefront's LDS
   instructions execute in order - each column's sum is taken in the stated
   order with no barrier between left entries. ds_add_f64 rounds as v_add_f64
   does and returns nothing, so no step waits for the one before; the loads of
   SG_AHEAD steps are issued ahead of their adds. An untouched column holds
   -0.0: a product is added as prod + 0.0 (never -0.0), so a touched column is
   never -0.0, and the row's columns come out in order by ballots. Rows next
   to each other share right rows: an XCD takes consecutive ones.
   The right rows bound it (12 bytes a product from L2 and the last-level
   cache): T P with 2048 columns, 5.0e9 products, 4.6 ms (13 TB/s); R A with
   4096 columns, 3.6e9 products, 5.6 ms (6.5 without the XCD order; A is
   60 MB); both and T P of the level above 47.1 ms with a barrier per left
   entry and a workgroup's lanes over one right row. Tiles of 512 / 2048
   columns: the setup takes 2 % / 4 % longer. */
__global__ __launch_bounds__(1024) void k_sg_wave(const int *__restrict__ large,
                                                  const int *__restrict__ Lrp,
                                                  const int *__restrict__ Lci,
                                                  const double *__restrict__ Lv,
                                                  const int *__restrict__ seg,
                                                  const int *__restrict__ Rci,
                                                  const double *__restrict__ Rv,
                                                  const int *__restrict__ u,
                                                  const int *__restrict__ uoff,
                                                  int *__restrict__ tcol,
                                                  double *__restrict__ tval, int W,
                                                  int serial_min, int only_left,
                                                  int *__restrict__ cnt)
{
    extern __shared__ double sg_acc[];
    __shared__ int wcnt[SG_TILES];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nt = blockDim.x >> 6;
    const int b0 = xcd_block(blockIdx.x, gridDim.x);
    const int r = large ? large[b0] : b0;
    const int eb = Lrp[r], ee = Lrp[r + 1];
    if (u[r] <= SG_CAP || (long long)u[r] < (long long)serial_min * (ee - eb)) return;
    if (only_left && cnt[r] != -1) return;   /* k_sg_hash took it */
    double *const acc = sg_acc + wv * W;
    for (int t = lane; t < W; t += 64) acc[t] = -0.0;
    __syncthreads();
    for (int e0 = eb; e0 < ee; e0 += 64) {
        const int e = e0 + lane;
        int s0 = 0, s1 = 0;
        double lv = 0.0;
        if (e < ee) {
            const int *const o = seg + (long long)Lci[e] * (nt + 1) + wv;
            s0 = o[0];
            s1 = o[1];
            lv = Lv[e];
        }
        unsigned long long todo = __ballot(s1 > s0);
        int f = 0, f1 = 0;
        double l = 0.0;
        while (todo || f < f1) {
            int cc[SG_AHEAD];
            double vv[SG_AHEAD], ll[SG_AHEAD];
#pragma unroll
            for (int d = 0; d < SG_AHEAD; d++) {
                if (f >= f1 && todo) {
                    const int t = __builtin_ctzll(todo);
                    todo &= todo - 1;
                    f = __builtin_amdgcn_readlane(s0, t);
                    f1 = __builtin_amdgcn_readlane(s1, t);
                    l = lane_double(lv, t);
                }
                const int p = f + lane;
                const int pc = min(p, f1 - 1);
                const int col = Rci[pc];
                cc[d] = p < f1 ? col : -1;
                vv[d] = Rv[pc];
                ll[d] = l;
                f += 64;
            }
#pragma unroll
            for (int d = 0; d < SG_AHEAD; d++)
                if (cc[d] >= 0)
                    __hip_atomic_fetch_add(&sg_acc[cc[d]], ll[d] * vv[d] + 0.0, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    }
    __syncthreads();
    int mine = 0;
    for (int t = lane; t < W; t += 64)
        mine += __popcll(__ballot(__double_as_longlong(acc[t]) != SG_UNTOUCHED));
    if (lane == 0) wcnt[wv] = mine;
    __syncthreads();
    int base = uoff[r], all = 0;
    for (int w = 0; w < nt; w++) {
        const int k = wcnt[w];
        if (w < wv) base += k;
        all += k;
    }
    for (int t = lane; t < W; t += 64) {
        const double v = acc[t];
        const bool have = __double_as_longlong(v) != SG_UNTOUCHED;
        const unsigned long long b = __ballot(have);
        if (have) {
            const int o = base + __popcll(b & ((1ull << lane) - 1));
            tcol[o] = wv * W + t;
            tval[o] = v;
        }
        base += __popcll(b);
    }
    if (threadIdx.x == 0) cnt[r] = all;
}

/* ------------------------------------------- dense operands

   Where both operands are filled well the products outnumber what LDS adds
   and gathered right rows can move, and the rows of C go through registers
   instead: R as a dense array, L in tiles of SGM_ROWS rows whose used columns
   are listed, a wavefront taking a tile's SGM_ROWS x 128 elements of C. An
   absent entry is a zero: its product is a zero and adds nothing (the sums
   start from +0 and are never -0), so each element is the stated sum in the
   stated order; the operands must be finite (an infinity times an absent
   zero is not zero), which is checked first. The pattern is the union of the
   right rows' column bits, taken apart from the values. */

/* flag[0] |= 1 if a value is not finite */
__global__ __launch_bounds__(BS) void k_sgm_finite(long long n, const double *__restrict__ v,
                                                   int *__restrict__ flag)
{
    bool bad = false;
    for (long long i = (long long)blockIdx.x * BS + threadIdx.x; i < n;
         i += (long long)gridDim.x * BS)
        bad = bad || !isfinite(v[i]);
    if (__ballot(bad) && (threadIdx.x & 63) == 0) atomicOr(flag, 1);
}

/* R's rows into Rd (pitch mp, zeroed) and their column bits (mw words of 64);
   a wavefront a row, bits gathered in LDS (4 mw words) */
__global__ __launch_bounds__(BS) void k_sgm_right(int n, const int *__restrict__ rp,
                                                  const int *__restrict__ ci,
                                                  const double *__restrict__ v, int mp, int mw,
                                                  double *__restrict__ Rd,
                                                  unsigned long long *__restrict__ bits)
{
    extern __shared__ unsigned sgm_bits[];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int r = blockIdx.x * (BS / 64) + wv;
    unsigned *const b = sgm_bits + wv * 2 * mw;
    for (int t = lane; t < 2 * mw; t += 64) b[t] = 0;
    __syncthreads();
    if (r < n)
        for (int e = rp[r] + lane; e < rp[r + 1]; e += 64) {
            const int c = ci[e];
            Rd[(size_t)r * mp + c] = v[e];
            atomicOr(&b[c >> 5], 1u << (c & 31));
        }
    __syncthreads();
    if (r < n)
        for (int t = lane; t < mw; t += 64)
            bits[(size_t)r * mw + t] = b[2 * t] | (unsigned long long)b[2 * t + 1] << 32;
}

/* L's rows into tiles, a workgroup a tile: Ld[(tile (K + 1) + k) SGM_ROWS +
   row in tile] (zeroed), and the tile's used k in ascending order (gathered as
   bits in LDS, kw words), filled up to a multiple of SGM_AHEAD with K, a row of
   zeros in Ld */
__global__ __launch_bounds__(BS) void k_sgm_left(int n, int K, int kw,
                                                 const int *__restrict__ rp,
                                                 const int *__restrict__ ci,
                                                 const double *__restrict__ v,
                                                 double *__restrict__ Ld, int pitch,
                                                 int *__restrict__ list, int *__restrict__ count)
{
    extern __shared__ unsigned sgm_used[];
    __shared__ int sh[BS / 64];
    const int tile = blockIdx.x, wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int t = threadIdx.x; t < kw; t += BS) sgm_used[t] = 0;
    __syncthreads();
    for (int q = wv; q < SGM_ROWS; q += BS / 64) {
        const int r = tile * SGM_ROWS + q;
        if (r >= n) break;
        const int b = rp[r + 1];
        for (int e = rp[r] + lane; e < b; e += 64) {
            const int k = ci[e];
            Ld[((size_t)tile * (K + 1) + k) * SGM_ROWS + q] = v[e];
            atomicOr(&sgm_used[k >> 5], 1u << (k & 31));
        }
    }
    __syncthreads();
    int *const o = list + (size_t)tile * pitch;
    int base = 0;
    for (int t0 = 0; t0 < kw; t0 += BS) {
        const int t = t0 + threadIdx.x;
        unsigned w = t < kw ? sgm_used[t] : 0u;
        int tot;
        int at = base + block_scan_excl(__popc(w), sh, &tot);
        for (; w; w &= w - 1) o[at++] = t * 32 + __builtin_ctz(w);
        base += tot;
    }
    const int end = (base + SGM_AHEAD - 1) / SGM_AHEAD * SGM_AHEAD;
    if ((int)threadIdx.x < end - base) o[base + threadIdx.x] = K;
    if (threadIdx.x == 0) count[tile] = end;
}

/* C's rows: column bits (the union over the left entries), the number of
   entries before each word, the columns and the count; a wavefront a row */
__global__ __launch_bounds__(BS) void k_sgm_pattern(int n, const int *__restrict__ rp,
                                                    const int *__restrict__ ci, int mw,
                                                    const unsigned long long *__restrict__ rbits,
                                                    const int *__restrict__ uoff,
                                                    unsigned long long *__restrict__ cbits,
                                                    int *__restrict__ before,
                                                    int *__restrict__ tcol, int *__restrict__ cnt)
{
    const int r = group_row(blockIdx.x, threadIdx.x, 64), lane = threadIdx.x & 63;
    if (r >= n) return;
    const int a = rp[r], b = rp[r + 1];
    int base = 0;
    for (int w0 = 0; w0 < mw; w0 += 64) {
        const int w = w0 + lane;
        const int wc = min(w, mw - 1);
        unsigned long long bits = 0;
        for (int e = a; e < b; e += 8) {
#pragma unroll
            for (int u = 0; u < 8; u++)
                bits |= rbits[(size_t)ci[min(e + u, b - 1)] * mw + wc];
        }
        if (w >= mw) bits = 0;
        int x = __popcll(bits);
        const int own = x;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(x, o, 64);
            if (lane >= o) x += y;
        }
        const int first = base + x - own;
        if (w < mw) {
            cbits[(size_t)r * mw + w] = bits;
            before[(size_t)r * mw + w] = first;
        }
        for (int t = 0; t < min(64, mw - w0); t++) {
            const unsigned lo = __builtin_amdgcn_readlane((int)bits, t);
            const unsigned hi = __builtin_amdgcn_readlane((int)(bits >> 32), t);
            const unsigned long long word = lo | (unsigned long long)hi << 32;
            const int at = __builtin_amdgcn_readlane(first, t);
            if ((word >> lane) & 1ull)
                tcol[uoff[r] + at + __popcll(word & ((1ull << lane) - 1))] = (w0 + t) * 64 + lane;
        }
        base += __builtin_amdgcn_readlane(x, 63);
    }
    if (lane == 0) cnt[r] = base;
}

/* The values: four wavefronts of a workgroup take four row tiles of the same
   128 columns (their right loads meet in L1); a left value is a scalar. The
   multiplier bounds it: 2048 x 4096 x 2048, 1.5 ms, 23 of 39 T operations/s
   (multiply and add apart); eight rows a tile and four right rows ahead 1.6,
   and 2.4 against 1.9 ms at 4096 columns. */
__global__ __launch_bounds__(BS) void k_sgm_values(int n, int K, int mp, int mw, int tiles,
                                                   const int *__restrict__ list, int pitch,
                                                   const int *__restrict__ count,
                                                   const double *__restrict__ Ld,
                                                   const double *__restrict__ Rd,
                                                   const unsigned long long *__restrict__ cbits,
                                                   const int *__restrict__ before,
                                                   const int *__restrict__ uoff,
                                                   double *__restrict__ tval)
{
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cols = mp / 128;
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int c = b % cols, tile = b / cols * (BS / 64) + wv;
    if (tile >= tiles) return;
    const int *const ks = list + (size_t)tile * pitch;
    const double *const Lt = Ld + (size_t)tile * (K + 1) * SGM_ROWS;
    const double *const Rt = Rd + c * 128 + lane;
    double acc[SGM_ROWS][2];
#pragma unroll
    for (int q = 0; q < SGM_ROWS; q++) acc[q][0] = acc[q][1] = 0.0;
    const int nk = count[tile];
    for (int e = 0; e < nk; e += SGM_AHEAD) {
        double rv[SGM_AHEAD][2];
        int kk[SGM_AHEAD];
#pragma unroll
        for (int u = 0; u < SGM_AHEAD; u++) {
            kk[u] = ks[e + u];
            const double *const row = Rt + (size_t)(kk[u] < K ? kk[u] : 0) * mp;
            rv[u][0] = row[0];
            rv[u][1] = row[64];
        }
#pragma unroll
        for (int u = 0; u < SGM_AHEAD; u++) {
            const double *const l = Lt + (size_t)kk[u] * SGM_ROWS;
#pragma unroll
            for (int q = 0; q < SGM_ROWS; q++) {
                acc[q][0] = acc[q][0] + l[q] * rv[u][0];
                acc[q][1] = acc[q][1] + l[q] * rv[u][1];
            }
        }
    }
#pragma unroll
    for (int q = 0; q < SGM_ROWS; q++) {
        const int r = tile * SGM_ROWS + q;
        if (r >= n) break;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int w = 2 * c + h;
            if (w >= mw) continue;
            const unsigned long long bits = cbits[(size_t)r * mw + w];
            if ((bits >> lane) & 1ull)
                tval[uoff[r] + before[(size_t)r * mw + w] +
                     __popcll(bits & ((1ull << lane) - 1))] = acc[q][h];
        }
    }
}

/* compact the rows from their product-count slots into C (G lanes a row) */
template <int G>
__global__ __launch_bounds__(BS) void k_sg_gather(int n, const int *__restrict__ uoff,
                                                  const int *__restrict__ Crp,
                                                  const int *__restrict__ tcol,
                                                  const double *__restrict__ tval,
                                                  int *__restrict__ ccol,
                                                  double *__restrict__ cval)
{
    const int row = group_row(blockIdx.x, threadIdx.x, G);
    const int lane = threadIdx.x & (G - 1);
    if (row >= n) return;
    const int s = uoff[row], d = Crp[row], len = Crp[row + 1] - d;
    for (int q = lane; q < len; q += G) {
        ccol[d + q] = tcol[s + q];
        cval[d + q] = tval[s + q];
    }
}

/* ------------------------------------------------------------ transpose */

/* A's rows by G lanes each */
template <int G>
__global__ __launch_bounds__(BS) void k_col_count(int n, const int *__restrict__ rp,
                                                  const int *__restrict__ ci,
                                                  int *__restrict__ cnt)
{
    for (long long i = group_row(blockIdx.x, threadIdx.x, G); i < n; i += row_step(gridDim.x, G)) {
        const int b = rp[i + 1];
        for (int e = rp[i] + (int)(threadIdx.x & (G - 1)); e < b; e += G)
            atomicAdd(&cnt[ci[e]], 1);
    }
}

template <int G>
__global__ __launch_bounds__(BS) void k_col_fill(int n, const int *__restrict__ rp,
                                                 const int *__restrict__ ci,
                                                 const double *__restrict__ v,
                                                 int *__restrict__ cursor, int *__restrict__ tcol,
                                                 double *__restrict__ tval)
{
    for (long long i = group_row(blockIdx.x, threadIdx.x, G); i < n; i += row_step(gridDim.x, G)) {
        const int b = rp[i + 1];
        for (int e = rp[i] + (int)(threadIdx.x & (G - 1)); e < b; e += G) {
            const int pos = atomicAdd(&cursor[ci[e]], 1);
            tcol[pos] = (int)i;
            tval[pos] = v[e];
        }
    }
}

/* Each row of the transpose in ascending column order (distinct columns): an
   entry's place is its rank among the row's entries. A wavefront a row of up
   to WAVE_RANK entries, compared lane against lane; longer rows are listed
   for k_rank_long. 16 384 rows of 75 entries: 473 us with a lane a row (to
   64 entries, the rest with the long ones), 31 so. */
__global__ __launch_bounds__(BS) void k_rank(int nr, const int *__restrict__ rp,
                                             const int *__restrict__ cin,
                                             const double *__restrict__ vin,
                                             int *__restrict__ col, double *__restrict__ val,
                                             int *__restrict__ longl, int *__restrict__ nlong)
{
    constexpr int Q = WAVE_RANK / 64;
    const int lane = threadIdx.x & 63;
    for (long long I = group_row(blockIdx.x, threadIdx.x, 64); I < nr;
         I += row_step(gridDim.x, 64)) {
        const int a = rp[I], len = rp[I + 1] - a;
        if (len > WAVE_RANK) {
            if (lane == 0) longl[atomicAdd(nlong, 1)] = (int)I;
            continue;
        }
        int c[Q], rank[Q];
#pragma unroll
        for (int q = 0; q < Q; q++) {
            c[q] = q * 64 + lane < len ? cin[a + q * 64 + lane] : INT_MAX;
            rank[q] = 0;
        }
#pragma unroll
        for (int f = 0; f < Q; f++) {
            if (f * 64 >= len) break;
            const int nf = min(64, len - f * 64);
            for (int t = 0; t < nf; t++) {
                const int d = __builtin_amdgcn_readlane(c[f], t);
#pragma unroll
                for (int q = 0; q < Q; q++) rank[q] += d < c[q] ? 1 : 0;
            }
        }
#pragma unroll
        for (int q = 0; q < Q; q++)
            if (q * 64 + lane < len) {
                col[a + rank[q]] = c[q];
                val[a + rank[q]] = vin[a + q * 64 + lane];
            }
    }
}

/* A long row per workgroup, m columns. Up to RANK_BITS of them: the row's
   columns set bits in LDS and an entry's rank is the number of bits below
   its own (2048 rows of 1291 entries, 4096 columns: 979 us by comparing all
   pairs, 24 so); more: ranks against the row's columns, RANK_CHUNK at a
   time. */
__global__ __launch_bounds__(BS) void k_rank_long(const int *__restrict__ longl, int m,
                                                  const int *__restrict__ rp,
                                                  const int *__restrict__ cin,
                                                  const double *__restrict__ vin,
                                                  int *__restrict__ col, double *__restrict__ val)
{
    __shared__ int buf[RANK_CHUNK];
    __shared__ int pre[RANK_CHUNK];
    __shared__ int sh[BS / 64];
    const int I = longl[blockIdx.x];
    const int a = rp[I], len = rp[I + 1] - a;
    if (m <= RANK_BITS) {
        unsigned *const bit = reinterpret_cast<unsigned *>(buf);
        const int words = (m + 31) >> 5;
        for (int t = threadIdx.x; t < words; t += BS) bit[t] = 0;
        __syncthreads();
        for (int e = threadIdx.x; e < len; e += BS) {
            const int c = cin[a + e];
            atomicOr(&bit[c >> 5], 1u << (c & 31));
        }
        __syncthreads();
        int base = 0;
        for (int t0 = 0; t0 < words; t0 += BS) {
            const int t = t0 + threadIdx.x;
            int tot;
            const int x = block_scan_excl(t < words ? __popc(bit[t]) : 0, sh, &tot);
            if (t < words) pre[t] = base + x;
            base += tot;
        }
        __syncthreads();
        for (int e = threadIdx.x; e < len; e += BS) {
            const int c = cin[a + e];
            const int rank = pre[c >> 5] + __popc(bit[c >> 5] & ((1u << (c & 31)) - 1));
            col[a + rank] = c;
            val[a + rank] = vin[a + e];
        }
        return;
    }
    for (int e0 = 0; e0 < len; e0 += BS) {
        const int e = e0 + threadIdx.x;
        const int c = e < len ? cin[a + e] : 0;
        int rank = 0;
        for (int k0 = 0; k0 < len; k0 += RANK_CHUNK) {
            const int nk = min(RANK_CHUNK, len - k0);
            __syncthreads();
            for (int t = threadIdx.x; t < nk; t += BS) buf[t] = cin[a + k0 + t];
            __syncthreads();
            if (e < len)
                for (int t = 0; t < nk; t++) rank += buf[t] < c ? 1 : 0;
        }
        if (e < len) {
            col[a + rank] = c;
            val[a + rank] = vin[a + e];
        }
    }
}

/* ------------------------------------------------ smoother S, omega */

/* s_ij = a_ij / d_i (CSRm::matrixVectorScaling, src/matrix/CSR.cu:520-545)
   and the largest 0 + sum_j |s_ij| in storage order (CSR.cu:386-416): row
   sums are >= 0, so their bit patterns order as the values do */
template <int G>
__global__ __launch_bounds__(BS) void k_sa_scale(int n, int per_block, const int *__restrict__ rp,
                                                 const double *__restrict__ av,
                                                 const double *__restrict__ D,
                                                 double *__restrict__ sv,
                                                 unsigned long long *__restrict__ norm)
{
    __shared__ unsigned long long part[BS / 64];
    unsigned long long top = 0;
    const int i1 = min(n, (int)(blockIdx.x + 1) * per_block);
    for (int i = blockIdx.x * per_block + threadIdx.x / G; i < i1; i += BS / G) {
        const double d = D[i];
        const int a = rp[i], b = rp[i + 1];
        double s = 0.0;
        if (G == 1) {
            for (int e = a; e < b; e++) {
                const double t = av[e] / d;
                sv[e] = t;
                s += fabs(t);
            }
        } else {
            for (int e0 = a; e0 < b; e0 += G) {
                const int e = e0 + (int)(threadIdx.x & (G - 1));
                double t = 0.0;
                if (e < b) {
                    t = av[e] / d;
                    sv[e] = t;
                }
                s = add_lanes_in_order(s, fabs(t), b - e0);
            }
        }
        const unsigned long long y = s > 0.0 ? (unsigned long long)__double_as_longlong(s) : 0ull;
        top = y > top ? y : top;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long y = __shfl_xor(top, o, 64);
        top = y > top ? y : top;
    }
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = top;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < BS / 64; w++) top = part[w] > top ? part[w] : top;
        if (top) atomicMax(norm, top);
    }
}

/* s_ij = -omega s_ij, plus 1 on the diagonal (_applyOmega,
   src/AMG/matchingAggregation.cu:64-80) */
template <int G>
__global__ __launch_bounds__(BS) void k_sa_omega(int n, const int *__restrict__ rp,
                                                 const int *__restrict__ ci, double omega,
                                                 double *__restrict__ sv)
{
    for (long long i = group_row(blockIdx.x, threadIdx.x, G); i < n; i += row_step(gridDim.x, G)) {
        const int b = rp[i + 1];
        for (int e = rp[i] + (int)(threadIdx.x & (G - 1)); e < b; e += G) {
            double t = -omega * sv[e];
            if (ci[e] == i) t += 1.;
            sv[e] = t;
        }
    }
}

__global__ __launch_bounds__(BS) void k_iota(int n, int *__restrict__ a)
{
    const int i = blockIdx.x * BS + threadIdx.x;
    if (i < n) a[i] = i;
}

__global__ __launch_bounds__(BS) void k_negate(long long n, double *__restrict__ v)
{
    const long long i = (long long)blockIdx.x * BS + threadIdx.x;
    if (i < n) v[i] = -v[i];
}

} // namespace

/* ================================================================ host */

namespace {

/* rows of a workgroup that takes several and ends with one atomic: about
   1024 workgroups of BS / 64 rows (a lane each: BS) to 256 */
int rows_per_block(int n, bool lng)
{
    const int step = lng ? BS / 64 : BS;
    return std::min(256, std::max(1, (n / 1024 + step - 1) / step) * step);
}

/* gather rows [0, n) from their product slots into (col, val) by rp */
void gather_rows(Ctx &c, int n, const int *uoff, const int *rp, const int *tcol,
                 const double *tval, long long nnz, int *col, double *val)
{
    if (n <= 0 || nnz <= 0) return;
    const double avg = (double)nnz / (double)n;
    const int G = avg <= 2 ? 1 : avg <= 8 ? 4 : avg <= 32 ? 16 : 64;
    const int gb = blocks_for((long long)n * G);
    switch (G) {
    case 1: k_sg_gather<1><<<gb, BS, 0, c.stream>>>(n, uoff, rp, tcol, tval, col, val); break;
    case 4: k_sg_gather<4><<<gb, BS, 0, c.stream>>>(n, uoff, rp, tcol, tval, col, val); break;
    case 16: k_sg_gather<16><<<gb, BS, 0, c.stream>>>(n, uoff, rp, tcol, tval, col, val); break;
    default: k_sg_gather<64><<<gb, BS, 0, c.stream>>>(n, uoff, rp, tcol, tval, col, val); break;
    }
    BCMG_CHECK_LAUNCH();
}

} // namespace

namespace {

/* all rows of C = L R with dense operands (every row long, one batch) */
void dense_product(Ctx &c, const CsrRef &L, const CsrRef &R, const int *uoff, int *tcol,
                   double *tval, int *cnt)
{
    const int n = L.n, K = L.m, mp = (R.m + 127) / 128 * 128, mw = (R.m + 63) / 64;
    const int tiles = (n + SGM_ROWS - 1) / SGM_ROWS, kw = (K + 31) / 32;
    const int pitch = (K + SGM_AHEAD - 1) / SGM_AHEAD * SGM_AHEAD;
    DBuf<double> Rd((size_t)K * mp), Ld((size_t)tiles * (K + 1) * SGM_ROWS);
    DBuf<unsigned long long> rbits((size_t)K * mw), cbits((size_t)n * mw);
    DBuf<int> before((size_t)n * mw), list((size_t)tiles * pitch), count(tiles);
    BCMG_HIP(hipMemsetAsync(Rd.get(), 0, sizeof(double) * (size_t)K * mp, c.stream));
    BCMG_HIP(hipMemsetAsync(Ld.get(), 0, sizeof(double) * (size_t)tiles * (K + 1) * SGM_ROWS,
                            c.stream));
    k_sgm_right<<<(K + BS / 64 - 1) / (BS / 64), BS, (size_t)(BS / 64) * 2 * mw * sizeof(unsigned),
                  c.stream>>>(K, R.rp, R.ci, R.v, mp, mw, Rd.get(), rbits.get());
    k_sgm_left<<<tiles, BS, sizeof(unsigned) * kw, c.stream>>>(n, K, kw, L.rp, L.ci, L.v, Ld.get(),
                                                               pitch, list.get(), count.get());
    k_sgm_pattern<<<(n + BS / 64 - 1) / (BS / 64), BS, 0, c.stream>>>(n, L.rp, L.ci, mw, rbits.get(), uoff,
                                                             cbits.get(), before.get(), tcol, cnt);
    const int grid = (tiles + BS / 64 - 1) / (BS / 64) * (mp / 128);
    k_sgm_values<<<grid, BS, 0, c.stream>>>(n, K, mp, mw, tiles, list.get(), pitch, count.get(),
                                            Ld.get(), Rd.get(), cbits.get(), before.get(), uoff,
                                            tval);
    BCMG_CHECK_LAUNCH();
}

} // namespace

/* Rows are taken in batches of at most per_pass output slots plus packing
   weights (a row over it is a batch of its own), so that the temporaries
   stay bounded and their offsets fit 32 bits; one batch writes C directly. */
void spgemm(Ctx &c, const CsrRef &L, const CsrRef &R, DevCsr &C, long long per_pass,
            bool right_unique, bool left_sorted)
{
    if (L.m != R.n) throw Error(BCMG_EINVAL, "spgemm: inner dimensions differ");
    if (per_pass <= 0) per_pass = SG_PER_PASS;
    if (per_pass > INT_MAX / 2) per_pass = INT_MAX / 2;
    const int n = L.n;
    C.n = n;
    C.m = R.m;
    C.row.alloc((size_t)n + 1);
    if (n == 0) {
        BCMG_HIP(hipMemsetAsync(C.row.get(), 0, sizeof(int), c.stream));
        C.nnz = 0;
        C.col.alloc(1);
        C.val.alloc(1);
        launch_block_nnz(c, C);
        return;
    }
    const long long mcols = R.m > 0 ? R.m : 1;
    /* Long rows whose accumulators fit LDS go to k_sg_wave when their left
       entries bring half a product per tile or more (below that most of its
       steps add a lane or none; at 1.2 per tile, 16 384 columns, it takes
       3.0 ms and the sorting form 4.9) and the tile pointers stay below R. */
    const int tiles = (int)std::min<long long>((mcols + SG_TILE - 1) / SG_TILE, SG_TILES);
    const int tile_w = (int)((mcols + 64ll * tiles - 1) / (64ll * tiles)) * 64;
    const bool lds = right_unique && mcols <= SG_LDS_COLS &&
                     (long long)R.n * (tiles + 1) <= 2ll * R.nnz;
    /* rows by hash where the right rows have four entries or more on average:
       a left entry is a step of a wavefront, and with one product each (the
       tentative prolongator) 2048 of them took 5.2 ms against 0.9 sorted; below
       four products per left entry and tile it also goes before k_sg_wave,
       which takes what has too many columns (T P with 16 384 columns and 19
       products per left entry: 3.0 ms
       against 1.1) */
    const bool hashed = right_unique && R.nnz >= 4ll * R.n;
    const int wmin = std::max(1, tiles / 2);
    const int smin = !right_unique ? 0 : !lds ? SG_SERIAL_MIN : hashed ? 4 * tiles : wmin;
    DBuf<int> u(n), sl(n), ws(n), cnt(n), large(n);
    /* Dense operands when the filled parts of both multiply to 1 / SGM_FILL or
       more and either fits SGM_ELEMS: 0.28 and 0.094 (2048 rows) win 4.5 ->
       2.0 and 5.6 -> 2.4 ms with all their preparation, 0.053 (1125 rows)
       breaks even, 0.011 loses (48^3's products 5.2 -> 6.3 ms). */
    const bool fill = right_unique && left_sorted && n >= SGM_ROWS && mcols >= 128 &&
                      mcols <= SG_LDS_COLS &&
                      (long long)n * L.m <= SGM_ELEMS && (long long)L.m * mcols <= SGM_ELEMS &&
                      (double)L.nnz * R.nnz * SGM_FILL >=
                          (double)n * L.m * ((double)R.n * (double)mcols);
    /* long-row count, row with too many products, long rows below smin, a
       value that is not finite */
    DBuf<int> flags(4);
    DBuf<unsigned long long> total(1);
    BCMG_HIP(hipMemsetAsync(flags.get(), 0, 4 * sizeof(int), c.stream));
    if (fill) {
        k_sgm_finite<<<std::min(1024, blocks_for(L.nnz)), BS, 0, c.stream>>>(L.nnz, L.v,
                                                                             flags.get() + 3);
        k_sgm_finite<<<std::min(1024, blocks_for(R.nnz)), BS, 0, c.stream>>>(R.nnz, R.v,
                                                                             flags.get() + 3);
        BCMG_CHECK_LAUNCH();
    }
    BCMG_HIP(hipMemsetAsync(total.get(), 0, sizeof(unsigned long long), c.stream));
    const bool lng = long_rows(n, L.nnz);
    const int per = rows_per_block(n, lng);
    (lng ? k_sg_count<64> : k_sg_count<1>)<<<(n + per - 1) / per, BS, 0, c.stream>>>(
        n, per, L.rp, L.ci, R.rp, mcols, u.get(), sl.get(), ws.get(), cnt.get(), large.get(),
        flags.get(), total.get(), flags.get() + 1, smin);
    BCMG_CHECK_LAUNCH();
    unsigned long long h_total = 0;
    int h_flags[4] = {0, 0, 0, 0};
    BCMG_HIP(hipMemcpyAsync(&h_total, total.get(), sizeof(h_total), hipMemcpyDeviceToHost,
                            c.stream));
    BCMG_HIP(hipMemcpyAsync(h_flags, flags.get(), 4 * sizeof(int), hipMemcpyDeviceToHost,
                            c.stream));
    BCMG_HIP(hipStreamSynchronize(c.stream));
    const int h_nlarge = h_flags[0];
    if (h_flags[1]) throw Error(BCMG_EUNSUP, "sparse product: a row with 2^30 products or more");
    /* batches of rows [lo, hi) by output slots and, per batch, its long rows
       (local ids) */
    std::vector<int> blo, bhi;
    std::vector<long long> bprod;
    std::vector<std::vector<int>> blarge;
    if ((long long)h_total <= per_pass) {
        blo.push_back(0);
        bhi.push_back(n);
        bprod.push_back((long long)h_total);   /* bounds the slots from above */
    } else {
        std::vector<int> hu(n), hw(n);
        BCMG_HIP(hipMemcpy(hu.data(), sl.get(), sizeof(int) * n, hipMemcpyDeviceToHost));
        BCMG_HIP(hipMemcpy(hw.data(), ws.get(), sizeof(int) * n, hipMemcpyDeviceToHost));
        long long acc = 0, slots = 0;
        int lo = 0;
        for (int i = 0; i < n; i++) {
            const long long cost = (long long)hu[i] + hw[i];
            if (i > lo && acc + cost > per_pass) {
                blo.push_back(lo);
                bhi.push_back(i);
                bprod.push_back(slots);
                lo = i;
                acc = 0;
                slots = 0;
            }
            acc += cost;
            slots += hu[i];
        }
        blo.push_back(lo);
        bhi.push_back(n);
        bprod.push_back(slots);
        std::vector<int> hl(h_nlarge);
        if (h_nlarge > 0)
            BCMG_HIP(hipMemcpy(hl.data(), large.get(), sizeof(int) * h_nlarge,
                               hipMemcpyDeviceToHost));
        std::sort(hl.begin(), hl.end());
        blarge.resize(blo.size());
        size_t q = 0;
        for (size_t b = 0; b < blo.size(); b++)
            while (q < hl.size() && hl[q] < bhi[b]) blarge[b].push_back(hl[q++] - blo[b]);
    }
    const size_t nbatch = blo.size();
    long long maxp = 1, maxrows = 1;
    for (size_t b = 0; b < nbatch; b++) {
        maxp = std::max(maxp, bprod[b]);
        maxrows = std::max<long long>(maxrows, bhi[b] - blo[b]);
    }
    DBuf<int> uoff((size_t)maxrows + 1), soff((size_t)maxrows + 1), brp;
    DBuf<int> tcol((size_t)maxp);
    DBuf<double> tval((size_t)maxp);
    std::vector<DBuf<int>> ocol(nbatch > 1 ? nbatch : 0);
    std::vector<DBuf<double>> oval(nbatch > 1 ? nbatch : 0);
    std::vector<long long> onnz(nbatch, 0);
    if (nbatch > 1) brp.alloc((size_t)maxrows + 1);
    DBuf<double> acc;
    DBuf<int> stamp;
    int dblocks = 0;
    DBuf<int> seg;
    for (size_t b = 0; b < nbatch; b++) {
        const int lo = blo[b], nr = bhi[b] - blo[b];
        const int *Lrp = L.rp + lo;
        exclusive_scan(c, sl.get() + lo, uoff.get(), nr, false);
        auto hash = [&](auto kern, int above, int upto, int below) {
            kern<<<(nr + BS / 64 - 1) / (BS / 64), BS, 0, c.stream>>>(
                nr, above, upto, below, Lrp, L.ci, L.v, R.rp, R.ci, R.v, u.get() + lo, uoff.get(),
                tcol.get(), tval.get(), cnt.get() + lo, flags.get() + 1);
        };
        if (hashed) {
            hash(k_sg_hash<512>, 0, 512, 0);
            hash(k_sg_hash<1024>, 512, SG_CAP, 0);
        }
        const long long S =
            hashed ? 0 : exclusive_scan(c, ws.get() + lo, soff.get(), nr, true);
        const int nb = (int)((S + SG_CAP - 1) / SG_CAP);
        if (nb > 0)
            k_sg_small<<<nb, BS, 0, c.stream>>>(nr, Lrp, L.ci, L.v, R.rp, R.ci, R.v,
                                                ws.get() + lo, soff.get(), uoff.get(),
                                                tcol.get(), tval.get(), cnt.get() + lo);
        BCMG_CHECK_LAUNCH();
        /* long rows: dense accumulators */
        const int *lrows = large.get();
        int nl = h_nlarge;
        DBuf<int> lbuf;
        if (nbatch > 1) {
            nl = (int)blarge[b].size();
            if (nl > 0) {
                lbuf.alloc(nl);
                BCMG_HIP(hipMemcpyAsync(lbuf.get(), blarge[b].data(), sizeof(int) * nl,
                                        hipMemcpyHostToDevice, c.stream));
            }
            lrows = lbuf.get();
        }
        if (fill && nbatch == 1 && nl == n && h_flags[3] == 0) {
            dense_product(c, L, R, uoff.get(), tcol.get(), tval.get(), cnt.get());
        } else if (nl > 0) {
            auto wave = [&](int least, int only_left) {
                if (!seg.get()) {
                    seg.alloc((size_t)R.n * (tiles + 1));
                    k_sg_seg<<<group_blocks(R.n, 64), BS, 0, c.stream>>>(R.n, R.rp, R.ci, tile_w,
                                                                          tiles, seg.get());
                }
                /* mostly long rows: by row, which keeps their order (the list
                   is in order of arrival) */
                const bool by_row = nl >= nr / 2;
                k_sg_wave<<<by_row ? nr : nl, 64 * tiles, sizeof(double) * tiles * tile_w,
                            c.stream>>>(by_row ? nullptr : lrows, Lrp, L.ci, L.v, seg.get(), R.ci,
                                        R.v, u.get() + lo, uoff.get(), tcol.get(), tval.get(),
                                        tile_w, least, only_left, cnt.get() + lo);
                BCMG_CHECK_LAUNCH();
            };
            if (lds && h_flags[2] < h_nlarge) wave(smin, 0);
            /* the others: by hash where their columns fit, the rest on dense
               accumulators */
            int rest = !lds || h_flags[2] > 0;
            if (rest && hashed) {
                BCMG_HIP(hipMemsetAsync(flags.get() + 1, 0, sizeof(int), c.stream));
                hash(k_sg_hash<1024>, SG_CAP, INT_MAX, lds ? smin : 0);
                BCMG_CHECK_LAUNCH();
                BCMG_HIP(hipMemcpyAsync(&rest, flags.get() + 1, sizeof(int),
                                        hipMemcpyDeviceToHost, c.stream));
                BCMG_HIP(hipStreamSynchronize(c.stream));
            }
            if (rest && lds && hashed) wave(wmin, 1);
            if (rest) {
                if (!acc.get()) {
                    /* dense accumulators: as many workgroups as the budget
                       allows, stamps cleared once for every batch */
                    const long long per = 12 * mcols;
                    dblocks = (int)std::min<long long>(
                        {(long long)h_nlarge, (long long)SG_DENSE_BLOCKS,
                         std::max<long long>(1, SG_DENSE_BYTES / per)});
                    acc.alloc((size_t)dblocks * mcols);
                    stamp.alloc((size_t)dblocks * mcols);
                    BCMG_HIP(hipMemsetAsync(stamp.get(), 0xff,
                                            sizeof(int) * (size_t)dblocks * mcols, c.stream));
                }
                k_sg_dense<<<std::min(nl, dblocks), BS, 0, c.stream>>>(
                    nl, lrows, Lrp, L.ci, L.v, R.rp, R.ci, R.v, u.get() + lo, uoff.get(),
                    tcol.get(), tval.get(), acc.get(), stamp.get(), mcols, lo, lds ? wmin : smin, lds ? 1 : 0,
                    hashed ? 1 : 0, cnt.get() + lo);
                BCMG_CHECK_LAUNCH();
            }
        }
        if (nbatch == 1) {
            const long long nnz = exclusive_scan(c, cnt.get(), C.row.get(), n, true);
            if (nnz > INT_MAX) throw Error(BCMG_EUNSUP, "sparse product: nnz above 2^31 - 1");
            C.nnz = (int)nnz;
            C.col.alloc(nnz > 0 ? (size_t)nnz : 1);
            C.val.alloc(nnz > 0 ? (size_t)nnz : 1);
            gather_rows(c, n, uoff.get(), C.row.get(), tcol.get(), tval.get(), nnz, C.col.get(),
                        C.val.get());
        } else {
            const long long nnz = exclusive_scan(c, cnt.get() + lo, brp.get(), nr, true);
            onnz[b] = nnz;
            ocol[b].alloc(nnz > 0 ? (size_t)nnz : 1);
            oval[b].alloc(nnz > 0 ? (size_t)nnz : 1);
            gather_rows(c, nr, uoff.get(), brp.get(), tcol.get(), tval.get(), nnz,
                        ocol[b].get(), oval[b].get());
        }
    }
    if (nbatch > 1) {
        const long long nnz = exclusive_scan(c, cnt.get(), C.row.get(), n, true);
        if (nnz > INT_MAX) throw Error(BCMG_EUNSUP, "sparse product: nnz above 2^31 - 1");
        C.nnz = (int)nnz;
        C.col.alloc(nnz > 0 ? (size_t)nnz : 1);
        C.val.alloc(nnz > 0 ? (size_t)nnz : 1);
        long long at = 0;
        for (size_t b = 0; b < nbatch; b++) {
            if (onnz[b] > 0) {
                BCMG_HIP(hipMemcpyAsync(C.col.get() + at, ocol[b].get(), sizeof(int) * onnz[b],
                                        hipMemcpyDeviceToDevice, c.stream));
                BCMG_HIP(hipMemcpyAsync(C.val.get() + at, oval[b].get(),
                                        sizeof(double) * onnz[b], hipMemcpyDeviceToDevice,
                                        c.stream));
            }
            at += onnz[b];
        }
    }
    C.group = lanes_for(n, C.nnz);
    launch_block_nnz(c, C);
    /* the temporaries are released on return, in the order of this stream */
}

void transpose_csr(Ctx &c, const CsrRef &A, DevCsr &T)
{
    const int nr = A.m;
    const size_t nz = A.nnz > 0 ? (size_t)A.nnz : 1;
    T.n = nr;
    T.m = A.n;
    T.nnz = A.nnz;
    T.row.alloc((size_t)nr + 1);
    T.col.alloc(nz);
    T.val.alloc(nz);
    DBuf<int> cnt(nr > 0 ? nr : 1), cursor((size_t)nr + 1), fcol(nz), longl(nr > 0 ? nr : 1);
    DBuf<double> fval(nz);
    DBuf<int> nlong(1);
    BCMG_HIP(hipMemsetAsync(cnt.get(), 0, sizeof(int) * (nr > 0 ? nr : 1), c.stream));
    BCMG_HIP(hipMemsetAsync(nlong.get(), 0, sizeof(int), c.stream));
    const bool lng = long_rows(A.n, A.nnz);
    const int gb = group_blocks(A.n, lng ? 64 : 1);
    if (A.n > 0)
        (lng ? k_col_count<64> : k_col_count<1>)<<<gb, BS, 0, c.stream>>>(A.n, A.rp, A.ci,
                                                                          cnt.get());
    BCMG_CHECK_LAUNCH();
    exclusive_scan(c, cnt.get(), T.row.get(), nr, false);
    BCMG_HIP(hipMemcpyAsync(cursor.get(), T.row.get(), sizeof(int) * ((size_t)nr + 1),
                            hipMemcpyDeviceToDevice, c.stream));
    if (A.n > 0)
        (lng ? k_col_fill<64> : k_col_fill<1>)<<<gb, BS, 0, c.stream>>>(
            A.n, A.rp, A.ci, A.v, cursor.get(), fcol.get(), fval.get());
    if (nr > 0)
        k_rank<<<group_blocks(nr, 64), BS, 0, c.stream>>>(nr, T.row.get(), fcol.get(),
                                                           fval.get(), T.col.get(), T.val.get(),
                                                           longl.get(), nlong.get());
    BCMG_CHECK_LAUNCH();
    int h_long = 0;
    BCMG_HIP(hipMemcpyAsync(&h_long, nlong.get(), sizeof(int), hipMemcpyDeviceToHost, c.stream));
    BCMG_HIP(hipStreamSynchronize(c.stream));
    if (h_long > 0)
        k_rank_long<<<h_long, BS, 0, c.stream>>>(longl.get(), A.n, T.row.get(), fcol.get(),
                                                 fval.get(), T.col.get(), T.val.get());
    BCMG_CHECK_LAUNCH();
    T.group = lanes_for(nr, A.nnz);
    launch_block_nnz(c, T);
}

double sa_smoother(Ctx &c, const DevCsr &A, const double *D, DBuf<double> &S)
{
    const int n = A.n;
    S.alloc(A.nnz > 0 ? (size_t)A.nnz : 1);
    DBuf<unsigned long long> nb(1);
    BCMG_HIP(hipMemsetAsync(nb.get(), 0, sizeof(unsigned long long), c.stream));
    const bool lng = long_rows(n, A.nnz);
    const int gb = group_blocks(n, lng ? 64 : 1);
    const int per = rows_per_block(n, lng);
    (lng ? k_sa_scale<64> : k_sa_scale<1>)<<<(n + per - 1) / per, BS, 0, c.stream>>>(
        n, per, A.row.get(), A.val.get(), D, S.get(), nb.get());
    BCMG_CHECK_LAUNCH();
    unsigned long long bits = 0;
    BCMG_HIP(hipMemcpyAsync(&bits, nb.get(), sizeof(bits), hipMemcpyDeviceToHost, c.stream));
    BCMG_HIP(hipStreamSynchronize(c.stream));
    double norm;
    std::memcpy(&norm, &bits, sizeof(norm));
    const double omega = 4.0 / (3.0 * norm);
    (lng ? k_sa_omega<64> : k_sa_omega<1>)<<<gb, BS, 0, c.stream>>>(n, A.row.get(), A.col.get(),
                                                                    omega, S.get());
    BCMG_CHECK_LAUNCH();
    return omega;
}

void launch_iota(hipStream_t s, int n, int *a)
{
    if (n <= 0) return;
    k_iota<<<blocks_for(n), BS, 0, s>>>(n, a);
    BCMG_CHECK_LAUNCH();
}

void launch_negate(hipStream_t s, long long n, double *v)
{
    if (n <= 0) return;
    k_negate<<<blocks_for(n), BS, 0, s>>>(n, v);
    BCMG_CHECK_LAUNCH();
}

} // namespace bcmg
