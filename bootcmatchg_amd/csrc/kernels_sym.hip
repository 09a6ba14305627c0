/*
 * kernels_sym.hip - symmetric stencils with varying coefficients: half of the
 * values, diagonal by diagonal.
 *
 * An uploaded operator whose columns take at most PAT_MAX offsets, closed
 * under negation, and whose entries (r, r - o) and (r - o, r) are the same
 * bits keeps, beside its CSR arrays, its diagonal and upper diagonals as
 * arrays over the rows and one mask byte per row. Row r's entry at offset -o
 * is read at position r - o of the diagonal o: the 7-point stencil streams
 * 4 values of 8 bytes and a byte per row instead of 7 values, 7 columns and a
 * row pointer (33 against 88 bytes beside the vectors; the lower values are
 * re-read from L2), without the pass through LDS and its barrier that the
 * CSR slices need. The products and their order are those of the CSR row, so
 * the results have the same bits; the L1 divisor in FP64 is the sum of the
 * row's magnitudes, formed in the same order as its array.
 *
 * Log-normal 7-point coefficients, FP64, 128^3 (2.1 M rows): product 26.4 ->
 * 16.0 us, L1 sweep 31.9 -> 20.2 us; 101^3: 16.8 -> 9.0 and 19.0 -> 11.6 us
 * (65 bytes a row in the sweep, 5.8 TB/s; the vectors and diagonals through
 * L2 and the last-level cache bound it).
 */
#include "kernels_common.h"

#include <algorithm>

namespace bcmg {

namespace {

/* offsets ascending; k0: position of offset 0; value of entry k >= k0 of row
   r at u[(k - k0) ld + r], of entry k < k0 at u[up[k] ld + r + off[k]] */
template <typename MT>
struct SymRef {
    const unsigned char *mask;
    const MT *u;
    long ld;
    int off[PAT_MAX];
    int up[PAT_MAX]; /* diagonal that holds entry k */
    InnerRows inner;
};

/* step 1: the diagonals and masks (rows that pad the last block get none) */
__global__ __launch_bounds__(BS) void k_sym_build(int n, const int *__restrict__ rp,
                                                  const int *__restrict__ ci,
                                                  const double *__restrict__ av, PatOffsets po,
                                                  int k, int k0, long ld,
                                                  unsigned char *__restrict__ mask,
                                                  double *__restrict__ u)
{
    const int r = blockIdx.x * BS + threadIdx.x;
    double v[PAT_MAX];
    unsigned m = 0;
#pragma unroll
    for (int q = 0; q < PAT_MAX; q++) v[q] = 0.0;
    if (r < n) {
        const int e1 = rp[r + 1];
        for (int e = rp[r]; e < e1; e++) {
            const int o = ci[e] - r;
#pragma unroll
            for (int q = 0; q < PAT_MAX; q++)
                if (q < k && po.d[q] == o) {
                    m |= 1u << q;
                    v[q] = av[e];
                }
        }
    }
    mask[r] = (unsigned char)m;
#pragma unroll
    for (int q = 0; q < PAT_MAX; q++)
        if (q >= k0 && q < k) u[(long)(q - k0) * ld + r] = v[q];
}

/* step 2: every lower entry equals its mirror image */
__global__ __launch_bounds__(BS) void k_sym_check(int n, const int *__restrict__ rp,
                                                  const int *__restrict__ ci,
                                                  const double *__restrict__ av, PatOffsets po,
                                                  int k, int k0, long ld,
                                                  const unsigned char *__restrict__ mask,
                                                  const double *__restrict__ u,
                                                  int *__restrict__ bad)
{
    const int r = blockIdx.x * BS + threadIdx.x;
    if (r >= n) return;
    int b = 0;
    const int e1 = rp[r + 1];
    for (int e = rp[r]; e < e1; e++) {
        const int c = ci[e], o = c - r;
        if (o >= 0) continue;
#pragma unroll
        for (int q = 0; q < PAT_MAX; q++)
            if (q >= k0 && q < k && po.d[q] == -o &&
                (!((mask[c] >> q) & 1u) ||
                 __double_as_longlong(u[(long)(q - k0) * ld + c]) != __double_as_longlong(av[e])))
                b = 1;
    }
    if (b) atomicOr(bad, 1);
}

template <typename T, int W>
struct SymVec {
    typedef T type __attribute__((ext_vector_type(W)));
    typedef type un __attribute__((aligned(sizeof(T))));
};

/* W consecutive elements from p (any alignment of T) */
template <typename T, int W>
__device__ __forceinline__ void load_run(const T *__restrict__ p, T (&v)[W])
{
    if constexpr (W == 1) {
        v[0] = *p;
    } else {
        const typename SymVec<T, W>::type q =
            *reinterpret_cast<const typename SymVec<T, W>::un *>(p);
#pragma unroll
        for (int w = 0; w < W; w++) v[w] = q[w];
    }
}

/* Row operations on a symmetric stencil, W rows per thread. Inside (every
   gather of the block stays in [0, n)) all loads go out at once; the first
   and last blocks load under the masks. SD: sum the magnitudes for the L1
   divisor. */
template <typename MT, typename VT, typename XT, int K, int W, bool SD>
__device__ __forceinline__ void sym_rows(int n, int r, bool inner, const SymRef<MT> &S,
                                         const XT *__restrict__ x, VT (&t)[W], VT (&sd)[W])
{
    unsigned m[W];
    XT g[K][W];
    MT v[K][W];
    if (inner) {
        if constexpr (W == 1) {
            m[0] = S.mask[r];
        } else {
            const unsigned mm = *reinterpret_cast<const unsigned short *>(S.mask + r);
            m[0] = mm & 0xFFu;
            m[1] = mm >> 8;
        }
#pragma unroll
        for (int k = 0; k < K; k++) {
            load_run<XT, W>(x + r + S.off[k], g[k]);
            load_run<MT, W>(S.u + (long)S.up[k] * S.ld + (S.off[k] < 0 ? r + S.off[k] : r), v[k]);
        }
    } else {
#pragma unroll
        for (int w = 0; w < W; w++) {
            m[w] = r + w < n ? S.mask[r + w] : 0u;
#pragma unroll
            for (int k = 0; k < K; k++) {
                g[k][w] = 0;
                v[k][w] = 0;
                if ((m[w] >> k) & 1u) {
                    const int c = r + w + S.off[k];
                    g[k][w] = x[c];
                    v[k][w] = S.u[(long)S.up[k] * S.ld + (S.off[k] < 0 ? c : r + w)];
                }
            }
        }
    }
#pragma unroll
    for (int w = 0; w < W; w++) {
        t[w] = 0;
        sd[w] = 0;
#pragma unroll
        for (int k = 0; k < K; k++)
            if ((m[w] >> k) & 1u) {
                t[w] = t[w] + (VT)v[k][w] * (VT)g[k][w];
                if (SD) sd[w] += fabs((VT)v[k][w]);
            }
    }
}

template <typename MT, typename VT, int OP, int K, int W, int DIV>
__global__ __launch_bounds__(BS) void k_rows_sym(int n, SymRef<MT> S, const VT *__restrict__ x,
                                                 const VT *__restrict__ f,
                                                 const VT *__restrict__ d, VT *__restrict__ y)
{
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = b * (BS * W);
    const int r = r0 + threadIdx.x * W;
    const bool inner = S.inner.holds(r0, BS * W);
    constexpr bool SD = OP == OP_JACOBI && DIV == DIV_L1;
    VT fr[W], xr[W], dr[W], t[W], sd[W];
#pragma unroll
    for (int w = 0; w < W; w++) {
        fr[w] = xr[w] = 0;
        dr[w] = 1;
    }
    if (inner) {
        if (OP != OP_SPMV) load_run<VT, W>(f + r, fr);
        if (OP == OP_JACOBI) load_run<VT, W>(x + r, xr);
        if (OP == OP_JACOBI && !SD) load_run<VT, W>(d + r, dr);
    } else {
#pragma unroll
        for (int w = 0; w < W; w++)
            if (r + w < n) {
                if (OP != OP_SPMV) fr[w] = f[r + w];
                if (OP == OP_JACOBI) xr[w] = x[r + w];
                if (OP == OP_JACOBI && !SD) dr[w] = d[r + w];
            }
    }
    sym_rows<MT, VT, VT, K, W, SD>(n, r, inner, S, x, t, sd);
    VT o[W];
#pragma unroll
    for (int w = 0; w < W; w++) {
        if (OP == OP_SPMV)
            o[w] = t[w];
        else if (OP == OP_RESID)
            o[w] = fr[w] - t[w];
        else
            o[w] = (fr[w] - t[w]) / (SD ? sd[w] : dr[w]) + xr[w];
    }
    if (W > 1 && inner) {
        typename SymVec<VT, W == 1 ? 2 : W>::type q;
#pragma unroll
        for (int w = 0; w < W; w++) q[w] = o[w];
        *reinterpret_cast<typename SymVec<VT, W == 1 ? 2 : W>::un *>(y + r) = q;
    } else {
#pragma unroll
        for (int w = 0; w < W; w++)
            if (r + w < n) y[r + w] = o[w];
    }
}

/* k_spmv_dots on a symmetric stencil (the same 256-row blocks and trees) */
template <int K, int KO, typename ZT>
__global__ __launch_bounds__(BS) void k_spmv_dots_sym(int n, SymRef<double> S,
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
    if (r < n) {
        const double zr = (double)z[r], rr = rv[r];
        const double tor = K > 2 ? to[r] : 0.0;
        double tr[1], unused[1];
        sym_rows<double, double, ZT, KO, 1, false>(n, r, S.inner.holds(r0, BS), S, z, tr,
                                                   unused);
        t[r] = tr[0];
        sdot[0] = rr * zr;
        sdot[1] = tr[0] * zr;
        if (K > 2) sdot[K - 1] = tor * zr;
    }
    block_reduce_store<K>(sdot, part + (size_t)b * K);
}

template <typename MT>
SymRef<MT> sym_ref(const DevCsr &A)
{
    const SymStencil &Y = A.sym;
    SymRef<MT> S;
    S.mask = Y.mask.get();
    if constexpr (std::is_same<MT, double>::value)
        S.u = Y.u.get();
    else
        S.u = Y.u32.get();
    S.ld = Y.ld;
    S.inner = inner_rows(A.n, Y.off[0], Y.off[Y.k - 1]);
    for (int k = 0; k < PAT_MAX; k++) {
        S.off[k] = k < Y.k ? Y.off[k] : 0;
        S.up[k] = k < Y.k ? std::abs(k - Y.k / 2) : 0;
    }
    return S;
}

/* rows from which an FP64 thread takes two rows (16-byte loads): sweep with
   1 / 2 rows 22.0 / 20.2 us at 2.1 M rows, 12.6 / 11.6 at 1 M, 6.3 / 5.8 at
   262 144, 5.2 / 5.1 at 42 875; FP32 keeps one (its 2.1 M-row V-cycle took
   656 us with one row, 669 with two) */
constexpr int SYM_WIDE = 1 << 17;

template <typename MT, typename VT, int OP, int K, int DIV>
void rows_sym_w(hipStream_t s, const DevCsr &A, const SymRef<MT> &S, const VT *x, const VT *f,
                const VT *d, VT *y)
{
    const int n = A.n;
    if (std::is_same<VT, double>::value && n >= SYM_WIDE)
        k_rows_sym<MT, VT, OP, K, 2, DIV><<<(n + 2 * BS - 1) / (2 * BS), BS, 0, s>>>(n, S, x, f, d,
                                                                                    y);
    else
        k_rows_sym<MT, VT, OP, K, 1, DIV><<<(n + BS - 1) / BS, BS, 0, s>>>(n, S, x, f, d, y);
}

template <typename MT, typename VT, int OP, int DIV>
void rows_sym_k(hipStream_t s, const DevCsr &A, const VT *x, const VT *f, const VT *d, VT *y)
{
    const SymRef<MT> S = sym_ref<MT>(A);
    const int k = A.sym.k;
    if (k <= 3)
        rows_sym_w<MT, VT, OP, 3, DIV>(s, A, S, x, f, d, y);
    else if (k <= 5)
        rows_sym_w<MT, VT, OP, 5, DIV>(s, A, S, x, f, d, y);
    else
        rows_sym_w<MT, VT, OP, 7, DIV>(s, A, S, x, f, d, y);
}

} // namespace

/* operators of fewer rows are not analysed: their launches are bound by
   latency and gain little */
constexpr int SYM_MIN_ROWS = 32768;

bool sym_candidate(const DevCsr &A)
{
    return A.n == A.m && A.n >= SYM_MIN_ROWS && A.nnz <= (long long)(PAT_MAX - 1) * A.n;
}

void make_sym(Ctx &c, DevCsr &A, const std::vector<int> &off)
{
    if (!sym_candidate(A) || A.cls.n > 0 || A.maxrow <= 0 || A.maxrow > PAT_MAX - 1) return;
    /* odd in number and closed under negation: the middle one is 0 */
    const int k = (int)off.size();
    if (k < 3 || k % 2 == 0) return;
    for (int q = 0; q < k; q++)
        if (off[q] != -off[k - 1 - q]) return;
    SymStencil &Y = A.sym;
    const int nblk = (A.n + BS - 1) / BS, k0 = k / 2;
    Y.ld = (long)nblk * BS;
    Y.mask.alloc((size_t)nblk * BS);
    Y.u.alloc((size_t)(k - k0) * Y.ld);
    DBuf<int> bad(1);
    PatOffsets po;
    for (int q = 0; q < PAT_MAX; q++) po.d[q] = q < k ? off[q] : 0;
    BCMG_HIP(hipMemsetAsync(bad.get(), 0, sizeof(int), c.stream));
    k_sym_build<<<nblk, BS, 0, c.stream>>>(A.n, A.row.get(), A.col.get(), A.val.get(), po, k, k0,
                                           Y.ld, Y.mask.get(), Y.u.get());
    k_sym_check<<<nblk, BS, 0, c.stream>>>(A.n, A.row.get(), A.col.get(), A.val.get(), po, k, k0,
                                           Y.ld, Y.mask.get(), Y.u.get(), bad.get());
    BCMG_CHECK_LAUNCH();
    BCMG_HIP(hipMemcpyAsync(c.h_ints, bad.get(), sizeof(int), hipMemcpyDeviceToHost, c.stream));
    BCMG_HIP(hipStreamSynchronize(c.stream));
    if (c.h_ints[0] != 0) {
        Y.mask.release();
        Y.u.release();
        return;
    }
    Y.k = A.noff = k;
    A.off_lo = off.front();
    A.off_hi = off.back();
    for (int q = 0; q < k; q++) Y.off[q] = off[q];
}

void SymStencil::make_lowp(hipStream_t s)
{
    if (k == 0) return;
    const size_t cnt = (size_t)(k - k / 2) * ld;
    if (!u32.get()) u32.alloc(cnt);
    launch_d2f(s, cnt, u.get(), u32.get());
}

template <typename VT>
bool sym_ok(const DevCsr &A, MatType mt)
{
    if (!A.use_sym()) return false;
    if constexpr (std::is_same<VT, double>::value)
        return mt == MT_F64;
    else
        return mt == MT_F32 && A.sym.u32.get() != nullptr;
}

template <typename VT>
void launch_rows_sym(hipStream_t s, const DevCsr &A, RowOp op, const VT *x, const VT *f,
                     const VT *d, VT *y, DivSource div)
{
    using MT = VT;
    if (op == OP_SPMV)
        rows_sym_k<MT, VT, OP_SPMV, DIV_ARRAY>(s, A, x, f, d, y);
    else if (op == OP_RESID)
        rows_sym_k<MT, VT, OP_RESID, DIV_ARRAY>(s, A, x, f, d, y);
    else if (std::is_same<VT, double>::value && div == DIV_L1)
        rows_sym_k<MT, VT, OP_JACOBI, std::is_same<VT, double>::value ? DIV_L1 : DIV_ARRAY>(
            s, A, x, f, d, y);
    else
        rows_sym_k<MT, VT, OP_JACOBI, DIV_ARRAY>(s, A, x, f, d, y);
    BCMG_CHECK_LAUNCH();
}

template <typename ZT>
void launch_spmv_dots_sym(hipStream_t s, const DevCsr &A, int k, const ZT *z, double *t,
                          const double *r, const double *to, double *part)
{
    const SymRef<double> S = sym_ref<double>(A);
    const int n = A.n, nb = (n + BS - 1) / BS, ko = A.sym.k;
    auto go = [&](auto kern) { kern<<<nb, BS, 0, s>>>(n, S, z, t, r, to, part); };
    if (k == 2)
        ko <= 3 ? go(k_spmv_dots_sym<2, 3, ZT>)
                : ko <= 5 ? go(k_spmv_dots_sym<2, 5, ZT>) : go(k_spmv_dots_sym<2, 7, ZT>);
    else
        ko <= 3 ? go(k_spmv_dots_sym<3, 3, ZT>)
                : ko <= 5 ? go(k_spmv_dots_sym<3, 5, ZT>) : go(k_spmv_dots_sym<3, 7, ZT>);
    BCMG_CHECK_LAUNCH();
}

#define BCMG_INSTANTIATE_SYM(T)                                                              \
    template bool sym_ok<T>(const DevCsr &, MatType);                                        \
    template void launch_rows_sym<T>(hipStream_t, const DevCsr &, RowOp, const T *,          \
                                     const T *, const T *, T *, DivSource);                  \
    template void launch_spmv_dots_sym<T>(hipStream_t, const DevCsr &, int, const T *,       \
                                          double *, const double *, const double *, double *);
BCMG_INSTANTIATE_SYM(double)
BCMG_INSTANTIATE_SYM(float)
#undef BCMG_INSTANTIATE_SYM

} // namespace bcmg
