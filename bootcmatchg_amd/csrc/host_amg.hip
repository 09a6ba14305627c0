/*
 * host_amg.hip - host orchestration of the AMG setup (bootstrap, coarsening)
 * and of the solve (V/H/W cycles, composite preconditioner, FCG v3).
 *
 * All device work is ordered on the context stream. The setup synchronises
 * only where a size is needed to allocate (coarse row count, coarse nnz);
 * the solve reads one scalar per FCG iteration (the residual norm) for the
 * stopping test, as the reference does (src/SOLVER/FCG.cu:558-565).
 */
#include "bcmg_internal.h"

#include <algorithm>
#include <cfloat>
#include <chrono>
#include <cmath>

namespace bcmg {

namespace {

/* src/AMG/AMG.cu:371-394 */
std::vector<int> grid_sweeps(int cycle_type, int max_levels)
{
    const int ml = max_levels - 1;
    std::vector<int> g(ml > 0 ? ml : 1, 1);
    if (cycle_type == 1) {
        for (int i = 0; i < ml; i++)
            if (i % 2 == 0) g[i] = 2;
    } else if (cycle_type == 2) {
        for (int i = 0; i < ml - 1; i++) g[i] = 2;
    }
    return g;
}

/* Event marks of the setup phases on the context stream, recorded only when
   Ctx::time_setup is set and read after the setup's last synchronisation.
   A phase is bracketed by a Scope; hierarchy h's marks add up in
   Boot::t_phase[h]. */
class SetupClock {
  public:
    explicit SetupClock(Ctx &c) : c_(c), on_(c.time_setup) {}
    ~SetupClock()
    {
        for (auto &m : marks_) {
            if (m.a) (void)hipEventDestroy(m.a);
            if (m.b) (void)hipEventDestroy(m.b);
        }
    }
    SetupClock(const SetupClock &) = delete;
    SetupClock &operator=(const SetupClock &) = delete;

    class Scope {
      public:
        Scope(SetupClock *k, int phase) : k_(k && k->on_ ? k : nullptr)
        {
            if (k_) idx_ = k_->open(phase);
        }
        ~Scope()
        {
            if (k_) k_->close(idx_);
        }
        Scope(const Scope &) = delete;
        Scope &operator=(const Scope &) = delete;

      private:
        SetupClock *k_;
        size_t idx_ = 0;
    };

    void set_hierarchy(int h) { hier_ = h; }
    void collect(Boot &B)
    {
        for (auto &t : B.t_phase) std::fill(t.begin(), t.end(), 0.0);
        for (const auto &m : marks_) {
            float ms = 0.f;
            if (!m.a || !m.b || hipEventElapsedTime(&ms, m.a, m.b) != hipSuccess) continue;
            if (m.hier >= (int)B.t_phase.size()) B.t_phase.resize(m.hier + 1);
            B.t_phase[m.hier].resize(PH_COUNT, 0.0);
            B.t_phase[m.hier][m.phase] += ms;
        }
    }

  private:
    struct Mark {
        int hier, phase;
        hipEvent_t a, b;
    };
    size_t open(int phase)
    {
        Mark m{hier_, phase, nullptr, nullptr};
        if (hipEventCreate(&m.a) == hipSuccess) (void)hipEventRecord(m.a, c_.stream);
        marks_.push_back(m);
        return marks_.size() - 1;
    }
    void close(size_t i)
    {
        Mark &m = marks_[i];
        if (hipEventCreate(&m.b) == hipSuccess) (void)hipEventRecord(m.b, c_.stream);
    }
    Ctx &c_;
    bool on_;
    int hier_ = 0;
    std::vector<Mark> marks_;
};

struct BuildState {
    int maxcoarsesize = 0;
    int ftcoarse = 1;
    SetupClock *clk = nullptr;
};

/* src/AMG/matchingAggregation.cu:18-60 */
void relax_prepare(Ctx &c, Level &lv, const DevCsr &A, int type)
{
    if (type == 0 || type == 4) {
        lv.D.ensure(A.n);
        launch_diag(c.stream, A, lv.D.get());
        lv.hasD = true;
    }
    if (type == 4) {
        lv.M.ensure(A.n);
        launch_abs_rowsum(c.stream, A, lv.M.get());
        lv.hasM = true;
    }
}

/* aggrsweeps pairwise sweeps (src/AMG/matchingAggregation.cu:211-295):
   A_{i+1} = R_i (A_i P_i), w_{i+1} = R_i w_i, P = P P_i. */
void matching_aggregation(Ctx &c, const bcmg_params &p, BuildState &bs, const DevCsr &A0,
                          DBuf<double> &w, DBuf<int> &aggP, DBuf<double> &pP, DevCsr &Aout)
{
    const int n0 = A0.n;
    const DevCsr *Ai = &A0;
    DevCsr cur;
    DBuf<double> wi;
    const double *wptr = w.get();
    for (int s = 0; s < p.aggrsweeps; s++) {
        const int n = Ai->n;
        DBuf<double> W(Ai->nnz > 0 ? Ai->nnz : 1);
        {
            SetupClock::Scope ph(bs.clk, PH_WEIGHTS);
            match_weights(c, *Ai, wptr, W.get());
        }
        DBuf<int> M(n), Ms(n);
        {
            SetupClock::Scope ph(bs.clk, PH_MATCHING);
            match_suitor(c, *Ai, W.get(), M.get(), Ms.get(), false);
        }
        W.release();
        DBuf<int> agg(n), members(2 * (size_t)n);
        DBuf<double> pv(n);
        int nc = 0;
        {
            SetupClock::Scope ph(bs.clk, PH_AGGREGATION);
            nc = aggregate_pairs(c, n, Ms.get(), wptr, agg.get(), pv.get(), members.get());
        }
        DevCsr Ac;
        {
            SetupClock::Scope ph(bs.clk, PH_GALERKIN);
            galerkin_pairwise(c, *Ai, agg.get(), pv.get(), members.get(), nc, Ac);
        }
        DBuf<double> wc(nc);
        {
            SetupClock::Scope ph(bs.clk, PH_AGGREGATION);
            restrict_w(c.stream, nc, members.get(), pv.get(), wptr, wc.get());
            if (s == 0) {
                aggP = std::move(agg);
                pP = std::move(pv);
            } else {
                compose_P(c.stream, n0, aggP.get(), pP.get(), agg.get(), pv.get());
            }
        }
        const double coarse_ratio = (double)n / (double)nc;
        cur = std::move(Ac);
        Ai = &cur;
        wi = std::move(wc);
        wptr = wi.get();
        if (coarse_ratio <= 1.2) bs.ftcoarse = 100;
        if ((double)nc <= (double)bs.ftcoarse * bs.maxcoarsesize) break;
    }
    w = std::move(wi);
    Aout = std::move(cur);
}

/* Smoothed prolongators for the levels the unsmoothed coarsening built
   (src/AMG/matchingAggregation.cu:353-390): on level j,
   S = I - omega D^-1 A_j with omega = 4 / (3 ||D^-1 A_j||_inf),
   P_j = S P_tent, R_j = P_j^T, A_{j+1} = (R_j A_j) P_j, and level j + 1's
   smoother data from the new A_{j+1} before level j + 1 is smoothed. The
   reference's infinity norm asserts (src/matrix/CSR.cu:402-404); this takes
   the body it left commented out there (largest sum of |s_ij| over a row). */
void smooth_prolongators(Ctx &c, const bcmg_params &p, Hierarchy &H, SetupClock *clk)
{
    const int levels = H.num_levels();
    for (int j = 0; j + 1 < levels; j++) {
        Level &lv = H.L[j];
        Level &next = H.L[j + 1];
        const DevCsr &A = lv.mat();
        const int n = A.n, nc = next.mat().n;
        double omega = 0.0;
        {
            SetupClock::Scope ph(clk, PH_AGGREGATION);
            DBuf<double> S;
            omega = sa_smoother(c, A, lv.D.get(), S);
            DBuf<int> iota((size_t)n + 1);
            launch_iota(c.stream, n + 1, iota.get());
            const CsrRef Sr{n, n, A.nnz, A.row.get(), A.col.get(), S.get()};
            const CsrRef Pt{n, nc, n, iota.get(), lv.agg.get(), lv.p.get()};
            spgemm(c, Sr, Pt, lv.Pneg);
            S.release();
            iota.release();
            transpose_csr(c, ref_of(lv.Pneg), lv.R);
        }
        DevCsr Ac;
        {
            SetupClock::Scope ph(clk, PH_GALERKIN);
            DevCsr T;
            spgemm(c, ref_of(lv.R), ref_of(A), T);
            spgemm(c, ref_of(T), ref_of(lv.Pneg), Ac);
        }
        launch_negate(c.stream, lv.Pneg.nnz, lv.Pneg.val.get());
        lv.smoothed = true;
        lv.omega = omega;
        next.Aown = std::move(Ac);
        next.hasD = next.hasM = false;
        {
            SetupClock::Scope ph(clk, PH_SMOOTHER);
            relax_prepare(c, next, next.Aown, p.relax_type);
        }
    }
}

/* src/AMG/matchingAggregation.cu:298-423 */
void adaptive_coarsening(Ctx &c, const bcmg_params &p, BuildState &bs, DevCsr &A,
                         const double *w_in, Hierarchy &H)
{
    const int n = A.n;
    DBuf<double> w(n);
    launch_copy(c.stream, n, w_in, w.get());
    H.L.clear();
    H.L.emplace_back();
    H.L[0].Aext = &A;
    DBuf<double> tmp(n);
    const double normw = a_norm(c, A, w.get(), tmp.get());
    tmp.release();
    {
        SetupClock::Scope ph(bs.clk, PH_SMOOTHER);
        relax_prepare(c, H.L[0], A, p.relax_type);
    }
    bs.ftcoarse = 1;
    double avcoarseratio = 0.0;
    int level = 0;
    if (!(normw > DBL_EPSILON))
        throw Error(BCMG_EINVAL, "||w||_A <= DBL_EPSILON: no hierarchy can be built "
                                 "(the reference asserts in Hierarchy::finalize_level)");
    for (level = 1; level < p.max_levels;) {
        H.L.emplace_back();
        Level &prev = H.L[level - 1];
        Level &next = H.L[level];
        const DevCsr &Aprev = prev.mat();
        matching_aggregation(c, p, bs, Aprev, w, prev.agg, prev.p, next.Aown);
        {
            SetupClock::Scope ph(bs.clk, PH_AGGREGATION);
            transpose_P(c, Aprev.n, next.Aown.n, prev.agg.get(), prev.p.get(), prev.R);
        }
        {
            SetupClock::Scope ph(bs.clk, PH_SMOOTHER);
            relax_prepare(c, next, next.Aown, p.relax_type);
        }
        const double size_coarse = next.Aown.n;
        avcoarseratio += Aprev.n / size_coarse;
        level++;
        if (size_coarse <= (double)bs.ftcoarse * bs.maxcoarsesize) break;
    }
    std::vector<DevCsr *> pending;
    if (p.aggrtype == 1 && level > 1) {
        /* the unsmoothed R tiles are replaced: resolve them first */
        for (int i = 0; i + 1 < level; i++) pending.push_back(&H.L[i].R);
        resolve_tiles(c, pending);
        pending.clear();
        smooth_prolongators(c, p, H, bs.clk);
        for (int i = 0; i + 1 < level; i++) {
            pending.push_back(&H.L[i].Pneg);
            pending.push_back(&H.L[i + 1].Aown);
        }
    }
    if (p.coarse_solver != p.relax_type) {
        SetupClock::Scope ph(bs.clk, PH_SMOOTHER);
        relax_prepare(c, H.L[level - 1], H.L[level - 1].mat(), p.coarse_solver);
    }
    for (int i = 0; i + 1 < level; i++) pending.push_back(&H.L[i].R);
    resolve_tiles(c, pending);
    pending.clear();
    for (int i = 1; i < level; i++) pending.push_back(&H.L[i].Aown);
    make_classes(c, pending);
    make_narrow(c, pending);
    double cx = 0, cw = 0;
    for (int i = 0; i < level; i++) {
        cx += H.L[i].mat().nnz;
        cw += std::pow(2.0, i) * H.L[i].mat().nnz;
    }
    H.op_cmplx = cx / H.L[0].mat().nnz;
    H.op_wcmplx = cw / H.L[0].mat().nnz;
    H.avg_cratio = avcoarseratio / (level - 1);
}

/* ------------------------------------------------------------ cycles */

template <typename VT>
struct LevelState {
    VT *x = nullptr, *x2 = nullptr;
    bool zero = true;
};

template <typename VT>
CycleBufs<VT> &bufs(Boot &B);
template <>
CycleBufs<double> &bufs<double>(Boot &B) { return B.b64; }
template <>
CycleBufs<float> &bufs<float>(Boot &B) { return B.b32; }

template <typename VT>
struct CycleRun {
    Ctx &c;
    Boot &B;
    const Hierarchy &H;
    std::vector<LevelState<VT>> &st;
    const VT *f0;               /* level-0 right-hand side */
    VT *final_out;              /* where the very last level-0 sweep should write */
};

/* `sweeps` Jacobi sweeps on level lv (src/AMG/relaxation.cu:211-285),
   ping-pong between st.x and st.x2. A sweep from a known-zero x is f / d
   (the SpMV of a zero vector is skipped; same values); when another sweep
   follows, the two run as one pass that forms f / d where the second sweep
   reads it (except on a streamed FP64 operator). A small level runs all its
   sweeps in one workgroup (same values, one launch). */
template <typename VT>
void relax_level(Ctx &c, const Level &lv, MatType mt, int type, int sweeps, const VT *f,
                 LevelState<VT> &s, VT *final_out, bool level0)
{
    const DevCsr &A = lv.mat();
    const VT *d = divisor<VT>(lv, type);
    if (sweeps == 0) return;
    const bool timing = level0 && c.time_smoother;
    int m = 0;
    for (int take; !timing && (take = slab_plan<VT>(A, mt, sweeps, s.zero, &m)) > 0;) {
        /* several sweeps a launch; over several workgroups the result goes
           to another buffer than x */
        const bool to_final = final_out && take == sweeps;
        VT *out = m >= A.n ? s.x : s.x2;
        if (to_final && (s.zero || m >= A.n || s.x != final_out)) out = final_out;
        launch_slab<VT>(c.stream, A, mt, m, take - (s.zero ? 1 : 0), s.zero, div_source(type), d,
                        f, s.x, out);
        if (out != s.x) {
            s.x2 = s.x;
            s.x = out;
        }
        s.zero = false;
        sweeps -= take;
        if (sweeps == 0) return;
    }
    if (relax_block_ok<VT>(A) && !timing) {
        VT *out = (final_out && s.x != final_out) ? final_out : s.x;
        launch_relax_block<VT>(c.stream, A, mt, d, f, s.x, out, sweeps, s.zero);
        if (out != s.x) {
            s.x2 = s.x;
            s.x = out;
        }
        s.zero = false;
        return;
    }
    /* timed: one event pair around the run of consecutive sweep launches
       (the first two sweeps from zero are then not fused, so that every
       sweep of the level falls inside the pair or is the zero sweep) */
    hipEvent_t e1 = nullptr;
    int timed = 0;
    for (int k = 0; k < sweeps; k++) {
        VT *out = s.x2;
        if (s.zero && k + 1 < sweeps && !timing && fuse_zero_sweeps<VT>(A, mt)) {
            /* the sweep from zero and the next one in one pass (same values:
               the first iterate f / d is formed where the second reads it) */
            k++;
            if (final_out && k == sweeps - 1 && s.x != final_out) out = final_out;
            launch_rows<VT>(c.stream, A, mt, OP_JACOBI_Z, nullptr, f, d, out, div_source(type));
            s.x2 = s.x;
            s.x = out;
            s.zero = false;
            continue;
        }
        if (final_out && k == sweeps - 1 && s.x != final_out) out = final_out;
        if (s.zero) {
            launch_jacobi_zero<VT>(c.stream, A, mt, f, d, out, div_source(type));
        } else {
            if (timing && !timed) {
                hipEvent_t e0 = c.next_event();
                e1 = c.next_event();
                BCMG_HIP(hipEventRecord(e0, c.stream));
            }
            launch_rows<VT>(c.stream, A, mt, OP_JACOBI, s.x, f, d, out, div_source(type));
            timed++;
        }
        s.x2 = s.x;
        s.x = out;
        s.zero = false;
    }
    if (timing && timed) {
        BCMG_HIP(hipEventRecord(e1, c.stream));
        c.ev_launches.push_back(timed);
    }
}

/* R's values in the cycle's type */
template <typename VT>
const VT *rvals(const DevCsr &R);
template <>
const double *rvals<double>(const DevCsr &R) { return R.val.get(); }
template <>
const float *rvals<float>(const DevCsr &R) { return R.val32.get(); }

/* Whether `sweeps` post-smoothing launches that start from iterate a (other
   buffer b) leave the result outside fo: relax_level redirects the last
   sweep into fo unless that sweep reads fo, and no sweep leaves it in a. */
template <typename VT>
bool post_lands_off(int sweeps, const VT *a, const VT *b, const VT *fo)
{
    if (!fo) return false;
    if (sweeps == 0) return a != fo;
    return ((sweeps - 1) % 2 == 0 ? a : b) == fo;
}

/* Where a launch that forms x + P x_c and sweeps puts its result: the other
   iterate, or the preconditioner's output fo when no launch follows
   (rest = 0). When the other iterate is that output and launches remain, a
   third level-0 buffer (the multiplicative composites leave xb[0] free):
   the remaining launches then alternate between two buffers that are not
   the output, so the last one writes the output and no copy follows. */
template <typename VT>
VT *third_buffer(Boot &B, const LevelState<VT> &s, VT *fo, int rest)
{
    if (fo && fo != s.x) {
        VT *third = bufs<VT>(B).xb[0].get();
        if (rest == 0) return fo;
        if (s.x2 == fo && third != s.x && third != fo) return third;
    }
    return s.x2;
}

/* inner-iteration tolerance of the K-cycle (src/SOLVER/GAMG_cycle.cu:5) */
constexpr double KCYCLE_RTOL = 0.25;

template <typename VT>
void cycle(CycleRun<VT> &R, int l, const VT *fin = nullptr);

/* K-cycle coarse correction on level m (0-based, not the coarsest): at most
   two flexible CG steps on A_m x = f_m preconditioned by the cycle from
   level m + 1 (inneritkcycle, src/SOLVER/FCG.cu:620-723). Every decision
   stays on the device (the iteration is captured in a graph): the second
   preconditioner application is always made, and weighted by 0 when the
   first step already meets the inner tolerance - the result is the
   reference's either way. The solution lands in the level's iterate. */
template <typename VT>
void kcycle_inner(CycleRun<VT> &R, int m)
{
    Ctx &c = R.c;
    Boot &B = R.B;
    CycleBufs<VT> &W = bufs<VT>(B);
    const DevCsr &A = R.H.L[m].mat();
    const MatType mt = level_mt(B, m);
    const int n = A.n;
    double *ks = B.kscal.get() + (size_t)m * KS_STRIDE;
    VT *w = W.kw[m].get(), *d0 = W.kd0[m].get(), *d1 = W.kd1[m].get();
    VT *v = W.kv[m].get(), *v1 = W.kv1[m].get();
    LevelState<VT> &s = R.st[m];
    launch_copy<VT>(c.stream, n, W.f[m].get(), w);
    launch_kdots<VT>(c, n, 1, w, nullptr, nullptr, w, ks + 0);
    auto apply = [&](VT *out) {
        s.zero = true;
        cycle<VT>(R, m + 1, w);
        if (s.zero)
            launch_fill<VT>(c.stream, n, VT(0), out);
        else
            launch_copy<VT>(c.stream, n, s.x, out);
    };
    apply(d0);
    launch_kdots<VT>(c, n, 1, w, nullptr, nullptr, d0, ks + 1);
    launch_rows<VT>(c.stream, A, mt, OP_SPMV, d0, nullptr, nullptr, v);
    launch_kdots<VT>(c, n, 1, d0, nullptr, nullptr, v, ks + 2);
    launch_kcycle_alpha(c.stream, ks, B.kscal.get() + KS_FLAG_GLOBAL);
    launch_kcycle_axpy<VT>(c.stream, n, ks, v, w);
    launch_kdots<VT>(c, n, 1, w, nullptr, nullptr, w, ks + 4);
    apply(d1);
    launch_rows<VT>(c.stream, A, mt, OP_SPMV, d1, nullptr, nullptr, v1);
    launch_kdots<VT>(c, n, 3, v, v1, w, d1, ks + 5);
    launch_kcycle_coef(c.stream, ks, KCYCLE_RTOL);
    launch_kcycle_combine<VT>(c.stream, n, ks, d0, d1, s.x);
    s.zero = false;
}

/* recursive cycle (src/SOLVER/GAMG_cycle.cu:25-140); l is 1-based; fin, when
   given, is the level's right-hand side (an inner K-cycle application) */
template <typename VT>
void cycle(CycleRun<VT> &R, int l, const VT *fin)
{
    Ctx &c = R.c;
    Boot &B = R.B;
    CycleBufs<VT> &W = bufs<VT>(B);
    const Hierarchy &H = R.H;
    const int L = H.num_levels();
    const Level &lv = H.L[l - 1];
    const MatType mt = level_mt(B, l - 1);
    LevelState<VT> &s = R.st[l - 1];
    const VT *f = fin ? fin : ((l == 1) ? R.f0 : W.f[l - 1].get());
    const bool top = (l == 1);
    if (l == L) {
        relax_level<VT>(c, lv, mt, B.coarse_solver, B.prm.relaxnumber_coarse, f, s,
                        top ? R.final_out : nullptr, top);
        return;
    }
    const DevCsr &A = lv.mat();
    /* R holds the prolongator values: FP32 whenever the cycle runs in FP32 */
    const MatType rmt = std::is_same<VT, double>::value ? MT_F64 : MT_F32;
    VT *fc = W.f[l].get();
    const bool timing = top && c.time_smoother;
    /* one workgroup relaxes the level: as a constant stencil, or any rows */
    const bool slab1 = !timing && slab_one<VT>(A, mt);
    const bool blk = slab1 || (relax_block_ok<VT>(A) && !timing);
    bool restricted = false;
    if (blk && B.prm.prerelax_sweeps > 0 && rows_sequential<VT>(lv.R)) {
        /* a one-workgroup level: pre-smoothing, residual and restriction in
           one launch (the separate launches' bits) */
        BlockFuse<VT> fu;
        fu.nc = lv.R.n;
        fu.rrp = lv.R.row.get();
        fu.rci = lv.R.col.get();
        fu.rv = rvals<VT>(lv.R);
        fu.fc = fc;
        if (slab1)
            launch_slab<VT>(c.stream, A, mt, A.n, B.prm.prerelax_sweeps - (s.zero ? 1 : 0),
                            s.zero, div_source(B.prm.relax_type), nullptr, f, s.x, s.x, fu);
        else
            launch_relax_block<VT>(c.stream, A, mt, divisor<VT>(lv, B.prm.relax_type), f, s.x,
                                   s.x, B.prm.prerelax_sweeps, s.zero, 1, 0, 1, nullptr, fu);
        s.zero = false;
        restricted = true;
    } else {
        relax_level<VT>(c, lv, mt, B.prm.relax_type, B.prm.prerelax_sweeps, f, s, nullptr, top);
    }
    if (!restricted) {
        const VT *rsrc = f;
        if (!s.zero) {
            /* a small level: residual and restriction in one launch */
            if (A.n <= SMALL_LEVEL_ROWS &&
                launch_resid_restrict<VT>(c.stream, A, mt, lv.R, s.x, f, fc)) {
                restricted = true;
            } else {
                launch_rows<VT>(c.stream, A, mt, OP_RESID, s.x, f, nullptr, W.res.get());
                rsrc = W.res.get();
            }
        }
        if (!restricted) launch_rows<VT>(c.stream, lv.R, rmt, OP_SPMV, rsrc, nullptr, nullptr, fc);
    }
    LevelState<VT> &sc = R.st[l];
    sc.zero = true;
    if (B.prm.cycle_type == 3 && l != L - 1) {
        kcycle_inner<VT>(R, l);
    } else {
        for (int i = 1; i <= B.num_grid_sweeps[l - 1]; i++) {
            cycle<VT>(R, l + 1);
            if (l == L - 1) break;
        }
    }
    bool prolong_in_block = false, prolong_in_sweep = false;
    int slab_m = 0, slab_n = 0; /* sweeps that a slab launch makes from x + P x_c */
    if (!sc.zero) {
        const bool fold = !lv.smoothed && B.prm.postrelax_sweeps > 0 && !timing;
        if (fold) slab_n = slab_plan<VT>(A, mt, B.prm.postrelax_sweeps, false, &slab_m);
        if (s.zero && !(fold && (blk || slab_n > 0))) {
            launch_fill<VT>(c.stream, A.n, VT(0), s.x);
            s.zero = false;
        }
        if (lv.smoothed) {
            /* x = x - (-P) x_c: the stored negated prolongator */
            launch_rows<VT>(c.stream, lv.Pneg, std::is_same<VT, double>::value ? MT_F64 : MT_F32,
                            OP_RESID, sc.x, s.x, nullptr, s.x2);
            std::swap(s.x, s.x2);
        } else if (slab_n > 0) {
            /* the prolongation folded into the first slab launch (below) */
        } else if (blk && B.prm.postrelax_sweeps > 0) {
            /* a one-workgroup level: the prolongation folded into the
               post-smoothing launch (below) */
            prolong_in_block = true;
        } else if (!blk && A.n <= SMALL_LEVEL_ROWS && B.prm.postrelax_sweeps > 0 &&
                   !(top && c.time_smoother) && rows_sequential<VT>(A)) {
            /* a small level: the prolongation folded into the first
               post-sweep (below) */
            prolong_in_sweep = true;
        } else if (top && post_lands_off(B.prm.postrelax_sweeps, s.x, s.x2, R.final_out) &&
                   !post_lands_off(B.prm.postrelax_sweeps, s.x2, s.x, R.final_out) && !blk) {
            /* into the other iterate: the post-smoothing's last sweep then
               writes the preconditioner's output itself (no copy after) */
            launch_prolong_to<VT>(c.stream, A.n, lv.agg.get(), pvals<VT>(lv), sc.x, s.x, s.x2);
            std::swap(s.x, s.x2);
        } else {
            launch_prolong<VT>(c.stream, A.n, lv.agg.get(), pvals<VT>(lv), sc.x, s.x);
        }
    }
    if (prolong_in_block) {
        BlockFuse<VT> fu;
        fu.agg = lv.agg.get();
        fu.p = pvals<VT>(lv);
        fu.xc = sc.x;
        VT *fo = top ? R.final_out : nullptr;
        VT *out = (fo && s.x != fo) ? fo : s.x;
        launch_relax_block<VT>(c.stream, A, mt, divisor<VT>(lv, B.prm.relax_type), f, s.x, out,
                               B.prm.postrelax_sweeps, s.zero, 1, 0, 1, nullptr, fu);
        if (out != s.x) {
            s.x2 = s.x;
            s.x = out;
        }
        s.zero = false;
        return;
    }
    if (slab_n > 0) {
        BlockFuse<VT> fu;
        fu.agg = lv.agg.get();
        fu.p = pvals<VT>(lv);
        fu.xc = sc.x;
        const int rest = B.prm.postrelax_sweeps - slab_n;
        VT *fo = top ? R.final_out : nullptr;
        VT *out = third_buffer<VT>(B, s, fo, rest);
        launch_slab<VT>(c.stream, A, mt, slab_m, slab_n, s.zero, div_source(B.prm.relax_type),
                        divisor<VT>(lv, B.prm.relax_type), f, s.x, out, fu);
        s.x2 = s.x;
        s.x = out;
        s.zero = false;
        relax_level<VT>(c, lv, mt, B.prm.relax_type, rest, f, s, fo, top);
        return;
    }
    if (prolong_in_sweep) {
        const int rest = B.prm.postrelax_sweeps - 1;
        VT *fo = top ? R.final_out : nullptr;
        VT *out = third_buffer<VT>(B, s, fo, rest);
        if (launch_jacobi_prolong<VT>(c.stream, A, mt, lv.agg.get(), pvals<VT>(lv), sc.x, s.x, f,
                                      divisor<VT>(lv, B.prm.relax_type), out)) {
            s.x2 = s.x;
            s.x = out;
            relax_level<VT>(c, lv, mt, B.prm.relax_type, rest, f, s, fo, top);
            return;
        }
        launch_prolong<VT>(c.stream, A.n, lv.agg.get(), pvals<VT>(lv), sc.x, s.x);
    }
    relax_level<VT>(c, lv, mt, B.prm.relax_type, B.prm.postrelax_sweeps, f, s,
                    top ? R.final_out : nullptr, top);
}

template <typename VT>
void run_hierarchy(Ctx &c, Boot &B, int k, std::vector<LevelState<VT>> &st, const VT *f0,
                   VT *final_out)
{
    CycleBufs<VT> &W = bufs<VT>(B);
    const Hierarchy &H = *B.H[k];
    for (int l = 1; l < H.num_levels(); l++) {
        st[l].x = W.xa[l].get();
        st[l].x2 = W.xb[l].get();
        st[l].zero = true;
    }
    CycleRun<VT> R{c, B, H, st, f0, final_out};
    cycle<VT>(R, 1);
}

/* composite preconditioner x <- B(r; x) (src/SOLVER/FCG.cu:112-187) in the
   compute type VT. When x_is_zero the content of x is treated as zero. */
template <typename VT>
void precond_apply_t(Ctx &c, Boot &B, const VT *r, VT *x, bool x_is_zero)
{
    CycleBufs<VT> &W = bufs<VT>(B);
    const int n = B.H[0]->L[0].mat().n;
    const int nh = (int)B.H.size();
    const size_t maxL = W.xa.size();
    std::vector<LevelState<VT>> st(maxL);
    if (B.prm.solver_type == 0 || B.prm.solver_type == 1) {
        st[0].x = x;
        st[0].x2 = W.xa[0].get();
        st[0].zero = x_is_zero;
        std::vector<int> order;
        for (int k = 0; k < nh; k++) order.push_back(k);
        if (B.prm.solver_type == 1)
            for (int k = nh - 1; k >= 0; k--) order.push_back(k);
        for (size_t t = 0; t < order.size(); t++) {
            const bool last = (t + 1 == order.size());
            run_hierarchy<VT>(c, B, order[t], st, r, last ? x : nullptr);
        }
        if (st[0].zero) {
            launch_fill<VT>(c.stream, n, VT(0), x);
        } else if (st[0].x != x) {
            launch_copy<VT>(c.stream, n, st[0].x, x);
        }
    } else {
        /* additive: every hierarchy starts from the same x; mean of results */
        W.xadd.ensure(n);
        W.xsave.ensure(n);
        launch_fill<VT>(c.stream, n, VT(0), W.xadd.get());
        if (!x_is_zero) launch_copy<VT>(c.stream, n, x, W.xsave.get());
        for (int k = 0; k < nh; k++) {
            st[0].x = W.xb[0].get();
            st[0].x2 = W.xa[0].get();
            st[0].zero = x_is_zero;
            if (!x_is_zero) launch_copy<VT>(c.stream, n, W.xsave.get(), st[0].x);
            run_hierarchy<VT>(c, B, k, st, r, nullptr);
            if (st[0].zero) launch_fill<VT>(c.stream, n, VT(0), st[0].x);
            launch_axpy<VT>(c.stream, n, VT(1), st[0].x, W.xadd.get());
        }
        launch_scale<VT>(c.stream, n, VT(1) / (VT)nh, W.xadd.get());
        launch_copy<VT>(c.stream, n, W.xadd.get(), x);
    }
}

template <typename VT>
void ensure_bufs(Boot &B, CycleBufs<VT> &W)
{
    size_t maxL = 0;
    for (auto &h : B.H) maxL = std::max(maxL, h->L.size());
    if (W.xa.size() < maxL) {
        W.xa.resize(maxL);
        W.xb.resize(maxL);
        W.f.resize(maxL);
    }
    for (size_t l = 0; l < maxL; l++) {
        size_t nl = 0;
        for (auto &h : B.H)
            if (l < h->L.size()) nl = std::max(nl, (size_t)h->L[l].mat().n);
        W.xa[l].ensure(nl);
        W.xb[l].ensure(nl);
        W.f[l].ensure(nl);
    }
    W.res.ensure(B.H[0]->L[0].mat().n);
    if (B.prm.cycle_type == 3) {
        for (auto *v : {&W.kw, &W.kd0, &W.kd1, &W.kv, &W.kv1}) {
            if (v->size() < maxL) v->resize(maxL);
            for (size_t l = 0; l < maxL; l++) {
                size_t nl = 0;
                for (auto &h : B.H)
                    if (l < h->L.size()) nl = std::max(nl, (size_t)h->L[l].mat().n);
                (*v)[l].ensure(nl);
            }
        }
    }
}

} // namespace

void Boot::drop_graphs()
{
    for (auto &g : gexec) {
        if (g) (void)hipGraphExecDestroy(g);
        g = nullptr;
    }
    graph_x = nullptr;
    drop_multi_graph(multi);
}

Boot::~Boot()
{
    drop_graphs();
    destroy_multi(multi);
}

void Boot::ensure_work()
{
    size_t maxL = 0;
    for (auto &h : H) maxL = std::max(maxL, h->L.size());
    kscal.ensure((maxL + 1) * KS_STRIDE);
    ensure_bufs<double>(*this, b64);
    if (prec != BCMG_PREC_FP64) {
        ensure_bufs<float>(*this, b32);
        const size_t n0 = H[0]->L[0].mat().n;
        r32.ensure(n0);
        z32.ensure(n0);
    }
}

double a_norm(Ctx &c, const DevCsr &A, const double *x, double *tmp)
{
    launch_rows(c.stream, A, OP_SPMV, x, nullptr, nullptr, tmp);
    c.red.ensure(1024 * 3 + 8);
    double *out = c.red.get() + 1024 * 3;
    launch_dots(c, A.n, 1, tmp, nullptr, nullptr, x, out);
    BCMG_HIP(hipMemcpyAsync(c.h_scalars, out, sizeof(double), hipMemcpyDeviceToHost, c.stream));
    BCMG_HIP(hipStreamSynchronize(c.stream));
    return std::sqrt(c.h_scalars[0]);
}

/* composite preconditioner on FP64 vectors; with a reduced-precision
   hierarchy r is rounded to FP32, the cycles run in FP32 and the result is
   widened back to FP64 */
void precond_apply(Ctx &c, Boot &B, const double *r, double *x, bool x_is_zero)
{
    if (B.prec == BCMG_PREC_FP64) {
        precond_apply_t<double>(c, B, r, x, x_is_zero);
        return;
    }
    const int n = B.H[0]->L[0].mat().n;
    launch_d2f(c.stream, n, r, B.r32.get());
    if (!x_is_zero) launch_d2f(c.stream, n, x, B.z32.get());
    precond_apply_t<float>(c, B, B.r32.get(), B.z32.get(), x_is_zero);
    launch_f2d(c.stream, n, B.z32.get(), x);
}

/* Convert the built hierarchy to the reduced-precision form: FP32 copies of
   every level's values (bfloat16 on levels >= 1 for BCMG_PREC_BF16), of the
   smoother divisors and of the prolongator values. */
void set_precision(Ctx &c, Boot &B, int prec)
{
    B.prec = prec;
    B.drop_graphs();
    if (prec == BCMG_PREC_FP64) return;
    /* level 0 (the caller's operator) and a hierarchy that several slots
       of the composite share are converted once */
    B.A0->make_lowp(c.stream, false);
    std::vector<const Hierarchy *> done;
    for (auto &Hp : B.H) {
        if (std::find(done.begin(), done.end(), Hp.get()) != done.end()) continue;
        done.push_back(Hp.get());
        Hierarchy &H = *Hp;
        for (int l = 0; l < H.num_levels(); l++) {
            Level &lv = H.L[l];
            DevCsr &A = l == 0 ? *B.A0 : lv.Aown;
            if (l > 0) A.make_lowp(c.stream, level_mt(B, l) == MT_BF16);
            const size_t n = A.n;
            if (lv.hasD) {
                lv.D32.ensure(n);
                launch_d2f(c.stream, n, lv.D.get(), lv.D32.get());
            }
            if (lv.hasM) {
                lv.M32.ensure(n);
                launch_d2f(c.stream, n, lv.M.get(), lv.M32.get());
            }
            if (l + 1 < H.num_levels()) {
                lv.p32.ensure(n);
                launch_d2f(c.stream, n, lv.p.get(), lv.p32.get());
                lv.R.make_lowp(c.stream, false);
                if (lv.smoothed) lv.Pneg.make_lowp(c.stream, false);
            }
        }
    }
    B.ensure_work();
    BCMG_HIP(hipStreamSynchronize(c.stream));
}

namespace {

/* src/BOOT/bootstrap.cu:5-44. The reference takes the A-norm after every
   one of the 15 applications, but only the last two enter the result (the
   ratio of the 15th to the 14th, and the scaling by the 15th), so only
   those are computed: the others are a SpMV, a product and a host wait
   each. The applications are the same launch sequence every time; from the
   second one on (the first has made every buffer) it is captured once as a
   HIP graph and replayed. */
void inner_iterations(Ctx &c, Boot &B, DBuf<double> &w)
{
    constexpr int IT = 15; /* bootBuildData::solver_it (src/AMG/AMG.cu:407) */
    const DevCsr &A = *B.A0;
    const int n = A.n;
    DBuf<double> x(n), rhs(n), tmp(n);
    launch_fill(c.stream, n, 1.0, x.get());
    launch_fill(c.stream, n, 0.0, rhs.get());
    /* direct launches: on the 128^3 bootstrap workload an application took
       0.93 ms either way, and capturing and instantiating its graph cost
       about 13 ms per bootstrap round, more than 15 replays could save */
    double normold = 0.0, normnew = 0.0, ratio = 1.0;
    for (int i = 1; i <= IT; i++) {
        precond_apply(c, B, rhs.get(), x.get(), false);
        if (i >= IT - 1) {
            normnew = a_norm(c, A, x.get(), tmp.get());
            if (i == IT) ratio = normnew / normold;
            normold = normnew;
        }
    }
    launch_scale(c.stream, n, 1. / normnew, x.get());
    launch_copy(c.stream, n, x.get(), w.get());
    BCMG_HIP(hipStreamSynchronize(c.stream));
    B.estimated_ratio = ratio;
}

} // namespace

/* src/BOOT/bootstrap.cu:46-90 with src/AMG/AMG.cu:426-448 */
void build_boot(Ctx &c, DevCsr &A, const bcmg_params &p, Boot &B)
{
    auto t0 = std::chrono::steady_clock::now();
    B.prm = p;
    B.A0 = &A;
    B.coarse_solver = p.coarse_solver;
    B.num_grid_sweeps = grid_sweeps(p.cycle_type, p.max_levels);
    SetupClock clk(c);
    BuildState bs;
    bs.clk = &clk;
    bs.maxcoarsesize = (int)(40 * std::pow((double)A.n, (double)1. / 3.));
    DBuf<double> w(A.n);
    launch_fill(c.stream, A.n, 1.0, w.get());
    B.estimated_ratio = 1.0;
    B.H.clear();
    B.ratio_after.clear();
    B.t_phase.clear();
    while (B.estimated_ratio > p.conv_ratio && (int)B.H.size() < p.max_hrc) {
        const int k = (int)B.H.size();
        clk.set_hierarchy(k);
        B.t_phase.emplace_back(PH_COUNT, 0.0);
        SetupClock::Scope ph(&clk, PH_HIER);
        if (k == 1) {
            /* no inner iterations follow the first hierarchy, so the second
               is built from the same w = 1 (src/BOOT/bootstrap.cu:68-75)
               and equals the first bit for bit: it shares its storage */
            B.H.push_back(B.H[0]);
        } else {
            B.H.push_back(std::make_shared<Hierarchy>());
            adaptive_coarsening(c, p, bs, A, w.get(), *B.H.back());
        }
        B.ensure_work();
        if (k > 0) {
            SetupClock::Scope in(&clk, PH_INNER);
            inner_iterations(c, B, w);
        }
        B.ratio_after.push_back(B.estimated_ratio);
    }
    B.ensure_work();
    const int n = A.n;
    B.v.ensure(n);
    B.w.ensure(n);
    B.d.ensure(n);
    B.q.ensure(n);
    B.r.ensure(n);
    B.scal.ensure(16);
    c.ensure_reductions(n);
    BCMG_HIP(hipStreamSynchronize(c.stream));
    clk.collect(B);
    B.t_setup_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
}

/* FCG v3 from x0 = 0 (src/SOLVER/FCG.cu:433-585) */
int fcg_solve(Ctx &c, Boot &B, const double *b, double *x, int *iters, double *resid,
              double *delta0_out)
{
    const DevCsr &A = *B.A0;
    const int n = A.n;
    double *scal = B.scal.get();
    double *v = B.v.get(), *w = B.w.get(), *d = B.d.get(), *q = B.q.get(), *r = B.r.get();
    /* scratch of the fused reductions; graphs hold its address */
    c.ensure_reductions(n);
    /* K-cycle breakdown flags (the reference exits on them) start clear */
    const bool kcyc = B.prm.cycle_type == 3;
    if (kcyc) {
        launch_fill<double>(c.stream, (int)B.kscal.n, 0.0, B.kscal.get());
        c.h_scalars[9] = 0.0;
    }
    /* x0 = 0: r = b - A 0 = b */
    launch_copy(c.stream, n, b, r);
    launch_fill(c.stream, n, 0.0, x);
    launch_dots(c, n, 1, r, nullptr, nullptr, r, scal + 7);
    BCMG_HIP(hipMemcpyAsync(c.h_scalars, scal + 7, sizeof(double), hipMemcpyDeviceToHost, c.stream));
    BCMG_HIP(hipStreamSynchronize(c.stream));
    const double delta0 = std::sqrt(c.h_scalars[0]);
    const double rhs_norm = delta0;
    if (delta0_out) *delta0_out = delta0;
    if (delta0 <= DBL_EPSILON * rhs_norm) {
        if (iters) *iters = 0;
        throw Error(BCMG_EZERORHS, "initial residual is zero (the reference exits)");
    }
    precond_apply(c, B, r, v, true);
    launch_spmv_dots<double>(c, A, 2, v, w, r, nullptr, scal);
    launch_fcg_first(c, n, scal, v, x, w, r);
    /* A reduced-precision iteration keeps r and z in the cycle's FP32 where
       the cycle meets FCG: the update writes r rounded beside r, the product
       and the update widen z as they read it (no conversion passes). */
    const bool z32 = B.prec != BCMG_PREC_FP64 && rows_sequential<double>(A);
    if (z32) launch_d2f(c.stream, n, r, B.r32.get());
    /* d, q take the first direction; the next one goes to the other pair */
    std::swap(v, d);
    std::swap(w, q);
    const double rtol = B.prm.rtol;
    const int max_iter = B.prm.itnlim;
    /* one FCG iteration (src/SOLVER/FCG.cu:497-565): preconditioner into the
       free direction slot, A z, the three products, the scalar recurrence,
       both merged axpys and ||r||, which is copied to pinned host memory */
    auto enqueue_iteration = [&](bool even) {
        double *z = even ? v : d;
        double *t = even ? w : q;
        const double *zo = even ? d : v;
        const double *to = even ? q : w;
        if (z32) {
            precond_apply_t<float>(c, B, B.r32.get(), B.z32.get(), true);
            launch_spmv_dots<float>(c, A, 3, B.z32.get(), t, r, to, scal);
            launch_fcg_update<float>(c, n, scal, zo, B.z32.get(), z, x, to, t, r, B.r32.get());
        } else {
            precond_apply(c, B, r, z, true);
            launch_spmv_dots<double>(c, A, 3, z, t, r, to, scal);
            launch_fcg_update<double>(c, n, scal, zo, z, z, x, to, t, r, nullptr);
        }
        BCMG_HIP(hipMemcpyAsync(c.h_scalars + 8, scal + 6, sizeof(double), hipMemcpyDeviceToHost,
                                c.stream));
        if (kcyc)
            BCMG_HIP(hipMemcpyAsync(c.h_scalars + 9, B.kscal.get() + KS_FLAG_GLOBAL,
                                    sizeof(double), hipMemcpyDeviceToHost, c.stream));
    };
    /* The iteration is the same launch sequence every time (two variants for
       the alternating direction slots), so it is captured once per composite
       and output vector as a HIP graph and replayed: the kernels then go out
       without per-launch host work. A composite's first solve launches
       directly: capturing and instantiating the graphs costs more than a
       solve's replays save on small operators (a setup-and-solve call pays
       it once), while repeated solves on a kept composite replay them. Event
       timing of the smoother needs the plain launches. */
    const bool graphs = c.use_graphs && !c.time_smoother && B.fcg_calls++ > 0;
    if (graphs && (B.graph_x != x || B.graph_red != c.red.get())) B.drop_graphs();
    B.restarts = 0;
    int iter = 0;  /* iterations after the first step, restarts included */
    int phase = 0; /* iterations since the last (re)start: selects the slot pair */
    double l2 = 0.0;
    bool run_loop = true;
    for (;;) {
        if (run_loop) do {
            const bool even = (phase % 2) == 0;
            if (graphs) {
                hipGraphExec_t &ge = B.gexec[even ? 0 : 1];
                if (!ge) {
                    hipGraph_t g = nullptr;
                    BCMG_HIP(hipStreamBeginCapture(c.stream, hipStreamCaptureModeThreadLocal));
                    try {
                        enqueue_iteration(even);
                    } catch (...) {
                        (void)hipStreamEndCapture(c.stream, &g);
                        if (g) (void)hipGraphDestroy(g);
                        throw;
                    }
                    BCMG_HIP(hipStreamEndCapture(c.stream, &g));
                    const hipError_t e = hipGraphInstantiate(&ge, g, nullptr, nullptr, 0);
                    (void)hipGraphDestroy(g);
                    BCMG_HIP(e);
                    B.graph_x = x;
                    B.graph_red = c.red.get();
                }
                BCMG_HIP(hipGraphLaunch(ge, c.stream));
            } else {
                enqueue_iteration(even);
            }
            BCMG_HIP(hipStreamSynchronize(c.stream));
            l2 = c.h_scalars[8];
            if (kcyc && c.h_scalars[9] != 0.0)
                throw Error(BCMG_EBREAKDOWN, "K-cycle inner iteration: indefinite preconditioner "
                                             "or matrix (the reference exits, FCG.cu:625-643)");
            iter++;
            phase++;
        } while (l2 > rtol * delta0 && iter < max_iter);
        /* With a reduced-precision hierarchy the recursively updated r can
           drift from b - A x; the stopping test is then confirmed on the
           true residual, and FCG restarts from it (first step again, same
           slot pairs) while it is above the tolerance. FP64 keeps the
           reference's recursive test unchanged. */
        if (B.prec == BCMG_PREC_FP64 || !std::isfinite(l2)) break;
        launch_true_residual(c, A, b, x, v, r, scal);
        BCMG_HIP(hipMemcpyAsync(c.h_scalars + 8, scal + 6, sizeof(double), hipMemcpyDeviceToHost,
                                c.stream));
        BCMG_HIP(hipStreamSynchronize(c.stream));
        l2 = c.h_scalars[8];
        if (l2 <= rtol * delta0 || iter >= max_iter || !std::isfinite(l2)) break;
        B.restarts++;
        precond_apply(c, B, r, d, true);
        launch_spmv_dots<double>(c, A, 2, d, q, r, nullptr, scal);
        launch_fcg_first(c, n, scal, d, x, q, r);
        if (z32) launch_d2f(c.stream, n, r, B.r32.get());
        BCMG_HIP(hipMemcpyAsync(c.h_scalars + 8, scal + 6, sizeof(double), hipMemcpyDeviceToHost,
                                c.stream));
        BCMG_HIP(hipStreamSynchronize(c.stream));
        l2 = c.h_scalars[8];
        iter++;
        phase = 0;
        /* a restart that already meets the test, or the limit, goes straight
           to the true-residual check */
        run_loop = l2 > rtol * delta0 && iter < max_iter;
    }
    if (iters) *iters = iter + 1;
    if (resid) *resid = l2;
    if (!std::isfinite(l2)) throw Error(BCMG_EBREAKDOWN, "non-finite residual");
    return BCMG_OK;
}

void Ctx::ensure_reductions(int n) { red.ensure(red_size_for(n)); }

hipEvent_t Ctx::next_event()
{
    if (ev_used == ev_pool.size()) {
        hipEvent_t e;
        BCMG_HIP(hipEventCreate(&e));
        ev_pool.push_back(e);
    }
    return ev_pool[ev_used++];
}

Ctx::~Ctx()
{
    for (auto e : ev_pool) (void)hipEventDestroy(e);
    if (h_scalars) (void)hipHostFree(h_scalars);
    if (h_ints) (void)hipHostFree(h_ints);
    red.release();
    iscratch.release();
    if (stream && own_stream) (void)hipStreamDestroy(stream);
}

} // namespace bcmg
