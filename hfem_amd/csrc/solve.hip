// Host side of the trace-system solver and of the Newton / DIRK drivers
// (declared in include/hfem_amd.h).  The reference binds GMRES, the
// preconditioner and the ordering from closed libraries (solvers/dgsolvers.cpp:16-20);
// their semantics here follow its MATLAB specifications (kernel/gmres_bilu0.m,
// computeBILU0.m, applyBILU0.m, computeMDFordering.m, mkBlockJacobi.m).  The
// drivers follow solveNonlinearProblem and solveUnsteadyProblem
// (solvers/dgsolvers.cpp:142-205, :221-444) with status codes in place of exit().
#include <algorithm>
#include <chrono>
#include <climits>
#include <cmath>
#include <utility>
#include <vector>

#include "ctx.h"

#define RC(x)                  \
    do {                       \
        int rc_ = (x);         \
        if (rc_) return rc_;   \
    } while (0)

static double now_ms()
{
    return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

static long trace_len(hfem_ctx *c) { return (long)c->hd.nf * c->d.nch * c->d.npf; }
static int trace_bsz(hfem_ctx *c) { return c->d.nch * c->d.npf; }

// Vectors and work arrays of the solver, allocated on first use.
static int ensure_vectors(hfem_ctx *c, int restart)
{
    SolverState &s = c->sv;
    const long N = trace_len(c);
    if (!s.x) HIPCHK(hfem_dalloc(&s.x, N));
    if (!s.b) HIPCHK(hfem_dalloc(&s.b, N));
    if (!s.t) HIPCHK(hfem_dalloc(&s.t, N));
    if (!s.d_info) HIPCHK(hfem_dalloc(&s.d_info, (size_t)c->hd.nf));
    for (auto &e : s.ev)
        if (!e) HIPCHK(hipEventCreate(&e));
    const size_t cols = (size_t)restart + 1;
    if (cols > (size_t)s.vcols) {
        // (no columns until all four are there, so that a call after a failed one tries again)
        auto release = [&] {
            s.vcols = 0;
            for (double **p : {&s.V, &s.dots, &s.coef}) {
                if (*p) (void)hipFree(*p);
                *p = nullptr;
            }
            if (s.h_dots) (void)hipHostFree(s.h_dots);
            s.h_dots = nullptr;
        };
        release();
        hipError_t e = hfem_dalloc(&s.V, N * cols);
        if (e == hipSuccess) e = hfem_dalloc(&s.dots, 2 * (size_t)gs_blocks(N) * cols);
        if (e == hipSuccess) e = hipHostMalloc((void **)&s.h_dots, sizeof(double) * (2 * cols + 1), hipHostMallocDefault);
        if (e == hipSuccess) e = hfem_dalloc(&s.coef, cols + 1);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            release();
            return hfem_fail(-2, "no memory for a Krylov basis of %zu vectors of %ld entries: %s", cols, N, hipGetErrorString(e));
        }
        s.vcols = (int)cols;
    }
    return 0;
}

static int require_system(hfem_ctx *c, const char *who)
{
    if (!c) return hfem_fail(-1, "%s: null context", who);
    if (!c->has_mesh) return hfem_fail(-3, "%s: mesh not set", who);
    return 0;
}

// ---------------------------------------------------------------- ordering

// Level schedules of the two BILU0 sweeps for the current ordering: a row's
// forward level is one more than the largest forward level of its neighbours
// numbered before it, its backward level likewise over the neighbours numbered
// after it.  Rows of one level never depend on each other.  Neighbours in the forward
// levels are the rows with a block on either side of the diagonal (a mesh's graph has
// both, a caller's need not): two rows with one differ in level by the order of their
// numbers, so a row that has both as neighbours may take them by level (ensure_schedule).
static int build_levels(hfem_ctx *c)
{
    SolverState &s = c->sv;
    const int n = c->hd.nf;
    const std::vector<int> &rp = s.rowpts, &ci = s.colind;
    std::vector<int> lv(n, 0), uv(n, 0);
    int nl = 0, nu = 0;
    for (int j = 0; j < n; j++) {
        const int r = s.o2u[j];
        int l = lv[r];
        for (int k = rp[r] + 1; k < rp[r + 1]; k++)
            if (s.u2o[ci[k]] < j) l = std::max(l, lv[ci[k]] + 1);
        lv[r] = l;
        nl = std::max(nl, l + 1);
        for (int k = rp[r] + 1; k < rp[r + 1]; k++)
            if (s.u2o[ci[k]] > j) lv[ci[k]] = std::max(lv[ci[k]], l + 1);
    }
    for (int j = n - 1; j >= 0; j--) {
        const int r = s.o2u[j];
        int l = 0;
        for (int k = rp[r] + 1; k < rp[r + 1]; k++)
            if (s.u2o[ci[k]] > j) l = std::max(l, uv[ci[k]] + 1);
        uv[r] = l;
        nu = std::max(nu, l + 1);
    }
    auto bucket = [&](const std::vector<int> &lev, int nlev, std::vector<int> &ptr, std::vector<int> &rows) {
        ptr.assign(nlev + 1, 0);
        for (int r = 0; r < n; r++) ptr[lev[r] + 1]++;
        for (int l = 0; l < nlev; l++) ptr[l + 1] += ptr[l];
        rows.assign(n, 0);
        std::vector<int> fill(ptr.begin(), ptr.end() - 1);
        for (int j = 0; j < n; j++) {                 // rows of a level in ordering sequence
            const int r = s.o2u[j];
            rows[fill[lev[r]]++] = r;
        }
    };
    bucket(lv, nl, s.lptr, s.lrows);
    bucket(uv, nu, s.uptr, s.urows);
    s.llev = std::move(lv);
    s.ulev = std::move(uv);
    s.sched_valid = false;
    s.prec = -2;                                       // factors belong to the previous ordering
    return 0;
}

// The ordering and the schedules of the BILU0 kernels on the device, for the current
// ordering (block-Jacobi needs none of them).
static int ensure_schedule(hfem_ctx *c)
{
    SolverState &s = c->sv;
    const bool fp32 = s.prec_fp32 != 0;
    if (s.sched_valid && (s.fnbr_valid || !fp32)) return 0;
    const int n = c->hd.nf;
    const std::vector<int> &rp = s.rowpts, &ci = s.colind;
    // the sweeps' rows in level order, each with the neighbours it reads by increasing
    // level (the last to be ready last)
    auto schedule = [&](const std::vector<int> &rows, const std::vector<int> &lev, bool lower, std::vector<int4> &sched,
                        std::vector<int2> &nbr) {
        sched.resize(n);
        nbr.clear();
        nbr.reserve(ci.size() / 2 + 1);
        for (int t = 0; t < n; t++) {
            const int r = rows[t], first = (int)nbr.size();
            for (int k = rp[r] + 1; k < rp[r + 1]; k++)
                if (lower ? s.u2o[ci[k]] < s.u2o[r] : s.u2o[ci[k]] > s.u2o[r]) nbr.push_back(make_int2(k, ci[k]));
            std::sort(nbr.begin() + first, nbr.end(), [&](const int2 &a, const int2 &b) {
                return lev[a.y] != lev[b.y] ? lev[a.y] < lev[b.y] : s.u2o[a.y] < s.u2o[b.y];
            });
            sched[t] = make_int4(r, rp[r], first, (int)nbr.size() - first);
        }
    };
    std::vector<int4> sched;
    std::vector<int2> nbr;
    // (each list of neighbours holds at most every off-diagonal block)
    auto upload = [&](int4 **d_sched, int2 **d_nbr) -> int {
        if (d_sched) {
            if (!*d_sched) HIPCHK(hfem_dalloc(d_sched, (size_t)n));
            HIPCHK(hipMemcpy(*d_sched, sched.data(), sizeof(int4) * n, hipMemcpyHostToDevice));
        }
        if (!*d_nbr) HIPCHK(hfem_dalloc(d_nbr, ci.size()));
        HIPCHK(hipMemcpy(*d_nbr, nbr.data(), sizeof(int2) * nbr.size(), hipMemcpyHostToDevice));
        return 0;
    };
    if (!s.sched_valid) {
        schedule(s.urows, s.ulev, false, sched, nbr);
        RC(upload(&s.d_usched, &s.d_unbr));
    }
    schedule(s.lrows, s.llev, true, sched, nbr);
    if (!s.sched_valid) {
        RC(upload(&s.d_lsched, &s.d_lnbr));
        if (!s.d_u2o) HIPCHK(hfem_dalloc(&s.d_u2o, (size_t)n));
        HIPCHK(hipMemcpy(s.d_u2o, s.u2o.data(), sizeof(int) * n, hipMemcpyHostToDevice));
        s.sched_valid = true;
        s.fnbr_valid = false;
    }
    // The single-precision factorisation's by increasing number: the order of a target's
    // updates, and with it the roundings, which can grow along the rows (solver.hip), then
    // do not depend on the levels.  In double precision, where they are far below the
    // solver's tolerances, by level: 27 ms against 29 on 16 464 p=3 tets.
    if (fp32) {
        for (const int4 &h : sched)
            std::sort(nbr.begin() + h.z, nbr.begin() + h.z + h.w,
                      [&](const int2 &a, const int2 &b) { return s.u2o[a.y] < s.u2o[b.y]; });
        RC(upload(nullptr, &s.d_fnbr));
        s.fnbr_valid = true;
    }
    return 0;
}

// Approximate minimum discarded fill (kernel/computeMDFordering.m): weight of row k
// = Frobenius norm of C(ik) C(kj) over pairs of distinct unnumbered neighbours
// ri, rj of k that are not neighbours of each other.
// A greedy order is a chain on the host: every row numbered changes its neighbours'
// weights, and the next is the lightest.  Per off-diagonal block e = (k, ri), from the mesh
// alone: rev, the position of (ri, k); far, which of row k's other blocks (bit j - rp[k] - 1)
// have columns that are not neighbours of ri, 64 bits a word.  live: a row's unnumbered
// neighbours likewise.
struct MdfRows {
    const std::vector<int> &rp, &ci;
    std::vector<int> rev, word;                 // word: a row's words in live; a block's in far are alike
    std::vector<unsigned long long> far, live;
    std::vector<long> fat;                      // a block's first word in far
    MdfRows(const std::vector<int> &rp_, const std::vector<int> &ci_) : rp(rp_), ci(ci_)
    {
        const int n = (int)rp.size() - 1;
        rev.assign(ci.size(), -1);
        fat.assign(ci.size(), 0);
        word.assign(n + 1, 0);
        long nf = 0;
        for (int k = 0; k < n; k++) {
            const int len = rp[k + 1] - rp[k] - 1, nw = (len + 63) / 64;
            word[k + 1] = word[k] + nw;
            for (int e = rp[k] + 1; e < rp[k + 1]; e++, nf += nw) fat[e] = nf;
        }
        live.assign(word[n], 0);
        far.assign(nf, 0);
        std::vector<int> owner(n, -1), place(n, 0), twin;   // twin: an earlier block of the same column
        for (int k = 0; k < n; k++) {
            const int d = rp[k] + 1, len = rp[k + 1] - d, nw = word[k + 1] - word[k];
            twin.assign(len, -1);
            for (int j = 0; j < len; j++) {
                const int c = ci[d + j];
                if (owner[c] == k) twin[j] = place[c];
                owner[c] = k;
                place[c] = j;
                live[word[k] + j / 64] |= 1ull << (j & 63);
            }
            for (int i = 0; i < len; i++) {
                unsigned long long *f = &far[fat[d + i]];
                std::copy(&live[word[k]], &live[word[k]] + nw, f);
                const int ri = ci[d + i];
                for (int m = rp[ri]; m < rp[ri + 1]; m++) {   // (ri itself, the diagonal, first)
                    for (int j = owner[ci[m]] == k ? place[ci[m]] : -1; j >= 0; j = twin[j]) f[j / 64] &= ~(1ull << (j & 63));
                    if (ci[m] == k && rev[d + i] < 0) rev[d + i] = m;
                }
            }
        }
    }
    double weight(const std::vector<double> &C, int k) const
    {
        const int d = rp[k] + 1, nw = word[k + 1] - word[k];
        const unsigned long long *lv = &live[word[k]];
        double s = 0.0;
        for (int wi = 0; wi < nw; wi++)
            for (unsigned long long bi = lv[wi]; bi; bi &= bi - 1) {
                const int i = 64 * wi + __builtin_ctzll(bi);
                const double a = rev[d + i] < 0 ? 0.0 : C[rev[d + i]];
                const unsigned long long *f = &far[fat[d + i]];
                for (int wj = 0; wj < nw; wj++)
                    for (unsigned long long bj = f[wj] & lv[wj]; bj; bj &= bj - 1) {
                        const double dc = a * C[d + 64 * wj + __builtin_ctzll(bj)];
                        s += dc * dc;
                    }
            }
        return std::sqrt(s);
    }
    // Row p has been numbered: it leaves the live neighbours of row k.
    void leave(int p, int k)
    {
        for (int m = rp[k] + 1; m < rp[k + 1]; m++)
            if (ci[m] == p) live[word[k] + (m - rp[k] - 1) / 64] &= ~(1ull << ((m - rp[k] - 1) & 63));
    }
};

// The lightest row, the lowest on ties (MATLAB's min, computeMDFordering.m:93), out of a
// tree of pairwise winners: a changed weight is carried up while it changes a winner.
// (16 464 p=3 tets, 34 104 rows: ordering on the host 27 ms with a balanced tree of all
// weights and the neighbours searched at every weight, 11 ms now; 4 410 rows 3.2 and 1.4.)
struct MdfTree {
    int base;
    std::vector<int> win;       // winners; leaf of row k at base + k; -1: none left
    const std::vector<double> &w;
    MdfTree(int n, const std::vector<double> &w_) : w(w_)
    {
        for (base = 1; base < n; base *= 2) {}
        win.assign(2 * base, -1);
        for (int k = 0; k < n; k++) win[base + k] = k;
        for (int q = base - 1; q > 0; q--) win[q] = better(win[2 * q], win[2 * q + 1]);
    }
    int better(int a, int b) const { return a < 0 ? b : b < 0 ? a : w[b] < w[a] ? b : a; }
    int lightest() const { return win[1]; }
    // after w[k] has changed, or (gone) to take k out
    void update(int k, bool gone)
    {
        int q = base + k;
        if (gone) win[q] = -1;
        for (q /= 2; q > 0; q /= 2) {
            const int b = better(win[2 * q], win[2 * q + 1]);
            if (b == win[q] && b != k) break;
            win[q] = b;
        }
    }
};

extern "C" int hfem_compute_ordering(hfem_ctx *c, int method)
{
    RC(require_system(c, "hfem_compute_ordering"));
    if (method != 0 && method != 1) return hfem_fail(-1, "hfem_compute_ordering: method %d (0 natural, 1 MDF)", method);
    HIPCHK(hipSetDevice(c->device));
    const double t0 = now_ms();
    SolverState &s = c->sv;
    const int n = c->hd.nf, bsz = trace_bsz(c);
    s.o2u.resize(n);
    s.u2o.resize(n);
    if (method == 0) {
        for (int i = 0; i < n; i++) s.o2u[i] = s.u2o[i] = i;
    } else {
        RC(ensure_vectors(c, 1));
        const long b2 = (long)bsz * bsz;
        if (!s.Dinv) HIPCHK(hfem_dalloc(&s.Dinv, (size_t)n * b2));
        if (!s.Cw) HIPCHK(hfem_dalloc(&s.Cw, (size_t)c->nblocks));
        HIPCHK(launch_block_inverse(n, bsz, c->rowstart, c->Hg, s.Dinv, s.d_info, c->stream));
        HIPCHK(launch_mdf_weights(n, bsz, c->rowstart, c->Hg, s.Dinv, s.Cw, c->stream));
        MdfRows mdf(s.rowpts, s.colind);   // (while the device forms the weights)
        std::vector<double> Cw(c->nblocks);
        std::vector<int> info(n);
        HIPCHK(hipMemcpyAsync(Cw.data(), s.Cw, sizeof(double) * Cw.size(), hipMemcpyDeviceToHost, c->stream));
        HIPCHK(hipMemcpyAsync(info.data(), s.d_info, sizeof(int) * n, hipMemcpyDeviceToHost, c->stream));
        HIPCHK(hipStreamSynchronize(c->stream));
        for (int i = 0; i < n; i++)
            if (info[i]) return hfem_fail(-4, "hfem_compute_ordering: diagonal block of row %d is singular", i);
        std::vector<double> w(n);
        std::vector<char> numbered(n, 0);
        for (int k = 0; k < n; k++) w[k] = mdf.weight(Cw, k);
        MdfTree tree(n, w);
        for (int l = 0; l < n; l++) {
            const int p = tree.lightest();
            tree.update(p, true);
            s.o2u[l] = p;
            numbered[p] = 1;
            for (int e = s.rowpts[p] + 1; e < s.rowpts[p + 1]; e++) {
                const int k = s.colind[e];
                if (numbered[k]) continue;
                mdf.leave(p, k);
                w[k] = mdf.weight(Cw, k);
                tree.update(k, false);
            }
        }
        for (int l = 0; l < n; l++) s.u2o[s.o2u[l]] = l;
    }
    s.order_method = method;
    RC(build_levels(c));
    s.ms_order = now_ms() - t0;
    return 0;
}

extern "C" int hfem_set_ordering(hfem_ctx *c, const int *o2u)
{
    RC(require_system(c, "hfem_set_ordering"));
    if (!o2u) return hfem_fail(-1, "hfem_set_ordering: null ordering");
    HIPCHK(hipSetDevice(c->device));
    SolverState &s = c->sv;
    const int n = c->hd.nf;
    std::vector<int> u2o(n, -1);
    for (int l = 0; l < n; l++) {
        if (o2u[l] < 0 || o2u[l] >= n || u2o[o2u[l]] >= 0)
            return hfem_fail(-1, "hfem_set_ordering: not a permutation of 0..%d", n - 1);
        u2o[o2u[l]] = l;
    }
    s.o2u.assign(o2u, o2u + n);
    s.u2o = u2o;
    s.order_method = 3;
    return build_levels(c);
}

extern "C" int hfem_get_ordering(hfem_ctx *c, int *o2u, int *nlevels)
{
    RC(require_system(c, "hfem_get_ordering"));
    const SolverState &s = c->sv;
    if (s.order_method < 0) return hfem_fail(-3, "hfem_get_ordering: no ordering computed");
    if (o2u) std::copy(s.o2u.begin(), s.o2u.end(), o2u);
    if (nlevels) {
        nlevels[0] = (int)s.lptr.size() - 1;
        nlevels[1] = (int)s.uptr.size() - 1;
    }
    return 0;
}

// ---------------------------------------------------------------- preconditioner

static int ensure_syncfree(hfem_ctx *c);
static int check_syncfree(hfem_ctx *c, const char *who);

extern "C" int hfem_precond_factor(hfem_ctx *c, int kind)
{
    RC(require_system(c, "hfem_precond_factor"));
    if (kind != -1 && kind != 0 && kind != 2)
        return hfem_fail(-1, "hfem_precond_factor: kind %d (-1 none, 0 BILU0, 2 block-Jacobi)", kind);
    HIPCHK(hipSetDevice(c->device));
    const double t0 = now_ms();
    SolverState &s = c->sv;
    RC(ensure_vectors(c, 1));
    const int n = c->hd.nf, bsz = trace_bsz(c);
    const long b2 = (long)bsz * bsz;
    if (kind == -1) {
        s.prec = -1;
        return 0;
    }
    if ((size_t)(kind == 0 ? bilu0_factor_lds(bsz) : block_inverse_lds(bsz)) > (size_t)c->maxlds)
        return hfem_fail(-1, "hfem_precond_factor: block size %d needs more LDS than the device offers", bsz);
    const bool fp32 = s.prec_fp32 != 0;
    s.prec = -2;   // until this factorisation has succeeded
    if (!fp32 && !s.Mg) HIPCHK(hfem_dalloc(&s.Mg, (size_t)c->nblocks * b2));
    if (fp32 && !s.Mg32) HIPCHK(hfem_dalloc(&s.Mg32, (size_t)c->nblocks * b2));
    if (kind == 2) {
        // block-Jacobi: inverses in FP64; single-precision factors are their FP32 copies
        if (!fp32) HIPCHK(launch_block_inverse(n, bsz, c->rowstart, c->Hg, s.Mg, s.d_info, c->stream));
        else {
            if (!s.Mg) HIPCHK(hfem_dalloc(&s.Mg, (size_t)c->nblocks * b2));
            HIPCHK(launch_block_inverse(n, bsz, c->rowstart, c->Hg, s.Mg, s.d_info, c->stream));
            HIPCHK(launch_to_float((long)n * b2, s.Mg, s.Mg32, c->stream));
        }
    } else {
        if (s.order_method < 0) RC(hfem_compute_ordering(c, 1));
        RC(ensure_schedule(c));
        // (sync-free: one persistent launch over the rows in forward-level order;
        // else one launch per level)
        if (s.sweep_mode == 1) RC(ensure_syncfree(c));
        unsigned *sync = s.sweep_mode == 1 ? s.sf_flags + (size_t)n : nullptr;
        if (!fp32) {
            HIPCHK(hipMemcpyAsync(s.Mg, c->Hg, sizeof(double) * c->nblocks * b2, hipMemcpyDeviceToDevice, c->stream));
            if (s.sweep_mode == 1)
                HIPCHK(launch_bilu0_factor_syncfree(bsz, c->rowstart, c->cols, s.d_u2o, s.d_lsched, s.d_lnbr, n, s.Mg, s.d_info,
                                                    s.sf_flags, sync, s.sweep_wgs, s.spin_limit, s.sf_err, c->stream));
            else
                for (size_t l = 0; l + 1 < s.lptr.size(); l++)
                    HIPCHK(launch_bilu0_factor_level(bsz, c->rowstart, c->cols, s.d_u2o, s.d_lsched, s.d_lnbr,
                                                     s.lptr[l], s.lptr[l + 1], s.Mg, s.d_info, c->stream));
        } else {
            // single precision (precPrecision 0): Hg rounded to FP32 and factored on
            // the FP32 MFMA
            HIPCHK(launch_to_float((long)c->nblocks * b2, c->Hg, s.Mg32, c->stream));
            if (s.sweep_mode == 1)
                HIPCHK(launch_bilu0_factor_syncfree(bsz, c->rowstart, c->cols, s.d_u2o, s.d_lsched, s.d_fnbr, n, s.Mg32,
                                                    s.d_info, s.sf_flags, sync, s.sweep_wgs, s.spin_limit, s.sf_err,
                                                    c->stream));
            else
                for (size_t l = 0; l + 1 < s.lptr.size(); l++)
                    HIPCHK(launch_bilu0_factor_level(bsz, c->rowstart, c->cols, s.d_u2o, s.d_lsched, s.d_fnbr,
                                                     s.lptr[l], s.lptr[l + 1], s.Mg32, s.d_info, c->stream));
        }
    }
    if (kind != 2) {
        // the sweeps' form of the upper blocks
        if (!fp32) HIPCHK(launch_bilu0_scale_upper(bsz, n, c->rowstart, c->cols, s.d_u2o, s.Mg, c->stream));
        else HIPCHK(launch_bilu0_scale_upper(bsz, n, c->rowstart, c->cols, s.d_u2o, s.Mg32, c->stream));
    }
    std::vector<int> info(n);
    HIPCHK(hipMemcpyAsync(info.data(), s.d_info, sizeof(int) * n, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    RC(check_syncfree(c, "hfem_precond_factor"));
    for (int i = 0; i < n; i++) {
        if (info[i] < 0)
            return hfem_fail(-4, "hfem_precond_factor: row %d has %d blocks, more than the factorisation takes", i,
                             -info[i]);
        if (info[i]) return hfem_fail(-4, "hfem_precond_factor: singular pivot block in row %d", i);
    }
    s.prec = kind;
    s.graph_dirty = true;
    s.ms_factor = now_ms() - t0;
    return 0;
}

// sys.precPrecision (preprocessing/initializestructs.cpp:476-486): 0 single-precision
// preconditioner factors (Mg_sp), 1 double.  Takes effect at the next factorisation.
extern "C" int hfem_set_precond_precision(hfem_ctx *c, int prec_precision)
{
    if (!c) return hfem_fail(-1, "hfem_set_precond_precision: null context");
    if (prec_precision != 0 && prec_precision != 1)
        return hfem_fail(-1, "hfem_set_precond_precision: %d (0 single, 1 double)", prec_precision);
    if ((prec_precision == 0) != (c->sv.prec_fp32 != 0)) c->sv.prec = -2;   // factors of the other precision are stale
    c->sv.prec_fp32 = prec_precision == 0;
    return 0;
}

// Buffers of the sync-free sweeps, allocated and cleared at their first use (before
// any graph capture: the clearing is a memset).
static int ensure_syncfree(hfem_ctx *c)
{
    SolverState &s = c->sv;
    const int n = c->hd.nf;
    if (s.lptr.empty() || s.lptr.back() != n || s.uptr.empty() || s.uptr.back() != n)
        return hfem_fail(-3, "sync-free BILU0 sweeps: the level lists do not cover the %d rows", n);
    if (!s.sf_flags) {
        HIPCHK(hfem_dalloc(&s.sf_flags, (size_t)n + 3));
        HIPCHK(hipMemset(s.sf_flags, 0, sizeof(unsigned) * ((size_t)n + 3)));
    }
    if (!s.sf_err) {
        HIPCHK(hfem_dalloc(&s.sf_err, 1));
        HIPCHK(hipMemset(s.sf_err, 0, sizeof(int)));
    }
    return 0;
}

// Whether a bounded wait of the sync-free sweeps gave up since the last check (the
// applications since then are invalid); clears the flag.  Synchronises the stream.
static int check_syncfree(hfem_ctx *c, const char *who)
{
    SolverState &s = c->sv;
    if (!s.sf_err) return 0;
    int e = 0;
    HIPCHK(hipStreamSynchronize(c->stream));
    HIPCHK(hipMemcpy(&e, s.sf_err, sizeof(int), hipMemcpyDeviceToHost));
    if (!e) return 0;
    HIPCHK(hipMemset(s.sf_err, 0, sizeof(int)));
    return hfem_fail(-5, "%s: a wait of the sync-free BILU0 sweeps gave up after %d polls; the preconditioner "
                     "applications are invalid", who, s.spin_limit);
}

// The two BILU0 sweeps: forward into s.t, backward into y; one launch per level
// (sweep_mode 0) or one persistent launch per sweep (sweep_mode 1).
static int bilu0_sweeps(hfem_ctx *c, const double *x, double *y)
{
    SolverState &s = c->sv;
    const int bsz = trace_bsz(c);
    if (s.sweep_mode == 1) {
        const int n = c->hd.nf;
        unsigned *sync = s.sf_flags + (size_t)n;
        if (s.prec_fp32)
            HIPCHK(launch_bilu0_syncfree(bsz, s.d_lsched, s.d_lnbr, s.d_usched, s.d_unbr, n, s.Mg32, x, s.t, y, sync,
                                         s.sweep_wgs, s.spin_limit, s.sf_err, c->stream));
        else
            HIPCHK(launch_bilu0_syncfree(bsz, s.d_lsched, s.d_lnbr, s.d_usched, s.d_unbr, n, s.Mg, x, s.t, y, sync,
                                         s.sweep_wgs, s.spin_limit, s.sf_err, c->stream));
        return 0;
    }
    for (size_t l = 0; l + 1 < s.lptr.size(); l++) {
        const int t0 = s.lptr[l], t1 = s.lptr[l + 1];
        if (s.prec_fp32) HIPCHK(launch_bilu0_lsolve_level(bsz, s.d_lsched, s.d_lnbr, t0, t1, s.Mg32, x, s.t, c->stream));
        else HIPCHK(launch_bilu0_lsolve_level(bsz, s.d_lsched, s.d_lnbr, t0, t1, s.Mg, x, s.t, c->stream));
    }
    for (size_t l = 0; l + 1 < s.uptr.size(); l++) {
        const int t0 = s.uptr[l], t1 = s.uptr[l + 1];
        if (s.prec_fp32) HIPCHK(launch_bilu0_usolve_level(bsz, s.d_usched, s.d_unbr, t0, t1, s.Mg32, s.t, y, c->stream));
        else HIPCHK(launch_bilu0_usolve_level(bsz, s.d_usched, s.d_unbr, t0, t1, s.Mg, s.t, y, c->stream));
    }
    return 0;
}

// How BILU0 runs: mode 1 (default) one persistent launch for the factorisation, whose
// workgroups wait on per-row ready flags, and one per sweep, whose workgroups wait on the
// vector entries themselves; each wait is bounded by spin_limit polls (0: the default
// 2^20), one that gives up making the next hfem_precond_factor / hfem_gmres /
// hfem_precond_apply fail; mode 0 one launch per level.  Same bits either way.  No
// counterpart in the reference.
extern "C" int hfem_set_bilu0_sweep(hfem_ctx *c, int mode, int spin_limit)
{
    if (!c) return hfem_fail(-1, "hfem_set_bilu0_sweep: null context");
    if (mode != 0 && mode != 1) return hfem_fail(-1, "hfem_set_bilu0_sweep: mode %d (0 level launches, 1 sync-free)", mode);
    if (spin_limit < 0) return hfem_fail(-1, "hfem_set_bilu0_sweep: spin_limit %d", spin_limit);
    c->sv.sweep_mode = mode;
    c->sv.spin_limit = spin_limit ? spin_limit : (1 << 20);
    c->sv.graph_dirty = true;
    return 0;
}

// Whether the BILU0 application replays a captured graph of its launches (1) or launches
// them one by one (0, default: the persistent sweeps are three launches, 4.4 us cheaper on
// 132 300 unknowns than a graph's launch and the copy out of its fixed output).  No
// counterpart in the reference.
extern "C" int hfem_set_apply_graph(hfem_ctx *c, int use)
{
    if (!c) return hfem_fail(-1, "hfem_set_apply_graph: null context");
    c->sv.use_graph = use != 0;
    c->sv.graph_dirty = true;
    return 0;
}

// y = M^{-1} x on device vectors (x and y distinct).
static int precond_apply_dev(hfem_ctx *c, const double *x, double *y)
{
    SolverState &s = c->sv;
    const int n = c->hd.nf, bsz = trace_bsz(c);
    const long N = trace_len(c);
    if (s.prec == -1) {
        HIPCHK(hipMemcpyAsync(y, x, sizeof(double) * N, hipMemcpyDeviceToDevice, c->stream));
    } else if (s.prec == 2) {
        if (s.prec_fp32) HIPCHK(launch_block_jacobi(n, bsz, s.Mg32, x, y, c->stream));
        else HIPCHK(launch_block_jacobi(n, bsz, s.Mg, x, y, c->stream));
    } else if (s.prec == 0) {
        const long bytes = sizeof(double) * N;
        if (s.sweep_mode == 1) RC(ensure_syncfree(c));
        if (s.use_graph) {
            // the launches of both sweeps as one graph from c->yv into s.gy
            // (captured after each factorisation; no memset nodes in it)
            if (s.graph_dirty || !s.apply_graph) {
                if (s.apply_graph) HIPCHK(hipGraphExecDestroy(s.apply_graph));
                s.apply_graph = nullptr;
                if (!s.gy) HIPCHK(hfem_dalloc(&s.gy, N));
                hipGraph_t g = nullptr;
                HIPCHK(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
                const int rc = bilu0_sweeps(c, c->yv, s.gy);
                hipError_t e = hipStreamEndCapture(c->stream, &g);
                if (rc) {
                    if (g) hipGraphDestroy(g);
                    return rc;
                }
                HIPCHK(e);
                e = hipGraphInstantiate(&s.apply_graph, g, nullptr, nullptr, 0);
                hipGraphDestroy(g);
                HIPCHK(e);
                s.graph_dirty = false;
            }
            if (x != c->yv) HIPCHK(hipMemcpyAsync(c->yv, x, bytes, hipMemcpyDeviceToDevice, c->stream));
            HIPCHK(hipGraphLaunch(s.apply_graph, c->stream));
            HIPCHK(hipMemcpyAsync(y, s.gy, bytes, hipMemcpyDeviceToDevice, c->stream));
        } else {
            RC(bilu0_sweeps(c, x, y));
        }
    } else {
        return hfem_fail(-3, "preconditioner not factored");
    }
    return 0;
}

extern "C" int hfem_precond_apply(hfem_ctx *c, const double *x, double *y)
{
    RC(require_system(c, "hfem_precond_apply"));
    if (!x || !y) return hfem_fail(-1, "hfem_precond_apply: null vector");
    HIPCHK(hipSetDevice(c->device));
    const long N = trace_len(c);
    HIPCHK(hipMemcpyAsync(c->xv, x, sizeof(double) * N, hipMemcpyHostToDevice, c->stream));
    RC(precond_apply_dev(c, c->xv, c->yv));
    HIPCHK(hipMemcpyAsync(y, c->yv, sizeof(double) * N, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    RC(check_syncfree(c, "hfem_precond_apply"));
    return 0;
}

// ---------------------------------------------------------------- GMRES

// Least squares min |beta e1 - Hbar y| over the (j+1) x j Hessenberg matrix by
// Givens rotations; returns the residual norm.
static double hessenberg_ls(int j, int ldh, const std::vector<double> &hh, double beta, std::vector<double> &y)
{
    std::vector<double> R(hh.begin(), hh.begin() + (size_t)ldh * j), g(j + 1, 0.0);
    g[0] = beta;
    for (int k = 0; k < j; k++) {
        const double a = R[k + ldh * k], b = R[k + 1 + ldh * k], r = std::hypot(a, b);
        const double cs = r == 0 ? 1.0 : a / r, sn = r == 0 ? 0.0 : b / r;
        for (int col = k; col < j; col++) {
            const double u = R[k + ldh * col], v = R[k + 1 + ldh * col];
            R[k + ldh * col] = cs * u + sn * v;
            R[k + 1 + ldh * col] = -sn * u + cs * v;
        }
        const double u = g[k], v = g[k + 1];
        g[k] = cs * u + sn * v;
        g[k + 1] = -sn * u + cs * v;
    }
    y.assign(j, 0.0);
    for (int k = j - 1; k >= 0; k--) {
        double t = g[k];
        for (int c2 = k + 1; c2 < j; c2++) t -= R[k + ldh * c2] * y[c2];
        y[k] = t / R[k + ldh * k];
    }
    return std::fabs(g[j]);
}

// Left-preconditioned restarted GMRES on Hg x = Rg (kernel/gmres_bilu0.m), x in the
// solver's device vector, zero initial guess.  orthog 0: modified Gram-Schmidt,
// 1: classical Gram-Schmidt applied twice.  flag: 0 converged, 1 iteration limit.
extern "C" int hfem_gmres(hfem_ctx *c, int restart, double tol, int maxit, int orthog, int *iters, double *rev,
                          int *flag)
{
    RC(require_system(c, "hfem_gmres"));
    if (restart < 1 || maxit < 1 || !(tol > 0)) return hfem_fail(-1, "hfem_gmres: restart, maxit and tol must be positive");
    if (orthog != 0 && orthog != 1) return hfem_fail(-1, "hfem_gmres: orthog %d (0 MGS, 1 ICGS)", orthog);
    if (c->sv.prec < -1) return hfem_fail(-3, "hfem_gmres: call hfem_precond_factor first");
    HIPCHK(hipSetDevice(c->device));
    const double t0 = now_ms();
    RC(ensure_vectors(c, restart));
    SolverState &s = c->sv;
    s.ms_matvec = s.ms_prec = 0;
    s.n_matvec = s.n_prec = 0;
    const long N = trace_len(c);
    const int nf = c->hd.nf, bsz = trace_bsz(c);
    auto matvec = [&](const double *x, double *y) -> int {
        HIPCHK(launch_bsr_matvec(nf, bsz, c->rowstart, c->cols, c->Hg, x, y, c->stream));
        return 0;
    };
    double *pa = s.dots, *pb = s.dots + (size_t)gs_blocks(N) * s.vcols;   // partial sums, taken in turn
    double *h1 = s.h_dots, *h2 = h1 + s.vcols, *hn2 = h2 + s.vcols;       // their totals, on the host
    const int ldh = restart + 1;
    std::vector<double> hh((size_t)ldh * restart), y;
    int it = 0, fl = -1;
    double res = 0.0, nrmb = 0.0, beta;
    RC(precond_apply_dev(c, c->Rg, s.b));                       // b = M \ Rg
    HIPCHK(launch_fill(N, 0.0, s.x, c->stream));
    while (true) {
        double *V0 = s.V;
        const bool first = it == 0;
        if (!first) {
            RC(matvec(s.x, c->yv));                              // r = b - M \ (Hg x); x = 0 at first
            RC(precond_apply_dev(c, c->yv, V0));
            HIPCHK(launch_axpby(N, 1.0, s.b, -1.0, V0, c->stream));
        }
        double *r = first ? s.b : V0;
        HIPCHK(launch_gs_project(N, 1, r, N, r, nullptr, pa, nullptr, c->stream));
        HIPCHK(launch_gs_scale(N, r, V0, pa, hn2, c->stream));
        HIPCHK(hipStreamSynchronize(c->stream));
        beta = std::sqrt(*hn2);
        if (first) nrmb = beta;
        if (beta == 0.0 || nrmb == 0.0) { fl = 0; res = 0.0; break; }
        std::fill(hh.begin(), hh.end(), 0.0);
        int jdone = 0;
        for (int j = 0; j < restart; j++) {
            double *vj = s.V + (long)j * N, *w = s.V + (long)(j + 1) * N;
            HIPCHK(hipEventRecord(s.ev[0], c->stream));
            RC(matvec(vj, c->yv));
            HIPCHK(hipEventRecord(s.ev[1], c->stream));
            RC(precond_apply_dev(c, c->yv, w));
            HIPCHK(hipEventRecord(s.ev[2], c->stream));
            if (orthog == 0) {
                HIPCHK(launch_gs_project(N, 1, s.V, N, w, nullptr, pa, nullptr, c->stream));
                for (int i = 0; i <= j; i++) {
                    HIPCHK(launch_gs_update(N, 1, s.V + (long)i * N, N, w, i < j ? s.V + (long)(i + 1) * N : nullptr, pa,
                                            pb, h1 + i, c->stream));
                    std::swap(pa, pb);
                }
            } else {
                HIPCHK(launch_gs_project(N, j + 1, s.V, N, w, nullptr, pa, nullptr, c->stream));
                HIPCHK(launch_gs_project(N, j + 1, s.V, N, w, pa, pb, h1, c->stream));
                HIPCHK(launch_gs_update(N, j + 1, s.V, N, w, nullptr, pb, pa, h2, c->stream));
            }
            HIPCHK(launch_gs_scale(N, w, w, pa, hn2, c->stream));
            HIPCHK(hipStreamSynchronize(c->stream));
            for (int i = 0; i <= j; i++) hh[i + (size_t)ldh * j] = orthog == 0 ? h1[i] : h1[i] + h2[i];
            const double hn = std::sqrt(*hn2);
            float e1 = 0, e2 = 0;
            HIPCHK(hipEventElapsedTime(&e1, s.ev[0], s.ev[1]));
            HIPCHK(hipEventElapsedTime(&e2, s.ev[1], s.ev[2]));
            s.ms_matvec += e1;
            s.ms_prec += e2;
            s.n_matvec++;
            s.n_prec++;
            hh[j + 1 + (size_t)ldh * j] = hn;
            jdone = j + 1;
            res = hessenberg_ls(j + 1, ldh, hh, beta, y);
            it++;
            if (rev) rev[it - 1] = res / nrmb;
            if (hn == 0.0 || res / nrmb <= tol) { fl = 0; break; }
            if (it >= maxit) { fl = 1; break; }
        }
        HIPCHK(hipMemcpyAsync(s.coef, y.data(), sizeof(double) * jdone, hipMemcpyHostToDevice, c->stream));
        HIPCHK(launch_multi_axpy(N, jdone, s.V, N, s.coef, 1.0, s.x, c->stream));   // x += V y
        if (fl >= 0) break;
    }
    HIPCHK(hipStreamSynchronize(c->stream));
    RC(check_syncfree(c, "hfem_gmres"));
    if (iters) *iters = it;
    if (flag) *flag = fl;
    s.ms_gmres = now_ms() - t0;
    return 0;
}

extern "C" int hfem_solver_stats(hfem_ctx *c, double *out)
{
    if (!c || !out) return hfem_fail(-1, "hfem_solver_stats: null argument");
    const SolverState &s = c->sv;
    const double v[7] = {s.ms_order, s.ms_factor, s.ms_gmres, s.ms_matvec, (double)s.n_matvec, s.ms_prec,
                         (double)s.n_prec};
    std::copy(v, v + 7, out);
    return 0;
}

extern "C" int hfem_read_trace_solution(hfem_ctx *c, double *x)
{
    RC(require_system(c, "hfem_read_trace_solution"));
    if (!c->sv.x || !x) return hfem_fail(-3, "hfem_read_trace_solution: no solution");
    HIPCHK(hipSetDevice(c->device));
    HIPCHK(hipStreamSynchronize(c->stream));
    HIPCHK(hipMemcpy(x, c->sv.x, sizeof(double) * trace_len(c), hipMemcpyDeviceToHost));
    return 0;
}

// ---------------------------------------------------------------- solution update and residual

extern "C" int hfem_update_solution(hfem_ctx *c, double alpha)
{
    RC(require_system(c, "hfem_update_solution"));
    if (!c->has_sol || !c->sv.x) return hfem_fail(-3, "hfem_update_solution: no solution or trace update");
    HIPCHK(hipSetDevice(c->device));
    const Dims &d = c->d;
    // UH += alpha duh (solvers/solutionupdate.cpp:75-77)
    HIPCHK(launch_axpby(trace_len(c), alpha, c->sv.x, 1.0, c->UH, c->stream));
    // getU on every element (:6-67), then getQ (assembly/elementassembly.cpp:1414-1479)
    HIPCHK(launch_update_u(c->hd.ne, d.npv, d.nc, d.nch, d.ndf, d.na, d.nb, c->ldx, c->elcon, c->X, c->sv.x, alpha,
                           c->UDG, c->stream));
    if (c->ph.fc_q != 0.0) {
        Master m{c->shapvt, c->shapvg, c->shapft, c->shapfg, c->perm, c->invperm};
        HIPCHK(launch_getq(c->d, m, c->ph, c->dgnodes, c->UDG, c->UH, c->SH, c->elcon, c->bf, 0, c->hd.ne, c->stream));
    }
    return 0;
}

extern "C" int hfem_get_q(hfem_ctx *c)
{
    RC(require_system(c, "hfem_get_q"));
    if (!c->has_sol || !c->has_master) return hfem_fail(-3, "hfem_get_q: master and solution must be set");
    HIPCHK(hipSetDevice(c->device));
    Master m{c->shapvt, c->shapvg, c->shapft, c->shapfg, c->perm, c->invperm};
    HIPCHK(launch_getq(c->d, m, c->ph, c->dgnodes, c->UDG, c->UH, c->SH, c->elcon, c->bf, 0, c->hd.ne, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return 0;
}

extern "C" int hfem_residual_norm(hfem_ctx *c, double *rNorm)
{
    RC(require_system(c, "hfem_residual_norm"));
    const int ne = c->hd.ne, nf = c->hd.nf;
    const Dims &d = c->d;
    RC(hfem_assemble_vector(c, 0, ne));   // residual rows only
    HIPCHK(launch_face_gather(nf, trace_bsz(c), d.nch, d.npf, d.nb, d.nb, c->f2e, c->einv, c->Rh, c->r, nullptr,
                              nullptr, c->stream));
    double s1 = 0, s2 = 0;
    RC(hfem_reduce_sum(c, ne, c->ru2, 0, &s1));
    RC(hfem_reduce_sum(c, trace_len(c), c->r, 1, &s2));
    if (rNorm) *rNorm = std::sqrt(s1 + s2);
    return 0;
}

// ---------------------------------------------------------------- Newton and DIRK

static int check_params(const hfem_solver_params *p)
{
    if (!p) return hfem_fail(-1, "solver parameters missing");
    if (!(p->newton_tol > 0) || p->newton_maxiter < 1 || p->restart < 1 || !(p->gmres_tol > 0) || p->gmres_maxit < 1)
        return hfem_fail(-1, "solver parameters: tolerances and iteration limits must be positive");
    if (p->precond != -1 && p->precond != 0 && p->precond != 2) return hfem_fail(-1, "solver parameters: precond %d", p->precond);
    if (p->prec_precision != 0 && p->prec_precision != 1)
        return hfem_fail(-1, "solver parameters: prec_precision %d (0 single, 1 double)", p->prec_precision);
    if (p->ordering != 0 && p->ordering != 1) return hfem_fail(-1, "solver parameters: ordering %d", p->ordering);
    if (p->orthog != 0 && p->orthog != 1) return hfem_fail(-1, "solver parameters: orthog %d", p->orthog);
    if (p->precision != HFEM_FP64 && p->precision != HFEM_MIXED) return hfem_fail(-1, "solver parameters: precision");
    if (p->quasi_newton && (p->qn_accuracy < 0 || p->qn_accuracy > 1 || !(p->qn_reuse_ratio >= 0)))
        return hfem_fail(-1, "solver parameters: quasi-Newton accuracy %d, reuse ratio", p->qn_accuracy);
    return 0;
}

extern "C" int hfem_solve_steady(hfem_ctx *c, const hfem_solver_params *p, int *converged, int *niter,
                                 double *history)
{
    RC(require_system(c, "hfem_solve_steady"));
    RC(check_params(p));
    const bool qn = p->quasi_newton != 0;
    if (qn) RC(hfem_quasi_newton_storage(c, p->qn_accuracy));
    const double alpha_min = 1.0e-4;
    const int true_max = p->true_newton_maxiter > 0 ? p->true_newton_maxiter : INT_MAX;
    double rNorm = p->newton_tol + 1.0;
    int it = 0, true_it = 0;
    // robustMode: reset at the start of a nonlinear solve; a failed line search goes
    // back to the previous iterate only while it is 0, or with quasi-Newton
    // (solvers/dgsolvers.cpp:114, :175-177)
    int robust = 0;
    // quasi-Newton bookkeeping (sys.linearSolvesClocks, sys.lastAssemblyAndPrecClocks)
    bool reuse = false;
    double lin_time = 0.0, jac_time = 0.0;
    auto now = [] { return std::chrono::steady_clock::now(); };
    auto secs = [](std::chrono::steady_clock::time_point t0) {
        return std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    };
    auto recompute_jacobian = [&] { reuse = false; lin_time = 0.0; };
    while (rNorm > p->newton_tol && it < p->newton_maxiter && true_it < true_max) {
        it++;
        const bool reused = reuse;
        if (!reused) true_it++;
        double oldNorm;
        auto t0 = now();
        if (!reused) {
            RC(hfem_assemble_linear_system(c, p->precision, &oldNorm));
            jac_time = secs(t0);
        } else {
            RC(hfem_assemble_rhs(c, &oldNorm));
        }
        if (!std::isfinite(oldNorm)) return hfem_fail(-5, "hfem_solve_steady: residual norm is NaN or Inf");
        if (c->sv.order_method < 0 || (p->reuse_ordering == 0) || c->sv.order_method != p->ordering)
            RC(hfem_compute_ordering(c, p->ordering));
        if (!reused) {
            auto t1 = now();
            RC(hfem_set_precond_precision(c, p->prec_precision));
            RC(hfem_precond_factor(c, p->precond));
            jac_time += secs(t1);
        }
        int gi = 0, gf = 0;
        auto t2 = now();
        RC(hfem_gmres(c, p->restart, p->gmres_tol, p->gmres_maxit, p->orthog, &gi, nullptr, &gf));
        lin_time += secs(t2);
        if (history) {
            history[HFEM_HIST * (it - 1)] = oldNorm;
            history[HFEM_HIST * (it - 1) + 2] = reused ? -gi : gi;
        }
        if (qn) {
            if (lin_time < p->qn_reuse_ratio * jac_time) reuse = true;
            else recompute_jacobian();
        }
        if (it == 1 && oldNorm < p->newton_tol) {
            rNorm = oldNorm;
            if (history) { history[1] = rNorm; history[3] = 0.0; history[4] = 0.0; }
            break;
        }
        double alpha = 1.0, applied = 0.0;
        int steps = 0;
        while (true) {
            RC(hfem_update_solution(c, alpha));
            applied += alpha;
            steps++;
            RC(hfem_residual_norm(c, &rNorm));
            if (!std::isfinite(rNorm) || (rNorm > oldNorm && rNorm > p->newton_tol)) {
                const double a = std::fabs(alpha / 2);
                alpha = -a;
                if (qn) recompute_jacobian();
                if (a < alpha_min) {
                    if (robust == 0 || qn) {
                        // back to the previous iterate (dgsolvers.cpp:175-180)
                        robust = 1;
                        alpha = -2.0 * std::fabs(alpha);
                        RC(hfem_update_solution(c, alpha));
                        applied += alpha;
                        steps++;
                    }
                    break;
                }
            } else {
                break;
            }
        }
        if (history) {
            history[HFEM_HIST * (it - 1) + 1] = rNorm;
            history[HFEM_HIST * (it - 1) + 3] = applied;
            history[HFEM_HIST * (it - 1) + 4] = steps;
        }
    }
    if (converged) *converged = rNorm < p->newton_tol;
    if (niter) *niter = it;
    return 0;
}

// DIRK coefficients of solvers/DIRKcoeff.cpp (d = inv(A) column-major, c = b inv(A), t).
static bool dirk_table(int nstage, int order, double *c, double *d, double *t)
{
    struct Tab { int s, o; double c[3], d[9], t[3]; };
    static const Tab tabs[] = {
        {1, 1, {1.0}, {1.0}, {1.0}},
        {1, 2, {2.0}, {2.0}, {0.5}},
        {2, 2, {0.0, 1.0}, {3.414213562373096, -8.242640687119289, 0.0, 3.414213562373096}, {0.292893218813452, 1.0}},
        {2, 3, {1.098076211353316, 0.633974596215561}, {1.267949192431123, 0.928203230275509, 0.0, 1.267949192431123},
         {0.788675134594813, 0.211324865405187}},
        {3, 3, {0.0, 0.0, 1.0},
         {2.294280360323567, -1.484721005721436, -8.556127801733982, 0.0, 2.294280360323568, 3.391748836909791, 0.0,
          0.0, 2.294280360323567},
         {0.435866521500000, 0.717933260750000, 1.0}},
        {3, 4, {0.445622407287714, 1.064177772475912, 0.120614758428183},
         {0.935822227524088, 0.497940606760015, -0.345865915800969, 0.0, 0.935822227524088, 2.867525668568206, 0.0,
          0.0, 0.935822227524088},
         {1.068579021301629, 0.5, -0.068579021301629}},
    };
    for (const Tab &tb : tabs)
        if (tb.s == nstage && tb.o == order) {
            for (int i = 0; i < nstage; i++) { c[i] = tb.c[i]; t[i] = tb.t[i]; }
            for (int i = 0; i < nstage * nstage; i++) d[i] = tb.d[i];
            return true;
        }
    return false;
}

extern "C" int hfem_dirk_step(hfem_ctx *c, double dt, int nstage, int order, const hfem_solver_params *p,
                              int *converged, int *newton_iters)
{
    RC(require_system(c, "hfem_dirk_step"));
    RC(check_params(p));
    double cc[3], d[9], tt[3];
    if (!(dt > 0)) return hfem_fail(-1, "hfem_dirk_step: dt must be positive");
    if (!dirk_table(nstage, order, cc, d, tt)) return hfem_fail(-1, "hfem_dirk_step: DIRK(%d,%d) not implemented", nstage, order);
    HIPCHK(hipSetDevice(c->device));
    const Dims &dm = c->d;
    const long ne = c->hd.ne, nu = ne * dm.npv * dm.nc;
    SolverState &s = c->sv;
    if (!s.UDGi) HIPCHK(hfem_dalloc(&s.UDGi, (size_t)nu));
    HIPCHK(hipMemcpyAsync(s.UDGi, c->UDG, sizeof(double) * nu, hipMemcpyDeviceToDevice, c->stream));
    const Phys saved = c->ph;
    auto D = [&](int i, int j) { return d[i + nstage * j]; };
    int total = 0, ok = 1;
    for (int st = 0; st < nstage; st++) {
        c->ph.fc_u = D(st, st) / dt;
        c->ph.fc_q = 1.0;
        c->ph.tdep = 1;
        // SH of the stage (solvers/dgsolvers.cpp:316-341) and zero q source (:344-349)
        double a, b, cf;
        if (st == 0) { a = D(0, 0) / dt; b = 0.0; cf = 0.0; }
        else if (st == 1) { a = (D(1, 0) + D(1, 1)) / dt; b = -D(1, 0) / dt; cf = 0.0; }
        else {
            const double r = D(2, 0) / D(1, 0);
            a = (D(2, 0) + D(2, 1) + D(2, 2)) / dt - r * (D(1, 0) + D(1, 1)) / dt;
            b = -D(2, 1) / dt;
            cf = r;
        }
        HIPCHK(launch_stage_source(ne, dm.npv, dm.nc, dm.ncu, a, s.UDGi, b, c->UDG, cf, c->SH, c->stream));
        int conv = 0, it = 0;
        int rc = hfem_solve_steady(c, p, &conv, &it, nullptr);
        total += it;
        if (rc) { c->ph = saved; return rc; }
        if (!conv) { ok = 0; break; }
    }
    c->ph = saved;
    if (converged) *converged = ok;
    if (newton_iters) *newton_iters = total;
    if (!ok) return hfem_fail(-6, "hfem_dirk_step: a DIRK stage did not converge");
    return 0;
}
