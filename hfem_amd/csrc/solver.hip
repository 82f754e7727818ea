// Trace-system solver kernels (gfx950): inverses of BSR diagonal blocks, MDF
// block weights, BILU0 factorisation and its triangular sweeps one level of the
// ordering at a time, block-Jacobi, the vector kernels of GMRES, the solution
// update (getU) and DIRK stage sources.
//
// BSR blocks are bsz x bsz column-major, rows = faces, the diagonal block first in
// each row (the reference's Hg layout, assembly/globalassembly.cpp:42-86).
#include "dinv_body.h"
#include "hfem_device.h"

#include <algorithm>
#include <type_traits>

namespace hfem {

constexpr int SV_THREADS = 256;

constexpr int FACTOR_MAXROW = 64;     // longest BSR row the factorisation takes

// A lane index the compiler cannot see through: address arithmetic formed from it stays
// where it is used (hoisted out of the row loops it fills the registers).
__device__ __forceinline__ int opaque(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// MFMA 16x16x4 operands: lane l supplies A(l%16, l/16) and B(l/16, l%16); result lane l,
// element v holds C(l/16 + 4v, l%16) (FP64) or C(4(l/16) + v, l%16) (FP32).
template <typename T> struct BlkMfma;
template <> struct BlkMfma<double> {
    typedef double v4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ v4 run(double a, double b, v4 c)
    {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lk, int v) { return lk + 4 * v; }
};
template <> struct BlkMfma<float> {
    typedef float v4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ v4 run(float a, float b, v4 c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lk, int v) { return 4 * lk + v; }
};

// ---- inverse of one block ----
//
// Blocked Gauss-Jordan with partial pivoting of an n x n block in LDS (column-major,
// stride n), in place up to the permutation and the row scales, by a workgroup of four
// waves.  Per panel of 16 columns wave 0 runs the pivot steps in registers (panel_steps,
// dinv_body.h); the panel then holds Gp = T(:, P), T the product of its elementary steps
// and P its pivot rows, and every other column a becomes T a = Abar + Gp a(P), Abar = a
// with the rows P zeroed: rank-16 updates of 16 x 16 tiles on the MFMA.
// In the BILU0 factorisation the inverse stands on the chain of dependent rows, so wave 0
// updates the next panel's columns itself and goes on while the other waves update the
// rest: one barrier per panel.  What the others do during the pivot steps is the
// caller's (idle(), by waves 1-3 once per panel).
// 45 x 45 FP64, alone on its CU: 23 us, of which the chain of the 45 pivot steps 15 us
// (0.33 us each) and wave 0's updates 2.4 us; with the block in LDS and a barrier around
// every pass (the earlier form) 95 us.
//
// LDS besides the block: the rows' scales, a pivot row's entries on their way (twice),
// per panel's parity the set of its pivot rows and the pivot rows of its steps, per row
// its step, per step its row, and a flag.
template <typename T>
struct InvShared {
    static constexpr int head(int rows) { return (int)((rows * sizeof(T) + 15) / 16 * 16); }
    static constexpr int bytes(int rows) { return head(rows) + 2 * 16 * (int)sizeof(T) + 4 * 8 + (2 * 16 + 2 * rows + 1) * 4; }
    T *scale, *buf;
    unsigned long long *set;
    int *prow, *lab, *pof, *sing;
    // mem: 16-byte aligned
    __device__ InvShared(void *mem, int rows)
    {
        scale = (T *)mem;
        buf = (T *)((char *)mem + head(rows));
        set = (unsigned long long *)(buf + 2 * 16);
        prow = (int *)(set + 4);
        lab = prow + 2 * 16;
        pof = lab + rows;
        sing = pof + rows;
    }
};

// NT: 16-row tiles (at least ceil(n / 16)).
// All threads call it with the block complete (a barrier before); out(i, c, v) receives
// every entry of the inverse once, rows along the lanes.  Returns 0, or 1 + the step of
// the first zero pivot (workgroup-uniform; the result is then finite but no inverse).
template <int NT, class IDLE, class OUT, typename T>
__device__ __forceinline__ int wg_inverse(int n, T *A, const InvShared<T> &sh, IDLE idle, OUT out)
{
    typedef BlkMfma<T> M;
    typedef typename M::v4 v4;
    constexpr int RPL = NT <= 4 ? 1 : 2;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nt = (n + 15) / 16;
    PanelState<T, RPL> ps;
    if (wv == 0) ps.init(n);
    // panel pb's update of tile column ct
    auto update = [&](int pb, int ct) {
        const int lr = opaque(lane & 15), lk = opaque(lane >> 4);
        const int kw = min(16, n - 16 * pb), col = min(16 * ct + lr, n - 1);
        const int *prow = sh.prow + (pb & 1) * 16;
        T *C = A + n * col;
        T b[4];
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
            const int k = 4 * ks + lk;
            b[ks] = C[prow[min(k, kw - 1)]];
            b[ks] = k < kw ? b[ks] : (T)0;
        }
        // the lane's rows 16 r + row(lk, v) among the pivot rows: bits 16 r + row(0, v)
        // of the set moved down by row(lk, 0)
        const unsigned long long set0 = sh.set[2 * (pb & 1)] >> M::row(lk, 0);
        const unsigned long long set1 = NT > 4 ? sh.set[2 * (pb & 1) + 1] >> M::row(lk, 0) : 0;
        v4 acc[NT];
#pragma unroll
        for (int r = 0; r < NT; r++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const T c = C[min(16 * r + M::row(lk, v), n - 1)];
                const unsigned long long set = r < 4 ? set0 : set1;
                acc[r][v] = (set >> (16 * (r & 3) + M::row(0, v))) & 1 ? (T)0 : c;
            }
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
            const int k = min(4 * ks + lk, kw - 1);
            T a[NT];
#pragma unroll
            for (int r = 0; r < NT; r++) a[r] = A[min(16 * r + lr, n - 1) + n * (16 * pb + k)];
#pragma unroll
            for (int r = 0; r < NT; r++) acc[r] = M::run(a[r], b[ks], acc[r]);
        }
        // (this wave alone touches the tile column between two barriers)
#pragma unroll
        for (int r = 0; r < NT; r++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int i = 16 * r + M::row(lk, v);
                if (i < n && 16 * ct + lr < n) C[i] = acc[r][v];
            }
    };
    for (int pb = 0;; pb++) {
        // the previous panel's update: its tile columns but the next panel's, which is wave
        // 0's, over waves 1-3 (after the last panel over all four)
        for (int ct = 0, d = 1; pb > 0 && ct < nt; ct++) {
            if (ct == pb - 1) continue;
            const int w = ct == pb ? 0 : d;
            if (ct != pb) d = d == 3 ? pb < nt : d + 1;
            if (wv == w) update(pb - 1, ct);
        }
        if (pb == nt) break;
        if (wv == 0) {
            const int kw = min(16, n - 16 * pb);
            T x[16][RPL];
#pragma unroll
            for (int j = 0; j < 16; j++)
#pragma unroll
                for (int q = 0; q < RPL; q++) x[j][q] = A[min(lane + 64 * q, n - 1) + n * min(16 * pb + j, n - 1)];
            const int pcv = panel_steps<T, RPL>(x, kw, 16 * pb, ps, sh.buf);
            // column k of the panel is in x[16 - kw + k] after kw rotations
            T *P = A + n * (16 * pb + kw - 16);
#pragma unroll
            for (int q = 0; q < RPL; q++)
                if (lane + 64 * q < n) {
#pragma unroll
                    for (int j = 0; j < 16; j++)
                        if (j >= 16 - kw) P[lane + 64 * q + n * j] = x[j][q];
                    sh.lab[lane + 64 * q] = ps.lab[q];
                    sh.scale[lane + 64 * q] = ps.scale[q];
                }
#pragma unroll
            for (int q = 0; q < RPL; q++) {
                const unsigned long long set = __ballot(ps.lab[q] >= 16 * pb);
                if (lane == 0) sh.set[2 * (pb & 1) + q] = set;
            }
            if (lane < kw) {
                sh.prow[(pb & 1) * 16 + lane] = pcv;
                sh.pof[16 * pb + lane] = pcv;
            }
            if (lane == 0) *sh.sing = ps.sing;
        } else {
            idle();
        }
        __syncthreads();
    }
    __syncthreads();
    int lab[RPL];
    T sc[RPL];
#pragma unroll
    for (int q = 0; q < RPL; q++) {
        lab[q] = sh.lab[min(lane + 64 * q, n - 1)];
        sc[q] = sh.scale[min(lane + 64 * q, n - 1)];
    }
    int pof[RPL];
#pragma unroll
    for (int q = 0; q < RPL; q++) pof[q] = sh.pof[min(lane + 64 * q, n - 1)];
    // the wave's columns c = wv, wv + 4, ..., four at a time
    for (int c0 = wv; c0 < n; c0 += 16) {
        T v[4][RPL];
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int q = 0; q < RPL; q++) v[u][q] = A[min(lane + 64 * q, n - 1) + n * min(c0 + 4 * u, n - 1)];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int c = c0 + 4 * u, cc = min(c, n - 1);
            int pc = __builtin_amdgcn_readlane(pof[0], cc & 63);
            if (RPL > 1 && cc >= 64) pc = __builtin_amdgcn_readlane(pof[RPL - 1], cc & 63);
#pragma unroll
            for (int q = 0; q < RPL; q++)
                if (c < n && lane + 64 * q < n) out(lab[q], pc, v[u][q] * sc[q]);
        }
    }
    return __builtin_amdgcn_readfirstlane(*sh.sing);
}

// ---- inverse of one block, entry by entry ----
//
// The inverse of the single-precision BILU0 factors: the same waves, panels and barriers,
// but every entry goes through the plain elimination's operations one by one,
// a - c (r pinv), on the vector ALU.  Along the rows of a factorisation roundings can
// grow: on 4 608 p=4 triangles (849 levels) those of single precision reach 3e-3 to 5e-3
// of M^-1 x, and the order of the sums alone moved a Newton iterate by 1e-6; this form's
// roundings are those of the unblocked elimination.  (Pivots, ties included, are chosen as
// if the rows were interchanged: pos is the place of a row.)
// The factorisation of those triangles: 13.1 ms (10.1 with the blocked inverse, 34.1 with
// the block in LDS and a barrier around every pass), of the 8^3 p=2 hexes 13.4 (9.6, 37.5).
template <typename T> struct StepShared;
template <>
struct StepShared<float> {
    static constexpr int bytes(int rows) { return (2 * 16 * rows + 2 * 16) * 4 + (2 * 16 + 2 * rows + 1) * 4; }
    float *c, *pinv;                 // per panel's parity: 16 pivot columns (0 in the pivot row), 16 reciprocals
    int *prow, *lab, *pof, *sing;    // per panel's parity: the pivot rows; per row its step; per step its row
    __device__ StepShared(void *mem, int rows)
    {
        c = (float *)mem;
        pinv = c + 2 * 16 * rows;
        prow = (int *)(pinv + 2 * 16);
        lab = prow + 2 * 16;
        pof = lab + rows;
        sing = pof + rows;
    }
};

// Entry `row` (wave-uniform) of a column held with rows lane + 64 q.
template <int RPL>
__device__ __forceinline__ float row_bcast(const float (&col)[RPL], int row)
{
    if constexpr (RPL == 1) return GJ<float>::bcast(col[0], row);
    else return GJ<float>::bcast(row < 64 ? col[0] : col[1], row & 63);
}

// The pivot steps k0 ... k0 + kw - 1 of a panel on one wave (rows lane + 64 q; the columns
// rotate through x: column k is left in x[16 - kw + k]).  Stores step k's pivot column to
// c[n k ...]; lane k returns its pivot row in prow, its reciprocal in pinvs.
template <int RPL>
struct PivotSteps {
    unsigned open[RPL];
    int pos[RPL], lab[RPL], sing;
    __device__ __forceinline__ void init(int n)
    {
        sing = 0;
#pragma unroll
        for (int q = 0; q < RPL; q++) {
            pos[q] = (threadIdx.x & 63) + 64 * q;
            open[q] = pos[q] < n ? ~0u : 0u;
            lab[q] = -1;
        }
    }
    __device__ __forceinline__ void run(float (&x)[16][RPL], int kw, int k0, int n, float *c, int &prow, float &pinvs)
    {
        const int lane = threadIdx.x & 63;
        unsigned key[RPL], m = 0;
        int p = 0;
        float pv = 0.0f, pinv = 0.0f, row1 = 0.0f;
        prow = 0;
        pinvs = 1.0f;
        auto search = [&](int stage, const float (&col)[RPL], const float (&next)[RPL]) {
            switch (stage) {
            case 0:
#pragma unroll
                for (int q = 0; q < RPL; q++) key[q] = pivot_key(col[q]) & open[q];
                m = key[0];
#pragma unroll
                for (int q = 1; q < RPL; q++) m = max(m, key[q]);
                m = key_max_step<0>(m);
                break;
            case 1: m = key_max_step<1>(m); m = key_max_step<2>(m); break;
            case 2: m = key_max_step<3>(m); m = key_max_step<4>(m); break;
            case 3: m = key_max_step<5>(m); break;
            case 4: {
                const unsigned mm = (unsigned)__builtin_amdgcn_readlane((int)m, 63);
                int ties = 0;
#pragma unroll
                for (int q = RPL - 1; q >= 0; q--) {
                    const unsigned long long b = __ballot(key[q] == mm);
                    p = b ? 64 * q + __ffsll((long long)b) - 1 : p;
                    ties += __popcll(b);
                }
                if (ties > 1) {
                    // the first in place (128 - pos > 0)
                    unsigned t[RPL], best = 0;
#pragma unroll
                    for (int q = 0; q < RPL; q++) {
                        t[q] = key[q] == mm ? 128u - (unsigned)pos[q] : 0u;
                        best = max(best, t[q]);
                    }
                    best = wave_max_key(best);
#pragma unroll
                    for (int q = 0; q < RPL; q++) {
                        const unsigned long long b = __ballot(t[q] == best);
                        p = b ? 64 * q + __ffsll((long long)b) - 1 : p;
                    }
                }
                break;
            }
            case 5:
                pv = row_bcast<RPL>(col, p);
                row1 = row_bcast<RPL>(next, p);
                break;
            case 6: pinv = pv == 0.0f ? 0.0f : 1.0f / pv; break;
            }
        };
        constexpr int NS = 7;
#pragma unroll
        for (int st = 0; st < NS; st++) search(st, x[0], x[1]);
#pragma unroll 1
        for (int k = 0; k < kw; k++) {
            bool mine[RPL];
            float cz[RPL], f[RPL], last[RPL];
            const float s1 = row1 * pinv;
            const int posp = RPL == 1 || p < 64 ? __builtin_amdgcn_readlane(pos[0], p & 63)
                                                : __builtin_amdgcn_readlane(pos[RPL - 1], p & 63);
#pragma unroll
            for (int q = 0; q < RPL; q++) {
                mine[q] = lane + 64 * q == p;
                cz[q] = mine[q] ? 0.0f : x[0][q];
                f[q] = mine[q] ? pinv : 1.0f;
                last[q] = mine[q] ? pinv : -x[0][q] * pinv;
                x[0][q] = mine[q] ? s1 : fmaf(-cz[q], s1, x[1][q]);
                open[q] = mine[q] ? 0u : open[q];
            }
            const int pk = p;
            const float pinvk = pinv;
            const bool zero = pv == 0.0f;
            // (after the last step: of a column that is none, unused)
#pragma unroll
            for (int st = 0; st < NS; st++) {
                // columns 2-15: st = 0 ... 6 takes two each, column 2 (the next step's second)
                // first
                search(st, x[0], x[1]);
                __builtin_amdgcn_sched_barrier(0);
                if (st == 0) {
#pragma unroll
                    for (int q = 0; q < RPL; q++) {
                        pos[q] = mine[q] ? k0 + k : pos[q] == k0 + k ? posp : pos[q];
                        lab[q] = mine[q] ? k0 + k : lab[q];
                        if (lane + 64 * q < n) c[n * k + lane + 64 * q] = cz[q];
                    }
                    sing = zero && !sing ? k0 + k + 1 : sing;
                    prow = lane == k ? pk : prow;
                    pinvs = lane == k ? pinvk : pinvs;
                }
#pragma unroll
                for (int j = 2 + 2 * st; j < 4 + 2 * st; j++) {
                    float y[RPL];
#pragma unroll
                    for (int q = 0; q < RPL; q++) y[q] = x[j][q] * f[q];
                    const float sj = row_bcast<RPL>(y, pk);
#pragma unroll
                    for (int q = 0; q < RPL; q++) x[j - 1][q] = fmaf(-cz[q], sj, y[q]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int q = 0; q < RPL; q++) x[15][q] = last[q];
        }
    }
};

// As wg_inverse.
template <int NT, class IDLE, class OUT>
__device__ __forceinline__ int wg_inverse(int n, float *A, const StepShared<float> &sh, IDLE idle, OUT out)
{
    constexpr int RPL = NT <= 4 ? 1 : 2;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int np = (n + 15) / 16, ng = (n + 3) / 4;
    PivotSteps<RPL> ps;
    if (wv == 0) ps.init(n);
    // panel pb's steps on columns 4 g ... 4 g + 3
    auto update = [&](int pb, int g) {
        const int kw = min(16, n - 16 * pb);
        const float *c = sh.c + (pb & 1) * 16 * n;
        float x[4][RPL], cn[RPL];
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int q = 0; q < RPL; q++) x[u][q] = A[min(lane + 64 * q, n - 1) + n * min(4 * g + u, n - 1)];
#pragma unroll
        for (int q = 0; q < RPL; q++) cn[q] = c[min(lane + 64 * q, n - 1)];
        const int pr = sh.prow[(pb & 1) * 16 + (lane & 15)];
        const float pi = sh.pinv[(pb & 1) * 16 + (lane & 15)];
#pragma unroll 2
        for (int k = 0; k < kw; k++) {
            const int p = __builtin_amdgcn_readlane(pr, k);
            const float pinv = GJ<float>::bcast(pi, k);
            float ck[RPL], f[RPL];
#pragma unroll
            for (int q = 0; q < RPL; q++) {
                ck[q] = cn[q];
                f[q] = lane + 64 * q == p ? pinv : 1.0f;
                cn[q] = c[min(lane + 64 * q, n - 1) + n * min(k + 1, kw - 1)];
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                float y[RPL];
#pragma unroll
                for (int q = 0; q < RPL; q++) y[q] = x[u][q] * f[q];
                const float s = row_bcast<RPL>(y, p);
#pragma unroll
                for (int q = 0; q < RPL; q++) x[u][q] = fmaf(-ck[q], s, y[q]);
            }
        }
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int q = 0; q < RPL; q++)
                if (4 * g + u < n && lane + 64 * q < n) A[lane + 64 * q + n * (4 * g + u)] = x[u][q];
    };
    for (int pb = 0;; pb++) {
        if (pb > 0 && pb < np) {
            // the next panel's columns over all four waves
            if (4 * pb + wv < ng) update(pb - 1, 4 * pb + wv);
            __syncthreads();
        }
        // the other columns over waves 1-3 (after the last panel over all four)
        for (int g = 0, d = pb < np; pb > 0 && g < ng; g++) {
            if (g >> 2 == pb - 1 || g >> 2 == pb) continue;
            if (wv == d) update(pb - 1, g);
            d = d == 3 ? pb < np : d + 1;
        }
        if (pb == np) break;
        if (wv == 0) {
            const int kw = min(16, n - 16 * pb);
            float x[16][RPL], pinvs;
            int prow;
#pragma unroll
            for (int j = 0; j < 16; j++)
#pragma unroll
                for (int q = 0; q < RPL; q++) x[j][q] = A[min(lane + 64 * q, n - 1) + n * min(16 * pb + j, n - 1)];
            ps.run(x, kw, 16 * pb, n, sh.c + (pb & 1) * 16 * n, prow, pinvs);
            float *P = A + n * (16 * pb + kw - 16);
#pragma unroll
            for (int q = 0; q < RPL; q++)
                if (lane + 64 * q < n) {
#pragma unroll
                    for (int j = 0; j < 16; j++)
                        if (j >= 16 - kw) P[lane + 64 * q + n * j] = x[j][q];
                    sh.lab[lane + 64 * q] = ps.lab[q];
                }
            if (lane < kw) {
                sh.prow[(pb & 1) * 16 + lane] = prow;
                sh.pinv[(pb & 1) * 16 + lane] = pinvs;
                sh.pof[16 * pb + lane] = prow;
            }
            if (lane == 0) *sh.sing = ps.sing;
        } else {
            idle();
        }
        __syncthreads();
    }
    __syncthreads();
    int lab[RPL], pof[RPL];
#pragma unroll
    for (int q = 0; q < RPL; q++) {
        lab[q] = sh.lab[min(lane + 64 * q, n - 1)];
        pof[q] = sh.pof[min(lane + 64 * q, n - 1)];
    }
    for (int c0 = wv; c0 < n; c0 += 16) {
        float v[4][RPL];
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int q = 0; q < RPL; q++) v[u][q] = A[min(lane + 64 * q, n - 1) + n * min(c0 + 4 * u, n - 1)];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int c = c0 + 4 * u, cc = min(c, n - 1);
            int pc = __builtin_amdgcn_readlane(pof[0], cc & 63);
            if (RPL > 1 && cc >= 64) pc = __builtin_amdgcn_readlane(pof[RPL - 1], cc & 63);
#pragma unroll
            for (int q = 0; q < RPL; q++)
                if (c < n && lane + 64 * q < n) out(lab[q], pc, v[u][q]);
        }
    }
    return __builtin_amdgcn_readfirstlane(*sh.sing);
}

// LDS of the factorisation's inverse.
template <typename T> using FactorInv = std::conditional_t<std::is_same<T, float>::value, StepShared<T>, InvShared<T>>;

// The block kernels' shapes by block size: CPW = columns per wave of four (and, for the
// MFMA products, k-steps of 4), RCH rows per lane.  A shape's unused columns cost their
// share of the work, so the block sizes of the element families (hfem_create takes no
// others) have one that fits: 8-16 (triangles p=1-3, tets p=1), 20 and 24 (triangles p=4,
// 5, hexes p=1), 30 (tets p=2), 45 (hexes p=2), 50 (tets p=3), 75 (tets p=4).
// launch(RCH, CPW) with integral constants.
constexpr int MAX_BLOCK = 80;

template <class F>
static hipError_t block_shape(int bsz, F launch)
{
#define SHAPE(R, C) launch(std::integral_constant<int, R>(), std::integral_constant<int, C>())
    if (bsz < 1 || bsz > MAX_BLOCK) return hipErrorInvalidValue;
    if (bsz <= 16) SHAPE(1, 4);
    else if (bsz <= 24) SHAPE(1, 6);
    else if (bsz <= 32) SHAPE(1, 8);
    else if (bsz <= 48) SHAPE(1, 12);
    else if (bsz <= 52) SHAPE(1, 13);
    else SHAPE(2, 20);
#undef SHAPE
    return hipGetLastError();
}

// Inverses of the diagonal blocks of Hg (block-Jacobi, mkBlockJacobi.m:9-11, and
// the MDF weights).  One workgroup per row.  34 104 blocks of 50 x 50: 4.6 ms with the
// earlier LDS form, 1.26 ms now (floor: 1.4 GB in and out, 0.28 ms).
template <int NT>
__global__ void __launch_bounds__(SV_THREADS, NT <= 4 ? 4 : 2)
block_inverse_kernel(int nrows, int bsz, const int *__restrict__ rowpts, const double *__restrict__ Hg,
                     double *__restrict__ Dinv, int *__restrict__ info)
{
    extern __shared__ __align__(16) double lds[];
    const int tid = threadIdx.x, nth = blockDim.x;
    const long b2 = (long)bsz * bsz;
    double *A = lds;
    const InvShared<double> sh(A + (b2 + 1) / 2 * 2, bsz);
    for (int row = blockIdx.x; row < nrows; row += gridDim.x) {
        const double *src = Hg + (long)rowpts[row] * b2;
        for (long i = tid; i < b2; i += nth) A[i] = src[i];
        __syncthreads();
        double *dst = Dinv + row * b2;
        const int r = wg_inverse<NT>(bsz, A, sh, [] {}, [&](int i, int c, double v) { dst[i + bsz * c] = v; });
        if (tid == 0 && info) info[row] = r;
        __syncthreads();
    }
}

// Broadcast lane `src` (wave-uniform) of a double to the whole wave.
__device__ __forceinline__ double wave_bcast(double v, int src)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, src);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), src);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// acc_i += sum_cc B[i + bsz cc] z[cc] for the lane's rows i = lane, lane + 64, with z
// held one entry per lane (z0 = z[lane], z1 = z[lane + 64]) and broadcast by readlane.
// The columns go in chunks of CH whose loads are all issued before the first
// multiply (addresses clamped into the block; columns past bsz are multiplied by
// zero), so a block costs ceil(bsz / CH) memory round trips instead of one per
// column pair.
template <int CH, bool TWO, typename TM>
__device__ __forceinline__ void wave_block_matvec_ch(int bsz, const TM *__restrict__ B, double z0, double z1,
                                                     double &acc0, double &acc1)
{
    const int lane = threadIdx.x & 63;
    const int r0 = lane < bsz ? lane : 0, r1 = lane + 64 < bsz ? lane + 64 : 0;
    double s0 = 0.0, s1 = 0.0;
    for (int c0 = 0; c0 < bsz; c0 += CH) {
        double v0[CH], v1[CH];
#pragma unroll
        for (int j = 0; j < CH; j++) {
            const long col = (long)bsz * min(c0 + j, bsz - 1);
            v0[j] = B[r0 + col];
            if (TWO) v1[j] = B[r1 + col];
        }
#pragma unroll
        for (int j = 0; j < CH; j++) {
            const int cc = c0 + j;
            double zj = wave_bcast(cc < 64 ? z0 : z1, cc & 63);
            zj = cc < bsz ? zj : 0.0;
            s0 += v0[j] * zj;
            if (TWO) s1 += v1[j] * zj;
        }
    }
    if (lane < bsz) acc0 += s0;
    if (TWO && lane + 64 < bsz) acc1 += s1;
}

template <typename TM>
__device__ __forceinline__ void wave_block_matvec(int bsz, const TM *__restrict__ B, double z0, double z1,
                                                  double &acc0, double &acc1)
{
    if (bsz > 64) wave_block_matvec_ch<16, true>(bsz, B, z0, z1, acc0, acc1);
    else wave_block_matvec_ch<64, false>(bsz, B, z0, z1, acc0, acc1);
}

// ---- BILU0 sweeps (kernel/applyBILU0.m) ----
//
// For row r of a sweep, with neighbours k taken by it (numbered before r in the
// forward sweep L y = x, after r in the backward sweep U v = y):
//   forward   z_r = b_r - sum_k L_rk z_k
//   backward  z_r = inv(U_rr) b_r - sum_k U~_rk z_k,  U~_rk = inv(U_rr) U_rk
// (upper blocks scaled by the factorisation's last step, bilu0_scale_upper_kernel,
// so that inv(U_rr) b_r is formed before the neighbours' z are needed).
//
// A sweep is bound by its chain of dependent rows (557 levels per sweep on 16 464
// p=3 tets, 5 597 on 24^3 periodic p=2 hexes), so a row is laid out for the time
// from its last neighbour's z to its own:
// * One workgroup of four waves per row; every wave takes a quarter of the columns
//   of every neighbour block (lane = block row), so what is left to do when the
//   last z arrives is a quarter of one block product, one barrier and a sum of four.
// * Blocks are loaded into registers before any wait, NPRE neighbours ahead.
// * The neighbours come in the order of their level (RowSched, built with the
//   levels), the last to be ready last.
// * z itself is the ready flag: a sweep that runs as one launch fills z with a bit
//   pattern no result has (SWEEP_EMPTY) and polls the entries it needs, so a hand-over is
//   one store and one load (about 0.45 us between any two CUs; a separate flag behind
//   a completed store, the earlier form, put three more round trips in each link).
// * Behind the last neighbour's z there is no branch, reload or readlane any more: taken
//   branches (some 30 cycles each) and readlanes (9) were two thirds of that path.
// Measured per application (two sweeps), FP64 factors: with a flag per row and one wave
// per whole block; with z as the flag and a quarter of each block per wave; now:
//   16 464 p=3 tets (block 50, 557 levels)         3.60 ms   1.81 ms   1.58 ms
//   8^3 periodic p=2 hexes (block 45, 370 levels)  2.68 ms   0.75 ms   0.61 ms
//   750 p=4 tets (block 75, 146 levels)            1.79 ms   0.64 ms   0.43 ms
//   4 608 p=4 triangles (block 20, 849 levels)     4.82 ms   1.42 ms   1.28 ms
//   512 p=2 triangles (block 12, 104 levels)       0.63 ms   0.20 ms   0.18 ms
// i.e. 0.75-0.9 us per link, of which the hand-over 0.45 us (a store and the load that
// sees it, between any two CUs); the large mesh is bound by reading its factors (4.6 GB)
// next to the chain.
struct RowSched {
    const int4 *rows;    // by ticket: row, its diagonal block, first entry in nbr, neighbours
    const int2 *nbr;     // block, column
};

// A signalling NaN: stored results are quieted, never equal to it.
constexpr unsigned long long SWEEP_EMPTY = 0x7ff4dead5eed0001ull;

// Until lane's *p is no longer SWEEP_EMPTY in any lane: its value.  Entries are read
// and written by agent-scope atomics (coherent across the XCDs).  At most spin_limit
// polls after the first; a wait that runs out, or any wait once another has (*err
// set), sets *err and returns.
__device__ __forceinline__ double wait_entry(const double *p, int spin_limit, int *err)
{
    auto load = [&] {
        return __hip_atomic_load((const unsigned long long *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    // (the ballot makes the loop's control wave-uniform; one exit that falls through: a
    // taken branch costs some 30 cycles)
    unsigned long long v = load();
    bool waiting = __ballot(v == SWEEP_EMPTY) != 0;
    const unsigned limit = (unsigned)spin_limit;
    unsigned spins = 0;
    while (__builtin_expect(waiting && spins < limit, 1)) {
        __builtin_amdgcn_s_sleep(1);
        spins++;
        if (__builtin_expect((spins & 63) == 0, 0) &&
            __builtin_amdgcn_readfirstlane(__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)))
            spins = limit;
        v = load();
        waiting = __ballot(v == SWEEP_EMPTY) != 0;
    }
    if (__builtin_expect(waiting, 0)) __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return __longlong_as_double((long long)v);
}

// Lane J of every row of 16 lanes to the whole row (DPP row_newbcast).
template <int J>
__device__ __forceinline__ double row16_bcast(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x150 + J, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x150 + J, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

template <class F, int... J>
__device__ __forceinline__ void for_columns(F f, std::integer_sequence<int, J...>)
{
    (f(std::integral_constant<int, J>()), ...);
}

// One row of a sweep, the ticket t's, by the whole workgroup.  The lane holds block
// rows lane (+ 64 with RCH 2); wave w the columns [w cpw, (w+1) cpw) of each block,
// cpw = ceil(bsz / 4) <= CPW.  Loads are clamped into the block and columns past the
// wave's multiplied by zero.  With one row per lane the wave's vector entries are fetched
// by every row of 16 lanes and broadcast in it by DPP (10 cycles a column with the
// multiplication; as readlanes 18).  Shared by the one-launch (WAIT) and level-launched
// kernels so that both compute the same bits.
template <bool BACKWARD, int RCH, int CPW, int NPRE, bool WAIT, typename TM>
__device__ __forceinline__ void sweep_row(int bsz, const RowSched &sch, int t, const TM *__restrict__ Mg,
                                          const double *__restrict__ b, double *z, double (*red)[64 * RCH],
                                          int spin_limit, int *err)
{
    constexpr int NW = SV_THREADS / 64;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const long b2 = (long)bsz * bsz;
    const int cpw = (bsz + NW - 1) / NW, c0 = wv * cpw;
    const int4 h = sch.rows[t];
    const int r = __builtin_amdgcn_readfirstlane(h.x), kd = __builtin_amdgcn_readfirstlane(h.y);
    const int first = __builtin_amdgcn_readfirstlane(h.z), cnt = __builtin_amdgcn_readfirstlane(h.w);
    // lane i: the row's neighbour i (fewer than FACTOR_MAXROW)
    const int2 nb = sch.nbr[first + max(min(lane, cnt - 1), 0)];
    auto block = [&](int i) { return __builtin_amdgcn_readlane(nb.x, i); };
    auto vec = [&](int i) { return z + (long)__builtin_amdgcn_readlane(nb.y, i) * bsz; };
    int rl[RCH];
#pragma unroll
    for (int q = 0; q < RCH; q++) rl[q] = min(lane + 64 * q, bsz - 1);
    // the vector entry this lane fetches
    constexpr bool DPP = RCH == 1;
    static_assert(!DPP || CPW <= 16, "columns per wave");
    const int le = DPP ? lane & 15 : lane, ce = min(c0 + min(le, cpw - 1), bsz - 1);
    const bool cv = le < cpw && c0 + le < bsz;
    auto load_share = [&](int blk, TM (&v)[CPW][RCH]) {
        const TM *B = Mg + (long)blk * b2;
#pragma unroll
        for (int j = 0; j < CPW; j++)
#pragma unroll
            for (int q = 0; q < RCH; q++) v[j][q] = B[rl[q] + (long)bsz * min(c0 + j, bsz - 1)];
    };
    auto add_share = [&](const TM (&v)[CPW][RCH], double ze, double (&acc)[RCH]) {
        const double zm = cv ? ze : 0.0;
        for_columns([&](auto J) {
            constexpr int j = J();
            double zj;
            if constexpr (DPP) zj = row16_bcast<j>(zm);
            else zj = wave_bcast(zm, j);
#pragma unroll
            for (int q = 0; q < RCH; q++) acc[q] += (double)v[j][q] * zj;
        }, std::make_integer_sequence<int, CPW>());
    };
    // the blocks of the last NPRE neighbours (base + i), the last to be waited for; the
    // last neighbour is always the last of them, so that no branch follows its z
    const int base = cnt - NPRE;
    TM v[NPRE][CPW][RCH];
#pragma unroll
    for (int i = 0; i < NPRE; i++)
        if (base + i >= 0) load_share(block(base + i), v[i]);
    double own[RCH], acc[RCH];
#pragma unroll
    for (int q = 0; q < RCH; q++) {
        own[q] = 0.0;
        acc[q] = 0.0;
    }
    if (BACKWARD) {
        TM dv[CPW][RCH];
        load_share(kd, dv);
        add_share(dv, b[(long)r * bsz + ce], own);
    } else if (wv == 0) {
#pragma unroll
        for (int q = 0; q < RCH; q++) own[q] = b[(long)r * bsz + rl[q]];
    }
    auto entry_of = [&](int i) { return WAIT ? wait_entry(vec(i) + ce, spin_limit, err) : vec(i)[ce]; };
    for (int i = 0; i < base; i++) {
        TM u[CPW][RCH];
        load_share(block(i), u);
        add_share(u, entry_of(i), acc);
    }
#pragma unroll
    for (int i = 0; i < NPRE; i++)
        if (base + i >= 0) add_share(v[i], entry_of(base + i), acc);
#pragma unroll
    for (int q = 0; q < RCH; q++) red[wv][lane + 64 * q] = own[q] - acc[q];
    __syncthreads();
    if (wv == 0) {
#pragma unroll
        for (int q = 0; q < RCH; q++) {
            double s = red[0][lane + 64 * q];
#pragma unroll
            for (int w = 1; w < NW; w++) s += red[w][lane + 64 * q];
            unsigned long long u = (unsigned long long)__double_as_longlong(s);
            u = u == SWEEP_EMPTY ? 0x7ff8000000000000ull : u;
            double *zr = z + (long)r * bsz + lane + 64 * q;
            if (lane + 64 * q < bsz) {
                if (WAIT) __hip_atomic_store((unsigned long long *)zr, u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                else *zr = __longlong_as_double((long long)u);
            }
        }
    }
}

// The rows of one level: tickets [t0, t1).
template <bool BACKWARD, int RCH, int CPW, int NPRE, typename TM>
__global__ void __launch_bounds__(SV_THREADS)
bilu0_sweep_kernel(int bsz, RowSched sch, int t0, int t1, const TM *__restrict__ Mg, const double *__restrict__ b,
                   double *z)
{
    __shared__ double red[SV_THREADS / 64][64 * RCH];
    for (int t = t0 + blockIdx.x; t < t1; t += gridDim.x) {
        sweep_row<BACKWARD, RCH, CPW, NPRE, false, TM>(bsz, sch, t, Mg, b, z, red, 0, nullptr);
        __syncthreads();
    }
}

// A whole sweep in one launch: the rows in ticket order -- the level lists
// concatenated, so every row comes after the rows it reads -- to persistent
// workgroups through an atomic ticket.  A wait that gives up (wait_entry) leaves a
// wrong result and *err set, which the host reports; every workgroup still runs to
// the end of the tickets.  No deadlock: a workgroup waits only on rows of smaller
// tickets, which were drawn by workgroups already running.
template <bool BACKWARD, int RCH, int CPW, int NPRE, typename TM>
__global__ void __launch_bounds__(SV_THREADS)
bilu0_sweep_syncfree_kernel(int bsz, RowSched sch, int n, const TM *__restrict__ Mg, const double *__restrict__ b,
                            double *z, unsigned *counter, int spin_limit, int *err)
{
    __shared__ double red[SV_THREADS / 64][64 * RCH];
    __shared__ int sticket;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // The ticket is drawn by the whole of wave 0 (a wave-uniform condition): the draw
    // adds 1 from lane 0 and 0 from the others, and lane 0's old value is the ticket.
    // Under "tid == 0" the structurizer may merge the draw across the back edge into
    // an inner loop that only lane 0 leaves.
    while (true) {
        if (wv == 0) sticket = __builtin_amdgcn_readfirstlane(atomicAdd(counter, lane == 0 ? 1u : 0u));
        // (also: wave 0 has summed the previous row's red before any wave writes it again)
        __syncthreads();
        const int t = __builtin_amdgcn_readfirstlane(sticket);
        if (t >= n) break;
        sweep_row<BACKWARD, RCH, CPW, NPRE, true, TM>(bsz, sch, t, Mg, b, z, red, spin_limit, err);
    }
}

// Fresh tickets for the two sweeps of an application and their empty results (a
// kernel, not a memset, so that the application can be captured in a graph).
__global__ void __launch_bounds__(SV_THREADS)
sweep_reset_kernel(unsigned *sync, long n, double *t, double *y)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sync[1] = 0;
        sync[2] = 0;
    }
    const double e = __longlong_as_double((long long)SWEEP_EMPTY);
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        t[i] = e;
        y[i] = e;
    }
}

// ---- BILU0 factorisation (kernel/computeBILU0.m) ----
//
// In the row-oriented form: row i takes, for each neighbour k numbered before it,
// L_ik = A_ik inv(U_kk), then A_ii -= L_ik U_ki and A_il -= L_ik U_kl for the later
// common neighbours l; finally A_ii is inverted.  The neighbours go by level: adjacent
// rows have different levels, in the order of their numbers, so every block receives
// its updates in an order the right-looking loop allows.
//
// Bound by its chain of dependent rows, like the sweeps (at 16 464 p=3 tets 557 links;
// its products would take 3 ms), so a row is laid out for the time from its last
// neighbour's flag to its own:
// * One workgroup of four waves per row.  The products run on the MFMA, 16 x 16 tiles;
//   a wave takes whole tile columns, so its B operands (inv(U_kk), U_kl) go from memory
//   straight into registers, all k-steps in flight, with no barrier behind the flag.
//   The A operands are in LDS: A_ik, staged before the wait, and -L_ik.
// * U_ki is fetched with inv(U_kk), each further target's operands during the product
//   before it.
// * The diagonal block stays in LDS until it is inverted there (wg_inverse); the last
//   neighbour's other targets are updated in that inverse's idle phases.
// * Which blocks are targets is found in registers (the column list of row k against
//   that of row i, lane by lane), before the wait.
// Blocks that other rows read go through agent-scope atomics (coherent across the
// XCDs); the row's flag is stored after every wave's stores have completed.
// FP64, before (all operands through LDS, target search by LDS scans, the inverse in
// LDS) and now: 16 464 p=3 tets (block 50, 557 levels) 86.9 and 27.0 ms; 8^3 periodic p=2
// hexes (block 45, 370 levels) 43.1 and 11.5 ms; 4 608 p=4 triangles (block 20, 849
// levels) 37.2 and 11.9 ms.  Of a row's time in the hexes (28 us): its first neighbour's
// flag to L 3.4 us, the targets 2.4 us, the inverse 22 us.

// Wait until *f holds `epoch`, for the factorisation's ready flags.  At most
// spin_limit polls; a wait that runs out, or any wait once another has (*err set), sets
// *err and returns.
__device__ __forceinline__ void wait_ready(const unsigned *f, unsigned epoch, int spin_limit, int *err)
{
    // (the polled values go through readfirstlane: a uniform loop)
    int spins = 0;
    while ((unsigned)__builtin_amdgcn_readfirstlane(
               __hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != epoch) {
        if (++spins > spin_limit ||
            ((spins & 63) == 0 && __builtin_amdgcn_readfirstlane(
                                      __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)))) {
            __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return;
        }
        __builtin_amdgcn_s_sleep(1);
    }
}

// Entry o of a block: a uniform base and an unsigned byte offset, so that a block's
// addresses are one register each.
template <typename T>
__device__ __forceinline__ T *entry(T *base, int o)
{
    return (T *)((char *)base + (unsigned)o * (unsigned)sizeof(T));
}
template <typename T>
__device__ __forceinline__ const T *entry(const T *base, int o)
{
    return (const T *)((const char *)base + (unsigned)o * (unsigned)sizeof(T));
}
template <typename T>
__device__ __forceinline__ T coh_load(const T *base, int o)
{
    return __hip_atomic_load(entry(base, o), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void coh_store(T *base, int o, T v)
{
    __hip_atomic_store(entry(base, o), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The workgroup's tiles of an n x n block product on the MFMA: NT = ceil(CPW / 4) tiles
// a side.  A wave takes tile column `wave` (NT 3, 4; NT 1: the first wave alone), one
// tile of four (NT 2), or tile column `wave` and its share of the fifth (NT 5).
template <typename T, int CPW>
struct BlockTiles {
    typedef BlkMfma<T> M;
    typedef typename M::v4 v4;
    static constexpr int NT = (CPW + 3) / 4, NCB = NT == 5 ? 2 : 1, TPW = NT <= 2 ? 1 : NT <= 4 ? NT : 7;
    static_assert(NT <= 5, "block size");
    int n, lr, lk, wv;
    __device__ BlockTiles(int n_) : n(n_)
    {
        const int lane = threadIdx.x & 63;
        lr = lane & 15;
        lk = lane >> 4;
        wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    }
    static constexpr __device__ int waves() { return NT == 1 ? 1 : NT == 3 ? 3 : 4; }
    __device__ bool active() const { return wv < waves(); }
    __device__ bool has(int s) const { return s < 6 || wv == 0; }
    __device__ int rt(int s) const { return NT == 2 ? wv >> 1 : s < 5 ? s : s == 5 ? wv : 4; }
    __device__ int cb(int s) const { return s < 5 ? 0 : 1; }
    __device__ int ct(int b) const { return b ? 4 : NT == 2 ? (wv & 1) : wv; }
    // B operands: every k-step of the wave's tile columns of a block in global memory
    template <typename S>
    __device__ __forceinline__ void load_b(const S *B, T (&b)[NCB][CPW]) const
    {
#pragma unroll
        for (int c = 0; c < NCB; c++) {
            const int col = min(ct(c) * 16 + opaque(lr), n - 1), k = opaque(lk);
#pragma unroll
            for (int ks = 0; ks < CPW; ks++) b[c][ks] = (T)coh_load(B, min(4 * ks + k, n - 1) + n * col);
        }
    }
    // acc += A b with A in LDS (rows past n are computed and not stored; k past n is
    // masked on the A side; every wave computes all TPW tiles -- no branch may stand
    // between MFMAs: the compiler was seen to leave out the wait for a result that is
    // read on the far side of a taken branch)
    __device__ __forceinline__ void product(const T *A, const T (&b)[NCB][CPW], v4 (&acc)[TPW]) const
    {
        const int lr = opaque(this->lr), lk = opaque(this->lk);
        int row[TPW];
#pragma unroll
        for (int s = 0; s < TPW; s++) row[s] = min(rt(s) * 16 + lr, n - 1);
        // (one k-step of operands ahead: all of them would fill the registers)
        T a[TPW], an[TPW];
        auto load_a = [&](int ks, T (&v)[TPW]) {
            const int k = 4 * ks + lk, kc = min(k, n - 1);
#pragma unroll
            for (int s = 0; s < TPW; s++) v[s] = A[row[s] + n * kc];
        };
        load_a(0, a);
#pragma unroll
        for (int ks = 0; ks < CPW; ks++) {
            if (ks + 1 < CPW) load_a(ks + 1, an);
#pragma unroll
            for (int s = 0; s < TPW; s++) acc[s] = M::run(4 * ks + lk < n ? a[s] : (T)0, b[cb(s)][ks], acc[s]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < TPW; s++) a[s] = an[s];
        }
    }
    // f(tile s, element v, offset in a block) for every entry of the wave's tiles
    template <class F>
    __device__ __forceinline__ void each(F f) const
    {
        const int lr = opaque(this->lr), lk = opaque(this->lk);
#pragma unroll
        for (int s = 0; s < TPW; s++)
            if (has(s))
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int i = rt(s) * 16 + M::row(lk, v), j = ct(cb(s)) * 16 + lr;
                    if (i < n && j < n) f(s, v, i + n * j);
                }
    }
};

// MDF block weights C(n) = ||inv(H_ii) H_n||_F for every block n of row i
// (kernel/computeMDFordering.m:14-20).  One workgroup per row, inv(H_ii) in LDS, the other
// blocks straight from memory into the B operands, the next block's while the current is
// multiplied; only sums of squares leave the registers.  Floor: reading the matrix, 1 ms for
// 34 104 rows of 50 x 50 blocks (4.8 GB); 8.9 ms as a dot product per thread out of LDS,
// 2.4 ms now.
constexpr int MDF_BATCH = 32;   // blocks between two barriers

template <int CPW>
__global__ void __launch_bounds__(SV_THREADS, CPW <= 16 ? 2 : 1)
mdf_weight_kernel(int nrows, int bsz, const int *__restrict__ rowpts, const double *__restrict__ Hg,
                  const double *__restrict__ Dinv, double *__restrict__ Cw)
{
    extern __shared__ double lds[];
    __shared__ double red[MDF_BATCH][SV_THREADS / 64];
    typedef BlockTiles<double, CPW> Tiles;
    const Tiles tl(bsz);
    const int tid = threadIdx.x, lane = tid & 63;
    const long b2 = (long)bsz * bsz;
    const bool act = tl.active();
    for (int row = blockIdx.x; row < nrows; row += gridDim.x) {
        const int n0 = __builtin_amdgcn_readfirstlane(rowpts[row]), n1 = __builtin_amdgcn_readfirstlane(rowpts[row + 1]);
        for (long i = tid; i < b2; i += SV_THREADS) lds[i] = Dinv[row * b2 + i];
        __syncthreads();
        for (int m0 = n0; m0 < n1; m0 += MDF_BATCH) {
            const int m1 = min(m0 + MDF_BATCH, n1);
            if (act) {
                double b[Tiles::NCB][CPW], bn[Tiles::NCB][CPW];
                tl.load_b(Hg + (long)m0 * b2, b);
                for (int n = m0; n < m1; n++) {
                    tl.load_b(Hg + (long)min(n + 1, m1 - 1) * b2, bn);
                    typename Tiles::v4 acc[Tiles::TPW];
#pragma unroll
                    for (int s = 0; s < Tiles::TPW; s++) acc[s] = (typename Tiles::v4){0.0, 0.0, 0.0, 0.0};
                    tl.product(lds, b, acc);
                    double s2 = 0.0;
                    tl.each([&](int s, int v, int) { s2 += acc[s][v] * acc[s][v]; });
                    for (int d = 32; d > 0; d >>= 1) s2 += __shfl_xor(s2, d);
                    if (lane == 0) red[n - m0][tl.wv] = s2;
#pragma unroll
                    for (int c = 0; c < Tiles::NCB; c++)
#pragma unroll
                        for (int ks = 0; ks < CPW; ks++) b[c][ks] = bn[c][ks];
                }
            }
            __syncthreads();
            if (m0 + tid < m1) {
                double s2 = 0.0;
                for (int w = 0; w < SV_THREADS / 64; w++) s2 += Tiles::waves() > w ? red[tid][w] : 0.0;
                Cw[m0 + tid] = sqrt(s2);
            }
            __syncthreads();
        }
    }
}

// The factorisation's last step for the sweeps: every upper block of row r becomes
// U~_rl = inv(U_rr) U_rl (inv(U_rr) is the row's diagonal block), in place, after
// the whole factorisation (the other rows' eliminations read the unscaled U_rl).
// One workgroup per row, as mdf_weight_kernel: inv(U_rr) in LDS (FP64 for either type of
// factors), the upper blocks straight from memory into the B operands, the next one's
// while the current is multiplied.  Floor: the upper blocks read and written and the
// diagonal ones read, 1 ms for 34 104 rows of 50 x 50 blocks (4.7 GB).  As a dot product
// per thread out of LDS and now: those 2.55 and 1.76 ms, 1 536 rows of 45 x 45 243 and
// 94 us, 375 of them in single precision 180 and 40, 7 008 of 20 x 20 in single precision
// 32 and 41 (a wave's one tile per block is too little to cover its latency; 0.01% of
// that solve, so there is one form).
template <int CPW, typename TM>
__global__ void __launch_bounds__(SV_THREADS, CPW <= 16 ? 2 : 1)
bilu0_scale_upper_kernel(int bsz, int n, const int *__restrict__ rowpts, const int *__restrict__ colind,
                         const int *__restrict__ u2o, TM *__restrict__ Mg)
{
    extern __shared__ double lds[];
    typedef BlockTiles<double, CPW> Tiles;
    const Tiles tl(bsz);
    const int lane = threadIdx.x & 63;
    const long b2 = (long)bsz * bsz;
    const bool act = tl.active();
    for (int r = blockIdx.x; r < n; r += gridDim.x) {
        // (loop control with barriers inside must be uniform)
        const int k0 = __builtin_amdgcn_readfirstlane(rowpts[r]);
        const int len = __builtin_amdgcn_readfirstlane(rowpts[r + 1]) - k0;
        const int o = __builtin_amdgcn_readfirstlane(u2o[r]);
        const TM *Ui = Mg + (long)k0 * b2;
        for (long i = threadIdx.x; i < b2; i += SV_THREADS) lds[i] = (double)Ui[i];
        __syncthreads();
        for (int q0 = 1; q0 < len; q0 += 64) {
            // lane l: whether block q0 + l is an upper one
            const int q = min(q0 + lane, len - 1);
            unsigned long long todo = __ballot(q0 + lane < len && u2o[colind[k0 + q]] > o);
            if (!todo) continue;
            int m = __ffsll((long long)todo) - 1;
            double b[Tiles::NCB][CPW], bn[Tiles::NCB][CPW];
            if (act) tl.load_b((const TM *)Mg + (long)(k0 + q0 + m) * b2, b);
            while (true) {
                TM *B = Mg + (long)(k0 + q0 + m) * b2;
                todo &= todo - 1;
                if (todo) m = __ffsll((long long)todo) - 1;
                typename Tiles::v4 acc[Tiles::TPW];
                if (act) {
                    tl.load_b((const TM *)Mg + (long)(k0 + q0 + m) * b2, bn);
#pragma unroll
                    for (int s = 0; s < Tiles::TPW; s++) acc[s] = (typename Tiles::v4){0.0, 0.0, 0.0, 0.0};
                    tl.product(lds, b, acc);
                    // (18 wait states behind an FP64 matrix instruction: the compiler leaves
                    // too few where its result is stored on the far side of a taken branch)
#pragma unroll
                    for (int s = 0; s < Tiles::TPW; s++) asm volatile("s_nop 15\n\ts_nop 3" : "+v"(acc[s]));
                }
                // (two waves read a tile column: both have their operands before either stores)
                if constexpr (Tiles::NT == 2 || Tiles::NT == 5) __syncthreads();
                if (act) tl.each([&](int s, int v, int i) { *entry(B, i) = (TM)acc[s][v]; });
                if (!todo) break;
#pragma unroll
                for (int c = 0; c < Tiles::NCB; c++)
#pragma unroll
                    for (int ks = 0; ks < CPW; ks++) b[c][ks] = bn[c][ks];
            }
        }
        __syncthreads();
    }
}

// dst[i] = src[i] for i < n by the workgroup, eight loads in flight per thread.
template <typename T>
__device__ __forceinline__ void wg_load_block_coh(T *dst, const T *src, long n)
{
    const int tid = threadIdx.x, nth = blockDim.x;
    for (long b = tid; b < n; b += 8L * nth) {
        T v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = coh_load(src, (int)min(b + (long)j * nth, n - 1));
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (b + (long)j * nth < n) dst[b + (long)j * nth] = v[j];
    }
}

template <typename T>
__host__ __device__ constexpr size_t factor_lds(int bsz)
{
    return ((size_t)3 * bsz * bsz * sizeof(T) + 15) / 16 * 16 + FactorInv<T>::bytes(bsz);
}

// The row of ticket t, by the whole workgroup (a barrier must lie between two calls).
// T: the factors' type (double, or float: the reference's single-precision
// preconditioner, precPrecision 0, preprocessing/initializestructs.cpp:476-486, on the
// FP32 MFMA).  Shared by the one-launch (WAIT) and level-launched kernels: the same bits.
template <typename T, int RCH, int CPW, bool WAIT>
__device__ __forceinline__ void factor_row(int n, const int *__restrict__ rowpts, const int *__restrict__ colind,
                                           const int *__restrict__ u2o, const RowSched &sch, int t, T *Mg,
                                           int *__restrict__ info, T *lds, const unsigned *flags, unsigned epoch,
                                           int spin_limit, int *err)
{
    typedef BlockTiles<T, CPW> Tiles;
    typedef typename Tiles::v4 v4;
    constexpr int TPW = Tiles::TPW, NCB = Tiles::NCB;
    const Tiles tl(n);
    const int tid = threadIdx.x, lane = tid & 63;
    const long b2 = (long)n * n;
    T *A = lds, *L = lds + b2, *Dg = lds + 2 * b2;
    const FactorInv<T> sh((char *)lds + ((size_t)3 * n * n * sizeof(T) + 15) / 16 * 16, n);
    const int4 h = sch.rows[t];
    const int ri = __builtin_amdgcn_readfirstlane(h.x), d0 = __builtin_amdgcn_readfirstlane(h.y);
    const int first = __builtin_amdgcn_readfirstlane(h.z), cnt = __builtin_amdgcn_readfirstlane(h.w);
    const int len = __builtin_amdgcn_readfirstlane(rowpts[ri + 1]) - d0;
    if (len > FACTOR_MAXROW) {
        // reported through info, the row is left as it is
        if (tid == 0) info[ri] = -len;
        return;
    }
    // lane l: column and number of the row's block l
    const int rcol = lane < len ? colind[d0 + lane] : -1, rord = lane < len ? u2o[rcol] : -1;
    const bool act = tl.active();
    T *Mii = Mg + (long)d0 * b2;
    wg_load_block_coh(Dg, (const T *)Mii, b2);
    constexpr int NT = Tiles::NT;
    // target block M_il -= L_ik U_kl (-L in LDS), tile column ct of it.  The product is summed
    // by itself: onto the target's larger entries its rounding doubled the FP32 factors'
    // error where the diagonal dominates.
    auto update_target = [&](T *Mil, const T *U, int ct) {
        const int lr = opaque(tl.lr), lk = opaque(tl.lk), j = ct * 16 + lr, jc = min(j, n - 1);
        T b[CPW];
        v4 c[NT], lu[NT];
#pragma unroll
        for (int ks = 0; ks < CPW; ks++) b[ks] = coh_load(U, min(4 * ks + lk, n - 1) + n * jc);
#pragma unroll
        for (int s = 0; s < NT; s++)
#pragma unroll
            for (int v = 0; v < 4; v++)
                c[s][v] = coh_load((const T *)Mil, min(s * 16 + Tiles::M::row(lk, v), n - 1) + n * jc);
        T a[NT], an[NT];
        auto load_a = [&](int ks, T (&x)[NT]) {
            const int kc = min(4 * ks + lk, n - 1);
#pragma unroll
            for (int s = 0; s < NT; s++) x[s] = L[min(s * 16 + lr, n - 1) + n * kc];
        };
        load_a(0, a);
#pragma unroll
        for (int s = 0; s < NT; s++) lu[s] = (v4){(T)0, (T)0, (T)0, (T)0};
#pragma unroll
        for (int ks = 0; ks < CPW; ks++) {
            if (ks + 1 < CPW) load_a(ks + 1, an);
#pragma unroll
            for (int s = 0; s < NT; s++) lu[s] = Tiles::M::run(4 * ks + lk < n ? a[s] : (T)0, b[ks], lu[s]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < NT; s++) a[s] = an[s];
        }
#pragma unroll
        for (int s = 0; s < NT; s++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int i = s * 16 + Tiles::M::row(lk, v);
                if (i < n && j < n) coh_store(Mil, i + n * j, (T)(c[s][v] + lu[s][v]));
            }
    };
    // the targets left of the current neighbour: those of the last one are updated next to
    // the inverse of the diagonal block, by waves 1-3
    unsigned long long todo = 0;
    int k0 = 0, km = -1, ct = 0, l = -1, w0 = 0;
    // the wave's next (target, tile column): they are dealt to the waves, ct counts tile
    // columns past the first of target l
    auto pair = [&]() -> bool {
        while (l < 0 || ct >= NT) {
            if (!todo) return false;
            if (l >= 0) ct -= NT;
            l = __ffsll((long long)todo) - 1;
            todo &= todo - 1;
        }
        update_target(Mg + (long)(d0 + l) * b2, Mg + (long)(k0 + __builtin_amdgcn_readlane(km, l)) * b2, ct);
        ct += 4 - w0;
        return true;
    };
    for (int q = 0; q < cnt; q++) {
        const int2 e = sch.nbr[first + q];
        T *Mik = Mg + (long)__builtin_amdgcn_readfirstlane(e.x) * b2;
        const int rk = __builtin_amdgcn_readfirstlane(e.y);
        k0 = __builtin_amdgcn_readfirstlane(rowpts[rk]);
        const int klen = min(__builtin_amdgcn_readfirstlane(rowpts[rk + 1]) - k0, FACTOR_MAXROW);
        const int ork = __builtin_amdgcn_readfirstlane(u2o[rk]);
        const int ncol = lane < klen ? colind[k0 + lane] : -2;
        // the previous neighbour's updates of A_ik are complete, and A, L free
        if (q > 0) {
            __builtin_amdgcn_s_waitcnt(0x0F70);   // s_waitcnt vmcnt(0)
            __syncthreads();
        }
        wg_load_block_coh(A, (const T *)Mik, b2);
        // lane l: (first) position of the row's column l in row k, and the mask of targets
        km = -1;
        for (int m = klen - 1; m > 0; m--) km = __builtin_amdgcn_readlane(ncol, m) == rcol ? m : km;
        todo = __ballot(lane < len && km > 0 && (lane == 0 || rord > ork));
        __syncthreads();
        if (WAIT) wait_ready(flags + rk, epoch, spin_limit, err);
        const bool diag = todo & 1;
        const T *Mki = Mg + (long)(k0 + (diag ? __builtin_amdgcn_readlane(km, 0) : 0)) * b2;   // U_ki
        todo &= ~1ull;
        T bd[NCB][CPW];
        if (act) {
            T bi[NCB][CPW];
            tl.load_b((const T *)Mg + (long)k0 * b2, bi);               // inv(U_kk)
            if (diag && NCB == 1) tl.load_b(Mki, bd);                   // (two tile columns of both do not fit)
            v4 lc[TPW];
#pragma unroll
            for (int s = 0; s < TPW; s++) lc[s] = (v4){(T)0, (T)0, (T)0, (T)0};
            tl.product(A, bi, lc);
            tl.each([&](int s, int v, int o) {
                L[o] = -lc[s][v];
                *entry(Mik, o) = lc[s][v];
            });
            if (diag && NCB > 1) tl.load_b(Mki, bd);
        }
        __syncthreads();
        if (act && diag) {
            v4 dg[TPW];
#pragma unroll
            for (int s = 0; s < TPW; s++) dg[s] = (v4){(T)0, (T)0, (T)0, (T)0};
            tl.product(L, bd, dg);
            tl.each([&](int s, int v, int o) { Dg[o] += dg[s][v]; });
        }
        w0 = q + 1 == cnt;
        ct = tl.wv - w0;
        l = -1;
        if (!w0)
            while (pair()) {}
    }
    __syncthreads();
    const int r = wg_inverse<NT>(n, Dg, sh, [&] { pair(); }, [&](int i, int c, T v) { coh_store(Mii, i + n * c, v); });
    if (tl.wv > 0)
        while (pair()) {}
    if (tid == 0) info[ri] = r;
}

// The rows of one level: tickets [t0, t1).
template <typename T, int RCH, int CPW>
__global__ void __launch_bounds__(SV_THREADS, RCH == 1 ? 2 : 1)
bilu0_factor_kernel(int bsz, const int *__restrict__ rowpts, const int *__restrict__ colind,
                    const int *__restrict__ u2o, RowSched sch, int t0, int t1, T *Mg, int *__restrict__ info)
{
    extern __shared__ __align__(16) double lds_raw[];
    for (int t = t0 + blockIdx.x; t < t1; t += gridDim.x) {
        factor_row<T, RCH, CPW, false>(bsz, rowpts, colind, u2o, sch, t, Mg, info, (T *)lds_raw, nullptr, 0, 0, nullptr);
        __syncthreads();
    }
}

// The whole factorisation in one launch: the rows in ticket order (the forward levels
// concatenated) to persistent workgroups through an atomic ticket, as in
// bilu0_sweep_syncfree_kernel.  Before reading row k's blocks every wave waits for k's
// ready flag, which holds the launch's epoch once all of k's blocks are final.  A row
// too long for the factorisation is reported through info and still published.
template <typename T, int RCH, int CPW>
__global__ void __launch_bounds__(SV_THREADS, RCH == 1 ? 2 : 1)
bilu0_factor_syncfree_kernel(int bsz, const int *__restrict__ rowpts, const int *__restrict__ colind,
                             const int *__restrict__ u2o, RowSched sch, int n, T *Mg, int *__restrict__ info,
                             unsigned *flags, const unsigned *epoch_p, unsigned *counter, int spin_limit, int *err)
{
    extern __shared__ __align__(16) double lds_raw[];
    __shared__ int sticket;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned epoch = __hip_atomic_load(epoch_p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // (loop control wave-uniform throughout: see bilu0_sweep_syncfree_kernel)
    while (true) {
        if (wv == 0) sticket = __builtin_amdgcn_readfirstlane(atomicAdd(counter, lane == 0 ? 1u : 0u));
        __syncthreads();
        const int t = __builtin_amdgcn_readfirstlane(sticket);
        if (t >= n) break;
        factor_row<T, RCH, CPW, true>(bsz, rowpts, colind, u2o, sch, t, Mg, info, (T *)lds_raw, flags, epoch,
                                      spin_limit, err);
        // publish the row once every wave's stores of it have completed (vmcnt 0:
        // device-scope stores are acknowledged at the coherence point)
        __builtin_amdgcn_s_waitcnt(0x0F70);   // s_waitcnt vmcnt(0)
        __syncthreads();
        if (wv == 0)
            __hip_atomic_store(flags + __builtin_amdgcn_readfirstlane(sch.rows[t].x), epoch, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    }
}

// A new epoch for the factorisation's ready flags (so that they are never cleared)
// and a fresh ticket.
__global__ void factor_reset_kernel(unsigned *sync)
{
    if (threadIdx.x == 0) {
        unsigned e = sync[0] + 1;
        sync[0] = e == 0 ? 1 : e;
        sync[1] = 0;
    }
}

// Block-Jacobi application y_i = inv(H_ii) x_i.  One wave per row.
template <typename TM>
__global__ void __launch_bounds__(SV_THREADS)
block_jacobi_kernel(int nrows, int bsz, const TM *__restrict__ Dinv, const double *__restrict__ x,
                    double *__restrict__ y)
{
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wpb = blockDim.x >> 6;
    const long b2 = (long)bsz * bsz;
    for (int r = blockIdx.x * wpb + wv; r < nrows; r += gridDim.x * wpb) {
        const double *xr = x + (long)r * bsz;
        const double z0 = lane < bsz ? xr[lane] : 0.0, z1 = lane + 64 < bsz ? xr[lane + 64] : 0.0;
        double a0 = 0.0, a1 = 0.0;
        wave_block_matvec(bsz, Dinv + (long)r * b2, z0, z1, a0, a1);
        if (lane < bsz) y[(long)r * bsz + lane] = a0;
        if (lane + 64 < bsz) y[(long)r * bsz + lane + 64] = a1;
    }
}

// ---- GMRES vector kernels ----

// The orthogonalisation is memory bound: classical Gram-Schmidt applied twice reads the
// basis three times (the projections; the update together with the projections of the
// updated w, the basis entries staying in registers; the update together with w's norm).
// No coefficient goes through the host between its launches: every kernel leaves one
// partial sum per workgroup and column, and the workgroups of the next kernel each add
// them up for themselves, in the same order (2 us out of the L2s at 512 workgroups and
// 16 columns, against a launch of its own for a reducing kernel); workgroup 0 also stores
// them to hout, host memory that is read after the iteration's one synchronisation.
// GMRES(30) with a projection kernel, a one-workgroup reduction, a copy and a
// synchronisation per set of coefficients, and now: 55 iterations on 1 705 200 unknowns
// 183 and 157 ms, 35 on 132 300 26.7 and 20.3 ms (the preconditioner's and the matrix's
// products 143 and 17.6 ms of them).

// tot[0..W) = sums over the nblk workgroups of the partial sums of columns i0 ... i0 + W - 1
// of k (zero past the last).  red: SV_THREADS doubles of LDS.
template <int W>
__device__ __forceinline__ void gs_totals(int nblk, int k, int i0, const double *__restrict__ partial, double *tot,
                                          double *red)
{
    const int tid = threadIdx.x, i = tid % W;
    double s = 0.0;
    if (i0 + i < k)
#pragma unroll 8
        for (int b = tid / W; b < nblk; b += SV_THREADS / W) s += partial[(long)b * k + i0 + i];
    red[tid] = s;
    __syncthreads();
#pragma unroll
    for (int st = SV_THREADS / 2; st >= W; st >>= 1) {
        if (tid < st) red[tid] += red[tid + st];
        __syncthreads();
    }
    if (tid < W) tot[tid] = red[tid];
    __syncthreads();
}

// The lanes halve the set of M columns they add up with every exchange (over distance D,
// D / 2, ...); lane l ends with the wave's sum of column l / (64 / M).
template <int M, int D>
__device__ __forceinline__ void gs_fold(double *acc, int lane)
{
    if constexpr (M > 1) {
        const bool up = lane & D;
#pragma unroll
        for (int j = 0; j < M / 2; j++) {
            const double give = up ? acc[j] : acc[j + M / 2], keep = up ? acc[j + M / 2] : acc[j];
            acc[j] = keep + __shfl_xor(give, D);
        }
        gs_fold<M / 2, D / 2>(acc, lane);
    } else if constexpr (D > 0) {
        acc[0] += __shfl_xor(acc[0], D);
        gs_fold<1, D / 2>(acc, lane);
    }
}

// v[j] = V_j[q], j < g <= KG; past the last a column of the last four (its coefficient is
// zero, its projection not used) or zero.
template <int KG>
__device__ __forceinline__ void gs_load(double (&v)[KG], const double *__restrict__ V, long ldv, long q, int g)
{
    constexpr int S = KG < 4 ? KG : 4;
#pragma unroll
    for (int j0 = 0; j0 < KG; j0 += S) {
        if (j0 < g) {
#pragma unroll
            for (int j = j0; j < j0 + S; j++) v[j] = V[min(j, g - 1) * ldv + q];
        } else {
#pragma unroll
            for (int j = j0; j < j0 + S; j++) v[j] = 0.0;
        }
    }
}

// partial[j] = sum over the workgroup of acc[j], j < g <= KG.  red: at least 4 KG doubles
// of LDS.
template <int KG>
__device__ __forceinline__ void gs_partials(double (&acc)[KG], int g, double *__restrict__ partial, double *red)
{
    const int tid = threadIdx.x, lane = tid & 63;
    gs_fold<KG, 32>(acc, lane);
    if (lane % (64 / KG) == 0) red[(tid >> 6) * KG + lane / (64 / KG)] = acc[0];
    __syncthreads();
    if (tid < g) partial[tid] = (red[tid] + red[KG + tid]) + (red[2 * KG + tid] + red[3 * KG + tid]);
    __syncthreads();
}

// The workgroup's slice of a vector of n entries.
__device__ __forceinline__ void gs_slice(long n, long &q0, long &q1)
{
    const long chunk = (n + gridDim.x - 1) / gridDim.x;
    q0 = min(blockIdx.x * chunk, n);
    q1 = min(q0 + chunk, n);
}

// pout: partial sums of V_i . w, i < k (V_i at V + i*ldv); with UPDATE after
// w -= sum_i h_i V_i, h out of the partial sums pin.
template <int KG, bool UPDATE>
__global__ void __launch_bounds__(SV_THREADS)
gs_project_kernel(long n, int k, const double *__restrict__ V, long ldv, double *__restrict__ w,
                  const double *__restrict__ pin, double *__restrict__ pout, double *__restrict__ hout)
{
    __shared__ double red[SV_THREADS], h[KG];
    const int tid = threadIdx.x;
    long q0, q1;
    gs_slice(n, q0, q1);
    if (UPDATE && k > KG)
        for (int i0 = 0; i0 < k; i0 += KG) {
            gs_totals<KG>(gridDim.x, k, i0, pin, h, red);
            const int g = min(KG, k - i0);
            if (blockIdx.x == 0 && tid < g) hout[i0 + tid] = h[tid];
            for (long q = q0 + tid; q < q1; q += SV_THREADS) {
                double s = 0.0;
                for (int j = 0; j < g; j++) s += h[j] * V[(i0 + j) * ldv + q];
                w[q] -= s;
            }
            __syncthreads();
        }
    const bool update = UPDATE && k <= KG;
    if (update) {
        gs_totals<KG>(gridDim.x, k, 0, pin, h, red);
        if (blockIdx.x == 0 && tid < k) hout[tid] = h[tid];
    }
    for (int i0 = 0; i0 < k; i0 += KG) {
        const int g = min(KG, k - i0);
        double acc[KG];
#pragma unroll
        for (int j = 0; j < KG; j++) acc[j] = 0.0;
        for (long q = q0 + tid; q < q1; q += SV_THREADS) {
            double v[KG];
            double wq = w[q];
            gs_load<KG>(v, V + i0 * ldv, ldv, q, g);
            if (update) {
                double s = 0.0;
#pragma unroll
                for (int j = 0; j < KG; j++) s = fma(h[j], v[j], s);
                wq -= s;
                w[q] = wq;
            }
#pragma unroll
            for (int j = 0; j < KG; j++) acc[j] = fma(v[j], wq, acc[j]);
        }
        gs_partials<KG>(acc, g, pout + (long)blockIdx.x * k + i0, red);
    }
}

// w -= sum_i h_i V_i, i < k, h out of the partial sums pin; pout: partial sums of w . w,
// or of d . w if d is given.
template <int KG>
__global__ void __launch_bounds__(SV_THREADS)
gs_update_kernel(long n, int k, const double *__restrict__ V, long ldv, double *__restrict__ w,
                 const double *__restrict__ d, const double *__restrict__ pin, double *__restrict__ pout,
                 double *__restrict__ hout)
{
    __shared__ double red[SV_THREADS], h[KG];
    const int tid = threadIdx.x;
    long q0, q1;
    gs_slice(n, q0, q1);
    double acc[1] = {0.0};
    for (int i0 = 0; i0 < k; i0 += KG) {
        gs_totals<KG>(gridDim.x, k, i0, pin, h, red);
        const int g = min(KG, k - i0);
        const bool last = i0 + KG >= k;
        if (blockIdx.x == 0 && tid < g) hout[i0 + tid] = h[tid];
        for (long q = q0 + tid; q < q1; q += SV_THREADS) {
            double v[KG], s = 0.0;
            const double w0 = w[q], dq = d && last ? d[q] : 0.0;
            gs_load<KG>(v, V + i0 * ldv, ldv, q, g);
#pragma unroll
            for (int j = 0; j < KG; j++) s = fma(h[j], v[j], s);
            const double wq = w0 - s;
            w[q] = wq;
            if (last) acc[0] = fma(d ? dq : wq, wq, acc[0]);
        }
        __syncthreads();
    }
    gs_partials<1>(acc, 1, pout + blockIdx.x, red);
}

// y = x / |x| (nothing if the norm is zero), the square of the norm out of the nblk
// partial sums pin, to *hout too.  x may be y.
__global__ void __launch_bounds__(SV_THREADS)
gs_scale_kernel(long n, int nblk, const double *x, double *y, const double *__restrict__ pin,
                double *__restrict__ hout)
{
    __shared__ double red[SV_THREADS], h[1];
    gs_totals<1>(nblk, 1, 0, pin, h, red);
    if (blockIdx.x == 0 && threadIdx.x == 0) *hout = h[0];
    if (h[0] == 0.0) return;
    const double f = 1.0 / sqrt(h[0]);
    for (long q = blockIdx.x * (long)SV_THREADS + threadIdx.x; q < n; q += (long)gridDim.x * SV_THREADS) y[q] = f * x[q];
}

// w += sign * sum_i coef[i] V_i
__global__ void __launch_bounds__(SV_THREADS)
multi_axpy_kernel(long n, int k, const double *__restrict__ V, long ldv, const double *__restrict__ coef,
                  double sign, double *__restrict__ w)
{
    for (long q = blockIdx.x * (long)blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) {
        double s = 0.0;
        for (int i = 0; i < k; i++) s += coef[i] * V[i * ldv + q];
        w[q] += sign * s;
    }
}

// y = a*x + b*y
__global__ void axpby_kernel(long n, double a, const double *__restrict__ x, double b, double *__restrict__ y)
{
    for (long q = blockIdx.x * (long)blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x)
        y[q] = a * x[q] + b * y[q];
}

__global__ void fill_kernel(long n, double v, double *__restrict__ y)
{
    for (long q = blockIdx.x * (long)blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) y[q] = v;
}

// ---- solution update (getU, solvers/solutionupdate.cpp:6-67) ----
// u_e <- u_e - alpha inv(D)F duh_e + alpha inv(D)Ru, with X = [inv(D)F  inv(D)Ru]
// row-major (na x ldx).  One workgroup per element.
__global__ void __launch_bounds__(SV_THREADS)
update_u_kernel(int ne, int npv, int nc, int nch, int ndf, int na, int nb, int ldx, const int *__restrict__ elcon,
                const double *__restrict__ X, const double *__restrict__ duh, double alpha, double *__restrict__ UDG)
{
    extern __shared__ double de[];
    const int tid = threadIdx.x, nth = blockDim.x;
    for (int e = blockIdx.x; e < ne; e += gridDim.x) {
        for (int q = tid; q < nb; q += nth) {
            const int j = q / nch, k = q % nch;
            de[q] = duh[(long)elcon[(long)e * ndf + j] * nch + k];
        }
        __syncthreads();
        const double *Xe = X + (long)e * na * ldx;
        for (int i = tid; i < na; i += nth) {
            const double *row = Xe + (long)i * ldx;
            double s = 0.0;
            for (int c = 0; c < nb; c++) s += row[c] * de[c];
            double *u = UDG + (long)e * npv * nc + i;
            *u = (*u - alpha * s) + alpha * row[nb];
        }
        __syncthreads();
    }
}

// DIRK stage source (solvers/dgsolvers.cpp:316-349): SH = a*UDGi + b*UDG + c*SH on the
// u components, 0 on the q components.
__global__ void stage_source_kernel(long ne, int npv, int nc, int ncu, double a, const double *__restrict__ UDGi,
                                    double b, const double *__restrict__ UDG, double c, double *__restrict__ SH)
{
    const long n = ne * npv * nc;
    for (long q = blockIdx.x * (long)blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) {
        const int comp = (int)((q / npv) % nc);
        SH[q] = comp < ncu ? (a * UDGi[q] + b * UDG[q]) + c * SH[q] : 0.0;
    }
}

// ---- launchers ----

static int grid_for(long n, int per = SV_THREADS)
{
    long g = (n + per - 1) / per;
    return (int)(g < 1 ? 1 : (g > 4096 ? 4096 : g));
}

static hipError_t set_lds(const void *fn, size_t bytes)
{
    return hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

size_t block_inverse_lds(int bsz)
{
    return sizeof(double) * (bsz * bsz + 1) / 16 * 16 + 16 + InvShared<double>::bytes(bsz);
}
size_t bilu0_factor_lds(int bsz) { return bsz <= MAX_BLOCK ? factor_lds<double>(bsz) : ~(size_t)0 / 2; }

hipError_t launch_block_inverse(int nrows, int bsz, const int *rowpts, const double *Hg, double *Dinv, int *info,
                                hipStream_t s)
{
    const size_t lds = block_inverse_lds(bsz);
    if (bsz < 1 || bsz > MAX_BLOCK) return hipErrorInvalidValue;
    const int nt = (bsz + 15) / 16;
    auto kernel = nt == 1 ? block_inverse_kernel<1> : nt == 2 ? block_inverse_kernel<2> : nt == 3 ? block_inverse_kernel<3>
                : nt == 4 ? block_inverse_kernel<4> : block_inverse_kernel<5>;
    hipError_t e = set_lds((const void *)kernel, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, dim3(std::min(nrows, 8192)), dim3(SV_THREADS), lds, s, nrows, bsz, rowpts, Hg, Dinv,
                       info);
    return hipGetLastError();
}

hipError_t launch_mdf_weights(int nrows, int bsz, const int *rowpts, const double *Hg, const double *Dinv,
                              double *Cw, hipStream_t s)
{
    return block_shape(bsz, [&](auto, auto C) {
        hipLaunchKernelGGL(mdf_weight_kernel<C()>, dim3(std::min(nrows, 8192)), dim3(SV_THREADS),
                           sizeof(double) * bsz * bsz, s, nrows, bsz, rowpts, Hg, Dinv, Cw);
    });
}

template <typename T>
static hipError_t factor_level(int bsz, const int *rowpts, const int *colind, const int *u2o, const RowSched &sch,
                               int t0, int t1, T *Mg, int *info, hipStream_t s)
{
    const size_t lds = factor_lds<T>(bsz);
    return block_shape(bsz, [&](auto R, auto C) {
        if (set_lds((const void *)bilu0_factor_kernel<T, R(), C()>, lds) == hipSuccess)
            hipLaunchKernelGGL((bilu0_factor_kernel<T, R(), C()>), dim3(std::min(t1 - t0, 8192)), dim3(SV_THREADS), lds,
                               s, bsz, rowpts, colind, u2o, sch, t0, t1, Mg, info);
    });
}

template <typename T>
static hipError_t factor_syncfree(int bsz, const int *rowpts, const int *colind, const int *u2o, const RowSched &sch,
                                  int n, T *Mg, int *info, unsigned *flags, unsigned *sync, int nwg, int spin_limit,
                                  int *err, hipStream_t s)
{
    if (n <= 0 || nwg <= 0) return hipErrorInvalidValue;
    const size_t lds = factor_lds<T>(bsz);
    hipLaunchKernelGGL(factor_reset_kernel, dim3(1), dim3(64), 0, s, sync);
    return block_shape(bsz, [&](auto R, auto C) {
        if (set_lds((const void *)bilu0_factor_syncfree_kernel<T, R(), C()>, lds) == hipSuccess)
            hipLaunchKernelGGL((bilu0_factor_syncfree_kernel<T, R(), C()>), dim3(std::min(n, nwg)), dim3(SV_THREADS),
                               lds, s, bsz, rowpts, colind, u2o, sch, n, Mg, info, flags, sync, sync + 1, spin_limit,
                               err);
    });
}

hipError_t launch_bilu0_factor_syncfree(int bsz, const int *rowpts, const int *colind, const int *u2o,
                                        const int4 *rows, const int2 *nbr, int n, double *Mg, int *info,
                                        unsigned *flags, unsigned *sync, int nwg, int spin_limit, int *err,
                                        hipStream_t s)
{
    return factor_syncfree(bsz, rowpts, colind, u2o, RowSched{rows, nbr}, n, Mg, info, flags, sync, nwg, spin_limit,
                           err, s);
}
hipError_t launch_bilu0_factor_syncfree(int bsz, const int *rowpts, const int *colind, const int *u2o,
                                        const int4 *rows, const int2 *nbr, int n, float *Mg, int *info,
                                        unsigned *flags, unsigned *sync, int nwg, int spin_limit, int *err,
                                        hipStream_t s)
{
    return factor_syncfree(bsz, rowpts, colind, u2o, RowSched{rows, nbr}, n, Mg, info, flags, sync, nwg, spin_limit,
                           err, s);
}

hipError_t launch_bilu0_factor_level(int bsz, const int *rowpts, const int *colind, const int *u2o, const int4 *rows,
                                     const int2 *nbr, int t0, int t1, double *Mg, int *info, hipStream_t s)
{
    return factor_level(bsz, rowpts, colind, u2o, RowSched{rows, nbr}, t0, t1, Mg, info, s);
}

hipError_t launch_bilu0_factor_level(int bsz, const int *rowpts, const int *colind, const int *u2o, const int4 *rows,
                                     const int2 *nbr, int t0, int t1, float *Mg, int *info, hipStream_t s)
{
    return factor_level(bsz, rowpts, colind, u2o, RowSched{rows, nbr}, t0, t1, Mg, info, s);
}

template <typename TM>
static hipError_t scale_upper(int bsz, int n, const int *rowpts, const int *colind, const int *u2o, TM *Mg,
                              hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    return block_shape(bsz, [&](auto, auto C) {
        hipLaunchKernelGGL((bilu0_scale_upper_kernel<C(), TM>), dim3(std::min(n, 8192)), dim3(SV_THREADS),
                           sizeof(double) * bsz * bsz, s, bsz, n, rowpts, colind, u2o, Mg);
    });
}
hipError_t launch_bilu0_scale_upper(int bsz, int n, const int *rowpts, const int *colind, const int *u2o,
                                    double *Mg, hipStream_t s)
{
    return scale_upper(bsz, n, rowpts, colind, u2o, Mg, s);
}
hipError_t launch_bilu0_scale_upper(int bsz, int n, const int *rowpts, const int *colind, const int *u2o,
                                    float *Mg, hipStream_t s)
{
    return scale_upper(bsz, n, rowpts, colind, u2o, Mg, s);
}

// Neighbours' shares a sweep keeps in registers (up to about 128 VGPRs of them; the
// sweeps' times hardly change between 2 and 4 at 50 columns).
constexpr int sweep_ahead(int rch, int cpw) { return rch > 1 ? 1 : cpw <= 6 ? 8 : cpw <= 8 ? 6 : cpw <= 12 ? 5 : 4; }

template <bool BACKWARD, typename TM>
static hipError_t sweep_level(int bsz, const RowSched &sch, int t0, int t1, const TM *Mg, const double *x, double *y,
                              hipStream_t s)
{
    return block_shape(bsz, [&](auto R, auto C) {
        constexpr int P = sweep_ahead(R(), C());
        hipLaunchKernelGGL((bilu0_sweep_kernel<BACKWARD, R(), C(), P, TM>), dim3(std::min(t1 - t0, 8192)),
                           dim3(SV_THREADS), 0, s, bsz, sch, t0, t1, Mg, x, y);
    });
}

hipError_t launch_bilu0_lsolve_level(int bsz, const int4 *rows, const int2 *nbr, int t0, int t1, const double *Mg,
                                     const double *x, double *y, hipStream_t s)
{
    return sweep_level<false>(bsz, RowSched{rows, nbr}, t0, t1, Mg, x, y, s);
}
hipError_t launch_bilu0_lsolve_level(int bsz, const int4 *rows, const int2 *nbr, int t0, int t1, const float *Mg,
                                     const double *x, double *y, hipStream_t s)
{
    return sweep_level<false>(bsz, RowSched{rows, nbr}, t0, t1, Mg, x, y, s);
}
hipError_t launch_bilu0_usolve_level(int bsz, const int4 *rows, const int2 *nbr, int t0, int t1, const double *Mg,
                                     const double *y, double *v, hipStream_t s)
{
    return sweep_level<true>(bsz, RowSched{rows, nbr}, t0, t1, Mg, y, v, s);
}
hipError_t launch_bilu0_usolve_level(int bsz, const int4 *rows, const int2 *nbr, int t0, int t1, const float *Mg,
                                     const double *y, double *v, hipStream_t s)
{
    return sweep_level<true>(bsz, RowSched{rows, nbr}, t0, t1, Mg, y, v, s);
}

// Both sweeps of one BILU0 application without level launches: x -> t (forward) ->
// y (backward).  sync: [1], [2] the tickets of the two sweeps.
template <typename TM>
static hipError_t sweeps_syncfree(int bsz, const RowSched &low, const RowSched &up, int n, const TM *Mg, const double *x,
                                  double *t, double *y, unsigned *sync, int nwg, int spin_limit, int *err,
                                  hipStream_t s)
{
    if (n <= 0 || nwg <= 0) return hipErrorInvalidValue;
    const int g = std::min(n, nwg);
    const long N = (long)n * bsz;
    hipLaunchKernelGGL(sweep_reset_kernel, dim3(grid_for(N)), dim3(SV_THREADS), 0, s, sync, N, t, y);
    return block_shape(bsz, [&](auto R, auto C) {
        constexpr int P = sweep_ahead(R(), C());
        hipLaunchKernelGGL((bilu0_sweep_syncfree_kernel<false, R(), C(), P, TM>), dim3(g), dim3(SV_THREADS), 0, s,
                           bsz, low, n, Mg, x, t, sync + 1, spin_limit, err);
        hipLaunchKernelGGL((bilu0_sweep_syncfree_kernel<true, R(), C(), P, TM>), dim3(g), dim3(SV_THREADS), 0, s,
                           bsz, up, n, Mg, t, y, sync + 2, spin_limit, err);
    });
}

hipError_t launch_bilu0_syncfree(int bsz, const int4 *lrows, const int2 *lnbr, const int4 *urows, const int2 *unbr,
                                 int n, const double *Mg, const double *x, double *t, double *y, unsigned *sync,
                                 int nwg, int spin_limit, int *err, hipStream_t s)
{
    return sweeps_syncfree(bsz, RowSched{lrows, lnbr}, RowSched{urows, unbr}, n, Mg, x, t, y, sync, nwg, spin_limit,
                           err, s);
}
hipError_t launch_bilu0_syncfree(int bsz, const int4 *lrows, const int2 *lnbr, const int4 *urows, const int2 *unbr,
                                 int n, const float *Mg, const double *x, double *t, double *y, unsigned *sync,
                                 int nwg, int spin_limit, int *err, hipStream_t s)
{
    return sweeps_syncfree(bsz, RowSched{lrows, lnbr}, RowSched{urows, unbr}, n, Mg, x, t, y, sync, nwg, spin_limit,
                           err, s);
}

template <typename TM>
static hipError_t bj(int nrows, int bsz, const TM *Dinv, const double *x, double *y, hipStream_t s)
{
    if (bsz > MAX_BLOCK) return hipErrorInvalidValue;
    const int wpb = SV_THREADS / 64;
    hipLaunchKernelGGL(block_jacobi_kernel<TM>, dim3(std::min((nrows + wpb - 1) / wpb, 8192)), dim3(SV_THREADS), 0,
                       s, nrows, bsz, Dinv, x, y);
    return hipGetLastError();
}
hipError_t launch_block_jacobi(int nrows, int bsz, const double *Dinv, const double *x, double *y, hipStream_t s)
{
    return bj(nrows, bsz, Dinv, x, y, s);
}
hipError_t launch_block_jacobi(int nrows, int bsz, const float *Dinv, const double *x, double *y, hipStream_t s)
{
    return bj(nrows, bsz, Dinv, x, y, s);
}

__global__ void to_float_kernel(long n, const double *__restrict__ x, float *__restrict__ y)
{
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        y[i] = (float)x[i];
}

hipError_t launch_to_float(long n, const double *x, float *y, hipStream_t s)
{
    hipLaunchKernelGGL(to_float_kernel, dim3(grid_for(n)), dim3(SV_THREADS), 0, s, n, x, y);
    return hipGetLastError();
}

// Workgroups of the orthogonalisation's kernels: two waves' worth of entries and more per
// wave, at most two workgroups per CU (every one adds up all workgroups' partial sums).
int gs_blocks(long n) { return (int)std::min<long>(512, (n + 511) / 512); }

// 1, 8, 16 or 32 columns at a time: the smallest that takes all k at once.
#define GS_COLUMNS(k, F)                                                                                             \
    if (k == 1) { constexpr int KG = 1; F; }                                                                         \
    else if (k <= 8) { constexpr int KG = 8; F; }                                                                    \
    else if (k <= 16) { constexpr int KG = 16; F; }                                                                  \
    else { constexpr int KG = 32; F; }

// pout: gs_blocks(n) * k partial sums of V_i . w, with pin given after w -= sum_i h_i V_i,
// h their totals (stored to hout).
hipError_t launch_gs_project(long n, int k, const double *V, long ldv, double *w, const double *pin, double *pout,
                             double *hout, hipStream_t s)
{
    const dim3 grid(gs_blocks(n)), wg(SV_THREADS);
    GS_COLUMNS(k, {
        if (pin) hipLaunchKernelGGL((gs_project_kernel<KG, true>), grid, wg, 0, s, n, k, V, ldv, w, pin, pout, hout);
        else hipLaunchKernelGGL((gs_project_kernel<KG, false>), grid, wg, 0, s, n, k, V, ldv, w, pin, pout, hout);
    })
    return hipGetLastError();
}

// w -= sum_i h_i V_i, then pout: gs_blocks(n) partial sums of d . w (w . w without d).
hipError_t launch_gs_update(long n, int k, const double *V, long ldv, double *w, const double *d, const double *pin,
                            double *pout, double *hout, hipStream_t s)
{
    const dim3 grid(gs_blocks(n)), wg(SV_THREADS);
    GS_COLUMNS(k, { hipLaunchKernelGGL(gs_update_kernel<KG>, grid, wg, 0, s, n, k, V, ldv, w, d, pin, pout, hout); })
    return hipGetLastError();
}

hipError_t launch_gs_scale(long n, const double *x, double *y, const double *pin, double *hout, hipStream_t s)
{
    hipLaunchKernelGGL(gs_scale_kernel, dim3(gs_blocks(n)), dim3(SV_THREADS), 0, s, n, gs_blocks(n), x, y, pin, hout);
    return hipGetLastError();
}

hipError_t launch_multi_axpy(long n, int k, const double *V, long ldv, const double *coef, double sign, double *w,
                             hipStream_t s)
{
    hipLaunchKernelGGL(multi_axpy_kernel, dim3(grid_for(n)), dim3(SV_THREADS), 0, s, n, k, V, ldv, coef, sign, w);
    return hipGetLastError();
}

hipError_t launch_axpby(long n, double a, const double *x, double b, double *y, hipStream_t s)
{
    hipLaunchKernelGGL(axpby_kernel, dim3(grid_for(n)), dim3(SV_THREADS), 0, s, n, a, x, b, y);
    return hipGetLastError();
}

hipError_t launch_fill(long n, double v, double *y, hipStream_t s)
{
    hipLaunchKernelGGL(fill_kernel, dim3(grid_for(n)), dim3(SV_THREADS), 0, s, n, v, y);
    return hipGetLastError();
}

hipError_t launch_update_u(int ne, int npv, int nc, int nch, int ndf, int na, int nb, int ldx, const int *elcon,
                           const double *X, const double *duh, double alpha, double *UDG, hipStream_t s)
{
    hipLaunchKernelGGL(update_u_kernel, dim3(std::min(ne, 8192)), dim3(SV_THREADS), sizeof(double) * nb, s, ne, npv,
                       nc, nch, ndf, na, nb, ldx, elcon, X, duh, alpha, UDG);
    return hipGetLastError();
}

hipError_t launch_stage_source(long ne, int npv, int nc, int ncu, double a, const double *UDGi, double b,
                               const double *UDG, double c, double *SH, hipStream_t s)
{
    hipLaunchKernelGGL(stage_source_kernel, dim3(grid_for(ne * npv * nc)), dim3(SV_THREADS), 0, s, ne, npv, nc, ncu,
                       a, UDGi, b, UDG, c, SH);
    return hipGetLastError();
}

}  // namespace hfem
