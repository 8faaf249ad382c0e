// The R <= 64 pivoted Cholesky + V^-1 (one 256-thread workgroup), shared by the
// standalone factor kernel (solve.hip) and the GEMM launches that run it in an
// extra workgroup (mttkrp.hip).
#pragma once
#include "dense_la.h"

namespace itcpd {

constexpr size_t FACTOR64_LDS = (size_t)(2 * 64 * 66) * 8;
// LDS of the unpivoted form alone: W (the sweeps' rows before it), D^-1, 16 doubles of reductions
constexpr int FACTOR64_UNPIV = 64 * 64 + 64 + 16;
constexpr size_t FACTOR64_UNPIV_LDS = (size_t)FACTOR64_UNPIV * 8;

// LDS written by lanes of one wave, then read by other lanes of the same wave: the wave's LDS
// operations complete in order, so only the compiler must keep them so.
__device__ __forceinline__ void lds_wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The triangular half of the inverse of a symmetric positive definite n x n matrix A = L D L^T:
// W = L^-1 and the reciprocals of D, in registers.  A thread holds 16 rows (16 grp ..) of one
// column col; rows and columns >= n are zero.  Eliminating index k, with r the k-th row and d =
// r_k: the rows i > k take a_il - r_i r_l / d (r_i, their column k, is their row k by symmetry),
// where column k counts as the identity's (r_k = 1, a_ik = 0 before).  So the columns below k
// collect W and those above the Schur complement, row k is final, and the row being eliminated,
// handed to every thread through LDS, is all that a step needs.  false when a pivot was not > low.
//
// Rows already eliminated take no part.  Updating them too (Gauss-Jordan) would leave A^-1 in
// place without a product, but its rows of size 1 / lambda_min then pass through every later
// update and the error of M A^-1, M = X A, grows with cond(A)^2: 1e-7 at cond(A) = 1e6 and
// wrong in the first digit at 1e9, where W^T D^-1 W, as the triangular inverse of a Cholesky
// factor, has 5e-11 and 4e-7.
//
// A step eliminates k and k + 1 together: p, q their rows, d1 = p_k, c = p_{k+1}, q' = q - (c /
// d1) p, the second pivot e' = q'_{k+1} = det / d1, det = d1 e - c^2, so that both reciprocals
// start at once: the element (i, l) takes a - p_i p_l / d1 - q'_i q'_l / e'.  With an odd n the
// index n is a 1 on the diagonal.  The step's critical chain is 1 / det, the next two rows'
// multiply-adds and their way through LDS: those rows go first and their reads are issued
// before the other rows are updated; d1 and e come from a running copy of the diagonal by
// readlane, not from the rows.
//
// The loop body is short on purpose: unrolled over all steps it is straight-line code that
// every launch fetches anew (27 us at n = 64).  So that registers are not indexed by k, every
// step rotates the rows by two (position j holds row 16 grp + (j + k) mod 16, the rows being
// eliminated sit at positions 0 and 1, the next ones at 2 and 3).  Each row is in LDS by column,
// and once more with its 16-entry groups twice in a row, so a rotated group is one run, and with
// zeros for the rows already eliminated.
//
// WAVES = 1: one wave, n <= 32, grp = lane >> 5, col = lane & 31, rows in LDS order, no
// barrier; WAVES = 4: a 256-thread workgroup, n <= 64, grp = wave, col = lane, one barrier a
// step (two row buffers), and p_i, q_i, which a wave's lanes share, by readlane from one
// LDS read (delivered to every lane they would take 512 cycles of the LDS port a step).
// rows: SWEEP_ROWS doubles of LDS.  KEEP_L: Lt[k ld + i] = L_ik, i > k, in LDS.  On return position
// j holds row sweep_row(n, grp, j) of W and rd the reciprocal of pivot col.
constexpr int SWEEP_BUF = 384;   // rows p, q by column and their runs of 128
constexpr int SWEEP_ROWS = 2 * SWEEP_BUF;

__device__ __forceinline__ int sweep_row(int n, int grp, int j) { return 16 * grp + ((j + n + (n & 1)) & 15); }

__device__ __forceinline__ double lane_double(double v, int k) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), k),
                            __builtin_amdgcn_readlane(__double2loint(v), k));
}
// Wave-wide sum / maximum by DPP row rotations and the four rows' values (uniform result):
// shorter chains than LDS shuffles.
template <int CTRL>
__device__ __forceinline__ double dpp_double(double v) {
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, false),
                            __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ double wave_sum_dpp(double v) {
    v += dpp_double<0x128>(v);   // row_ror:8
    v += dpp_double<0x124>(v);
    v += dpp_double<0x122>(v);
    v += dpp_double<0x121>(v);
    return (lane_double(v, 0) + lane_double(v, 16)) + (lane_double(v, 32) + lane_double(v, 48));
}
__device__ __forceinline__ double wave_max_dpp(double v) {
    v = fmax(v, dpp_double<0x128>(v));
    v = fmax(v, dpp_double<0x124>(v));
    v = fmax(v, dpp_double<0x122>(v));
    v = fmax(v, dpp_double<0x121>(v));
    return fmax(fmax(lane_double(v, 0), lane_double(v, 16)), fmax(lane_double(v, 32), lane_double(v, 48)));
}
__device__ __forceinline__ double newton_rcp(double d) {
    // the estimate's error e (< 2^-20) cubed
    const double y = __builtin_amdgcn_rcp(d), e = fma(-d, y, 1.0);
    return fma(y, fma(e, e, e), y);
}

template <int WAVES, bool KEEP_L>
__device__ __forceinline__ bool sweep_triangular(double (&a)[16], int n, int grp, int col, double low, double* rows,
                                                 double& rd, double* Lt = nullptr, int ld = 0) {
    auto sync = [] {
        if (WAVES == 1) lds_wave_order();
        else __syncthreads();
    };
    const int at = 32 * (col >> 4) + (col & 15);   // this column's place in a row's runs
    auto put = [&](double* buf, int q, int k, double v) {   // row q of the pair k, k + 1
        const double run = col > k + 1 ? v : 0.0;
        buf[64 * q + col] = v;
        buf[128 + 128 * q + at] = run;
        buf[128 + 128 * q + at + 16] = run;
    };
    double dg = 0.0;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const bool here = 16 * grp + i == col;
        a[i] = here && (n & 1) && col == n ? 1.0 : a[i];
        dg = here ? a[i] : dg;
    }
    if (col >> 4 == grp) rows[SWEEP_BUF + col] = dg;
    if (grp == 0) {
        put(rows, 0, 0, a[0]);
        put(rows, 1, 0, a[1]);
    }
    sync();
    dg = rows[SWEEP_BUF + col];
    rd = 0.0;
    const int lane = threadIdx.x & 63;
    // the rows' entries of this column and of this group
    double pl, ql;
    auto fetch = [&](const double* buf, int k, double (&p)[16], double (&q)[16]) {
        const double* run = buf + 128 + 32 * grp + (k & 15);
        pl = buf[col];
        ql = buf[64 + col];
        if (WAVES == 4) {
            p[0] = run[lane & 15];
            q[0] = run[128 + (lane & 15)];
        } else {
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                p[j] = run[j];
                q[j] = run[128 + j];
            }
        }
    };
    double pa[16], qa[16], pb[16], qb[16];
    fetch(rows, 0, pa, qa);
    sync();   // the diagonal's place is the next rows'
    bool pos = true;
    // the step of rows k, k + 1 in (p, q); the next two go to (pn, qn)
    auto step = [&](int k, double (&p)[16], double (&q)[16], double (&pn)[16], double (&qn)[16]) {
        const double d1 = lane_double(dg, k), e = lane_double(dg, k + 1), c = lane_double(pl, k + 1);
        const double det = fma(d1, e, -c * c);
        pos = pos && d1 > low && det > low * d1;
        const double r1 = newton_rcp(d1), r2 = d1 * newton_rcp(det), m = c * r1;
        const double q2 = fma(-m, pl, ql);
        double t1 = pl * r1, t2 = q2 * r2;
        const bool c1 = col == k, c2 = col == k + 1;
        const double l0 = t1, l1 = t2;   // above the diagonal, L's columns k and k + 1
        // the diagonal as the rows' own updates; four waves after the next rows, which wait for less
        if (WAVES == 1) dg = fma(-q2, l1, fma(-pl, l0, dg));
        t1 = c1 ? r1 : (c2 ? 0.0 : t1);
        t2 = c1 ? -m * r2 : (c2 ? r2 : t2);
        const double keep = c1 || c2 ? 0.0 : 1.0;
        const double ps = p[0], qs = fma(-m, p[0], q[0]);
        auto multiplier = [&](int j) {
            if (WAVES == 4) {
                p[j] = lane_double(ps, j);
                q[j] = lane_double(qs, j);
            } else {
                q[j] = fma(-m, p[j], q[j]);
            }
        };
        multiplier(2);
        multiplier(3);
        double* next = rows + SWEEP_BUF * ((k / 2 + 1) & 1);
        if ((k + 2) >> 4 == grp) {
            const double v2 = fma(-p[2], t1, a[2] * keep), v3 = fma(-p[3], t1, a[3] * keep);
            put(next, 0, k + 2, fma(-q[2], t2, v2));
            put(next, 1, k + 2, fma(-q[3], t2, v3));
        }
        if (WAVES == 4) {
            __builtin_amdgcn_sched_barrier(0);
            dg = fma(-q2, l1, fma(-pl, l0, dg));
        }
        // rows k and k + 1 of W: their multipliers are zero, so they are final from here on
        const bool own = k >> 4 == grp, below = col < k;
        a[0] = own ? (c1 ? 1.0 : (below ? pl : 0.0)) : a[0] * keep;
        a[1] = own ? (c1 ? -m : (c2 ? 1.0 : (below ? q2 : 0.0))) : a[1] * keep;
        rd = c1 ? r1 : (c2 ? r2 : rd);
        if (KEEP_L && own) {
            Lt[k * ld + col] = l0;
            Lt[(k + 1) * ld + col] = l1;
        }
        sync();
        fetch(next, k + 2, pn, qn);
        // a <- a keep - p t1 - q t2 in passes of 16 independent operations
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 16; ++j)
            if (j != 2 && j != 3) multiplier(j);
#pragma unroll
        for (int j = 2; j < 16; ++j) a[j] *= keep;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 16; ++j) a[j] = fma(-p[j], t1, a[j]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 16; ++j) a[j] = fma(-q[j], t2, a[j]);
        __builtin_amdgcn_sched_barrier(0);
        const double x0 = a[0], x1 = a[1];
#pragma unroll
        for (int j = 0; j < 14; ++j) a[j] = a[j + 2];
        a[14] = x0;
        a[15] = x1;
    };
#pragma unroll 1
    for (int k = 0;; k += 4) {
        step(k, pa, qa, pb, qb);
        if (k + 2 >= n) break;
        step(k + 2, pb, qb, pa, qa);
        if (k + 4 >= n) break;
    }
    return pos;
}

// W = L^-1 in LDS as the operand of W^T D^-1 W: entry (r, k) of rows of ld (32 or 64) doubles,
// odd rows with their 16-column groups swapped in pairs, so that two rows of a read meet
// distinct banks.
__device__ __forceinline__ int tri_at(int ld, int r, int k) { return r * ld + (k ^ ((r & 1) << 4)); }

// One Newton step Z <- Z + Z (I - V Z) for the inverse Z of V = Hadamard of the Grams of modes !=
// mode, by the 256 threads of a workgroup on MFMA; returns the thread's share of ||I - V Z||_F^2.
// D: 64 x 64 doubles of LDS.
//
// W is a left inverse of L to rounding (each of its columns is a substitution) and a right one only
// to eps cond(V), so V W^T D^-1 W is off the identity by up to eps cond(V)^1.5; after the step
// by that squared plus the step's own eps cond(V).  X from M = X V, worst of 6 seeds, without / with / by
// the pivoted substitution: cond(V) 1e6 1e-10 / 1e-11 / 2e-11; 5e7 9e-8 / 5e-10 / 1e-9; 1e9 4e-6 / 2e-8 /
// 2e-8.  Up to NEWTON_COND all are within a few units of eps cond(V), and the step would cost, us: R =
// 10 3.6, 24 6.0, 37 8.6, 64 11.6.
constexpr double NEWTON_COND = 1e5;
__device__ __forceinline__ double newton_inverse(const GramSet& gs, int mode, int R, double* Z, double* D) {
    const int l = threadIdx.x & 63, c = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = 16 * w + c;   // this lane's row of the left operands
    d4 acc[4];
    double dsq = 0.0;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[b][v] = 16 * w + g + 4 * v == 16 * b + c ? 1.0 : 0.0;
    for (int k0 = 0; k0 < R; k0 += 16) {   // four k-steps' loads in flight
        double a[4], z[4][4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int k = k0 + 4 * s + g;
            a[s] = k < R && i < R ? -1.0 : 0.0;
#pragma unroll
            for (int b = 0; b < 4; ++b) z[s][b] = Z[k < R && 16 * b + c < R ? k * R + 16 * b + c : 0];
        }
        for (int m = 0; m < gs.N; ++m) {
            if (m == mode) continue;
            const double* __restrict__ G = gs.G[m];
            double v[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) v[s] = G[k0 + 4 * s + g < R && i < R ? (k0 + 4 * s + g) * R + i : 0];
#pragma unroll
            for (int s = 0; s < 4; ++s) a[s] *= v[s];
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int b = 0; b < 4; ++b)
                acc[b] = mfma_f64(a[s], k0 + 4 * s + g < R && 16 * b + c < R ? z[s][b] : 0.0, acc[b]);
    }
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = 16 * w + g + 4 * v, j = 16 * b + c;
            if (r < R && j < R) dsq = fma(acc[b][v], acc[b][v], dsq);
            D[r * 64 + j] = acc[b][v];
            acc[b][v] = r < R && j < R ? Z[r * R + j] : 0.0;
        }
    __syncthreads();
    for (int k0 = 0; k0 < R; k0 += 16) {
        double a[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int k = k0 + 4 * s + g;
            a[s] = Z[k < R && i < R ? i * R + k : 0];
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int k = k0 + 4 * s + g;
#pragma unroll
            for (int b = 0; b < 4; ++b) acc[b] = mfma_f64(k < R && i < R ? a[s] : 0.0, D[k * 64 + 16 * b + c], acc[b]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = 16 * w + g + 4 * v, j = 16 * b + c;
            if (r < R && j < R) Z[r * R + j] = acc[b][v];
        }
    return dsq;
}

// Unpivoted V^-1 for the R <= 64 row solves (one 256-thread workgroup; the first wave alone
// up to R = 32).
//
// It stands in for the pivoted factorisation (xPSTRF, absolute tolerance tol) only
// when that one provably keeps every pivot: each pivoted pivot is a diagonal entry
// of a Schur complement of V, hence >= lambda_min(V), and lambda_min(V) >=
// 1 / ||V^-1||_F.  The computed inverse is trusted while ||V||_F ||V^-1||_F < cond_max;
// the bound must exceed 2 tol plus the pivots' rounding (64 R eps max V_ii); every
// unpivoted pivot must be > 0; and past NEWTON_COND, where a Newton step follows, the
// ||I - V V^-1||_F^2 before it must be below eps cond(V).  Then the solution (the unique
// minimiser) is the pivoted path's up to rounding (eps cond(V)), and V^-1 and finfo are
// written; otherwise it returns false and writes nothing but V^-1 (which the caller's
// pivoted path overwrites or leaves unused).  Uniform result.
//
// Bound by its chain of R / 2 steps, 0.5 us each, on one wave per SIMD.  The Hadamard-reduce of
// 64 x 64 x 64 that carries it takes, us: R = 10 7.2, 16 8.6, 24 11.5, 37 17.9, 64 25.5 (Gauss-Jordan
// 6.6, 7.8, 9.4, 16.2, 22.8; the blocked Cholesky, triangular inverse and product of them
// before that 11 at R = 10, 17 at 24, 19 at 37, 29 at 64).
// SMALL = false: R > 32 only, in a kernel whose registers the one-wave form would not fit.
template <bool SMALL = true>
__device__ __forceinline__ bool factor64_unpivoted(const GramSet& gs, int mode, int R, double tol,
                                                   double* __restrict__ Vinv, int* __restrict__ finfo,
                                                   double* S, double cond_max = 1e12) {
    double* red = S + 64 * 64 + 64;   // behind W (before it the sweeps' rows) and D^-1
    const int t = threadIdx.x, l = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const bool one = SMALL && R <= 32;
    if (!one || w == 0) {
        const int grp = one ? l >> 5 : w, col = one ? l & 31 : l;
        // V in the mode order of the pivoted path's Hadamard; two modes' loads in flight
        double a[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) a[i] = 1.0;
        for (int m0 = 0; m0 < gs.N; m0 += 2) {
            const bool on0 = m0 != mode, on1 = m0 + 1 < gs.N && m0 + 1 != mode;
            const double* __restrict__ G0 = gs.G[m0];
            const double* __restrict__ G1 = on1 ? gs.G[m0 + 1] : G0;
            double g0[16], g1[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int r = 16 * grp + i, x = (r < R && col < R) ? r * R + col : 0;
                g0[i] = G0[x];
                g1[i] = G1[x];
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                if (!on0) g0[i] = 1.0;
                if (!on1) g1[i] = 1.0;
                a[i] = (a[i] * g0[i]) * g1[i];
            }
        }
        double vsq = 0.0, dmax = 0.0, zsq = 0.0;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int r = 16 * grp + i;
            if (r >= R || col >= R) a[i] = 0.0;
            vsq = fma(a[i], a[i], vsq);
            if (r == col) dmax = fmax(dmax, a[i]);
        }
        double rd;
        const bool pos = one ? sweep_triangular<1, false>(a, R, grp, col, 0.0, S, rd)
                             : sweep_triangular<4, false>(a, R, grp, col, 0.0, S, rd);
        // V^-1 = W^T D^-1 W by upper tiles, 16 rows of W (4 k-steps) read ahead of their products
        double* dinv = S + 64 * 64;
        const int ld = one ? 32 : 64, c = l & 15, g = l >> 4;
        auto sync = [&] {
            if (one) lds_wave_order();
            else __syncthreads();
        };
        sync();
        if (grp == 0) dinv[col] = rd;
#pragma unroll
        for (int i = 0; i < 16; ++i) S[tri_at(ld, sweep_row(R, grp, i), col)] = a[i];
        sync();
        auto tile = [&](int ta, int tb, const d4& z) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int ra = 16 * ta + g + 4 * v, rb = 16 * tb + c;
                if (ra >= R || rb >= R) continue;
                Vinv[ra * R + rb] = z[v];
                if (ta != tb) Vinv[rb * R + ra] = z[v];
                zsq = fma(ta == tb ? z[v] : 2.0 * z[v], z[v], zsq);
            }
        };
        // rows 16 kb .. of a column block of W, and the same times D^-1
        auto load = [&](double (&x)[4], int kb, int t) {
#pragma unroll
            for (int s = 0; s < 4; ++s) x[s] = S[tri_at(ld, 16 * kb + 4 * s + g, 16 * t + c)];
        };
        auto scaled = [&](const double (&x)[4], int kb, double (&y)[4]) {
#pragma unroll
            for (int s = 0; s < 4; ++s) y[s] = x[s] * dinv[16 * kb + 4 * s + g];
        };
        auto product = [&](const double (&x)[4], const double (&y)[4], d4& z) {
#pragma unroll
            for (int s = 0; s < 4; ++s) z = mfma_f64(x[s], y[s], z);
        };
        const d4 zero = (d4){0.0, 0.0, 0.0, 0.0};
        if (one) {
            double x00[4], x10[4], x11[4], y[4];
            d4 z00 = zero, z01 = zero, z11 = zero;
            load(x00, 0, 0);
            load(x10, 1, 0);
            load(x11, 1, 1);
            scaled(x00, 0, y);
            product(x00, y, z00);
            if (R > 16) {
                scaled(x11, 1, y);
                product(x10, y, z01);
                product(x11, y, z11);
                scaled(x10, 1, y);
                product(x10, y, z00);
                tile(0, 1, z01);
                tile(1, 1, z11);
            }
            tile(0, 0, z00);
        } else {
            constexpr int ZT[4][3][2] = {{{0, 0}, {0, 3}, {-1, -1}},
                                         {{0, 1}, {1, 3}, {2, 3}},
                                         {{1, 1}, {0, 2}, {-1, -1}},
                                         {{1, 2}, {2, 2}, {3, 3}}};   // 20 k-steps a wave
            const int nt = (R + 15) / 16;
#pragma unroll 1
            for (int q = 0; q < 3; ++q) {
                const int ta = ZT[w][q][0], tb = ZT[w][q][1];
                if (ta < 0 || tb >= nt) continue;
                d4 z = zero;
                double x0[4], w0[4], x1[4], w1[4], y[4];
                load(x0, tb, ta);
                load(w0, tb, tb);
                for (int kb = tb; kb < nt; kb += 2) {
                    const int k1 = kb + 1 < 4 ? kb + 1 : 3, k2 = kb + 2 < 4 ? kb + 2 : 3;   // past the last: not used
                    load(x1, k1, ta);
                    load(w1, k1, tb);
                    scaled(w0, kb, y);
                    product(x0, y, z);
                    if (kb + 1 >= nt) break;
                    load(x0, k2, ta);
                    load(w0, k2, tb);
                    scaled(w1, k1, y);
                    product(x1, y, z);
                }
                tile(ta, tb, z);
            }
        }
        vsq = wave_sum_dpp(vsq);
        zsq = wave_sum_dpp(zsq);
        dmax = wave_max_dpp(dmax);
        if (l == 0) {
            red[w] = vsq;
            red[4 + w] = dmax;
            red[8 + w] = zsq;
            if (w == 0) red[12] = pos ? 0.0 : 1.0;
        }
    }
    __syncthreads();
    double vs = red[0], dmax = red[4], zs = red[8];
    if (!one)
        for (int q = 1; q < 4; ++q) {
            vs += red[q];
            dmax = fmax(dmax, red[4 + q]);
            zs += red[8 + q];
        }
    const double vF = sqrt(vs), zF = sqrt(zs);
    bool cert = red[12] == 0.0 && zF > 0.0 && zF < __builtin_inf() &&
                1.0 / zF > 2.0 * tol + 64.0 * R * 0x1p-52 * dmax && vF * zF < cond_max;
    if (cert && vF * zF > NEWTON_COND) {
        const double d = wave_sum_dpp(newton_inverse(gs, mode, R, Vinv, S));
        if (l == 0) red[w] = d;
        __syncthreads();
        cert = (red[0] + red[1]) + (red[2] + red[3]) < 0x1p-52 * vF * zF;
    }
    if (cert && t == 0) {
        finfo[0] = R;
        finfo[1] = 0;
        finfo[2] = R;
    }
    __syncthreads();   // S is reused by the pivoted path
    return cert;
}

// Pivoted Cholesky for R <= 64 (dpstrf semantics as k_factor: absolute tolerance,
// the first step only checks d > 0): pivot p is the remaining index with the
// largest V(p,p) - sum_t U(t,p)^2 (first index on ties).  Right-looking on
// registers: thread (w, l) holds rows 16w..16w+15 of column l of the Schur
// complement; each step the wave owning row p hands it to all waves through LDS,
// u_l = S(p, l) / U(j,j) for the remaining l, and every thread applies the rank-1
// update to its 16 entries.  The pivot search runs redundantly in every wave on
// identical data (the same u, the same running sums), so all waves agree without
// communication.  UbT(l, j) = U(j, l) (zero for finished l) with ld 66.
// Output in pivoted order: Uperm(j, t) = u^(j)_{piv[t]}, invdiag(j) = 1/U(j,j);
// with Vinv, also V^-1 (R x R).  On rank deficiency all four waves build the QR
// data.
// Device function so that a GEMM launch can run it in one extra workgroup
// (256 threads, FACTOR64_LDS bytes of dynamic LDS).
__device__ __forceinline__ void factor64_dev(GramSet gs, int mode, int R, double tol,
                                          double* __restrict__ Uperm, double* __restrict__ Vinv,
                                          double* __restrict__ invdiag, int* __restrict__ piv,
                                          int* __restrict__ finfo, double* __restrict__ W,
                                          double* __restrict__ qtau, double* __restrict__ ztau,
                                          int* __restrict__ jpvt, double* vwork,
                                          bool try_unpivoted = true) {
    constexpr int LDT = 66;
    extern __shared__ double S[];   // V (ld R), later U^-1 (ld LDT): 64 x LDT | UbT: 64 x LDT
    __shared__ double diagU[64];
    __shared__ double invdU[64];
    __shared__ double rowb[2][64];
    __shared__ int pivS[64];
    __shared__ int s_rank;
    __shared__ double redv[256];
    __shared__ int redi[256];
    double* UbT = S + 64 * LDT;
    const int t = threadIdx.x, l = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    if (Vinv && try_unpivoted && factor64_unpivoted(gs, mode, R, tol, Vinv, finfo, S)) return;
    fill_hadamard<256>(S, gs, mode, R * R);
    __syncthreads();
    d16 sr;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int m = 16 * w + i;
        sr[i] = (m < R && l < R) ? S[m * R + l] : 0.0;
    }
    bool rem = l < R;
    const double vdiag = rem ? S[l * R + l] : 0.0;
    double sumsq = 0.0;
    uint64_t remmask = R >= 64 ? ~0ull : ((1ull << R) - 1);
    int rank = R;
    // Software pipelined: at the top of step j the registers hold the Schur
    // complement with the updates of steps < j-1 applied; step j-1's rank-1 update
    // (this wave's 16 entries of row p_{j-1} in rw, coefficient cu = u_l /
    // U(j-1,j-1)) is pending.  The owner of row p_j corrects just that entry before
    // handing the row over, and every wave applies the pending update after the
    // barrier, while its LDS reads are in flight.  The pivot search needs only the
    // running sums.
    // One step; rc holds the pending row values, the new ones go to rn (the loop
    // below alternates two register sets instead of copying).  False when the
    // pivot fails the tolerance test (rank = j).
    double cu = 0.0;
    auto step = [&](int j, const d16& rc, d16& rn) -> bool {
        double d;
        const int p = wave_first_max(rem ? vdiag - sumsq : -__builtin_inf(), d);
        const bool bad = (p >= R) || !((remmask >> p) & 1) || ((j == 0) ? !(d > 0.0) : !(d > tol));
        if (bad) { rank = j; return false; }
        if (w == (p >> 4)) rowb[j & 1][l] = fma(-rc[p & 15], cu, sr[p & 15]);
        remmask &= ~(1ull << p);
        if (l == p) rem = false;
        __syncthreads();
        // rows of finished indices take the update too (never read again), so the
        // 16 row values are plain loads with no per-row condition
        const double* rb = rowb[j & 1];
        const double rl = rb[l];
#pragma unroll
        for (int i = 0; i < 16; ++i) rn[i] = rb[16 * w + i];
#pragma unroll
        for (int i = 0; i < 16; ++i) sr[i] = fma(-rc[i], cu, sr[i]);
        // 1/sqrt(d) from the hardware estimate (relative error < 2^-22) and two
        // Newton steps y <- y + y (1/2 - d y^2 / 2); U(j,j) = d / sqrt(d).  d > 0
        // here; the clamp keeps the estimate finite below 2^-1020.
        const double dc = fmax(d, 0x1p-1020);
        const double h = 0.5 * dc;
        double y = __builtin_amdgcn_rsq(dc);
        y = fma(y, fma(-h * y, y, 0.5), y);
        y = fma(y, fma(-h * y, y, 0.5), y);
        const double inv = y, ujj = dc * y;
        const double u = rem ? rl * inv : 0.0;
        sumsq = fma(u, u, sumsq);
        cu = u * inv;
        if (t == 0) { diagU[j] = ujj; invdU[j] = inv; pivS[j] = p; }
        if (w == 0 && l < R) UbT[l * LDT + j] = u;
        return true;
    };
    d16 rwa, rwb;
#pragma unroll
    for (int i = 0; i < 16; ++i) { rwa[i] = 0.0; rwb[i] = 0.0; }
    for (int j = 0; j < R; j += 2) {
        if (!step(j, rwa, rwb)) break;
        if (j + 1 >= R || !step(j + 1, rwb, rwa)) break;
    }
    if (t == 0) s_rank = rank;
    __syncthreads();
    if (s_rank == R) {
        for (int j = t; j < R; j += 256) {
            invdiag[j] = invdU[j];
            piv[j] = pivS[j];
        }
        if (!Vinv) {
            for (int x = t; x < R * R; x += 256) {
                const int j = x / R, tt = x % R;
                double v = 0.0;
                if (tt > j) v = UbT[pivS[tt] * LDT + j];
                else if (tt == j) v = diagU[j];
                Uperm[x] = v;
            }
        } else {
            // V^-1 = P U^-1 U^-T P^T for the MFMA row solves.  U in pivoted order,
            // Up(i, k) = U(i, piv k) = UbT(piv k, i) for i < k < R (identity beyond
            // R), is read in place; U^-1 goes to Ui (the S region, ld LDT) by 16 x 16
            // blocks: diagonal blocks by substitution (wave b, lane c: column c of
            // block b), then X_ij = -X_ii sum_{k=i+1..j} Up_ik X_kj by block
            // diagonals on MFMA; finally the upper tiles of Z = U^-1 U^-T on MFMA
            // (Z(a, b) sums over k >= max(a, b) only) and Vinv(piv a, piv b) =
            // Vinv(piv b, piv a) = Z(a, b).  f64 16x16x4 MFMA layout: A lane (c, g)
            // = A[c][k0+g], B lane = B[k0+g][c], result v = D[g+4v][c]; the result of
            // one product is the B operand of the next one as it stands (k0 = 4v).
            const int c = l & 15, g = l >> 4;
            double* Ui = S;
            if (t >= R && t < 64) invdU[t] = 1.0;
            for (int x = t; x < 64 * 64; x += 256) {
                const int i = x >> 6, k = x & 63;
                if ((i >> 4) > (k >> 4)) Ui[i * LDT + k] = 0.0;
            }
            __syncthreads();
            if (l < 16) {
                const int b0 = 16 * w;
                int pk[16];
#pragma unroll
                for (int k = 0; k < 16; ++k) pk[k] = (b0 + k < R) ? pivS[b0 + k] * LDT : -1;
                double xv[16];
#pragma unroll
                for (int i = 15; i >= 0; --i) {
                    double acc0 = (i == l) ? 1.0 : 0.0, acc1 = 0.0;
#pragma unroll
                    for (int k = i + 1; k < 16; ++k) {
                        const double uik = pk[k] >= 0 ? UbT[pk[k] + b0 + i] : 0.0;
                        if (k & 1) acc1 -= uik * xv[k];
                        else acc0 -= uik * xv[k];
                    }
                    xv[i] = (i <= l) ? (acc0 + acc1) * invdU[b0 + i] : 0.0;
                }
#pragma unroll
                for (int i = 0; i < 16; ++i) Ui[(b0 + i) * LDT + b0 + l] = xv[i];
            }
            __syncthreads();
            for (int dd = 1; dd < 4; ++dd) {
                const int bi = w, bj = w + dd;
                if (bj < 4) {
                    const int i = 16 * bi + c;
                    d4 acc = (d4){0.0, 0.0, 0.0, 0.0};
                    for (int bk = bi + 1; bk <= bj; ++bk)
#pragma unroll
                        for (int k0 = 0; k0 < 16; k0 += 4) {
                            const int kk = 16 * bk + k0 + g;
                            const double a = (kk < R && i < R) ? UbT[pivS[kk] * LDT + i] : 0.0;
                            acc = mfma_f64(a, Ui[kk * LDT + 16 * bj + c], acc);
                        }
                    d4 out = (d4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        out = mfma_f64(-Ui[(16 * bi + c) * LDT + 16 * bi + 4 * v + g], acc[v], out);
#pragma unroll
                    for (int v = 0; v < 4; ++v) Ui[(16 * bi + g + 4 * v) * LDT + 16 * bj + c] = out[v];
                }
                __syncthreads();
            }
            // upper tiles (ta <= tb) of Z, 20 k-steps per wave
            constexpr int ZT[4][3][2] = {{{0, 0}, {0, 3}, {-1, -1}},
                                         {{0, 1}, {1, 3}, {2, 3}},
                                         {{1, 1}, {0, 2}, {-1, -1}},
                                         {{1, 2}, {2, 2}, {3, 3}}};
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const int ta = ZT[w][q][0], tb = ZT[w][q][1];
                if (ta < 0 || 16 * tb >= R) continue;
                d4 acc = (d4){0.0, 0.0, 0.0, 0.0};
                for (int k0 = 16 * tb; k0 < 64; k0 += 4)
                    acc = mfma_f64(Ui[(16 * ta + c) * LDT + k0 + g], Ui[(16 * tb + c) * LDT + k0 + g], acc);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int ra = 16 * ta + g + 4 * v, rb = 16 * tb + c;
                    if (ra < R && rb < R) {
                        Vinv[pivS[ra] * R + pivS[rb]] = acc[v];
                        if (ta != tb) Vinv[pivS[rb] * R + pivS[ra]] = acc[v];
                    }
                }
            }
        }
        if (t == 0) { finfo[0] = R; finfo[1] = 0; finfo[2] = R; }
        return;
    }
    qr_fallback<256>(gs, mode, R, W, qtau, ztau, jpvt, vwork, finfo, redv, redi, s_rank);
}


}  // namespace itcpd
