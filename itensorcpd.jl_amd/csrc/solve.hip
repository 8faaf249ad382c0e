// Per-mode update on the device: the R x R normal-equation solve, row_norm,
// the Gram refresh, and (after the last mode) the fit and the convergence check.
//
// Reference semantics restated here:
//  * solve_ls_problem -> ldiv_solve!! (algebra/ldiv_solve.jl:13-29):
//    cholesky(Hermitian(V), RowMaximum(), check=true, tol=1e-6) \ M^T, i.e. LAPACK
//    xPSTRF (upper) + xPOTRS; when the pivoted Cholesky stops early (rank < R)
//    the bare `catch` falls back to qr(V, ColumnNorm()) \ M^T, whose Julia
//    implementation is the xGELSY scheme: xGEQP3, rank by incremental condition
//    estimation (xLAIC1) at rcond = R*eps, complete orthogonal decomposition
//    (xTZRZF), Q^T (xORMQR), triangular solve, Z^T (xORMRZ), un-permute.
//    (LAPACK 3.x as shipped with OpenBLAS 0.3.x is the third-party code the
//    reference calls; its published algorithms are restated, not linked.)
//  * row_norm (math_tools/row_norm.jl:4-24): lambda_r = sqrt(sum_i X(i,r)^2),
//    A = X ./ lambda.
//  * post_solve (algorithms/als_algorithms/standard/tensor.jl:46-49): G_n = A_n^T A_n.
//  * check_converge (converge_checks/fit_check.jl:24-66, no_check.jl:8-20,
//    converge_checks.jl:5-11).
#include "dense_la.h"
#include "factor64.h"
#include "inverse.h"

namespace itcpd {

// The certified inverse of inverse.h stands for the pivoted factorisation: its status,
// finfo[3] = 1, and true; else finfo[3] = 0 and the pivoted kernel goes on.
__device__ __forceinline__ bool wide_exit(const double* __restrict__ stat, int nb, int R, double tol,
                                          int* __restrict__ finfo) {
    const bool ok = wide_certified(stat, nb, R, tol);
    if (threadIdx.x == 0) {
        finfo[3] = ok ? 1 : 0;
        if (ok) {
            finfo[0] = R;
            finfo[1] = 0;
            finfo[2] = R;
        }
    }
    return ok;
}

// ------------------------------------------------------------ factorisation
// One workgroup.  Builds V = Hadamard of the Grams of modes != mode, factors it
// with pivoted Cholesky (upper, right-looking, pivot = largest remaining diagonal,
// first index on ties; stop when the pivot is <= tol, or <= 0 / NaN at the first
// step).  Full rank: U (row-major, ld R) and piv are written, finfo[1] = 0.
// Otherwise the column-pivoted QR solve data are prepared in W (column-major):
// Householder vectors below the diagonal, T11 and the RZ vectors above it, with
// qtau, ztau, jpvt, and finfo[2] = numerical rank; finfo[1] = 1.
__global__ __launch_bounds__(FACTOR_THREADS) void k_factor(GramSet gs, int mode, int R, double tol,
                                                           double* __restrict__ U,
                                                           double* __restrict__ invdiag,
                                                           int* __restrict__ piv,
                                                           int* __restrict__ finfo,
                                                           double* __restrict__ W,
                                                           double* __restrict__ qtau,
                                                           double* __restrict__ ztau,
                                                           int* __restrict__ jpvt, double* vwork,
                                                           const double* __restrict__ stat, int nb,
                                                           const DevCheck* __restrict__ chk) {
    if (chk->done) return;
    if (wide_exit(stat, nb, R, tol, finfo)) return;
    __shared__ double redv[FACTOR_THREADS];
    __shared__ int redi[FACTOR_THREADS];
    const int t = threadIdx.x;
    constexpr int NT = FACTOR_THREADS;
    double* S = U;  // full symmetric R x R, row-major
    int* pv = piv;

    // V = ones .* G_m for m != mode, in mode order (MttkrpAlgorithm.jl:38-47)
    fill_hadamard<NT>(S, gs, mode, R * R);
    for (int i = t; i < R; i += NT) pv[i] = i;
    __syncthreads();

    int rank = R;
    for (int j = 0; j < R; ++j) {
        const int p = block_argmax<NT>(j, R, [&](int i) { return S[i * R + i]; }, redv, redi);
        const double d = (p < R) ? S[p * R + p] : __builtin_nan("");
        const bool bad = (j == 0) ? !(d > 0.0) : !(d > tol);
        if (bad) { rank = j; break; }
        if (p != j) {
            // symmetric swap of indices j and p in the trailing block, and of
            // columns j and p in the finished rows 0..j-1 of U
            for (int k = t; k < R; k += NT) {
                if (k >= j) {
                    const double a = S[j * R + k];
                    S[j * R + k] = S[p * R + k];
                    S[p * R + k] = a;
                }
            }
            __syncthreads();
            for (int k = t; k < R; k += NT) {
                const double a = S[k * R + j];
                S[k * R + j] = S[k * R + p];
                S[k * R + p] = a;
            }
            if (t == 0) {
                const int q = pv[j];
                pv[j] = pv[p];
                pv[p] = q;
            }
            __syncthreads();
        }
        const double ujj = sqrt(S[j * R + j]);
        const double inv = 1.0 / ujj;
        __syncthreads();
        if (t == 0) S[j * R + j] = ujj;
        for (int k = j + 1 + t; k < R; k += NT) S[j * R + k] *= inv;
        __syncthreads();
        // trailing update of both triangles: S(k,l) -= U(j,k) U(j,l)
        const int n = R - j - 1;
        for (int x = t; x < n * n; x += NT) {
            const int k = j + 1 + x / n, l = j + 1 + x % n;
            S[k * R + l] -= S[j * R + k] * S[j * R + l];
        }
        __syncthreads();
    }

    if (rank == R) {
        // U = the factor (upper triangle of S; strict lower triangle zeroed)
        for (int x = t; x < R * R; x += NT) {
            const double v = (x % R) >= (x / R) ? S[x] : 0.0;
            U[x] = v;
        }
        for (int j = t; j < R; j += NT) invdiag[j] = 1.0 / S[j * R + j];
        if (t == 0) { finfo[0] = R; finfo[1] = 0; finfo[2] = R; }
        return;
    }
    qr_fallback<NT>(gs, mode, R, W, qtau, ztau, jpvt, vwork, finfo, redv, redi, rank);
}

// Pivoted Cholesky for 64 < R <= 128: the register form of factor64_dev on 16
// waves.  Thread (w, l) holds rows 16 (w >> 1) .. + 15 of column l + 64 (w & 1)
// of the Schur complement (V from the Grams, straight into registers); each step
// the two waves owning row p hand it to all waves through LDS and every thread
// applies the rank-1 update (one step late, as in factor64_dev).  Every wave runs
// the pivot search over all 128 candidates (columns l and l + 64 of each lane) on
// identical data.  Same pivot rule and outputs as k_factor: Uperm(j, t) =
// U(j, piv t) in pivoted order, invdiag, piv; on rank deficiency the QR data.
constexpr int F128_LDT = 129;
constexpr size_t F128_LDS = (size_t)128 * F128_LDT * 8;

__global__ __launch_bounds__(1024) void k_factor128(GramSet gs, int mode, int R, double tol,
                                                    double* __restrict__ Uperm,
                                                    double* __restrict__ invdiag,
                                                    int* __restrict__ piv, int* __restrict__ finfo,
                                                    double* __restrict__ W, double* __restrict__ qtau,
                                                    double* __restrict__ ztau, int* __restrict__ jpvt,
                                                    double* vwork, const double* __restrict__ stat, int nb,
                                                    const DevCheck* __restrict__ chk) {
    if (chk->done) return;
    if (wide_exit(stat, nb, R, tol, finfo)) return;
    constexpr int LDT = F128_LDT;
    extern __shared__ double UbT[];   // UbT(l, j) = U(j, l), 128 x LDT
    __shared__ double diagU[128];
    __shared__ double invdU[128];
    __shared__ double rowb[2][128];
    __shared__ int pivS[128];
    __shared__ int s_rank;
    __shared__ double redv[1024];
    __shared__ int redi[1024];
    const int t = threadIdx.x, l = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int h = w & 1, row0 = 16 * (w >> 1);
    const int col = l + 64 * h;

    d16 sr;
    double vda = 0.0, vdb = 0.0;
    {
        double v[16];
        double da = 1.0, db = 1.0;
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = 1.0;
        for (int m = 0; m < gs.N; ++m) {
            if (m == mode) continue;
            const double* __restrict__ G = gs.G[m];
            double gv[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int row = row0 + i;
                gv[i] = (row < R && col < R) ? G[row * R + col] : 0.0;
            }
            const double ga = l < R ? G[l * R + l] : 0.0;
            const double gb = l + 64 < R ? G[(l + 64) * R + l + 64] : 0.0;
#pragma unroll
            for (int i = 0; i < 16; ++i) v[i] *= gv[i];
            da *= ga;
            db *= gb;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) sr[i] = v[i];
        vda = l < R ? da : 0.0;
        vdb = l + 64 < R ? db : 0.0;
    }
    // remaining indices: bit l of maska (index l) and of maskb (index 64 + l)
    uint64_t maska = R >= 64 ? ~0ull : ((1ull << R) - 1);
    uint64_t maskb = R >= 128 ? ~0ull : ((1ull << (R - 64)) - 1);
    double suma = 0.0, sumb = 0.0, cu = 0.0;
    int rank = R;
    // rc: the pending row (step j-1's row p, this thread's 16 rows), applied with cu
    d16 rc;
#pragma unroll
    for (int i = 0; i < 16; ++i) rc[i] = 0.0;
    for (int j = 0; j < R; ++j) {
        double d;
        const bool rema = (maska >> l) & 1, remb = (maskb >> l) & 1;
        const int p = wave_first_max2(rema ? vda - suma : -__builtin_inf(),
                                      remb ? vdb - sumb : -__builtin_inf(), d);
        const bool live = p < 64 ? ((maska >> p) & 1) : (p < 128 && ((maskb >> (p - 64)) & 1));
        const bool bad = (p >= R) || !live || ((j == 0) ? !(d > 0.0) : !(d > tol));
        if (bad) { rank = j; break; }
        if ((w >> 1) == (p >> 4)) rowb[j & 1][col] = fma(-rc[p & 15], cu, sr[p & 15]);
        if (p < 64) maska &= ~(1ull << p);
        else maskb &= ~(1ull << (p - 64));
        __syncthreads();
        const double* rb = rowb[j & 1];
        const double rla = rb[l], rlb = rb[l + 64];
#pragma unroll
        for (int i = 0; i < 16; ++i) sr[i] = fma(-rc[i], cu, sr[i]);
#pragma unroll
        for (int i = 0; i < 16; ++i) rc[i] = rb[row0 + i];
        // 1/sqrt(d): hardware estimate and two Newton steps (as factor64_dev)
        const double dc = fmax(d, 0x1p-1020);
        const double hh = 0.5 * dc;
        double y = __builtin_amdgcn_rsq(dc);
        y = fma(y, fma(-hh * y, y, 0.5), y);
        y = fma(y, fma(-hh * y, y, 0.5), y);
        const double inv = y, ujj = dc * y;
        const double ua = ((maska >> l) & 1) ? rla * inv : 0.0;
        const double ub = ((maskb >> l) & 1) ? rlb * inv : 0.0;
        suma = fma(ua, ua, suma);
        sumb = fma(ub, ub, sumb);
        cu = (h ? ub : ua) * inv;
        if (t == 0) { diagU[j] = ujj; invdU[j] = inv; pivS[j] = p; }
        if (w == 0) {
            if (l < R) UbT[l * LDT + j] = ua;
            if (l + 64 < R) UbT[(l + 64) * LDT + j] = ub;
        }
    }
    if (t == 0) s_rank = rank;
    __syncthreads();
    if (s_rank == R) {
        for (int j = t; j < R; j += 1024) {
            invdiag[j] = invdU[j];
            piv[j] = pivS[j];
        }
        for (int x = t; x < R * R; x += 1024) {
            const int j = x / R, tt = x - j * R;
            double v = 0.0;
            if (tt > j) v = UbT[pivS[tt] * LDT + j];
            else if (tt == j) v = diagU[j];
            Uperm[x] = v;
        }
        if (t == 0) { finfo[0] = R; finfo[1] = 0; finfo[2] = R; }
        return;
    }
    qr_fallback<1024>(gs, mode, R, W, qtau, ztau, jpvt, vwork, finfo, redv, redi, s_rank);
}

__global__ __launch_bounds__(256) void k_factor64(GramSet gs, int mode, int R, double tol,
                                                  double* __restrict__ Uperm,
                                                  double* __restrict__ Vinv,
                                                  double* __restrict__ invdiag,
                                                  int* __restrict__ piv, int* __restrict__ finfo,
                                                  double* __restrict__ W, double* __restrict__ qtau,
                                                  double* __restrict__ ztau, int* __restrict__ jpvt,
                                                  double* vwork, const DevCheck* __restrict__ chk) {
    // no test of the done flag: the factorisation writes only the row solves' inputs
    // (V^-1, pivots, status), which the later kernels of a finished run ignore, and
    // the test's round trip would precede the Gram loads
    (void)chk;
    factor64_dev(gs, mode, R, tol, Uperm, Vinv, invdiag, piv, finfo, W, qtau, ztau, jpvt, vwork);
}

// Row solves and Gram tiles (no cross-block communication inside the kernel):
// block b takes row tiles of rpb = 4 * RPW rows; each wave solves RPW rows at once
// (their dependency chains interleave), x_i = V^{-1} m_i through U^T z = P^T m_i,
// U w = z, x = P w (xPOTRS on the pivoted factor, reciprocal diagonal); m_i is kept
// in Msum when given.
// X is written to global memory and to an LDS tile whose X^T X is accumulated
// into gram_part[b].  The QR fallback applies Q^T, T11^{-1}, Z^T row by row.
template <int RQ, int RPW>
__device__ __forceinline__ void solve_rows_dev(
    const double* __restrict__ Msrc, int64_t In, int R,
    const double* __restrict__ Ug, const double* __restrict__ invdiag, const int* __restrict__ piv,
    const int* __restrict__ finfo, const double* __restrict__ W, const double* __restrict__ qtau,
    const double* __restrict__ ztau, const int* __restrict__ jpvt, int u_in_lds,
    double* __restrict__ X, double* __restrict__ Msum, double* __restrict__ gram_part, int grams,
    int nparts = 1, int64_t pstride = 0) {
    constexpr int RPB = 4 * RPW;
    extern __shared__ double lds[];
    const int t = threadIdx.x;
    const int lane = t & 63, wave = t >> 6;
    const bool fallback = finfo[1] != 0;
    double* Xs = lds;                                   // RPB x R tile
    double* Us = lds + (size_t)RPB * R;                 // R x (R+1) when u_in_lds
    const int ldu = R + 1;
    const double* U = Ug;
    int uld = R;
    if (!fallback && u_in_lds) {
        for (int x0 = t; x0 < R * R; x0 += 256 * 16) {
            double v[16];
#pragma unroll
            for (int k = 0; k < 16; ++k) v[k] = (x0 + 256 * k < R * R) ? Ug[x0 + 256 * k] : 0.0;
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const int x = x0 + 256 * k;
                if (x < R * R) Us[(x / R) * ldu + (x % R)] = v[k];
            }
        }
        U = Us;
        uld = ldu;
    }
    __syncthreads();
    int pk[RQ];
    double ivd[RQ];
#pragma unroll
    for (int q = 0; q < RQ; ++q) {
        const int k = lane + 64 * q;
        pk[q] = (k < R) ? (fallback ? jpvt[k] : piv[k]) : 0;
        ivd[q] = (k < R && !fallback) ? invdiag[k] : 0.0;
    }
    const int rk = fallback ? finfo[2] : R;
    double* gp = gram_part + (int64_t)blockIdx.x * R * R;
    bool first_tile = true;
    for (int64_t i0 = (int64_t)blockIdx.x * RPB; i0 < In; i0 += (int64_t)gridDim.x * RPB) {
        const int nr = (int)((In - i0) < RPB ? (In - i0) : RPB);
        const int rbase = wave * RPW;
        double y[RPW][RQ];
#pragma unroll
        for (int rr = 0; rr < RPW; ++rr)
#pragma unroll
            for (int q = 0; q < RQ; ++q) {
                const int k = lane + 64 * q;
                const bool ok = rbase + rr < nr && k < R;
                const int64_t off = ok ? i0 + rbase + rr + In * (fallback ? k : pk[q]) : 0;
                double m = Msrc[off];
#pragma unroll 1
                for (int b = 1; b < nparts; ++b) m += Msrc[(int64_t)b * pstride + off];
                y[rr][q] = m;
            }
        if (Msum) {
#pragma unroll
            for (int rr = 0; rr < RPW; ++rr)
#pragma unroll
                for (int q = 0; q < RQ; ++q) {
                    const int k = lane + 64 * q;
                    if (rbase + rr < nr && k < R)
                        Msum[i0 + rbase + rr + In * (fallback ? k : pk[q])] = y[rr][q];
                }
        }
        if (!fallback) {
            // forward: U^T z = y (rows interleaved)
            for (int j = 0; j < R; ++j) {
                double uj[RQ];
#pragma unroll
                for (int q = 0; q < RQ; ++q) {
                    const int k = lane + 64 * q;
                    uj[q] = (k > j && k < R) ? U[j * uld + k] : 0.0;
                }
                const double ij = bcast<RQ>(ivd, j);
#pragma unroll
                for (int rr = 0; rr < RPW; ++rr) {
                    const double zj = bcast<RQ>(y[rr], j) * ij;
#pragma unroll
                    for (int q = 0; q < RQ; ++q) {
                        const int k = lane + 64 * q;
                        if (k == j) y[rr][q] = zj;
                        else y[rr][q] -= uj[q] * zj;
                    }
                }
            }
            // backward: U w = z
            for (int j = R - 1; j >= 0; --j) {
                double uj[RQ];
#pragma unroll
                for (int q = 0; q < RQ; ++q) {
                    const int k = lane + 64 * q;
                    uj[q] = (k < j) ? U[k * uld + j] : 0.0;
                }
                const double ij = bcast<RQ>(ivd, j);
#pragma unroll
                for (int rr = 0; rr < RPW; ++rr) {
                    const double wj = bcast<RQ>(y[rr], j) * ij;
#pragma unroll
                    for (int q = 0; q < RQ; ++q) {
                        const int k = lane + 64 * q;
                        if (k == j) y[rr][q] = wj;
                        else y[rr][q] -= uj[q] * wj;
                    }
                }
            }
        } else {
#pragma unroll
            for (int rr = 0; rr < RPW; ++rr) fallback_apply<RQ>(y[rr], lane, R, rk, W, qtau, ztau);
        }
#pragma unroll
        for (int rr = 0; rr < RPW; ++rr) {
            if (rbase + rr >= nr) continue;
            const int64_t i = i0 + rbase + rr;
#pragma unroll
            for (int q = 0; q < RQ; ++q) {
                const int k = lane + 64 * q;
                if (k < R) {
                    X[i + In * pk[q]] = y[rr][q];
                    Xs[(rbase + rr) * R + pk[q]] = y[rr][q];
                }
            }
        }
        if (grams) {
            __syncthreads();
            for (int x = t; x < R * R; x += 256) {
                const int r = x % R, r2 = x / R;
                double sacc = 0.0;
                for (int ii = 0; ii < nr; ++ii) sacc += Xs[ii * R + r] * Xs[ii * R + r2];
                gp[x] = first_tile ? sacc : gp[x] + sacc;
            }
        }
        __syncthreads();
        first_tile = false;
    }
}

template <int RQ, int RPW>
__global__ __launch_bounds__(256) void k_solve(
    const double* __restrict__ Msrc, int64_t In, int R,
    const double* __restrict__ Ug, const double* __restrict__ invdiag, const int* __restrict__ piv,
    const int* __restrict__ finfo, const double* __restrict__ W, const double* __restrict__ qtau,
    const double* __restrict__ ztau, const int* __restrict__ jpvt, int u_in_lds,
    double* __restrict__ X, const DevCheck* __restrict__ chk) {
    if (chk->done || finfo[3] == 1) return;   // certified: k_solve_inv solved the rows
    solve_rows_dev<RQ, RPW>(Msrc, In, R, Ug, invdiag, piv, finfo, W, qtau, ztau, jpvt, u_in_lds, X, nullptr,
                            nullptr, 0);
}

// Row solves for R <= RT <= 64.  Cholesky case: X = M V^-1 on FP64 MFMA with the
// explicit V^-1 the factor kernel formed.  Blocks of 256 threads take 16-row
// tiles (grid stride); wave w < RT/16 owns output columns 16w..16w+15 and keeps
// its V^-1 column panel in registers for all tiles (the other waves only join the
// barriers).  f64 16x16x4 layout: A lane (c, g) = A[c][k0+g], B lane =
// B[k0+g][c], result v = D[g+4v][c].  The wave's result tile is, as it stands,
// the A operand of X^T X over the tile's rows (k0 = 4v), so the block's Gram
// partial needs only the other waves' tiles from LDS; it stays in registers
// across tiles and is written once.  All loads of a tile are issued before the
// first MFMA.  M is copied to Msum when asked.  QR fallback case: the same
// blocks run the row-by-row fallback solve (16-row tiles as well, so the Gram
// partials line up), with dynamic LDS for its 16 x R tile.
template <int RT>
__device__ __forceinline__ bool solve_mfma_rows(const double* __restrict__ Msrc, int64_t In, int R,
                                                const double* __restrict__ Vinv, double* __restrict__ X,
                                                double* __restrict__ Msum, double* __restrict__ gram_part,
                                                int grams, int nparts, int64_t pstride,
                                                const int* __restrict__ finfo,
                                                const DevCheck* __restrict__ chk) {
    constexpr int NT = RT / 16, KS = RT / 4, LDX = RT + 2;
    __shared__ double Xs[16 * LDX];
    __shared__ double Ms[16 * LDX];   // the tile's rows of M when M comes as partials
    // the done flag and the factorisation's status are requested with the first
    // tile's operands and tested before the first store: false = QR fallback
    const int gdone = chk->done, gfb = finfo[1];
    bool first = true;
    const int t = threadIdx.x, l = t & 63, c = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const bool active = w < NT;
    const int col = 16 * w + c;
    const bool colok = active && col < R;
    double bv[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const int k = 4 * ks + g;
        bv[ks] = (colok && k < R) ? Vinv[k * R + col] : 0.0;
    }
    d4 gacc[NT];
#pragma unroll
    for (int tb = 0; tb < NT; ++tb) gacc[tb] = (d4){0.0, 0.0, 0.0, 0.0};
    for (int64_t i0 = (int64_t)blockIdx.x * 16; i0 < In; i0 += (int64_t)gridDim.x * 16) {
        if (nparts > 1) {
            // M = sum of the partials in increasing order (as k_sum_parts): wave w
            // sums columns 16w..16w+15 of the tile's rows, 8 partials of each of its
            // 4 entries in flight, into LDS
            if (active) {
                const int64_t ia = i0 + c;
                const bool aok = ia < In;
                double sv[4] = {0.0, 0.0, 0.0, 0.0};
                const double* src[4];
                bool in[4];
#pragma unroll
                for (int h = 0; h < 4; ++h) {
                    const int k = 16 * w + 4 * h + g;
                    in[h] = aok && k < R;
                    src[h] = Msrc + (in[h] ? ia + In * k : 0);
                }
                int b = 0;
#pragma unroll 1
                for (; b + 8 <= nparts; b += 8) {
                    double v[4][8];
#pragma unroll
                    for (int h = 0; h < 4; ++h)
#pragma unroll
                        for (int z = 0; z < 8; ++z) v[h][z] = src[h][(int64_t)(b + z) * pstride];
#pragma unroll
                    for (int h = 0; h < 4; ++h)
#pragma unroll
                        for (int z = 0; z < 8; ++z) sv[h] += in[h] ? v[h][z] : 0.0;
                }
#pragma unroll 1
                for (; b < nparts; ++b)
#pragma unroll
                    for (int h = 0; h < 4; ++h) sv[h] += in[h] ? src[h][(int64_t)b * pstride] : 0.0;
#pragma unroll
                for (int h = 0; h < 4; ++h) Ms[c * LDX + 16 * w + 4 * h + g] = sv[h];
            }
            __syncthreads();
        }
        d4 acc = (d4){0.0, 0.0, 0.0, 0.0};
        const int64_t ia = i0 + c;
        const bool aok = ia < In;
        double av[KS];
        if (active) {
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const int k = 4 * ks + g;
                av[ks] = nparts > 1 ? Ms[c * LDX + k] : ((aok && k < R) ? Msrc[ia + In * k] : 0.0);
            }
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) acc = mfma_f64(av[ks], bv[ks], acc);
        }
        if (first) {
            first = false;
            if (gdone) return true;
            if (gfb) return false;
        }
        if (active) {
            if (Msum) {
#pragma unroll
                for (int ks = 4 * w; ks < 4 * w + 4; ++ks) {
                    const int k = 4 * ks + g;
                    if (aok && k < R) Msum[ia + In * k] = av[ks];
                }
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int64_t row = i0 + g + 4 * v;
                if (row < In && colok) X[row + In * col] = acc[v];
            }
        }
        if (grams) {
            // rows >= In and columns >= R of acc are zero (their operands were)
            if (active) {
#pragma unroll
                for (int v = 0; v < 4; ++v) Xs[(g + 4 * v) * LDX + col] = acc[v];
            }
            __syncthreads();
            if (active) {
#pragma unroll
                for (int tb = 0; tb < NT; ++tb)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        gacc[tb] = mfma_f64(acc[v], Xs[(4 * v + g) * LDX + 16 * tb + c], gacc[tb]);
            }
            __syncthreads();
        } else if (nparts > 1) {
            __syncthreads();   // Ms is rewritten by the next tile
        }
    }
    if (gdone) return true;
    if (gfb) return false;
    if (grams && active) {
        double* gp = gram_part + (int64_t)blockIdx.x * R * R;
#pragma unroll
        for (int tb = 0; tb < NT; ++tb)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = 16 * w + g + 4 * v, r2 = 16 * tb + c;
                if (r < R && r2 < R) gp[r * R + r2] = gacc[tb][v];
            }
    }
    return true;
}

template <int RT>
__global__ __launch_bounds__(256) void k_solve_mfma(const double* __restrict__ Msrc, int64_t In, int R,
                                                    const double* __restrict__ Vinv,
                                                    const int* __restrict__ finfo,
                                                    const double* __restrict__ W,
                                                    const double* __restrict__ qtau,
                                                    const double* __restrict__ ztau,
                                                    const int* __restrict__ jpvt,
                                                    double* __restrict__ X, double* __restrict__ Msum,
                                                    double* __restrict__ gram_part, int grams,
                                                    int nparts, int64_t pstride,
                                                    const DevCheck* __restrict__ chk) {
    if (!solve_mfma_rows<RT>(Msrc, In, R, Vinv, X, Msum, gram_part, grams, nparts, pstride, finfo, chk))
        solve_rows_dev<1, 4>(Msrc, In, R, nullptr, nullptr, nullptr, finfo, W, qtau, ztau, jpvt, 0, X, Msum,
                             gram_part, grams, nparts, pstride);
}

// row_norm + post_solve across blocks, after the row solves:
// lambda_r = sqrt(sum_b gram_part[b](r,r)) (every block, fixed order); block k
// writes its slice of G = S ./ (lambda lambda^T) (S = sum_b gram_part[b]) and of the
// rows A = X ./ lambda, At; with `inner_part` it also sums <M, A .* lambda> over
// its rows.  hold (nullable): nonzero when X was not set, and the CPD stays as it is.
__global__ __launch_bounds__(256) void k_finalize(const double* __restrict__ gram_part, int nb,
                                                  const double* __restrict__ X,
                                                  const double* __restrict__ Msum, int64_t In, int R,
                                                  int Rp, double* __restrict__ A,
                                                  double* __restrict__ At, double* __restrict__ lam,
                                                  double* __restrict__ Gout,
                                                  double* __restrict__ inner_part,
                                                  const int* __restrict__ hold,
                                                  const DevCheck* __restrict__ chk) {
    if (chk->done || (hold && *hold)) return;
    extern __shared__ double lamS[];
    __shared__ double red[256];
    const int t = threadIdx.x;
    const int64_t RR = (int64_t)R * R;
    for (int r = t; r < R; r += 256) {
        lamS[r] = sqrt(sum_parts_at(gram_part, RR, nb, (int64_t)r * R + r));
        if (blockIdx.x == 0) lam[r] = lamS[r];
    }
    __syncthreads();
    const int64_t gchunk = (RR + gridDim.x - 1) / gridDim.x;
    const int64_t g0 = (int64_t)blockIdx.x * gchunk;
    const int64_t g1 = g0 + gchunk < RR ? g0 + gchunk : RR;
    for (int64_t x = g0 + t; x < g1; x += 256) {
        const double sacc = sum_parts_at(gram_part, RR, nb, x);
        const int r = (int)(x % R), r2 = (int)(x / R);
        Gout[x] = sacc / (lamS[r] * lamS[r2]);
    }
    const int64_t rchunk = (In + gridDim.x - 1) / gridDim.x;
    const int64_t i0 = (int64_t)blockIdx.x * rchunk;
    const int64_t i1 = i0 + rchunk < In ? i0 + rchunk : In;
    const int nr = (int)(i1 > i0 ? i1 - i0 : 0);
    double inner = 0.0;
    for (int x0 = t; x0 < nr * R; x0 += 256 * 4) {
        double xv[4], mv[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int x = x0 + 256 * k;
            const bool ok = x < nr * R;
            const int64_t off = ok ? i0 + (x % nr) + In * (x / nr) : 0;
            xv[k] = ok ? X[off] : 0.0;
            mv[k] = (ok && inner_part) ? Msum[off] : 0.0;
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int x = x0 + 256 * k;
            if (x >= nr * R) continue;
            const int ii = x % nr, r = x / nr;
            const int64_t i = i0 + ii;
            const double a = xv[k] / lamS[r];
            A[i + In * r] = a;
            At[i * Rp + r] = a;
            if (inner_part) inner += mv[k] * (a * lamS[r]);
        }
    }
    if (inner_part) {
        inner = block_sum<256>(inner, red);
        if (t == 0) inner_part[blockIdx.x] = inner;
    }
}

// k_finalize when every load of a block fits one round trip: nb <= 32 Gram
// partials, R <= 256, a Gram chunk of at most 256 entries and at most 2048 row
// entries per block.  The done flag, the partials of the diagonal (thread t < R:
// entry (t, t)) and of the block's chunk (one entry per thread) and the block's
// rows of X (and M) are all requested before the first wait; the sums run in
// increasing partial order as in k_finalize, so the results are the same.
__global__ __launch_bounds__(256) void k_finalize_1rt(const double* __restrict__ gram_part, int nb,
                                                      const double* __restrict__ X,
                                                      const double* __restrict__ Msum, int64_t In, int R,
                                                      int Rp, double* __restrict__ A,
                                                      double* __restrict__ At, double* __restrict__ lam,
                                                      double* __restrict__ Gout,
                                                      double* __restrict__ inner_part,
                                                      const int* __restrict__ hold,
                                                      const DevCheck* __restrict__ chk) {
    __shared__ double lamS[256];
    __shared__ double red[256];
    const int t = threadIdx.x;
    const int done = chk->done | (hold ? *hold : 0);
    const int64_t RR = (int64_t)R * R;
    const bool dr = t < R;
    const int64_t xd = dr ? (int64_t)t * R + t : 0;
    const int64_t gchunk = (RR + gridDim.x - 1) / gridDim.x;
    const int64_t g0 = (int64_t)blockIdx.x * gchunk;
    const int64_t g1 = g0 + gchunk < RR ? g0 + gchunk : RR;
    const int64_t xg = g0 + t;
    const bool gr = xg < g1;
    const int64_t rchunk = (In + gridDim.x - 1) / gridDim.x;
    const int64_t i0 = (int64_t)blockIdx.x * rchunk;
    const int64_t i1 = i0 + rchunk < In ? i0 + rchunk : In;
    const int nr = (int)(i1 > i0 ? i1 - i0 : 0);
    // unconditional loads from clamped (valid) addresses, masked afterwards: no
    // branch separates a load from its use, so all are in flight together
    double dv[32], gv[32], xv[8], mv[8];
#pragma unroll
    for (int k = 0; k < 32; ++k) {
        const int64_t kb = (int64_t)(k < nb ? k : 0) * RR;
        dv[k] = gram_part[kb + xd];
        gv[k] = gram_part[kb + (gr ? xg : 0)];
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int x = t + 256 * q;
        const bool ok = x < nr * R;
        const int64_t off = ok ? i0 + (x % nr) + In * (x / nr) : 0;
        xv[q] = X[off];
        mv[q] = Msum[off];
    }
    double ds = 0.0, gsum = 0.0;
#pragma unroll
    for (int k = 0; k < 32; ++k) {
        if (k < nb) {
            ds += dv[k];
            gsum += gv[k];
        }
    }
    if (done) return;
    if (dr) {
        lamS[t] = sqrt(ds);
        if (blockIdx.x == 0) lam[t] = lamS[t];
    }
    __syncthreads();
    if (gr) Gout[xg] = gsum / (lamS[(int)(xg % R)] * lamS[(int)(xg / R)]);
    double inner = 0.0;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int x = t + 256 * q;
        if (x >= nr * R) continue;
        const int ii = x % nr, r = x / nr;
        const int64_t i = i0 + ii;
        const double a = xv[q] / lamS[r];
        A[i + In * r] = a;
        At[i * Rp + r] = a;
        if (inner_part) inner += mv[q] * (a * lamS[r]);
    }
    if (inner_part) {
        inner = block_sum<256>(inner, red);
        if (t == 0) inner_part[blockIdx.x] = inner;
    }
}

// NoCheck's state after a sweep.
__device__ __forceinline__ void count_sweep(DevCheck* chk) {
    chk->iter += 1;
    chk->sweeps += 1;
    if (chk->iter == chk->max_counter) {
        chk->iter = 0;
        chk->done = 1;
    }
}

// After the last mode of a sweep: the fit from <T,X> (sum of the finalize blocks'
// partials, fixed order) and ||X||^2 = lambda^T (G_0 .* ... .* G_{N-1}) lambda, then
// the check update (FitCheck) or the sweep count (NoCheck).
constexpr int FIT_THREADS = 1024;   // R = 64: 5.3 us (6.3 with 256)
__global__ __launch_bounds__(FIT_THREADS) void k_fit(const double* __restrict__ inner_part, int nbf, int R,
                                             GramSet gs, const double* __restrict__ lam,
                                             double* __restrict__ scal, DevCheck* __restrict__ chk,
                                             double* __restrict__ trace, int trace_cap) {
    if (chk->done) return;
    __shared__ double red[FIT_THREADS / 64];
    const int t = threadIdx.x;
    if (chk->kind == ITCPD_CHECK_NONE) {
        if (t == 0) count_sweep(chk);
        return;
    }
    double fs = 0.0;
    const double inner = t == 0 ? sum_parts_at(inner_part, 1, nbf, 0) : 0.0;
    for (int x0 = t; x0 < R * R; x0 += FIT_THREADS * 4) {
        double h[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) h[k] = 1.0;
        for (int m = 0; m < gs.N; ++m) {
            const double* __restrict__ G = gs.G[m];
            double g[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int x = x0 + FIT_THREADS * k;
                g[k] = G[x < R * R ? x : 0];
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) h[k] *= g[k];
        }
        double l1[4], l2[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int x = x0 + FIT_THREADS * k;
            l1[k] = lam[(x < R * R ? x : 0) % R];
            l2[k] = lam[(x < R * R ? x : 0) / R];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (x0 + FIT_THREADS * k < R * R) fs += h[k] * (l1[k] * l2[k]);
    }
    fs = wave_sum_dpp(fs);
    if ((t & 63) == 0) red[t >> 6] = fs;
    __syncthreads();
    if (t == 0) {
        for (int k = 1; k < FIT_THREADS / 64; ++k) fs += red[k];
        check_update(chk, inner, fs, scal, trace, trace_cap);
    }
}

// The whole update of a short mode in one workgroup, R <= RT <= 32: row solve, Gram, row_norm
// and after the last mode the fit.  Wave w takes rows 16w..16w+15 with their tile of X in
// registers throughout: as the product's result it is both operands of X^T X (k0 = 4v), so
// only the waves' Gram tiles meet in LDS.  Otherwise the same as k_solve_mfma, k_finalize and
// k_fit, whose launches cost more than their work here.
template <int RT>
__global__ __launch_bounds__(RT == 16 ? 1024 : 512) void k_update_small(
    const double* __restrict__ Msrc, int nparts, int64_t pstride, int In, int R, int Rp,
    const double* __restrict__ Vinv, const int* __restrict__ finfo, const double* __restrict__ W,
    const double* __restrict__ qtau, const double* __restrict__ ztau, const int* __restrict__ jpvt, double* X,
    double* __restrict__ A, double* __restrict__ At, double* __restrict__ lam, double* __restrict__ Gout,
    int mode, GramSet gs, int fit, double* __restrict__ scal, DevCheck* __restrict__ chk,
    double* __restrict__ trace, int trace_cap) {
    constexpr int NT = RT / 16, KS = RT / 4, NP = NT * (NT + 1) / 2, LDS_ = RT + 1, NH = RT * RT / 256;
    __shared__ double part[(RT == 16 ? 16 : 8) * NP * 256];
    __shared__ double S[RT * LDS_];
    __shared__ double lamS[RT];
    __shared__ double red[32];
    const int t = threadIdx.x, nthr = blockDim.x, l = t & 63, c = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int nt = (In + 15) / 16;
    const bool active = w < nt;
    // every load of the usual path is requested before the first wait
    const int done = chk->done, kind = chk->kind, gfb = finfo[1];
    const bool want_fit = fit && kind != ITCPD_CHECK_NONE;
    const int ia = 16 * w + c;
    auto sum_m = [&](int row, int k) {   // M(row, k): the partials in increasing order
        const bool ok = row < In && k < R;
        const double* src = Msrc + (ok ? row + (int64_t)In * k : 0);
        double v = src[0];
        for (int b = 1; b < nparts; ++b) v += src[b * pstride];
        return ok ? v : 0.0;
    };
    double av[KS], bv[NT][KS], md[NT][4], h[NH];
    d4 acc[NT];
#pragma unroll
    for (int tb = 0; tb < NT; ++tb) acc[tb] = (d4){0.0, 0.0, 0.0, 0.0};
    if (active) {
        const double* src[KS];
        bool ok[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int k = 4 * ks + g;
            ok[ks] = ia < In && k < R;
            src[ks] = Msrc + (ok[ks] ? ia + (int64_t)In * k : 0);
            av[ks] = src[ks][0];
#pragma unroll
            for (int tb = 0; tb < NT; ++tb) {
                const int col = 16 * tb + c;
                const double v = Vinv[k < R && col < R ? k * R + col : 0];
                bv[tb][ks] = k < R && col < R ? v : 0.0;
            }
        }
        int b = 1;
        for (; b + 4 <= nparts; b += 4) {
            double v[KS][4];
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                for (int z = 0; z < 4; ++z) v[ks][z] = src[ks][(b + z) * pstride];
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                for (int z = 0; z < 4; ++z) av[ks] += v[ks][z];
        }
        for (; b < nparts; ++b)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) av[ks] += src[ks][b * pstride];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) av[ks] = ok[ks] ? av[ks] : 0.0;
    }
    if (want_fit) {
#pragma unroll
        for (int q = 0; q < NH; ++q) h[q] = 1.0;
        for (int m = 0; m < gs.N; ++m) {
            if (m == mode) continue;
#pragma unroll
            for (int q = 0; q < NH; ++q) {
                const int x = t + nthr * q;
                h[q] *= gs.G[m][x < R * R ? x : 0];
            }
        }
#pragma unroll
        for (int tb = 0; tb < NT; ++tb)
#pragma unroll
            for (int v = 0; v < 4; ++v) md[tb][v] = active ? sum_m(16 * w + g + 4 * v, 16 * tb + c) : 0.0;
    }
    if (done) return;
    if (!gfb) {
        if (active) {
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                for (int tb = 0; tb < NT; ++tb) acc[tb] = mfma_f64(av[ks], bv[tb][ks], acc[tb]);
        }
    } else {   // QR fallback, row by row: lane k holds column k; then the tile as above
        const int rk = finfo[2], pk = l < R ? jpvt[l] : 0;
        for (int rr = 0; rr < 16; ++rr) {
            const int row = 16 * w + rr;
            if (row >= In) break;
            double y[1] = {sum_m(row, l)};
            fallback_apply<1>(y, l, R, rk, W, qtau, ztau);
            if (l < R) X[row + (int64_t)In * pk] = y[0];
        }
        __syncthreads();
#pragma unroll
        for (int tb = 0; tb < NT; ++tb)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = 16 * w + g + 4 * v, col = 16 * tb + c;
                acc[tb][v] = row < In && col < R ? X[row + (int64_t)In * col] : 0.0;
            }
    }
    if (active) {   // rows >= In and columns >= R of acc are zero
        d4 ga[NP];
#pragma unroll
        for (int q = 0; q < NP; ++q) ga[q] = (d4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int tb = 0, q = 0; tb < NT; ++tb)
#pragma unroll
                for (int ta = 0; ta <= tb; ++ta, ++q) ga[q] = mfma_f64(acc[ta][v], acc[tb][v], ga[q]);
#pragma unroll
        for (int q = 0; q < NP; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) part[(w * NP + q) * 256 + 64 * v + l] = ga[q][v];
    }
    __syncthreads();
    for (int x = t; x < NP * 256; x += nthr) {
        double s = 0.0;
        for (int k = 0; k < nt; ++k) s += part[k * NP * 256 + x];
        const int q = x >> 8, tb = q > 0, ta = q > 1;   // tiles (0, 0), (0, 1), (1, 1)
        const int r = 16 * ta + ((x >> 4) & 3) + 4 * ((x >> 6) & 3), r2 = 16 * tb + (x & 15);
        S[r * LDS_ + r2] = s;
        if (ta != tb) S[r2 * LDS_ + r] = s;
    }
    __syncthreads();
    if (t < R) {
        lamS[t] = sqrt(S[t * LDS_ + t]);
        lam[t] = lamS[t];
    }
    __syncthreads();
    double fs = 0.0, inner = 0.0;
#pragma unroll
    for (int q = 0; q < NH; ++q) {
        const int x = t + nthr * q;
        if (x >= R * R) continue;
        const int r = x % R, r2 = x / R;
        const double ll = lamS[r] * lamS[r2], gx = S[r * LDS_ + r2] / ll;
        Gout[x] = gx;
        if (want_fit) fs += h[q] * gx * ll;
    }
    if (active) {
#pragma unroll
        for (int tb = 0; tb < NT; ++tb) {
            const int col = 16 * tb + c;
            if (col >= R) continue;
            const double lc = lamS[col];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = 16 * w + g + 4 * v;
                if (row >= In) continue;
                const double a = acc[tb][v] / lc;
                A[row + (int64_t)In * col] = a;
                At[(int64_t)row * Rp + col] = a;
                if (want_fit) inner += md[tb][v] * (a * lc);
            }
        }
    }
    if (!fit) return;
    if (want_fit) {
        fs = wave_sum_dpp(fs);
        inner = wave_sum_dpp(inner);
        if (l == 0) {
            red[w] = fs;
            red[16 + w] = inner;
        }
        __syncthreads();
        if (t == 0) {
            for (int k = 1; k < nthr / 64; ++k) {
                fs += red[k];
                inner += red[16 + k];
            }
            check_update(chk, inner, fs, scal, trace, trace_cap);
        }
    } else if (t == 0) {
        count_sweep(chk);
    }
}

// ------------------------------------- CPDiffCheck / CPAngleCheck (CP vs CP)
// The previous sweep's CPD against the current one: cp_cp_contract
// (cp_contract.jl:32-52) is the Hadamard product over modes of the cross Grams
// C_q = A_prev,q^T A_q, and <X_prev, X> = lambda_prev^T (.* C_q) lambda.
struct FacPair {
    const double* P[ITCPD_MAX_ORDER];   // previous factors, rank fastest (Rp x I_q)
    const double* C[ITCPD_MAX_ORDER];   // current factors, rank fastest
    int64_t I[ITCPD_MAX_ORDER];
};

// Cross-Gram partials over row chunks: block (x, chunk, q), thread e = 256 x + t
// for the entry (r, r2) = (e / R, e % R) of C_q; a wave's threads share r (one
// broadcast load of the previous factor per row) and read consecutive r2.
__global__ __launch_bounds__(256) void k_cross_gram(FacPair fp, int R, int Rp, int chunks,
                                                    double* __restrict__ part,
                                                    const DevCheck* __restrict__ chk) {
    if (chk->done || !chk->has_prev) return;
    const int q = blockIdx.z, ch = blockIdx.y;
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= R * R) return;
    const int r = e / R, r2 = e % R;
    const int64_t In = fp.I[q];
    const int64_t per = (In + chunks - 1) / chunks;
    const int64_t i0 = (int64_t)ch * per;
    const int64_t i1 = i0 + per < In ? i0 + per : In;
    const double* __restrict__ P = fp.P[q];
    const double* __restrict__ Cc = fp.C[q];
    double a[4] = {0.0, 0.0, 0.0, 0.0};
    int64_t i = i0;
    for (; i + 4 <= i1; i += 4) {
        double x[4], y[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            x[k] = P[(i + k) * Rp + r];
            y[k] = Cc[(i + k) * Rp + r2];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) a[k] += x[k] * y[k];
    }
    for (; i < i1; ++i) a[0] += P[i * Rp + r] * Cc[i * Rp + r2];
    part[((int64_t)q * chunks + ch) * R * R + e] = (a[0] + a[1]) + (a[2] + a[3]);
}

// cp_diff_check.jl:20-71 / cp_angle_check.jl:20-73 after the sweep (one thread).
static __device__ void cp_check_update(DevCheck* chk, double cross, double fact_square, double* trace,
                                       int trace_cap) {
    chk->iter += 1;
    const int sweep = chk->sweeps;
    chk->sweeps += 1;
    const bool angle = chk->kind == ITCPD_CHECK_CPANGLE;
    if (!chk->has_prev) {
        // the first call stores PrevCP and its norm and returns false
        chk->has_prev = 1;
        chk->norm_prev = angle ? sqrt(fact_square) : fact_square;
        if (trace && sweep < trace_cap) trace[sweep] = __builtin_nan("");
        return;
    }
    double cur;
    if (!angle) {
        const double nres = sqrt(fabs(chk->norm_prev + fact_square - 2.0 * fabs(cross)));
        cur = 1.0 - nres / sqrt(fabs(chk->norm_prev));
        chk->norm_prev = fact_square;
    } else {
        const double ncur = sqrt(fact_square);
        double th = cross / (ncur * chk->norm_prev);
        th = th > 1.0 ? 1.0 : th;
        cur = acos(th);
        chk->norm_prev = ncur;
    }
    const double delta = fabs(chk->lastfit - cur);
    chk->lastfit = cur;
    if (trace && sweep < trace_cap) trace[sweep] = cur;
    if (delta < chk->tolerance) {
        chk->counter += 1;
        if (chk->counter >= 2) {
            chk->total_iter = chk->iter;
            chk->iter = 0;
            chk->counter = 0;
            chk->final_fit = chk->lastfit;
            chk->lastfit = 0.0;
            chk->has_prev = 0;
            chk->done = 1;
            return;
        }
    } else {
        chk->counter = 0;
    }
    if (chk->iter >= chk->max_counter) {
        chk->total_iter = chk->iter;
        chk->iter = 0;
        chk->counter = 0;
        chk->final_fit = chk->lastfit;
        chk->lastfit = 0.0;
        chk->has_prev = 0;
    }
}

// ||X||^2 = lambda^T (.* G_q) lambda (norm_factors, converge_checks.jl:5-11) and,
// with a previous CPD, <X_prev, X> from the cross-Gram partials (fixed order);
// then the check's state update.
__global__ __launch_bounds__(256) void k_cp_check(const double* __restrict__ part, int chunks, int R,
                                                  GramSet gs, const double* __restrict__ lam,
                                                  const double* __restrict__ lamprev,
                                                  DevCheck* __restrict__ chk, double* __restrict__ trace,
                                                  int trace_cap) {
    if (chk->done) return;
    __shared__ double red[256];
    const int t = threadIdx.x;
    const bool have = chk->has_prev != 0;
    const int64_t RR = (int64_t)R * R;
    double fs = 0.0, cr = 0.0;
    for (int x = t; x < R * R; x += 256) {
        const int r = x / R, r2 = x % R;
        double h = 1.0;
        for (int m = 0; m < gs.N; ++m) h *= gs.G[m][x];
        fs += h * (lam[r] * lam[r2]);
        if (have) {
            double c = 1.0;
            for (int m = 0; m < gs.N; ++m) {
                double sacc = 0.0;
                for (int ch = 0; ch < chunks; ++ch) sacc += part[((int64_t)m * chunks + ch) * RR + x];
                c *= sacc;
            }
            cr += c * (lamprev[r] * lam[r2]);
        }
    }
    const double fact_square = block_sum<256>(fs, red);
    const double cross = block_sum<256>(cr, red);
    if (t == 0) cp_check_update(chk, cross, fact_square, trace, trace_cap);
}

// ------------------------------------------------ row_norm + Gram partials
// lambda from the per-block sums of squares; A = X ./ lambda (column-major,
// Rp columns) and At (rank fastest); Gram partial over this block's rows; for
// the fit, <M, A .* lambda> over this block's rows.
__global__ __launch_bounds__(256) void k_normalize(const double* __restrict__ X, int64_t In, int R,
                                                   int Rp, const double* __restrict__ sumsq_part,
                                                   int nsp, int rows_per_block, double* __restrict__ A,
                                                   double* __restrict__ At, double* __restrict__ lam,
                                                   double* __restrict__ gram_part,
                                                   const double* __restrict__ M, int want_inner,
                                                   double* __restrict__ inner_part, int normalize,
                                                   const DevCheck* __restrict__ chk) {
    if (chk && chk->done) return;
    extern __shared__ double lds[];
    double* lamS = lds;            // R
    double* As = lds + R;          // rows_per_block x R (row-major)
    __shared__ double red[256];
    const int t = threadIdx.x;
    for (int r = t; r < R; r += 256) {
        if (normalize) {
            double s = 0.0;
            for (int b = 0; b < nsp; ++b) s += sumsq_part[(int64_t)b * R + r];
            lamS[r] = sqrt(s);
        } else {
            lamS[r] = 1.0;
        }
    }
    __syncthreads();
    if (normalize && blockIdx.x == 0)
        for (int r = t; r < R; r += 256) lam[r] = lamS[r];
    double inner = 0.0;
    double* gp = gram_part + (int64_t)blockIdx.x * R * R;
    bool first_tile = true;
    for (int64_t i0 = (int64_t)blockIdx.x * rows_per_block; i0 < In;
         i0 += (int64_t)gridDim.x * rows_per_block) {
        const int nr = (int)((In - i0) < rows_per_block ? (In - i0) : rows_per_block);
        for (int x = t; x < nr * R; x += 256) {
            const int ii = x % nr, r = x / nr;
            const int64_t i = i0 + ii;
            const double a = normalize ? X[i + In * r] / lamS[r] : X[i + In * r];
            As[ii * R + r] = a;
            if (normalize) A[i + In * r] = a;
            At[i * Rp + r] = a;
            if (want_inner) inner += M[i + In * r] * (a * lamS[r]);
        }
        __syncthreads();
        for (int x = t; x < R * R; x += 256) {
            const int r = x % R, r2 = x / R;
            double s = 0.0;
            for (int ii = 0; ii < nr; ++ii) s += As[ii * R + r] * As[ii * R + r2];
            gp[x] = first_tile ? s : gp[x] + s;
        }
        first_tile = false;
        __syncthreads();
    }
    if (want_inner) {
        const double v = block_sum<256>(inner, red);
        if (t == 0) inner_part[blockIdx.x] = v;
    }
}

// Sums the Gram partials into G_mode; after the last mode also evaluates the fit
// and advances the check state (FitCheck / NoCheck), recording the fit trace.
__global__ __launch_bounds__(256) void k_gram_final(const double* __restrict__ gram_part, int nb,
                                                    int R, double* __restrict__ Gout, GramSet gs,
                                                    int mode, const double* __restrict__ lam,
                                                    const double* __restrict__ inner_part,
                                                    int do_check, double* __restrict__ scal,
                                                    DevCheck* __restrict__ chk,
                                                    double* __restrict__ trace, int trace_cap) {
    if (chk && chk->done) return;
    __shared__ double red[256];
    const int t = threadIdx.x;
    if (gram_part) {   // null: the partials were already summed into Gout by a wider launch
        for (int x = t; x < R * R; x += 256) {
            double s = 0.0;
            for (int b = 0; b < nb; ++b) s += gram_part[(int64_t)b * R * R + x];
            Gout[x] = s;
        }
    }
    if (!do_check) return;
    __threadfence_block();
    __syncthreads();
    if (chk->kind == ITCPD_CHECK_NONE) {
        if (t == 0) count_sweep(chk);
        return;
    }
    // ||X||^2 = lambda^T (G_0 .* ... .* G_{N-1}) lambda   (converge_checks.jl:5-11)
    double fs = 0.0;
    for (int x = t; x < R * R; x += 256) {
        const int r = x % R, r2 = x / R;
        double h = gs.G[0][x];
        for (int m = 1; m < gs.N; ++m) h *= gs.G[m][x];
        fs += h * (lam[r] * lam[r2]);
    }
    const double fact_square = block_sum<256>(fs, red);
    if (t == 0) {
        double inner = 0.0;
        for (int b = 0; b < nb; ++b) inner += inner_part[b];
        check_update(chk, inner, fact_square, scal, trace, trace_cap);
    }
}

// --------------------------------------------------------------- init (RNG)
__global__ __launch_bounds__(256) void k_random_normal(double* __restrict__ X, int64_t In, int R,
                                                       uint64_t seed, int mode) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;   // e = i + In * r
    if (e >= In * R) return;
    uint32_t c[4] = {(uint32_t)e, (uint32_t)((uint64_t)e >> 32), (uint32_t)mode, 0u};
    philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
    const uint64_t a = ((uint64_t)c[0] << 32) | c[1];
    const uint64_t b = ((uint64_t)c[2] << 32) | c[3];
    const double u1 = (double)((a >> 11) + 1) * 1.1102230246251565e-16;  // (0, 1]
    const double u2 = (double)(b >> 11) * 1.1102230246251565e-16;        // [0, 1)
    X[e] = sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
}
// reconstruct.jl:2-9: X(i_1..i_N) = sum_r lambda_r prod_n A_n(i_n, r), column-major,
// one element per thread, plus sigma * N(0,1) from the Philox stream keyed by
// (seed, element index) when sigma > 0.  Written as FP64 or FP32.
struct RecoArgs {
    const double* A[ITCPD_MAX_ORDER];
    int64_t dims[ITCPD_MAX_ORDER];
    int N;
};
template <typename OT>
__global__ __launch_bounds__(256) void k_reconstruct(RecoArgs ra, int R, const double* __restrict__ lam,
                                                     int64_t nel, double sigma, uint64_t seed,
                                                     OT* __restrict__ out) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= nel) return;
    int64_t idx[ITCPD_MAX_ORDER];
    int64_t t = e;
    for (int n = 0; n < ra.N; ++n) {
        idx[n] = t % ra.dims[n];
        t /= ra.dims[n];
    }
    double x = 0.0;
    for (int r = 0; r < R; ++r) {
        double pr = lam[r];
        for (int n = 0; n < ra.N; ++n) pr *= ra.A[n][idx[n] + ra.dims[n] * r];
        x += pr;
    }
    if (sigma > 0.0) {
        uint32_t c[4] = {(uint32_t)e, (uint32_t)((uint64_t)e >> 32), 0x6E6F6973u, 0u};
        philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
        const uint64_t a = ((uint64_t)c[0] << 32) | c[1];
        const uint64_t b = ((uint64_t)c[2] << 32) | c[3];
        const double u1 = (double)((a >> 11) + 1) * 1.1102230246251565e-16;
        const double u2 = (double)(b >> 11) * 1.1102230246251565e-16;
        x += sigma * sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
    }
    out[e] = (OT)x;
}

// The same sum as a tiled outer product: the modes split into a left group [0, s) and
// a right group [s, N), X = (left KRP) diag(lambda) (right KRP)^T with the element at
// l + ML r.  A 256-thread block computes 64 x 64 elements; per chunk of 16 ranks the
// block builds its 64 left rows (lambda_r prod A_m) and 64 right rows in LDS, and
// thread (tx, ty) accumulates elements (l0 + tx + 16 i, r0 + ty + 16 j).  The noise
// is the per-element Philox draw of k_reconstruct.
struct RecoSplit {
    const double* A[ITCPD_MAX_ORDER];
    int64_t dims[ITCPD_MAX_ORDER];
    int N, s;
    int64_t ML, MR;
};
__device__ __forceinline__ double reco_noise(int64_t e, double sigma, uint64_t seed) {
    uint32_t c[4] = {(uint32_t)e, (uint32_t)((uint64_t)e >> 32), 0x6E6F6973u, 0u};
    philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
    const uint64_t a = ((uint64_t)c[0] << 32) | c[1];
    const uint64_t b = ((uint64_t)c[2] << 32) | c[3];
    const double u1 = (double)((a >> 11) + 1) * 1.1102230246251565e-16;
    const double u2 = (double)(b >> 11) * 1.1102230246251565e-16;
    return sigma * sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
}
template <typename OT>
__global__ __launch_bounds__(256) void k_reconstruct_tiled(RecoSplit ra, int R, const double* __restrict__ lam,
                                                           double sigma, uint64_t seed, OT* __restrict__ out) {
    __shared__ double Ls[16][65];
    __shared__ double Rs[16][65];
    __shared__ int idxL[64][ITCPD_MAX_ORDER];
    __shared__ int idxR[64][ITCPD_MAX_ORDER];
    const int t = threadIdx.x;
    const int64_t l0 = (int64_t)blockIdx.x * 64, r0 = (int64_t)blockIdx.y * 64;
    if (t < 64) {
        int64_t x = l0 + t;
        for (int m = 0; m < ra.s; ++m) {
            idxL[t][m] = (int)(x % ra.dims[m]);
            x /= ra.dims[m];
        }
    } else if (t < 128) {
        int64_t x = r0 + (t - 64);
        for (int m = ra.s; m < ra.N; ++m) {
            idxR[t - 64][m] = (int)(x % ra.dims[m]);
            x /= ra.dims[m];
        }
    }
    const int tx = t & 15, ty = t >> 4;
    double acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0.0;
    for (int rc = 0; rc < R; rc += 16) {
        __syncthreads();
        // 16 ranks x 64 rows per side: thread t fills (rank k = t >> 4, rows 4 (t & 15) ..)
        {
            const int k = t >> 4, rr = rc + k;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int x = 4 * (t & 15) + q;
                double lv = 0.0, rv = 0.0;
                if (rr < R) {
                    lv = lam[rr];
                    for (int m = 0; m < ra.s; ++m) lv *= ra.A[m][idxL[x][m] + ra.dims[m] * rr];
                    rv = 1.0;
                    for (int m = ra.s; m < ra.N; ++m) rv *= ra.A[m][idxR[x][m] + ra.dims[m] * rr];
                }
                Ls[k][x] = lv;
                Rs[k][x] = rv;
            }
        }
        __syncthreads();
#pragma unroll 4
        for (int k = 0; k < 16; ++k) {
            double a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = Ls[k][tx + 16 * i];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = Rs[k][ty + 16 * j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fma(a[i], b[j], acc[i][j]);
        }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int64_t r = r0 + ty + 16 * j;
        if (r >= ra.MR) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int64_t l = l0 + tx + 16 * i;
            if (l >= ra.ML) continue;
            const int64_t e = l + ra.ML * r;
            double x = acc[i][j];
            if (sigma > 0.0) x += reco_noise(e, sigma, seed);
            out[e] = (OT)x;
        }
    }
}

// per-block sums of squares of the columns of X (for the init's row_norm)
__global__ __launch_bounds__(256) void k_col_sumsq(const double* __restrict__ X, int64_t In, int R,
                                                   int rows_per_block, double* __restrict__ part) {
    const int64_t i0 = (int64_t)blockIdx.x * rows_per_block;
    const int64_t i1 = i0 + rows_per_block < In ? i0 + rows_per_block : In;
    for (int r = threadIdx.x; r < R; r += 256) {
        double s = 0.0;
        for (int64_t i = i0; i < i1; ++i) s += X[i + In * r] * X[i + In * r];
        part[(int64_t)blockIdx.x * R + r] = s;
    }
}

// V = Hadamard of the Grams of modes != mode (compute_krp hook)
__global__ __launch_bounds__(256) void k_hadamard_grams(GramSet gs, int mode, int R,
                                                        double* __restrict__ V) {
    const int x = blockIdx.x * 256 + threadIdx.x;
    if (x >= R * R) return;
    double v = 1.0;
    for (int m = 0; m < gs.N; ++m)
        if (m != mode) v *= gs.G[m][x];
    V[x] = v;
}

// ----------------------------------------------------------------- fit hook
__global__ __launch_bounds__(256) void k_fit_hook(const double* __restrict__ M,
                                                  const double* __restrict__ AN, int64_t In, int R,
                                                  const double* __restrict__ lam, GramSet gs,
                                                  double ref, double* __restrict__ scal) {
    __shared__ double red[256];
    const int t = threadIdx.x;
    double inner = 0.0;
    for (int64_t x = t; x < In * R; x += 256) {
        const int r = (int)(x / In);
        inner += M[x] * (AN[x] * lam[r]);
    }
    inner = block_sum<256>(inner, red);
    double fs = 0.0;
    for (int x = t; x < R * R; x += 256) {
        const int r = x % R, r2 = x / R;
        double h = gs.G[0][x];
        for (int m = 1; m < gs.N; ++m) h *= gs.G[m][x];
        fs += h * (lam[r] * lam[r2]);
    }
    fs = block_sum<256>(fs, red);
    if (t == 0) {
        scal[0] = inner;
        scal[1] = fs;
        scal[2] = 1.0 - sqrt(fabs(ref * ref + fs - 2.0 * fabs(inner))) / ref;
    }
}

// ---------------------------------------------------------------- launchers
namespace {

GramSet grams_of(itcpd_plan* p) {
    GramSet gs{};
    gs.N = p->N;
    for (int m = 0; m < p->N; ++m) gs.G[m] = p->G[m];
    return gs;
}

int rows_per_block_for(int R) {
    int rpb = 32;
    while (rpb > 1 && (size_t)(rpb * R + R) * 8 > 120 * 1024) rpb >>= 1;
    return rpb;
}

// Number of row-normalisation blocks: capped so the Gram partials stay bounded.
int norm_blocks(int64_t In, int R, int rpb) {
    int64_t nb = cdiv(In, rpb);
    int64_t cap = (int64_t)1 << 25;
    cap = cap / ((int64_t)R * R);
    if (cap > 64) cap = 64;
    if (cap < 1) cap = 1;
    return (int)(nb < cap ? nb : cap);
}

int solve_blocks(int64_t In) {
    int64_t nb = cdiv(In, 4);
    return (int)(nb < 128 ? nb : 128);
}

}  // namespace

int launch_factor(itcpd_plan* p, int mode) { return launch_factor_on(p, mode, p->stream); }

// CPDiffCheck / CPAngleCheck after the last mode of a sweep: cross Grams against
// the held previous CPD, the check update, then PrevCP <- the current CPD.
int launch_cp_check(itcpd_plan* p) {
    const int R = (int)p->R, N = p->N;
    FacPair fp{};
    for (int q = 0; q < N; ++q) {
        fp.P[q] = p->Atprev[q];
        fp.C[q] = p->At[q];
        fp.I[q] = p->dims[q];
    }
    const unsigned nx = (unsigned)cdiv((int64_t)R * R, 256);
    hipLaunchKernelGGL(k_cross_gram, dim3(nx, (unsigned)p->xg_chunks, (unsigned)N), dim3(256), 0, p->stream,
                       fp, R, (int)p->Rp, p->xg_chunks, p->xg_part, p->chk);
    ITCPD_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_cp_check, dim3(1), dim3(256), 0, p->stream, p->xg_part, p->xg_chunks, R, grams_of(p),
                       p->lam, p->lamprev, p->chk, p->fit_trace, p->trace_cap);
    ITCPD_HIP(hipGetLastError());
    for (int q = 0; q < N; ++q)
        ITCPD_HIP(hipMemcpyAsync(p->Atprev[q], p->At[q], (size_t)(p->dims[q] * p->Rp) * 8,
                                 hipMemcpyDeviceToDevice, p->stream));
    ITCPD_HIP(hipMemcpyAsync(p->lamprev, p->lam, (size_t)p->Rp * 8, hipMemcpyDeviceToDevice, p->stream));
    return ITCPD_OK;
}

int launch_factor_on(itcpd_plan* p, int mode_in, hipStream_t st) {
    const int R = (int)p->R;
    // a set V override: the factorisation of that matrix (as the Hadamard of {V}
    // with mode 1 skipped), else of the Hadamard of the other Grams
    GramSet gs = grams_of(p);
    int mode = mode_in;
    if (p->v_override) {
        gs.G[0] = p->v_override;
        gs.G[1] = p->v_override;
        gs.N = 2;
        mode = 1;
    }
    double* W = p->qr_aux;
    double* qtau = W + (size_t)R * R;
    double* ztau = qtau + R;
    double* vwork = ztau + R;
    if (R <= 64) {
        hipLaunchKernelGGL(k_factor64, dim3(1), dim3(256), FACTOR64_LDS,
                           st, gs, mode, R, 1e-6, p->U, p->Upad, p->invdiag, p->piv,
                           p->finfo, W, qtau, ztau, p->piv + R, vwork, p->chk);
    } else {
        // V^-1 by blocks; the pivoted factorisation only when it is not certified
        const int nb = (int)cdiv(R, 64);
        const size_t half = (size_t)(64 * nb) * (64 * nb);
        hipLaunchKernelGGL(k_inv_first, dim3((unsigned)nb, (unsigned)nb), dim3(256), INV_LDS, st, gs, mode, R, nb, p->inv_buf,
                           p->inv_stat, p->chk);
        for (int k = 1; k < nb; ++k)
            hipLaunchKernelGGL(k_inv_step, dim3((unsigned)(nb - k), (unsigned)nb), dim3(256), INV_LDS, st, k, R, nb,
                               p->inv_buf + ((k - 1) & 1) * half, p->inv_buf + (k & 1) * half, p->inv_stat, p->chk);
        // into U: the pivoted kernels write it only when they do not exit on the certificate
        hipLaunchKernelGGL(k_inv_product, dim3((unsigned)inv_tiles(R)), dim3(256), 0, st, R, nb, p->inv_buf, p->U,
                           p->inv_stat, p->chk);
        ITCPD_HIP(hipGetLastError());
        if (R <= 128)
            hipLaunchKernelGGL(k_factor128, dim3(1), dim3(1024), F128_LDS, st, gs, mode, R, 1e-6, p->U, p->invdiag,
                               p->piv, p->finfo, W, qtau, ztau, p->piv + R, vwork, p->inv_stat, nb, p->chk);
        else
            hipLaunchKernelGGL(k_factor, dim3(1), dim3(FACTOR_THREADS), 0, st, gs, mode, R, 1e-6, p->U, p->invdiag,
                               p->piv, p->finfo, W, qtau, ztau, p->piv + R, vwork, p->inv_stat, nb, p->chk);
    }
    ITCPD_HIP(hipGetLastError());
    return ITCPD_OK;
}

namespace {

// rows per wave in the row solves (fewer for large R to bound registers)
template <int RQ>
// 64 < R <= 128: one row per wave, so a mode of a few hundred rows spreads over
// as many workgroups (each stages U in LDS; 4 interleaved rows per wave left most
// CUs idle at I = 224)
constexpr int rpw_of() { return RQ == 2 ? 1 : (RQ <= 4 ? 4 : (RQ == 8 ? 2 : 1)); }
int rpb_of(int R) { return 4 * (R <= 64 ? 4 : (R <= 128 ? 1 : (R <= 256 ? 4 : (R <= 512 ? 2 : 1)))); }

// Block count of the row solves, capped so that the per-block Gram partials stay
// within 2^25 doubles.
int solve_nb(int64_t In, int R) {
    int64_t cap = ((int64_t)1 << 25) / ((int64_t)R * R);
    cap = cap < 1 ? 1 : (cap > 256 ? 256 : cap);
    // R <= 64: 16-row tiles, both in k_solve_mfma and in k_solve's fallback path
    const int64_t nb = cdiv(In, R <= 64 ? 16 : rpb_of(R));
    return (int)(nb < cap ? nb : cap);
}
// 32 rows and 256 Gram entries (one per thread) a block, which is k_finalize_1rt's form while
// the partials are few; at most 16 blocks for R <= 64, 128 above.  Measured: R = 24, I = 20
// 5.2 us (5.8 with one block); R = 128, I = 224 with 64 blocks 7.9 us (45 with 7 blocks and
// 56 partials).
int finalize_nb(int64_t In, int R) {
    return (int)std::min<int64_t>(R > 64 ? 128 : 16, std::max(cdiv(In, 32), cdiv((int64_t)R * R, 256)));
}

// Row ranges of the Gram products: one up to 2048 rows, at most 64 (and within gram_part).
int gram_parts(int64_t In, int R) {
    const int64_t cap = std::max<int64_t>(1, ((int64_t)1 << 25) / ((int64_t)R * R));
    return (int)std::min<int64_t>(std::min<int64_t>(64, cap), std::max<int64_t>(1, cdiv(In, 2048)));
}
unsigned gram_tiles(int R) {
    const unsigned nt = (unsigned)cdiv(R, 16);
    return nt * (nt + 1) / 2;
}

// R > 64: X = M V^-1 when the inverse is certified, else the substitution / QR row solves;
// one of the two launches finds that the other has the rows.
template <int RQ>
int run_solve_k(itcpd_plan* p, int mode, const double* Msrc) {
    const int64_t In = p->dims[mode];
    const int R = (int)p->R;
    hipLaunchKernelGGL(k_solve_inv, dim3((unsigned)cdiv(In, 16), (unsigned)cdiv(cdiv(R, 16), 4)), dim3(256), 0,
                       p->stream, Msrc, In, R, p->U, p->finfo, p->X, p->chk);
    const bool u_lds = R <= 128;
    constexpr int RPW = rpw_of<RQ>();
    const size_t lds = (size_t)4 * RPW * R * 8 + (u_lds ? (size_t)R * (R + 1) * 8 : 0);
    double* W = p->qr_aux;
    hipLaunchKernelGGL((k_solve<RQ, RPW>), dim3(solve_nb(In, R)), dim3(256), lds, p->stream, Msrc, In, R, p->U,
                       p->invdiag, p->piv, p->finfo, W, W + (size_t)R * R, W + (size_t)R * R + R,
                       (const int*)(p->piv + R), u_lds ? 1 : 0, p->X, p->chk);
    ITCPD_HIP(hipGetLastError());
    return ITCPD_OK;
}

// R <= 64: one launch; the kernel takes the Cholesky (MFMA) or the QR-fallback path
// from the factor kernel's status.
template <int RT>
int run_solve_rows(itcpd_plan* p, int mode, const double* Msrc, int nparts, int64_t stride, bool grams,
                   bool keep_m) {
    const int64_t In = p->dims[mode];
    const int R = (int)p->R;
    const int nb = solve_nb(In, R);
    double* Msum = keep_m ? p->Msum : (double*)nullptr;
    double* W = p->qr_aux;
    hipLaunchKernelGGL((k_solve_mfma<RT>), dim3(nb), dim3(256), (size_t)16 * R * 8, p->stream, Msrc, In, R,
                       p->Upad, p->finfo, W, W + (size_t)R * R, W + (size_t)R * R + R,
                       (const int*)(p->piv + R), p->X, Msum, p->gram_part, grams ? 1 : 0, nparts, stride,
                       p->chk);
    ITCPD_HIP(hipGetLastError());
    return ITCPD_OK;
}

int run_apply(itcpd_plan* p, int mode, const double* Msrc, int nparts, int64_t stride, bool grams,
              bool keep_m) {
    const int R = (int)p->R;
    if (p->RT == 16) return run_solve_rows<16>(p, mode, Msrc, nparts, stride, grams, keep_m);
    if (p->RT == 32) return run_solve_rows<32>(p, mode, Msrc, nparts, stride, grams, keep_m);
    if (p->RT == 64) return run_solve_rows<64>(p, mode, Msrc, nparts, stride, grams, keep_m);
    if (R <= 128) return run_solve_k<2>(p, mode, Msrc);
    if (R <= 256) return run_solve_k<4>(p, mode, Msrc);
    if (R <= 512) return run_solve_k<8>(p, mode, Msrc);
    return run_solve_k<16>(p, mode, Msrc);
}

// One workgroup for the whole update: while its matrix products (In RT) and M's partials
// through one CU stay below what the separate launches cost.
bool update_small_ok(const itcpd_plan* p, int mode, int nparts) {
    const int64_t In = p->dims[mode];
    return p->RT && p->RT <= 32 && In * p->RT <= 4096 && In * p->R * nparts <= ((int64_t)1 << 15);
}
template <int RT>
int run_update_small(itcpd_plan* p, int mode, const double* Msrc, int nparts, int64_t stride, bool fit) {
    const int64_t In = p->dims[mode];
    const int R = (int)p->R;
    double* W = p->qr_aux;
    hipLaunchKernelGGL((k_update_small<RT>), dim3(1), dim3(64 * std::max<unsigned>(4, (unsigned)cdiv(In, 16))), 0,
                       p->stream, Msrc, nparts, stride, (int)In, R, (int)p->Rp, p->Upad, p->finfo, W,
                       W + (size_t)R * R, W + (size_t)R * R + R, (const int*)(p->piv + R), p->X, p->A[mode],
                       p->At[mode], p->lam, p->G[mode], mode, grams_of(p), fit ? 1 : 0, p->scal, p->chk,
                       p->fit_trace, p->trace_cap);
    ITCPD_HIP(hipGetLastError());
    return ITCPD_OK;
}

// row_norm of X from nb Gram partials, with <M, X> for the fit when asked
int run_finalize(itcpd_plan* p, int mode, int nb, const double* Mkept, bool fit, const int* hold = nullptr) {
    const int64_t In = p->dims[mode];
    const int R = (int)p->R;
    const int nbf = finalize_nb(In, R);
    const bool one_rt = nb <= 32 && R <= 256 && cdiv((int64_t)R * R, nbf) <= 256 && cdiv(In, nbf) * R <= 2048;
    hipLaunchKernelGGL(one_rt ? k_finalize_1rt : k_finalize, dim3(nbf), dim3(256), one_rt ? 0 : (size_t)R * 8,
                       p->stream, p->gram_part, nb, p->X, Mkept, In, R, (int)p->Rp, p->A[mode], p->At[mode],
                       p->lam, p->G[mode], fit ? p->inner_part : (double*)nullptr, hold, p->chk);
    ITCPD_HIP(hipGetLastError());
    return ITCPD_OK;
}
// the same with X's Gram by a launch of its own
int run_gram_finalize(itcpd_plan* p, int mode, const double* Mkept, bool fit, const int* hold = nullptr) {
    const int R = (int)p->R;
    GramJobs gj{};
    gj.X[0] = p->X;
    gj.S[0] = p->gram_part;
    gj.I[0] = p->dims[mode];
    const int nb = gram_parts(p->dims[mode], R);
    hipLaunchKernelGGL(k_gram_mfma, dim3(gram_tiles(R), (unsigned)nb), dim3(256), 0, p->stream, gj, R, nb, p->chk);
    ITCPD_HIP(hipGetLastError());
    return run_finalize(p, mode, nb, Mkept, fit, hold);
}

}  // namespace

int launch_row_norm(itcpd_plan* p, int mode, const int* hold) {
    return run_gram_finalize(p, mode, p->X, false, hold);
}

int launch_solve(itcpd_plan* p, int mode, const double* Msrc, int nparts, int64_t stride,
                 bool finalize, bool fit_after, int next_factor) {
    const int R = (int)p->R;
    int rc;
    // the R <= 64 row solves sum up to SOLVE_MAX_PARTS partials as they load M
    if (nparts > 1 && !(p->RT && nparts <= SOLVE_MAX_PARTS)) {
        const int64_t n = p->dims[mode] * p->R;
        if ((rc = launch_sum_parts(p, MSrc{Msrc, nparts, stride}, n, p->M))) return rc;
        Msrc = p->M;
        nparts = 1;
    }
    const bool cp_check = p->check_kind == ITCPD_CHECK_CPDIFF || p->check_kind == ITCPD_CHECK_CPANGLE;
    if (finalize && update_small_ok(p, mode, nparts)) {
        const bool fit = fit_after && !cp_check;
        rc = p->RT == 16 ? run_update_small<16>(p, mode, Msrc, nparts, stride, fit)
                         : run_update_small<32>(p, mode, Msrc, nparts, stride, fit);
        if (!rc && fit_after && cp_check) rc = launch_cp_check(p);
        return rc || next_factor < 0 ? rc : launch_factor(p, next_factor);
    }
    rc = run_apply(p, mode, Msrc, nparts, stride, finalize, fit_after);
    if (rc || !finalize) return rc;
    const int64_t In = p->dims[mode];
    const bool fit = fit_after && !cp_check;
    // R > 64: the Gram of X by its own launch; M is still where the solve read it
    if ((rc = p->RT ? run_finalize(p, mode, solve_nb(In, R), p->Msum, fit)
                    : run_gram_finalize(p, mode, Msrc, fit)))
        return rc;
    const int nbf = finalize_nb(In, R);
    if (fit_after && cp_check) {
        if ((rc = launch_cp_check(p))) return rc;
    } else if (fit_after) {
        hipLaunchKernelGGL(k_fit, dim3(1), dim3(FIT_THREADS), 0, p->stream, p->inner_part, nbf, R, grams_of(p),
                           p->lam, p->scal, p->chk, p->fit_trace, p->trace_cap);
        ITCPD_HIP(hipGetLastError());
    }
    if (next_factor >= 0) return launch_factor(p, next_factor);
    return ITCPD_OK;
}

int launch_update_mode(itcpd_plan* p, int mode, bool fit_after, const double* Msrc, int nparts,
                       int64_t stride) {
    int rc;
    if ((rc = launch_factor(p, mode))) return rc;
    return launch_solve(p, mode, Msrc, nparts, stride, true, fit_after, -1);
}

int launch_normalize(itcpd_plan* p, int mode, const double* Xsrc, bool fit_after) {
    const int64_t In = p->dims[mode];
    const int R = (int)p->R;
    const int rpb = rows_per_block_for(R);
    const int nb2 = norm_blocks(In, R, rpb);
    const int nsp = solve_blocks(In);
    const size_t lds = (size_t)(R + rpb * R) * 8;
    hipLaunchKernelGGL(k_normalize, dim3(nb2), dim3(256), lds, p->stream, Xsrc, In, R, (int)p->Rp,
                       p->sumsq_part, nsp, rpb, p->A[mode], p->At[mode], p->lam, p->gram_part,
                       p->M, fit_after ? 1 : 0, p->inner_part, 1, p->chk);
    ITCPD_HIP(hipGetLastError());
    // the Gram partials summed over the chip (in block order, as k_gram_final would), then
    // the check on one workgroup
    int rc;
    if ((rc = launch_sum_parts(p, MSrc{p->gram_part, nb2, (int64_t)R * R}, (int64_t)R * R, p->G[mode])))
        return rc;
    hipLaunchKernelGGL(k_gram_final, dim3(1), dim3(256), 0, p->stream, (const double*)nullptr, nb2, R,
                       p->G[mode], grams_of(p), mode, p->lam, p->inner_part, fit_after ? 1 : 0,
                       p->scal, p->chk, p->fit_trace, p->trace_cap);
    ITCPD_HIP(hipGetLastError());
    return ITCPD_OK;
}

// Gram cache seeding (optimizers/als_optimizers/standard/tensor.jl:12) and the
// rank-fastest copies of the factors.
//
// One launch for the copies and one for the Grams of every mode of at most 2048 rows; longer
// modes sum row ranges.  Was a row-normalisation and a single-workgroup sum per mode: 3 x 89
// us at 512^3 rank 64, 3 x 290 us at 200^3 rank 150.
int launch_seed_grams(itcpd_plan* p) {
    const int R = (int)p->R;
    TransposeJobs tj{};
    GramJobs gj{};
    int64_t imax = 0;
    for (int m = 0; m < p->N; ++m) {
        tj.A[m] = gj.X[m] = p->A[m];
        tj.At[m] = p->At[m];
        tj.I[m] = gj.I[m] = p->dims[m];
        gj.S[m] = p->G[m];
        imax = std::max(imax, p->dims[m]);
    }
    hipLaunchKernelGGL(k_rank_fast, dim3((unsigned)cdiv(imax, 32), (unsigned)cdiv(R, 32), (unsigned)p->N), dim3(256),
                       0, p->stream, tj, R, (int)p->Rp);
    ITCPD_HIP(hipGetLastError());
    if (gram_parts(imax, R) == 1) {
        hipLaunchKernelGGL(k_gram_mfma, dim3(gram_tiles(R), 1, (unsigned)p->N), dim3(256), 0, p->stream, gj, R, 1,
                           (const DevCheck*)nullptr);
        ITCPD_HIP(hipGetLastError());
        return ITCPD_OK;
    }
    for (int m = 0; m < p->N; ++m) {
        const int nb = gram_parts(p->dims[m], R);
        GramJobs one{};
        one.X[0] = p->A[m];
        one.I[0] = p->dims[m];
        one.S[0] = nb == 1 ? p->G[m] : p->gram_part;
        hipLaunchKernelGGL(k_gram_mfma, dim3(gram_tiles(R), (unsigned)nb), dim3(256), 0, p->stream, one, R, nb,
                           (const DevCheck*)nullptr);
        ITCPD_HIP(hipGetLastError());
        if (nb == 1) continue;
        if (int rc = launch_sum_parts(p, MSrc{p->gram_part, nb, (int64_t)R * R}, (int64_t)R * R, p->G[m])) return rc;
    }
    return ITCPD_OK;
}

__global__ void k_reset_flags(DevCheck* __restrict__ chk) {
    chk->done = 0;
    chk->nan_flag = 0;
}
int launch_reset_flags(itcpd_plan* p) {
    hipLaunchKernelGGL(k_reset_flags, dim3(1), dim3(1), 0, p->stream, p->chk);
    ITCPD_HIP(hipGetLastError());
    return ITCPD_OK;
}

// random_factors (cpd.jl:48-60): draw, row_norm, lambda from the last mode.
int launch_random_init(itcpd_plan* p, uint64_t seed) {
    const int R = (int)p->R;
    const int rpb = rows_per_block_for(R);
    for (int m = 0; m < p->N; ++m) {
        const int64_t In = p->dims[m];
        hipLaunchKernelGGL(k_random_normal, dim3((unsigned)cdiv(In * R, 256)), dim3(256), 0,
                           p->stream, p->X, In, R, seed, m);
        ITCPD_HIP(hipGetLastError());
        const int nsp = solve_blocks(In);
        const int per = (int)cdiv(In, nsp);
        hipLaunchKernelGGL(k_col_sumsq, dim3(nsp), dim3(256), 0, p->stream, p->X, In, R, per,
                           p->sumsq_part);
        ITCPD_HIP(hipGetLastError());
        const int nb2 = norm_blocks(In, R, rpb);
        const size_t lds = (size_t)(R + rpb * R) * 8;
        hipLaunchKernelGGL(k_normalize, dim3(nb2), dim3(256), lds, p->stream, p->X, In, R,
                           (int)p->Rp, p->sumsq_part, nsp, rpb, p->A[m], p->At[m], p->lam,
                           p->gram_part, p->M, 0, p->inner_part, 1, (const DevCheck*)nullptr);
        ITCPD_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_gram_final, dim3(1), dim3(256), 0, p->stream, p->gram_part, nb2, R,
                           p->G[m], grams_of(p), m, p->lam, p->inner_part, 0, p->scal,
                           (DevCheck*)nullptr, (double*)nullptr, 0);
        ITCPD_HIP(hipGetLastError());
    }
    return ITCPD_OK;
}

int launch_fit_only(itcpd_plan* p, const double* Mlast, double ref_norm) {
    const int N = p->N;
    hipLaunchKernelGGL(k_fit_hook, dim3(1), dim3(256), 0, p->stream, Mlast, p->A[N - 1],
                       p->dims[N - 1], (int)p->R, p->lam, grams_of(p), ref_norm, p->scal);
    ITCPD_HIP(hipGetLastError());
    return ITCPD_OK;
}

int launch_hadamard(itcpd_plan* p, int mode, double* V) {
    const int R = (int)p->R;
    hipLaunchKernelGGL(k_hadamard_grams, dim3((unsigned)cdiv((int64_t)R * R, 256)), dim3(256), 0,
                       p->stream, grams_of(p), mode, R, V);
    ITCPD_HIP(hipGetLastError());
    return ITCPD_OK;
}

// Column sums of squares of X in the block partition the row solve uses.
int launch_col_sumsq(itcpd_plan* p, int mode, const double* X) {
    const int64_t In = p->dims[mode];
    const int nsp = solve_blocks(In);
    const int per = (int)cdiv(In, nsp);
    hipLaunchKernelGGL(k_col_sumsq, dim3(nsp), dim3(256), 0, p->stream, X, In, (int)p->R, per,
                       p->sumsq_part);
    ITCPD_HIP(hipGetLastError());
    return ITCPD_OK;
}


int launch_reconstruct(int order, const int64_t* dims, int64_t rank, const double* const* factors_dev,
                       const double* lambda_dev, void* out, int out_elt, double sigma, uint64_t seed,
                       hipStream_t st) {
    RecoArgs ra{};
    ra.N = order;
    int64_t nel = 1;
    for (int n = 0; n < order; ++n) {
        ra.A[n] = factors_dev[n];
        ra.dims[n] = dims[n];
        nel *= dims[n];
    }
    // the tiled form when both groups of modes are large enough to fill 64-element tiles:
    // the split whose groups are closest in size, the right group's tiles along y
    RecoSplit rs{};
    rs.N = order;
    int best_s = 0;
    double best = 1e300;
    for (int sp = 1; sp < order; ++sp) {
        double ml = 1.0, mr = 1.0;
        for (int n = 0; n < sp; ++n) ml *= (double)dims[n];
        for (int n = sp; n < order; ++n) mr *= (double)dims[n];
        const double d = fabs(log(ml) - log(mr));
        if (mr / 64.0 <= 65535.0 && d < best) { best = d; best_s = sp; }
    }
    if (best_s > 0) {
        rs.s = best_s;
        rs.ML = 1;
        rs.MR = 1;
        for (int n = 0; n < order; ++n) {
            rs.A[n] = factors_dev[n];
            rs.dims[n] = dims[n];
            if (n < best_s) rs.ML *= dims[n];
            else rs.MR *= dims[n];
        }
        const int64_t gx = cdiv(rs.ML, 64), gy = cdiv(rs.MR, 64);
        if (rs.ML >= 64 && rs.MR >= 64 && gx <= 0x7FFFFFFF) {
            const dim3 grid((unsigned)gx, (unsigned)gy);
            if (out_elt == 8)
                hipLaunchKernelGGL(k_reconstruct_tiled<double>, grid, dim3(256), 0, st, rs, (int)rank, lambda_dev,
                                   sigma, seed, (double*)out);
            else
                hipLaunchKernelGGL(k_reconstruct_tiled<float>, grid, dim3(256), 0, st, rs, (int)rank, lambda_dev,
                                   sigma, seed, (float*)out);
            ITCPD_HIP(hipGetLastError());
            return ITCPD_OK;
        }
    }
    if (out_elt == 8)
        hipLaunchKernelGGL(k_reconstruct<double>, dim3((unsigned)cdiv(nel, 256)), dim3(256), 0, st, ra,
                           (int)rank, lambda_dev, nel, sigma, seed, (double*)out);
    else
        hipLaunchKernelGGL(k_reconstruct<float>, dim3((unsigned)cdiv(nel, 256)), dim3(256), 0, st, ra,
                           (int)rank, lambda_dev, nel, sigma, seed, (float*)out);
    ITCPD_HIP(hipGetLastError());
    return ITCPD_OK;
}

}  // namespace itcpd
