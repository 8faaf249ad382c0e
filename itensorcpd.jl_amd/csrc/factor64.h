// The R <= 64 pivoted Cholesky + V^-1 (one 256-thread workgroup), shared by the
// standalone factor kernel (solve.hip) and the GEMM launches that run it in an
// extra workgroup (mttkrp.hip).
#pragma once
#include "dense_la.h"

namespace itcpd {

constexpr size_t FACTOR64_LDS = (size_t)(2 * 64 * 66) * 8;
// LDS of the unpivoted form alone: V / U / U^-1 (64 x 66) and 144 doubles of
// reductions, 1/U(j,j) and the broadcast row
constexpr int FACTOR64_RED = 64 * 66;
constexpr size_t FACTOR64_UNPIV_LDS = (size_t)(64 * 66 + 144) * 8;

// The blocked inverse of a symmetric positive definite matrix of at most 64 rows in LDS (one
// 256-thread workgroup; S: the matrix padded to 64 with the identity, ld 66; nbk = its
// 16-row panels; red = S + FACTOR64_RED with red[12] = 0 on entry).  Unpivoted Cholesky
// V = U^T U, then U^-1 in place.  Per 16-row panel kb: wave 0 factors the whole block row in
// registers (lane l holds column l; row j comes through LDS), the trailing update A(ib, jb)
// -= U(kb, ib)^T U(kb, jb) runs on FP64 MFMA.  Then the diagonal blocks of U^-1 by
// substitution (one wave each), the off-diagonal blocks block row by block row from the
// bottom, X(i, j) = -X(i, i) sum_{i<k<=j} U(i, k) X(k, j) (row i of U is read before it is
// overwritten).  red[12] = 1 when a pivot was not > 0; 1/U(j,j) in red[16 + j].
__device__ __forceinline__ void inv64_core(double* S, double* red, int nbk) {
    constexpr int LDT = 66;
    const int t = threadIdx.x, l = t & 63, c = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    double* invd = red + 16;      // 1/U(j,j), 64 doubles
    double* rowj = red + 80;      // one row of the block row, 64 doubles
    for (int kb = 0; kb < nbk; ++kb) {
        const int b0 = 16 * kb;
        if (w == 0) {
            // Block row kb (rows b0..b0+15, all 64 columns): lane l holds column l.
            // Step j: row j goes through LDS (lane l writes A(b0+j, l)); d =
            // A(b0+j, b0+j), 1/sqrt(d) from the hardware estimate and two Newton
            // steps, U(b0+j, l) = A(b0+j, l)/sqrt(d) for l > b0+j, and rows i > j take
            // A(b0+i, l) -= A(b0+j, b0+i) A(b0+j, l) / d.  Lanes l < b0 (finished
            // columns) compute along on values nobody reads and store zeros.
            double col[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) col[i] = S[(b0 + i) * LDT + l];
            bool pos = true;
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                rowj[l] = col[j];
                const double d = rowj[b0 + j];
                double bi[16];
#pragma unroll
                for (int i = j + 1; i < 16; ++i) bi[i] = rowj[b0 + i];
                pos = pos && d > 0.0;
                const double dc = fmax(d, 0x1p-1020);
                const double h = 0.5 * dc;
                double y = __builtin_amdgcn_rsq(dc);
                y = fma(y, fma(-h * y, y, 0.5), y);
                y = fma(y, fma(-h * y, y, 0.5), y);
                const double u = l > b0 + j ? col[j] * y : (l == b0 + j ? dc * y : 0.0);
                const double ncu = -(u * y);
#pragma unroll
                for (int i = j + 1; i < 16; ++i) col[i] = fma(bi[i], ncu, col[i]);
                col[j] = u;
                invd[b0 + j] = y;
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) S[(b0 + i) * LDT + l] = l >= b0 + i ? col[i] : 0.0;
            if (!pos) red[12] = 1.0;
        }
        __syncthreads();
        // trailing update of the upper blocks kb < ib <= jb (round-robin over waves).
        // f64 16x16x4 layout: A lane (c, g) = A[c][k0+g], B lane = B[k0+g][c], result
        // v = D[g+4v][c]
        if (kb + 1 < nbk) {
            int idx = 0;
            for (int ib = kb + 1; ib < nbk; ++ib)
                for (int jb = ib; jb < nbk; ++jb, ++idx) {
                    if ((idx & 3) != w) continue;
                    d4 acc;
#pragma unroll
                    for (int v = 0; v < 4; ++v) acc[v] = S[(16 * ib + g + 4 * v) * LDT + 16 * jb + c];
#pragma unroll
                    for (int k0 = 0; k0 < 16; k0 += 4)
                        acc = mfma_f64(-S[(b0 + k0 + g) * LDT + 16 * ib + c], S[(b0 + k0 + g) * LDT + 16 * jb + c],
                                       acc);
#pragma unroll
                    for (int v = 0; v < 4; ++v) S[(16 * ib + g + 4 * v) * LDT + 16 * jb + c] = acc[v];
                }
            __syncthreads();
        }
    }
    // diagonal blocks of U^-1, wave w block w: lane c computes column c by
    // substitution (zero below the diagonal; the four 16-lane groups alike)
    if (w < nbk) {
        const int b0 = 16 * w;
        double xv[16];
#pragma unroll
        for (int i = 15; i >= 0; --i) {
            double acc0 = (i == c) ? 1.0 : 0.0, acc1 = 0.0;
#pragma unroll
            for (int k = i + 1; k < 16; ++k) {
                const double uik = S[(b0 + i) * LDT + b0 + k];
                if (k & 1) acc1 -= uik * xv[k];
                else acc0 -= uik * xv[k];
            }
            xv[i] = (i <= c) ? (acc0 + acc1) * invd[b0 + i] : 0.0;
        }
        // (the wave's own reads of U(w, w) precede these writes)
#pragma unroll
        for (int i = 0; i < 16; ++i) S[(b0 + i) * LDT + b0 + c] = xv[i];
    }
    __syncthreads();
    // off-diagonal blocks of U^-1, block row bi from the bottom, wave w column
    // bi + 1 + w: X_ij = -X_ii sum_{k=i+1..j} U_ik X_kj, from row i of U and the
    // finished rows below; row i is overwritten after every wave has read it
    for (int bi = nbk - 2; bi >= 0; --bi) {
        const int bj = bi + 1 + w;
        d4 out = (d4){0.0, 0.0, 0.0, 0.0};
        if (bj < nbk) {
            const int i = 16 * bi + c;
            d4 acc = (d4){0.0, 0.0, 0.0, 0.0};
            for (int bk = bi + 1; bk <= bj; ++bk)
#pragma unroll
                for (int k0 = 0; k0 < 16; k0 += 4) {
                    const int kk = 16 * bk + k0 + g;
                    acc = mfma_f64(S[i * LDT + kk], S[kk * LDT + 16 * bj + c], acc);
                }
#pragma unroll
            for (int v = 0; v < 4; ++v) out = mfma_f64(-S[(16 * bi + c) * LDT + 16 * bi + 4 * v + g], acc[v], out);
        }
        __syncthreads();
        if (bj < nbk) {
#pragma unroll
            for (int v = 0; v < 4; ++v) S[(16 * bi + g + 4 * v) * LDT + 16 * bj + c] = out[v];
        }
        __syncthreads();
    }
}

// The upper 16 x 16 tiles of Z = U^-1 U^-T from inv64_core's S on FP64 MFMA (Z(a, b) sums
// over k >= max(a, b)): store(ra, rb, value, ta != tb) for the tiles ta <= tb below nbk.
template <typename F>
__device__ __forceinline__ void inv64_tiles(const double* S, int nbk, F store) {
    constexpr int LDT = 66;
    const int t = threadIdx.x, l = t & 63, c = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    constexpr int ZT[4][3][2] = {{{0, 0}, {0, 3}, {-1, -1}},
                                 {{0, 1}, {1, 3}, {2, 3}},
                                 {{1, 1}, {0, 2}, {-1, -1}},
                                 {{1, 2}, {2, 2}, {3, 3}}};
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const int ta = ZT[w][q][0], tb = ZT[w][q][1];
        if (ta < 0 || tb >= nbk) continue;
        d4 acc = (d4){0.0, 0.0, 0.0, 0.0};
        for (int k0 = 16 * tb; k0 < 16 * nbk; k0 += 4)
            acc = mfma_f64(S[(16 * ta + c) * LDT + k0 + g], S[(16 * tb + c) * LDT + k0 + g], acc);
#pragma unroll
        for (int v = 0; v < 4; ++v) store(16 * ta + g + 4 * v, 16 * tb + c, acc[v], ta != tb);
    }
}

// Unpivoted V = U^T U and V^-1 = U^-1 U^-T for the R <= 64 row solves (one 256-thread
// workgroup; V, then U, then U^-1 in S, FACTOR64_UNPIV_LDS bytes with red behind it).
//
// It stands in for the pivoted factorisation (xPSTRF, absolute tolerance tol) only
// when that one provably keeps every pivot: each pivoted pivot is a diagonal entry
// of a Schur complement of V, hence >= lambda_min(V), and lambda_min(V) >=
// 1 / ||V^-1||_F.  The computed inverse is trusted while ||V||_F ||V^-1||_F < 1e12;
// the bound must exceed 2 tol plus the pivots' rounding (64 R eps max V_ii); every
// unpivoted pivot must be > 0.  Then the solution (the unique minimiser) is the
// pivoted path's up to rounding, and V^-1, invdiag, piv (identity) and finfo are
// written; otherwise it returns false and writes nothing but V^-1 (which the
// caller's pivoted path overwrites or leaves unused).  Uniform result.
//
// Bound by its serial chain (about 2 us per 16-row panel), so only the ceil(R / 16)
// panels that hold any of V are worked on.  In the launch that it rides, us: R = 10,
// 11 (20 with all four panels); R = 24, 17 (21); R = 37, 19 (21).
__device__ __forceinline__ bool factor64_unpivoted(const GramSet& gs, int mode, int R, double tol,
                                                   double* __restrict__ Vinv, double* __restrict__ invdiag,
                                                   int* __restrict__ piv, int* __restrict__ finfo, double* S) {
    constexpr int LDT = 66;
    double* red = S + FACTOR64_RED;   // [0, 16) scalars, then 1/U(j,j) and the broadcast row
    const int t = threadIdx.x, l = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int nbk = (R + 15) >> 4;   // 16-row panels that hold any of V; the rest stay the identity
    if (t == 0) red[12] = 0.0;   // set by wave 0 when a pivot is not > 0
    // V (mode order of the Hadamard as the pivoted path), identity beyond R; thread
    // (w, l) fills column l of rows w, w + 4, ...; two modes' loads in flight at once
    {
        double v[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) v[k] = 1.0;
        for (int m0 = 0; m0 < gs.N; m0 += 2) {
            const bool on0 = m0 != mode, on1 = m0 + 1 < gs.N && m0 + 1 != mode;
            const double* __restrict__ G0 = gs.G[m0];
            const double* __restrict__ G1 = on1 ? gs.G[m0 + 1] : G0;
            double g0[16], g1[16];
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const int i = w + 4 * k;
                const int x = (i < R && l < R) ? i * R + l : 0;
                g0[k] = G0[x];
                g1[k] = G1[x];
            }
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                if (!on0) g0[k] = 1.0;
                if (!on1) g1[k] = 1.0;
            }
#pragma unroll
            for (int k = 0; k < 16; ++k) v[k] = (v[k] * g0[k]) * g1[k];
        }
        double vsq = 0.0, dmax = 0.0;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const int i = w + 4 * k;
            const bool in = i < R && l < R;
            const double x = in ? v[k] : (i == l ? 1.0 : 0.0);
            S[i * LDT + l] = x;
            if (in) {
                vsq = fma(x, x, vsq);
                if (i == l) dmax = fmax(dmax, x);
            }
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            vsq += __shfl_xor(vsq, o);
            dmax = fmax(dmax, __shfl_xor(dmax, o));
        }
        if (l == 0) {
            red[w] = vsq;
            red[4 + w] = dmax;
        }
    }
    __syncthreads();
    inv64_core(S, red, nbk);
    const double* invd = red + 16;
    // both halves of V^-1, and ||V^-1||_F^2 over the R x R block
    double zsq = 0.0;
    inv64_tiles(S, nbk, [&](int ra, int rb, double z, bool off) {
        if (ra < R && rb < R) {
            Vinv[ra * R + rb] = z;
            if (off) Vinv[rb * R + ra] = z;
            zsq = fma((off ? 2.0 : 1.0) * z, z, zsq);
        }
    });
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) zsq += __shfl_xor(zsq, o);
    if (l == 0) red[8 + w] = zsq;
    __syncthreads();
    const double vF = sqrt((red[0] + red[1]) + (red[2] + red[3]));
    const double dmax = fmax(fmax(red[4], red[5]), fmax(red[6], red[7]));
    const double zF = sqrt((red[8] + red[9]) + (red[10] + red[11]));
    const bool cert = red[12] == 0.0 && zF > 0.0 && zF < __builtin_inf() &&
                      1.0 / zF > 2.0 * tol + 64.0 * R * 0x1p-52 * dmax && vF * zF < 1e12;
    if (cert) {
        for (int j = t; j < R; j += 256) {
            invdiag[j] = invd[j];
            piv[j] = j;
        }
        if (t == 0) { finfo[0] = R; finfo[1] = 0; finfo[2] = R; }
    }
    __syncthreads();   // red and S are reused by the pivoted path
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
    if (Vinv && try_unpivoted && factor64_unpivoted(gs, mode, R, tol, Vinv, invdiag, piv, finfo, S)) return;
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
