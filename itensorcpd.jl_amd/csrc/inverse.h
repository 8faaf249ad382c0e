// V^-1 for 64 < R <= 1024 by block Gauss-Jordan elimination over the chip, the row solves
// X = M V^-1 and the Gram products X^T X on FP64 MFMA (included by solve.hip).
//
// The pivoted Cholesky that the reference runs is a chain of R dependent steps on one
// workgroup; for the well-conditioned V of most sweeps its pivoting changes nothing.  So, as
// factor64_unpivoted does for R <= 64, V^-1 is first formed without pivoting and kept only
// when that provably loses no pivot (wide_certified); else the pivoted kernels run.
//
// V is padded to Rq = 64 nb with the identity and kept as nb x nb blocks of 64.  Launch k
// (k_inv_step) reads the blocks of buffer k & 1, the inverse P of the pivot block (k, k), and
// writes buffer (k + 1) & 1:
//   (k, k) <- P,  (k, j) <- P A_kj,  (i, k) <- -A_ik P,  (i, j) <- A_ij - A_ik P A_kj,
// one workgroup per block; the one of block (k + 1, k + 1) goes on to invert it (sweep_inverse).
// After nb launches the buffer holds V^-1.  The pivot blocks are the Schur complements of
// the unpivoted block factorisation, so their Cholesky pivots are those of V.
//
// Bound by the chain of nb pivot-block inverses (18-27 us a launch).  Whole factorisation
// with the pivoted kernel's early exit, us: R = 128 76 (197 for the pivoted one), R = 150 79
// (931); row solves, Gram and finalize: R = 128, I = 224 31 (145), R = 150, I = 200 29 (244).
#pragma once
#include "dense_la.h"
#include "factor64.h"
#include "gemm64.h"

namespace itcpd {

constexpr int INV_LD = 66;
constexpr int INV_TILE = 64 * INV_LD;
// three 64 x 64 tiles and the inverse's broadcast rows
constexpr size_t INV_LDS = (size_t)(3 * INV_TILE + SWEEP_ROWS) * 8;


// Sums (or maxima) of v over the workgroup's four waves by red[0..3]; thread 0 gets it.
__device__ __forceinline__ double block4_sum(double v, double* red) {
    const int t = threadIdx.x;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if ((t & 63) == 0) red[t >> 6] = v;
    __syncthreads();
    v = (red[0] + red[1]) + (red[2] + red[3]);
    __syncthreads();
    return v;
}

// Inverts the rb x rb pivot block of the 64 x 64 tile S into P (identity beyond rb).
__device__ __forceinline__ void inv_pivot(const double* S, double* rows, int rb, double* __restrict__ P,
                                          double* __restrict__ flag) {
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
    double a[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int r = 16 * w + i;
        a[i] = r < rb && l < rb ? S[r * INV_LD + l] : 0.0;
    }
    const bool pos = sweep_inverse<4>(a, rb, w, l, rows);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int r = sweep_row(rb, w, i);
        P[r * 64 + l] = r < rb && l < rb ? -a[i] : (r == l ? 1.0 : 0.0);
    }
    if (threadIdx.x == 0) flag[0] = pos ? 0.0 : 1.0;
}

// V = Hadamard of the Grams of modes != mode in blocks, identity beyond R; block (0, 0) is
// inverted right away.
__global__ __launch_bounds__(256) void k_inv_first(GramSet gs, int mode, int R, int nb, double* __restrict__ V,
                                                   double* __restrict__ P, double* __restrict__ stat,
                                                   const DevCheck* __restrict__ chk) {
    if (chk->done) return;
    extern __shared__ __attribute__((aligned(16))) double S[];
    __shared__ double red[4];
    const int t = threadIdx.x, l = t & 63, w = t >> 6;
    const int bi = blockIdx.x, bj = blockIdx.y, Rq = 64 * nb;
    double v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = 1.0;
    for (int m = 0; m < gs.N; ++m) {
        if (m == mode) continue;
        const double* __restrict__ G = gs.G[m];
        double g[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const int i = 64 * bi + w + 4 * k, j = 64 * bj + l;
            g[k] = G[i < R && j < R ? (int64_t)i * R + j : 0];
        }
#pragma unroll
        for (int k = 0; k < 16; ++k) v[k] *= g[k];
    }
    double vsq = 0.0, dmax = 0.0;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const int i = 64 * bi + w + 4 * k, j = 64 * bj + l;
        const bool in = i < R && j < R;
        const double x = in ? v[k] : (i == j ? 1.0 : 0.0);
        V[(int64_t)i * Rq + j] = x;
        if (bi == 0 && bj == 0) S[(w + 4 * k) * INV_LD + l] = x;
        if (in) {
            vsq = fma(x, x, vsq);
            if (i == j) dmax = fmax(dmax, x);
        }
    }
    vsq = block4_sum(vsq, red);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) dmax = fmax(dmax, __shfl_xor(dmax, o));
    if (l == 0) red[w] = dmax;
    __syncthreads();
    if (t == 0) {
        stat[bi * nb + bj] = vsq;
        stat[nb * nb + bi * nb + bj] = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
    }
    if (bi == 0 && bj == 0) inv_pivot(S, S + INV_TILE, R < 64 ? R : 64, P, stat + 3 * nb * nb);
}

__global__ __launch_bounds__(256) void k_inv_step(int k, int R, int nb, const double* __restrict__ src,
                                                  double* __restrict__ dst, const double* __restrict__ P,
                                                  double* __restrict__ Pnext, double* __restrict__ stat,
                                                  const DevCheck* __restrict__ chk) {
    if (chk->done) return;
    extern __shared__ __attribute__((aligned(16))) double S[];
    __shared__ double red[4];
    double* Pt = S;                // P, later the next pivot block
    double* At = S + INV_TILE;     // A_ik, then A_ik P
    double* Bt = At + INV_TILE;    // A_kj
    double* rows = Bt + INV_TILE;
    const int t = threadIdx.x, l = t & 63, c = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int bi = blockIdx.x, bj = blockIdx.y;
    const int64_t Rq = 64 * (int64_t)nb;
    const bool prow = bi == k, pcol = bj == k;
    auto load = [&](double* d, const double* s, int64_t ld) {
        double v[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) v[q] = s[(w + 4 * q) * ld + l];
#pragma unroll
        for (int q = 0; q < 16; ++q) d[(w + 4 * q) * INV_LD + l] = v[q];
    };
    load(Pt, P, 64);
    if (!prow) load(At, src + 64 * bi * Rq + 64 * k, Rq);
    if (!pcol) load(Bt, src + 64 * k * Rq + 64 * bj, Rq);
    // row block w (16 rows) of a product of two tiles, lane layout D[g + 4 v][c] per column block
    d4 acc[4];
    auto product = [&](const double* L, const double* M) {
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[b] = (d4){0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
        for (int k0 = 0; k0 < 64; k0 += 4) {
            const double a = L[(16 * w + c) * INV_LD + k0 + g];
#pragma unroll
            for (int b = 0; b < 4; ++b) acc[b] = mfma_f64(a, M[(k0 + g) * INV_LD + 16 * b + c], acc[b]);
        }
    };
    double aij[4][4];
    if (!prow && !pcol) {
        const double* s = src + 64 * bi * Rq + 64 * bj;
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) aij[b][v] = s[(16 * w + g + 4 * v) * Rq + 16 * b + c];
    }
    __syncthreads();
    if (prow && pcol) {
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[b][v] = Pt[(16 * w + g + 4 * v) * INV_LD + 16 * b + c];
    } else if (prow) {
        product(Pt, Bt);
    } else {
        product(At, Pt);
        if (pcol) {
#pragma unroll
            for (int b = 0; b < 4; ++b) acc[b] = -acc[b];
        } else {
            // A_ik P replaces this wave's own rows of A_ik (no other wave reads them)
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int v = 0; v < 4; ++v) At[(16 * w + g + 4 * v) * INV_LD + 16 * b + c] = acc[b][v];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            product(At, Bt);
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[b][v] = aij[b][v] - acc[b][v];
        }
    }
    double* d = dst + 64 * bi * Rq + 64 * bj;
    double zsq = 0.0;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = 16 * w + g + 4 * v, j = 16 * b + c;
            d[i * Rq + j] = acc[b][v];
            if (64 * bi + i < R && 64 * bj + j < R) zsq = fma(acc[b][v], acc[b][v], zsq);
        }
    if (k == nb - 1) {
        zsq = block4_sum(zsq, red);
        if (t == 0) stat[2 * nb * nb + bi * nb + bj] = zsq;
        return;
    }
    if (bi == k + 1 && bj == k + 1) {
        __syncthreads();   // every wave is done with P
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) Pt[(16 * w + g + 4 * v) * INV_LD + 16 * b + c] = acc[b][v];
        __syncthreads();
        const int rb = R - 64 * (k + 1) < 64 ? R - 64 * (k + 1) : 64;
        inv_pivot(Pt, rows, rb, Pnext, stat + 3 * nb * nb + k + 1);
    }
}

// factor64_unpivoted's certificate from the statistics (see there): uniform over the
// workgroup.  Every pivot of the pivoted factorisation is >= lambda_min(V) >= 1 / ||V^-1||_F.
__device__ __forceinline__ bool wide_certified(const double* __restrict__ stat, int nb, int R, double tol) {
    __shared__ int ok;
    const int t = threadIdx.x;
    if (t < 64) {
        double vsq = 0.0, dmax = 0.0, zsq = 0.0, bad = 0.0;
        for (int x = t; x < nb * nb; x += 64) {
            vsq += stat[x];
            dmax = fmax(dmax, stat[nb * nb + x]);
            zsq += stat[2 * nb * nb + x];
        }
        if (t < nb) bad = stat[3 * nb * nb + t];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            vsq += __shfl_xor(vsq, o);
            dmax = fmax(dmax, __shfl_xor(dmax, o));
            zsq += __shfl_xor(zsq, o);
            bad += __shfl_xor(bad, o);
        }
        const double vF = sqrt(vsq), zF = sqrt(zsq);
        if (t == 0)
            ok = bad == 0.0 && zF > 0.0 && zF < __builtin_inf() &&
                 1.0 / zF > 2.0 * tol + 64.0 * R * 0x1p-52 * dmax && vF * zF < 1e12;
    }
    __syncthreads();
    return ok != 0;
}

// Row solves X = M V^-1 with the certified inverse: wave w of block (x, y) takes the 16 x 16
// tile of rows 16 x .. and columns 16 (4 y + w) .. over k < R, 16 k-steps of both operands
// in flight.  Latency-bound (a few hundred rows): one tile per wave spreads a mode over
// In R / 1024 workgroups.
__global__ __launch_bounds__(256) void k_solve_inv(const double* __restrict__ M, int64_t In, int R,
                                                   const double* __restrict__ Vinv, int64_t Rq,
                                                   const int* __restrict__ finfo, double* __restrict__ X,
                                                   const DevCheck* __restrict__ chk) {
    if (chk->done || finfo[3] != 1) return;
    const int t = threadIdx.x, l = t & 63, c = l & 15, g = l >> 4;
    const int col = 16 * (4 * blockIdx.y + (t >> 6)) + c;
    const int64_t i0 = (int64_t)blockIdx.x * 16;
    if (col - c >= R) return;
    const int64_t ia = i0 + c < In ? i0 + c : In - 1;
    const double* __restrict__ Vc = Vinv + (col < R ? col : R - 1);
    d4 acc[2] = {(d4){0.0, 0.0, 0.0, 0.0}, (d4){0.0, 0.0, 0.0, 0.0}};
    for (int k0 = 0; k0 < R; k0 += 64) {
        double a[16], b[16];
#pragma unroll
        for (int s = 0; s < 16; ++s) {
            const int k = k0 + 4 * s + g, kc = k < R ? k : R - 1;
            a[s] = M[ia + In * kc];
            b[s] = Vc[kc * Rq];
        }
#pragma unroll
        for (int s = 0; s < 16; ++s) {
            const bool in = k0 + 4 * s + g < R;
            acc[s & 1] = mfma_f64(in ? a[s] : 0.0, in ? b[s] : 0.0, acc[s & 1]);
        }
    }
    if (col >= R) return;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int64_t row = i0 + g + 4 * v;
        if (row < In) X[row + In * col] = acc[0][v] + acc[1][v];
    }
}

// Gram products S_z = X_z^T X_z of column-major I_z x R matrices (blockIdx.z), one workgroup
// per upper 16 x 16 tile and row range (blockIdx.y): part y goes to S + y R^2.  The four
// waves split the rows in 16-row stages, lane (c, g) reading four consecutive rows of columns
// 16 ta + c and 16 tb + c, and add up through LDS.
struct GramJobs {
    const double* X[ITCPD_MAX_ORDER];
    double* S[ITCPD_MAX_ORDER];
    int64_t I[ITCPD_MAX_ORDER];
};
__global__ __launch_bounds__(256) void k_gram_mfma(GramJobs jobs, int R, int nparts,
                                                   const DevCheck* __restrict__ chk) {
    if (chk && chk->done) return;
    const int t = threadIdx.x, l = t & 63, c = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    int tb = 0, ta = blockIdx.x;
    while (ta > tb) { ta -= tb + 1; ++tb; }   // tiles (0,0), (0,1), (1,1), (0,2), ...
    const double* __restrict__ X = jobs.X[blockIdx.z];
    const int64_t In = jobs.I[blockIdx.z];
    const int ca = 16 * ta + c < R ? 16 * ta + c : R - 1, cb = 16 * tb + c < R ? 16 * tb + c : R - 1;
    const double* __restrict__ pa = X + In * ca;
    const double* __restrict__ pb = X + In * cb;
    const int64_t nst = (In + 15) / 16;
    const int64_t per = (nst + nparts - 1) / nparts;
    int64_t s0 = (int64_t)blockIdx.y * per, s1 = s0 + per < nst ? s0 + per : nst;
    const int64_t wper = s1 > s0 ? (s1 - s0 + 3) / 4 : 0;
    s0 = s0 + w * wper < s1 ? s0 + w * wper : s1;
    s1 = s0 + wper < s1 ? s0 + wper : s1;
    d4 acc[1] = {(d4){0.0, 0.0, 0.0, 0.0}};
    const int64_t full = In / 16 < s1 ? In / 16 : s1;
    int64_t s = s0;
    for (; s + 2 <= full; s += 2) {
        double a[2][4], b[2][4];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            ld_run4<double, 4>(pa + 16 * (s + u) + 4 * g, a[u]);
            ld_run4<double, 4>(pb + 16 * (s + u) + 4 * g, b[u]);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q) acc[0] = mfma_f64(a[u][q], b[u][q], acc[0]);
    }
    for (; s < s1; ++s) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int64_t i = 16 * s + 4 * g + q, ic = i < In ? i : In - 1;
            const double a = pa[ic], b = pb[ic];
            acc[0] = mfma_f64(i < In ? a : 0.0, i < In ? b : 0.0, acc[0]);
        }
    }
    __shared__ d4 red[1][64];
    if (!sum_waves<1>(acc, red, w, l)) return;
    double* S = jobs.S[blockIdx.z] + (int64_t)blockIdx.y * R * R;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int r = 16 * ta + g + 4 * v, r2 = 16 * tb + c;
        if (r < R && r2 < R) {
            S[(int64_t)r * R + r2] = acc[0][v];
            S[(int64_t)r2 * R + r] = acc[0][v];
        }
    }
}

// Rank-fastest copies of column-major factors (At[i][r] = A[i + I r]), one 32 x 32 tile per
// workgroup through LDS; blockIdx.z = the mode.
struct TransposeJobs {
    const double* A[ITCPD_MAX_ORDER];
    double* At[ITCPD_MAX_ORDER];
    int64_t I[ITCPD_MAX_ORDER];
};
__global__ __launch_bounds__(256) void k_rank_fast(TransposeJobs jobs, int R, int Rp) {
    __shared__ double tile[32][33];
    const int x = threadIdx.x & 31, y = threadIdx.x >> 5;
    const int64_t In = jobs.I[blockIdx.z];
    const int64_t i0 = (int64_t)blockIdx.x * 32;
    const int r0 = blockIdx.y * 32;
    if (i0 >= In) return;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int r = r0 + y + 8 * q;
        if (i0 + x < In && r < R) tile[y + 8 * q][x] = jobs.A[blockIdx.z][i0 + x + In * r];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int64_t i = i0 + y + 8 * q;
        if (i < In && r0 + x < R) jobs.At[blockIdx.z][i * Rp + r0 + x] = tile[x][y + 8 * q];
    }
}

}  // namespace itcpd
