// V^-1 for 64 < R <= 1024 by blocks over the chip, the row solves X = M V^-1 and the Gram
// products X^T X on FP64 MFMA (included by solve.hip).
//
// The pivoted Cholesky that the reference runs is a chain of R dependent steps on one
// workgroup; for the well-conditioned V of most sweeps its pivoting changes nothing.  So, as
// factor64_unpivoted does for R <= 64, V^-1 is first formed without pivoting and kept only
// when that provably loses no pivot (wide_certified); else the pivoted kernels run.
//
// V is padded to Rq = 64 nb with the identity and kept as nb x nb blocks of 64.  Its Cholesky
// factor's inverse N = D^-1/2 L^-1 (lower triangular) comes row of blocks by row of blocks, one
// launch each; block row k of buffer k & 1 ends as
//   (k, k) N_kk = C^-1,  (k, j) N_kj = C^-1 A_kj (j > k: rows of the factor, j < k: of N),
// C the Cholesky factor of the pivot block A_kk, and the next launch takes A_ij - N_ki^T N_kj
// below it (A_ik counting as zero: the identity's column).  A workgroup (k, j) eliminates a pivot
// block of its own (sweep_triangular) and solves with its factor by 16-row blocks, so nothing
// waits for another one.  At cond(V) = 2e10 that leaves 1e-7 of X; multiplying by an explicit
// C^-1, of 64 rows or of 16 without the correction, up to 100 times more, and updating the
// rows above (Gauss-Jordan) nothing that is right.  V^-1 = N^T N by tiles over the chip.
//
// Bound by the chain of nb eliminations (28-31 us a launch, the last one less).  Whole
// factorisation with the pivoted kernel's early exit, us: R = 128 69 (197 for the pivoted one), R =
// 150 88 (931); row solves, Gram and finalize: R = 128, I = 224 31 (145), R = 150, I = 200 29
// (244).
#pragma once
#include "dense_la.h"
#include "factor64.h"
#include "gemm64.h"

namespace itcpd {

constexpr int INV_LD = 66;
constexpr int INV_TILE = 64 * INV_LD;
// two 64 x 64 tiles and the elimination's rows
constexpr size_t INV_LDS = (size_t)(2 * INV_TILE + SWEEP_ROWS) * 8;

// Statistics of the certificate: ||V||_F^2 and the largest diagonal entry of every block, a flag
// per pivot block (nonzero: a pivot was not positive), ||V^-1||_F^2 of every tile of 16.
struct InvStat {
    double *vsq, *dmax, *bad, *zsq;
    __host__ __device__ InvStat(double* s, int nb) : vsq(s), dmax(s + nb * nb), bad(s + 2 * nb * nb), zsq(bad + nb) {}
};
inline __host__ __device__ int inv_tiles(int R) {
    const int nt = (R + 15) / 16;
    return nt * (nt + 1) / 2;
}
size_t inv_stat_elems(int64_t R) {
    const int64_t nb = cdiv(R, 64);
    return (size_t)(2 * nb * nb + nb + inv_tiles((int)R));
}

// Block (k, j) of N: the pivot block A_kk in x (row 16 w + i, column l at i) and, with panel (j
// != k), A_kj in y, wave w its columns 16 w .. in the products' layout (y[b][v]: row 16 b + g +
// 4 v, column 16 w + c), which is also what the next product reads.  The rows of 16 block b: r =
// A_b - sum_{b' < b} L_bb' Y_b', Y_b = W_bb r + W_bb (r - L_bb W_bb r) (the diagonal blocks of
// L^-1 are the inverses of L's).  Lt, Wt: tiles in LDS; dst: the block's place, ld Rq.
__device__ __forceinline__ void inv_row(double (&x)[16], d4 (&y)[4], int rb, bool panel, double* Lt, double* Wt,
                                        double* rows, double* __restrict__ dst, int64_t Rq,
                                        double* __restrict__ flag) {
    const int l = threadIdx.x & 63, c = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
    for (int i = 0; i < 16; ++i)
        if (16 * w + i >= rb || l >= rb) x[i] = 0.0;
    double rd;
    const bool pos = sweep_triangular<4, true>(x, rb, w, l, 0.0, rows, rd, Lt, INV_LD);
    const double sc = sqrt(rd);
    if (!panel) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int r = sweep_row(rb, w, i);
            dst[r * Rq + l] = x[i] * __shfl(sc, r);
        }
        if (threadIdx.x == 0) flag[0] = pos ? 0.0 : 1.0;
        return;
    }
    __syncthreads();   // the elimination's rows are read no more
#pragma unroll
    for (int i = 0; i < 16; ++i) Wt[sweep_row(rb, w, i) * INV_LD + l] = x[i];
    if (w == 0) rows[l] = sc;
    __syncthreads();
    auto lower = [&](int i, int k) {   // -L_ik, zero past the last row
        const double v = Lt[k * INV_LD + i];
        return k < rb && i > k ? -v : (i == k ? -1.0 : 0.0);
    };
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        d4 r = y[b], z = (d4){0.0, 0.0, 0.0, 0.0};
        double wv[4], lv[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            wv[s] = Wt[(16 * b + c) * INV_LD + 16 * b + 4 * s + g];
            lv[s] = lower(16 * b + c, 16 * b + 4 * s + g);
        }
#pragma unroll
        for (int q = 0; q < b; ++q)
#pragma unroll
            for (int s = 0; s < 4; ++s) r = mfma_f64(lower(16 * b + c, 16 * q + 4 * s + g), y[q][s], r);
#pragma unroll
        for (int s = 0; s < 4; ++s) z = mfma_f64(wv[s], r[s], z);
#pragma unroll
        for (int s = 0; s < 4; ++s) r = mfma_f64(lv[s], z[s], r);
#pragma unroll
        for (int s = 0; s < 4; ++s) z = mfma_f64(wv[s], r[s], z);
        y[b] = z;
    }
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = 16 * b + g + 4 * v;
            dst[r * Rq + 16 * w + c] = y[b][v] * rows[r];
        }
}

// V = Hadamard of the Grams of modes != mode in blocks on and above the diagonal, identity
// beyond R; block row 0 goes on to its rows of N.
__global__ __launch_bounds__(256) void k_inv_first(GramSet gs, int mode, int R, int nb, double* __restrict__ V,
                                                   double* __restrict__ stat, const DevCheck* __restrict__ chk) {
    const int bi = blockIdx.x, bj = blockIdx.y, Rq = 64 * nb;
    if (bi > bj || chk->done) return;
    extern __shared__ __attribute__((aligned(16))) double S[];
    __shared__ double red[2][4];
    const InvStat st(stat, nb);
    const int t = threadIdx.x, l = t & 63, c = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    double vsq = 0.0, dmax = 0.0;
    // 16 elements of block (ci, cj), element i at (row(i), column) of it
    auto hadamard = [&](int ci, int cj, auto row, int column, bool own, double (&x)[16]) {
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] = 1.0;
        for (int m = 0; m < gs.N; ++m) {
            if (m == mode) continue;
            const double* __restrict__ G = gs.G[m];
            double v[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int r = 64 * ci + row(i), q = 64 * cj + column;
                v[i] = G[r < R && q < R ? (int64_t)r * R + q : 0];
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) x[i] *= v[i];
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int r = 64 * ci + row(i), q = 64 * cj + column;
            if (r >= R || q >= R) {
                x[i] = r == q ? 1.0 : 0.0;
            } else if (own) {
                vsq = fma(x[i], x[i], vsq);
                if (r == q) dmax = fmax(dmax, x[i]);
            }
            if (own && bi > 0) V[(int64_t)r * Rq + q] = x[i];
        }
    };
    double x[16], e[16];
    const bool panel = bj > 0;
    if (panel) hadamard(bi, bj, [&](int i) { return 16 * (i >> 2) + g + 4 * (i & 3); }, 16 * w + c, true, e);
    if (bi == 0) hadamard(0, 0, [&](int i) { return 16 * w + i; }, l, !panel, x);
    vsq = wave_sum_dpp(vsq);
    dmax = wave_max_dpp(dmax);
    if (l == 0) {
        red[0][w] = vsq;
        red[1][w] = dmax;
    }
    __syncthreads();
    if (t == 0) {
        st.vsq[bi * nb + bj] = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
        st.dmax[bi * nb + bj] = fmax(fmax(red[1][0], red[1][1]), fmax(red[1][2], red[1][3]));
    }
    if (bi > 0) return;
    d4 y[4];
    if (panel)
#pragma unroll
        for (int i = 0; i < 16; ++i) y[i >> 2][i & 3] = e[i];
    inv_row(x, y, 64, panel, S, S + INV_TILE, S + 2 * INV_TILE, V + 64 * bj, Rq, st.bad);
}

// Launch k >= 1: A_ij - N_{k-1,i}^T N_{k-1,j} for the blocks of rows i >= k that later rows read
// (j >= i and j < k), then block row k's rows of N.  Grid: x the rows from k, y the columns.
__global__ __launch_bounds__(256) void k_inv_step(int k, int R, int nb, const double* __restrict__ src,
                                                  double* __restrict__ dst, double* __restrict__ stat,
                                                  const DevCheck* __restrict__ chk) {
    const int bi = k + blockIdx.x, bj = blockIdx.y;
    if ((bj >= k && bj < bi) || chk->done) return;
    extern __shared__ __attribute__((aligned(16))) double S[];
    double* Ti = S;                // N_{k-1,i}
    double* Tj = S + INV_TILE;     // N_{k-1,j}
    const InvStat st(stat, nb);
    const int t = threadIdx.x, l = t & 63, c = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int64_t Rq = 64 * (int64_t)nb;
    const bool pivot = bi == k, panel = bj != k;
    {
        const double* si = src + 64 * (k - 1) * Rq + 64 * bi;
        const double* sj = src + 64 * (k - 1) * Rq + 64 * bj;
        double v[16], u[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            v[q] = si[(w + 4 * q) * Rq + l];
            u[q] = sj[(w + 4 * q) * Rq + l];
        }
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            Ti[(w + 4 * q) * INV_LD + l] = v[q];
            Tj[(w + 4 * q) * INV_LD + l] = u[q];
        }
    }
    // this wave's columns of block (i, j) and its rows of the pivot block, less their products
    d4 y[4], pv[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) y[b] = pv[b] = (d4){0.0, 0.0, 0.0, 0.0};
    if (bj != k - 1) {   // the column of row k - 1's pivot counts as zero
        const double* s = src + 64 * bi * Rq + 64 * bj + 16 * w + c;
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) y[b][v] = s[(16 * b + g + 4 * v) * Rq];
    }
    if (pivot) {
        const double* s = src + 64 * k * Rq + 64 * k + c;
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) pv[b][v] = s[(16 * w + g + 4 * v) * Rq + 16 * b];
    }
    __syncthreads();
    if (panel) {
#pragma unroll 4
        for (int k0 = 0; k0 < 64; k0 += 4) {
            const double q = Tj[(k0 + g) * INV_LD + 16 * w + c];
#pragma unroll
            for (int b = 0; b < 4; ++b) y[b] = mfma_f64(-Ti[(k0 + g) * INV_LD + 16 * b + c], q, y[b]);
        }
    }
    double* d = dst + 64 * bi * Rq + 64 * bj;
    if (!pivot) {   // not panel: j = k < i, which is not needed and has left above
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) d[(16 * b + g + 4 * v) * Rq + 16 * w + c] = y[b][v];
        return;
    }
#pragma unroll 4
    for (int k0 = 0; k0 < 64; k0 += 4) {
        const double q = -Ti[(k0 + g) * INV_LD + 16 * w + c];
#pragma unroll
        for (int b = 0; b < 4; ++b) pv[b] = mfma_f64(q, Ti[(k0 + g) * INV_LD + 16 * b + c], pv[b]);
    }
    __syncthreads();   // every wave is done with the tiles
    double x[16];      // the wave's 16 rows, from the products' layout to one column per lane
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v) Ti[(16 * w + g + 4 * v) * INV_LD + 16 * b + c] = pv[b][v];
    lds_wave_order();
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = Ti[(16 * w + i) * INV_LD + l];
    inv_row(x, y, R - 64 * k < 64 ? R - 64 * k : 64, panel, Ti, Tj, Tj + INV_TILE, d, Rq, st.bad + k);
}

// Tile x of the upper 16 x 16 tiles of V^-1 = N^T N (R x R), row block r of N in buffer r & 1:
// the four waves split the rows from the tile's column block on (N is lower triangular).
__global__ __launch_bounds__(256) void k_inv_product(int R, int nb, const double* __restrict__ buf, double* __restrict__ Z,
                                                     double* __restrict__ stat, const DevCheck* __restrict__ chk) {
    if (chk->done) return;
    __shared__ d4 red[1][64];
    const int t = threadIdx.x, l = t & 63, c = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    int tb = 0, ta = blockIdx.x;
    while (ta > tb) { ta -= tb + 1; ++tb; }
    const int64_t Rq = 64 * (int64_t)nb;
    d4 acc[1] = {(d4){0.0, 0.0, 0.0, 0.0}};
    for (int r0 = 16 * tb + 16 * w; r0 < R; r0 += 64) {   // 16 rows: the ones past R are zero
        const double* __restrict__ Nr = buf + ((r0 >> 6) & 1) * Rq * Rq + (int64_t)r0 * Rq;
        double x[4], y[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            x[s] = Nr[(4 * s + g) * Rq + 16 * ta + c];
            y[s] = Nr[(4 * s + g) * Rq + 16 * tb + c];
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) acc[0] = mfma_f64(x[s], y[s], acc[0]);
    }
    if (!sum_waves<1>(acc, red, w, l)) return;
    double zsq = 0.0;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int r = 16 * ta + g + 4 * v, r2 = 16 * tb + c;
        if (r >= R || r2 >= R) continue;
        const double z = acc[0][v];
        Z[(int64_t)r * R + r2] = z;
        if (ta != tb) Z[(int64_t)r2 * R + r] = z;
        zsq = fma(ta == tb ? z : 2.0 * z, z, zsq);
    }
    zsq = wave_sum_dpp(zsq);
    if (l == 0) InvStat(stat, nb).zsq[blockIdx.x] = zsq;
}

// factor64_unpivoted's certificate from the statistics (see there): every pivot of the pivoted
// factorisation is >= lambda_min(V) >= 1 / ||V^-1||_F.  Up to WIDE_COND the product with V^-1 has the
// error of the pivoted path's substitution; it can have 40 times that at 2e9, 500 at 3e10.
// Unit columns stay below R / (2 tol).  Uniform over the workgroup.
constexpr double WIDE_COND = 1e8;
__device__ __forceinline__ bool wide_certified(const double* __restrict__ stat, int nb, int R, double tol) {
    __shared__ int ok;
    const int t = threadIdx.x;
    if (t < 64) {
        const InvStat st(const_cast<double*>(stat), nb);
        double vsq = 0.0, dmax = 0.0, zsq = 0.0, bad = 0.0;
        for (int x = t; x < nb * nb; x += 64) {   // the blocks above the diagonal count twice
            const int bi = x / nb, bj = x - bi * nb;
            if (bi > bj) continue;
            vsq = fma(bi < bj ? 2.0 : 1.0, st.vsq[x], vsq);
            dmax = fmax(dmax, st.dmax[x]);
        }
#pragma unroll 4
        for (int x = t; x < inv_tiles(R); x += 64) zsq += st.zsq[x];
        if (t < nb) bad = st.bad[t];
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
                 1.0 / zF > 2.0 * tol + 64.0 * R * 0x1p-52 * dmax && vF * zF < WIDE_COND;
    }
    __syncthreads();
    return ok != 0;
}

// Row solves X = M V^-1 with the certified inverse: wave w of block (x, y) takes the 16 x 16
// tile of rows 16 x .. and columns 16 (4 y + w) .. over k < R, 16 k-steps of both operands
// in flight.  Latency-bound (a few hundred rows): one tile per wave spreads a mode over
// In R / 1024 workgroups.
__global__ __launch_bounds__(256) void k_solve_inv(const double* __restrict__ M, int64_t In, int R,
                                                   const double* __restrict__ Vinv,
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
            b[s] = Vc[(int64_t)kc * R];
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
