// Leverage-score-sampled ALS (LevScoreSampled, krp_lev_score_sampled.jl:9-57): the
// device side of one projected least-squares step, and the leverage-score
// probabilities that drive the sampling (math_tools/probability.jl:3-10).  The
// sampling itself (StatsBase.sample with Weights in the reference) is host logic.
//
// One step for mode n with ns sampled index tuples of the other modes:
//   K_s(s, r) = prod_q A_q(samples(s, q), r)            pivot_hadamard, had_contract.jl:277-295
//   B(s, i)   = T(i at mode n, samples(s, :))           fused_flatten_sample, pivot_mapping.jl:90-118
//                                                       (stored transposed: ns x I_n)
//   normal:  X = ldiv_solve(K_s^T K_s, (B^T K_s)^T)^T   ProjectionAlgorithm.jl:56-58
//   else:    X = (qr(K_s, ColumnNorm()) \ B)^T          ProjectionAlgorithm.jl:60
// then row_norm into the plan's CPD.  The normal form reuses the plan's pivoted
// Cholesky / QR-fallback factorisation and row solves with V = K_s^T K_s; the QR
// form runs LAPACK dgelsy's steps (column-pivoted Householder QR, rank by
// incremental condition estimation at rcond = min(m, n) eps, RZ reduction of the
// trapezoid, minimum-norm solution) in one workgroup.
#include "dense_la.h"
#include "factor64.h"
#include "internal.h"

namespace itcpd {

namespace {

constexpr int SNT = 512;   // threads of the one-workgroup QR kernels
constexpr double EPS64 = 2.220446049250313e-16;

struct OtherModes {
    const double* A[ITCPD_MAX_ORDER];   // column-major factors of the other modes (ld = dim)
    int64_t dim[ITCPD_MAX_ORDER];
    int64_t tstride[ITCPD_MAX_ORDER];   // element stride of that mode in T
    int n;
};

// K_s, column-major ns x R.
__global__ __launch_bounds__(256) void k_pivot_hadamard(OtherModes om, const int* __restrict__ smp,
                                                        int64_t ns, int R, double* __restrict__ Ks,
                                                        const DevCheck* __restrict__ chk) {
    if (chk->done) return;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= ns * R) return;
    const int r = (int)(idx / ns);
    const int64_t s = idx - (int64_t)r * ns;
    double v = 1.0;
    for (int q = 0; q < om.n; ++q) v *= om.A[q][smp[s + ns * q] + om.dim[q] * r];
    Ks[idx] = v;
}

// B(s, i) = T(sampled fiber s, element i of mode n), column-major ns x In.
template <typename TT>
__global__ __launch_bounds__(256) void k_sample_fibers(const TT* __restrict__ T, OtherModes om,
                                                       int64_t mstride, int64_t In,
                                                       const int* __restrict__ smp, int64_t ns,
                                                       double* __restrict__ B,
                                                       const DevCheck* __restrict__ chk) {
    if (chk->done) return;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= ns * In) return;
    const int64_t i = idx / ns;
    const int64_t s = idx - i * ns;
    int64_t off = i * mstride;
    for (int q = 0; q < om.n; ++q) off += (int64_t)smp[s + ns * q] * om.tstride[q];
    B[idx] = (double)T[off];
}

// C(i, j) = sum_s A(s, i) B(s, j) (A: ns x m, B: ns x n, both ld ns; C: m x n), one
// wave per output element, lanes over s.
__global__ __launch_bounds__(256) void k_gemm_tn(const double* __restrict__ A, const double* __restrict__ B,
                                                 int64_t ns, int m, int n, double* __restrict__ C,
                                                 const DevCheck* __restrict__ chk) {
    if (chk->done) return;
    const int64_t w = ((int64_t)blockIdx.x * 256 + threadIdx.x) >> 6;
    const int lane = threadIdx.x & 63;
    if (w >= (int64_t)m * n) return;
    const int i = (int)(w % m), j = (int)(w / m);
    const double* a = A + ns * i;
    const double* b = B + ns * j;
    double s = 0.0;
    for (int64_t k = lane; k < ns; k += 64) s = fma(a[k], b[k], s);
    s = wave_sum(s);
    if (lane == 0) C[i + (int64_t)m * j] = s;
}

// A 16-sample chunk of a column over the four lanes g: value q is sample chunk_at(g, q), so
// that each of the two 16-byte loads takes 64 consecutive bytes of a column (columns a power of
// two apart share a cache set: what a load leaves of a line is evicted before the next one).
typedef double dvu2 __attribute__((ext_vector_type(2), aligned(8)));
__device__ __forceinline__ int chunk_at(int g, int q) { return 2 * g + (q & 1) + 8 * (q >> 1); }
__device__ __forceinline__ void ld_chunk(const double* __restrict__ p, int g, double (&x)[4]) {
    const dvu2 a = *reinterpret_cast<const dvu2*>(p + 2 * g), b = *reinterpret_cast<const dvu2*>(p + 8 + 2 * g);
    x[0] = a.x; x[1] = a.y; x[2] = b.x; x[3] = b.y;
}

// V = K^T K (n x n, upper tiles and their mirror) and M = B^T K (In x n, column-major) of the
// sampled step: one workgroup per 16 x 16 tile, eight waves over 16-sample chunks of column c
// of each operand.  ns = 1024, n = 32, In = 256: 10.3 us, bound by the latency of its two
// rounds of loads.
__global__ __launch_bounds__(512) void k_sampled_products(const double* __restrict__ K, const double* __restrict__ B,
                                                          int64_t ns, int n, int64_t In, double* __restrict__ V,
                                                          double* __restrict__ M, const DevCheck* __restrict__ chk) {
    if (chk->done) return;
    __shared__ double part[8][256];
    const int t = threadIdx.x, l = t & 63, c = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int nt = (n + 15) / 16, ngram = nt * (nt + 1) / 2;
    const bool gram = (int)blockIdx.x < ngram;
    int tb = 0;
    int64_t ta = blockIdx.x;
    if (gram) {
        while (ta > tb) { ta -= tb + 1; ++tb; }
    } else {
        tb = (int)((ta - ngram) % nt);
        ta = (ta - ngram) / nt;
    }
    // columns past the end read a valid one: their products are not stored
    const int64_t na = gram ? n : In, ca = 16 * ta + c < na ? 16 * ta + c : na - 1;
    const int cb = 16 * tb + c < n ? 16 * tb + c : n - 1;
    const double* __restrict__ pa = (gram ? K : B) + ns * ca;
    const double* __restrict__ pb = K + ns * cb;
    d4 acc = (d4){0.0, 0.0, 0.0, 0.0};
    int64_t s = 16 * w;
    for (; s + 400 <= ns; s += 512) {
        double a[4][4], b[4][4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            ld_chunk(pa + s + 128 * u, g, a[u]);
            ld_chunk(pb + s + 128 * u, g, b[u]);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q) acc = mfma_f64(a[u][q], b[u][q], acc);
    }
    for (; s < ns; s += 128) {
        double a[4], b[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int64_t sq = s + chunk_at(g, q);
            const bool ok = sq < ns;
            a[q] = pa[ok ? sq : ns - 1];
            b[q] = pb[ok ? sq : ns - 1];
            if (!ok) a[q] = b[q] = 0.0;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) acc = mfma_f64(a[q], b[q], acc);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) part[w][64 * v + l] = acc[v];
    __syncthreads();
    if (t >= 256) return;
    double sum = 0.0;
#pragma unroll
    for (int k = 0; k < 8; ++k) sum += part[k][t];
    const int64_t r = 16 * ta + ((t >> 4) & 3) + 4 * (t >> 6);
    const int r2 = 16 * tb + (t & 15);
    if (r >= na || r2 >= n) return;
    if (gram) {
        V[r * n + r2] = sum;
        V[(int64_t)r2 * n + r] = sum;
    } else {
        M[r + In * r2] = sum;
    }
}

// V^-1 of the normal equations.  info = {n, 0, n} when certified, else info[1] = 1.  Certified
// means ||V||_F ||V^-1||_F < 1e8, so cond(K) < 1e4, and V^-1 solves to eps cond(V), 1e-8 at
// worst: k_sampled_correct's one correction squares that, below the rounding of the QR solve
// it replaces (1e-13; both sides of the certificate measure 6e-14 .. 1.5e-13 on low-rank
// tensors), and K has full rank by the QR's test (n eps).
// gs: V as the only Gram of a mode 0, beside a mode 1.
__global__ __launch_bounds__(256) void k_sampled_inverse(GramSet gs, int n, double* __restrict__ Vinv,
                                                         int* __restrict__ info, const DevCheck* __restrict__ chk) {
    if (chk->done) return;
    __shared__ double S[FACTOR64_UNPIV];
    if (!factor64_unpivoted(gs, 1, n, 0.0, Vinv, info, S, 1e8) && threadIdx.x == 0) info[1] = 1;
}

// Corrected normal equations for 16 rows of X (one workgroup): X_0 = M V^-1, the residual
// E = B - K X_0^T of every sample in FP64, X = X_0 + (E^T K) V^-1.  The waves take
// 16-sample chunks; a chunk of E comes out of its product as the operand of the next one
// (sample chunk_at(g, v), row c), so it never leaves the registers.  Bound by the matrix cores of
// the In / 16 CUs it runs on: ns = 1024, n = 32, In = 256, 21.8 us (31.7 with
// 8-byte loads of the chunks).  The column-pivoted QR, its application and rank test took 610
// us there (74 launches); they still solve what k_sampled_inverse does not certify.
// four waves for RT = 64, whose two chunks in flight need more than 256 registers
constexpr int correct_threads(int rt) { return rt == 64 ? 256 : 512; }
template <int RT>
__global__ __launch_bounds__(correct_threads(RT)) void k_sampled_correct(const double* __restrict__ K, const double* __restrict__ B,
                                                         int64_t ns, int n, int64_t In, const double* __restrict__ M,
                                                         const double* __restrict__ Vinv, const int* __restrict__ info,
                                                         double* __restrict__ X, const DevCheck* __restrict__ chk) {
    constexpr int NT = RT / 16, KS = RT / 4, LD = RT + 2, NTHR = correct_threads(RT), NW = NTHR / 64;
    if (chk->done || info[1] != 0) return;
    __shared__ double X0[16 * LD];
    __shared__ double part[NW * NT * 256];
    const int t = threadIdx.x, l = t & 63, c = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int64_t i0 = 16 * (int64_t)blockIdx.x, ic = i0 + c < In ? i0 + c : In - 1;
    // tile tb of (16 x RT operand rows `row(k)`) V^-1; zero beyond n
    auto times_vinv = [&](auto row, int tb) {
        d4 acc = (d4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int k = 4 * ks + g, r = 16 * tb + c;
            const bool ok = k < n && r < n;
            const double b = Vinv[ok ? k * n + r : 0];
            acc = mfma_f64(k < n ? row(k) : 0.0, ok ? b : 0.0, acc);
        }
        return acc;
    };
    d4 x0 = (d4){0.0, 0.0, 0.0, 0.0};
    if (w < NT) {
        x0 = times_vinv([&](int k) { return M[ic + In * k]; }, w);
#pragma unroll
        for (int v = 0; v < 4; ++v) X0[(g + 4 * v) * LD + 16 * w + c] = x0[v];
    }
    __syncthreads();
    double xb[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) xb[ks] = X0[c * LD + 4 * ks + g];
    d4 acc[NT];
#pragma unroll
    for (int tb = 0; tb < NT; ++tb) acc[tb] = (d4){0.0, 0.0, 0.0, 0.0};
    const double* __restrict__ pB = B + ns * ic;
    const double* __restrict__ pa[KS];   // columns past n: valid, met by zeros of xb
    const double* __restrict__ pk[NT];   // columns past n: valid, not stored
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) pa[ks] = K + ns * (4 * ks + g < n ? 4 * ks + g : n - 1);
#pragma unroll
    for (int tb = 0; tb < NT; ++tb) pk[tb] = K + ns * (16 * tb + c < n ? 16 * tb + c : n - 1);
    struct Chunk {
        double ka[KS], kb[NT][4], b[4];
    };
    const int pc = chunk_at(c & 3, c >> 2);   // row g + 4v of the product is sample chunk_at(g, v)
    auto load = [&](int64_t s0, Chunk& h) {
        if (s0 + 16 <= ns) {
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) h.ka[ks] = pa[ks][s0 + pc];
            ld_chunk(pB + s0, g, h.b);
#pragma unroll
            for (int tb = 0; tb < NT; ++tb) ld_chunk(pk[tb] + s0, g, h.kb[tb]);
        } else {   // samples past the end: the last one
            const int64_t sa = s0 + pc < ns ? s0 + pc : ns - 1;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) h.ka[ks] = pa[ks][sa];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int64_t s = s0 + chunk_at(g, v) < ns ? s0 + chunk_at(g, v) : ns - 1;
                h.b[v] = pB[s];
#pragma unroll
                for (int tb = 0; tb < NT; ++tb) h.kb[tb][v] = pk[tb][s];
            }
        }
    };
    auto step = [&](int64_t s0, const Chunk& h) {
        d4 pr = (d4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) pr = mfma_f64(h.ka[ks], xb[ks], pr);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const double e = s0 + chunk_at(g, v) < ns ? h.b[v] - pr[v] : 0.0;
#pragma unroll
            for (int tb = 0; tb < NT; ++tb) acc[tb] = mfma_f64(e, h.kb[tb][v], acc[tb]);
        }
    };
    Chunk h0, h1;   // the next chunk's loads in flight behind the current one's products
    int64_t s0 = 16 * (int64_t)w;
    if (s0 < ns) load(s0, h0);
    for (; s0 < ns; s0 += 32 * NW) {
        const int64_t s1 = s0 + 16 * NW, s2 = s0 + 32 * NW;
        if (s1 < ns) load(s1, h1);
        step(s0, h0);
        if (s1 >= ns) break;
        if (s2 < ns) load(s2, h0);
        step(s1, h1);
    }
#pragma unroll
    for (int tb = 0; tb < NT; ++tb)
#pragma unroll
        for (int v = 0; v < 4; ++v) part[(w * NT + tb) * 256 + 64 * v + l] = acc[tb][v];
    __syncthreads();
    // the waves' sums, as the next product's rows: X0 is read no more
    for (int x = t; x < NT * 256; x += NTHR) {
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < NW; ++k) s += part[k * NT * 256 + x];
        X0[(((x >> 4) & 3) + 4 * ((x >> 6) & 3)) * LD + 16 * (x >> 8) + (x & 15)] = s;
    }
    __syncthreads();
    if (w < NT) {
        const d4 dx = times_vinv([&](int k) { return X0[c * LD + k]; }, w);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int64_t i = i0 + g + 4 * v;
            const int r = 16 * w + c;
            if (i < In && r < n) X[i + In * r] = x0[v] + dx[v];
        }
    }
}

// Householder reflector of x = (x[0], x[1 .. len)) (xLARFG): x[0] <- beta,
// x[1 .. len) <- v (v[0] = 1 implicit); returns tau (0 when the tail is zero).
template <int NT>
__device__ double house(double* x, int len, double* redv) {
    const int t = threadIdx.x;
    double xs = 0.0;
    for (int k = 1 + t; k < len; k += NT) xs += x[k] * x[k];
    const double xnorm2 = block_sum<NT>(xs, redv);
    const double alpha = x[0];
    double tau = 0.0, beta = alpha, scal = 0.0;
    if (xnorm2 > 0.0) {
        beta = -copysign(hypot(alpha, sqrt(xnorm2)), alpha);
        tau = (beta - alpha) / beta;
        scal = 1.0 / (alpha - beta);
    }
    __syncthreads();
    if (xnorm2 > 0.0)
        for (int k = 1 + t; k < len; k += NT) x[k] *= scal;
    if (t == 0) x[0] = beta;
    __syncthreads();
    return tau;
}

// C <- (I - tau u u^T) C for the ncols columns of C (rows 0 .. len-1, ld ldc), with
// u = (1, v[1 .. len)); one wave per column.
template <int NT>
__device__ void house_left(const double* v, int len, double tau, double* C, int64_t ldc, int64_t ncols) {
    if (tau != 0.0) {
        const int t = threadIdx.x, ln = t & 63;
        for (int64_t j = t >> 6; j < ncols; j += NT / 64) {
            double* c = C + ldc * j;
            double s = 0.0;
            for (int k = ln; k < len; k += 64) s += (k == 0 ? 1.0 : v[k]) * c[k];
            const double f = tau * wave_sum(s);
            for (int k = ln; k < len; k += 64) c[k] -= f * (k == 0 ? 1.0 : v[k]);
        }
    }
    __syncthreads();
}

// Householder QR of W (m x n, ld) with column pivoting (xGEQP3 / xLAQP2: largest
// remaining partial column norm first, norms downdated and recomputed when the
// downdate loses accuracy) or without.  tau[min(m, n)], jpvt[n].
template <int NT>
__device__ void geqp3(double* W, int m, int n, int64_t ld, bool pivot, double* tau, int* jpvt,
                      double* vn1, double* vn2, double* redv, int* redi) {
    const int t = threadIdx.x;
    for (int j = t; j < n; j += NT) jpvt[j] = j;
    if (pivot) {
        for (int j = t >> 6; j < n; j += NT / 64) {
            const int ln = t & 63;
            double ss = 0.0;
            for (int k = ln; k < m; k += 64) ss += W[k + ld * j] * W[k + ld * j];
            ss = wave_sum(ss);
            if (ln == 0) { vn1[j] = sqrt(ss); vn2[j] = sqrt(ss); }
        }
    }
    __syncthreads();
    const double tol3z = 1.0536712127723509e-08;   // sqrt(eps)
    const int kmax = m < n ? m : n;
    for (int i = 0; i < kmax; ++i) {
        if (pivot) {
            const int p = block_argmax<NT>(i, n, [&](int j) { return fabs(vn1[j]); }, redv, redi);
            const int pvt = (p < n) ? p : i;
            if (pvt != i) {
                for (int k = t; k < m; k += NT) {
                    const double a = W[k + ld * pvt];
                    W[k + ld * pvt] = W[k + ld * i];
                    W[k + ld * i] = a;
                }
                if (t == 0) {
                    const int q = jpvt[pvt]; jpvt[pvt] = jpvt[i]; jpvt[i] = q;
                    vn1[pvt] = vn1[i];
                    vn2[pvt] = vn2[i];
                }
            }
            __syncthreads();
        }
        double* col = W + i + ld * i;
        const double ti = house<NT>(col, m - i, redv);
        if (t == 0) tau[i] = ti;
        if (i + 1 < n) house_left<NT>(col, m - i, ti, col + ld, ld, n - i - 1);
        if (pivot) {
            for (int j = i + 1 + (t >> 6); j < n; j += NT / 64) {
                const int ln = t & 63;
                const double v1 = vn1[j];
                if (v1 != 0.0) {
                    double temp = fabs(W[i + ld * j]) / v1;
                    temp = fmax(1.0 - temp * temp, 0.0);
                    const double q = v1 / vn2[j];
                    if (temp * q * q <= tol3z) {
                        double ss = 0.0;
                        for (int k = i + 1 + ln; k < m; k += 64) ss += W[k + ld * j] * W[k + ld * j];
                        ss = wave_sum(ss);
                        if (ln == 0) { vn1[j] = sqrt(ss); vn2[j] = vn1[j]; }
                    } else if (ln == 0) {
                        vn1[j] = v1 * sqrt(temp);
                    }
                }
            }
            __syncthreads();
        }
    }
}

// qr(K, ColumnNorm()) \ B as LAPACK dgelsy, factor part (one workgroup): K (m x n) in
// W is overwritten by the column-pivoted QR (tau, jpvt), the numerical rank goes to
// info[0], and for rank < n the rk x n trapezoid is reduced to [T11 0] Z (ztau).  With
// `factored` the column-pivoted QR is already in W / tau / jpvt (the grid-wide steps).
template <int NT>
__global__ __launch_bounds__(NT) void k_lsq_qr_factor(double* __restrict__ W, int m, int n,
                                                      double* __restrict__ tau, double* __restrict__ ztau,
                                                      double* __restrict__ vwork, int* __restrict__ jpvt,
                                                      int* __restrict__ info, int factored,
                                                      const DevCheck* __restrict__ chk) {
    if (chk->done) return;
    __shared__ double redv[NT];
    __shared__ int redi[NT];
    __shared__ int s_rank;
    const int t = threadIdx.x;
    const int64_t ld = m;
    const int kq = m < n ? m : n;
    double* vn1 = vwork;
    double* vn2 = vwork + n;
    if (!factored) geqp3<NT>(W, m, n, ld, true, tau, jpvt, vn1, vn2, redv, redi);

    // numerical rank: incremental condition estimation on R, rcond = min(m, n) eps.  For
    // kq <= 64 wave 0 runs it on an LDS copy of R's triangle, lane k holding entry k of
    // both estimate vectors (the dot products as wave sums); above that thread 0 runs it
    // in column order on global memory.
    __shared__ double r_lds[64 * 64];
    const bool small = kq <= 64;
    if (small) {
        for (int x = t; x < kq * kq; x += NT) {
            const int a = x % kq, b = x / kq;
            r_lds[x] = a <= b ? W[a + ld * b] : 0.0;
        }
    }
    __syncthreads();
    const double rcond = (double)kq * EPS64;
    if (small && t < 64) {
        const int lane = t;
        double xm = lane == 0 ? 1.0 : 0.0, xM = xm;
        double smax = fabs(r_lds[0]);
        double smin = smax;
        int rk = 0;
        if (kq > 0 && smax != 0.0) {
            rk = 1;
            while (rk < kq) {
                const int i = rk;
                const double rki = lane < i ? r_lds[lane + kq * i] : 0.0;
                const double amin = wave_sum(xm * rki), amax = wave_sum(xM * rki);
                const double gamma = r_lds[i + kq * i];
                double sminpr, s1, c1, smaxpr, s2, c2;
                laic1(2, amin, smin, gamma, &sminpr, &s1, &c1);
                laic1(1, amax, smax, gamma, &smaxpr, &s2, &c2);
                if (smaxpr * rcond > sminpr) break;
                if (lane < i) {
                    xm *= s1;
                    xM *= s2;
                } else if (lane == i) {
                    xm = c1;
                    xM = c2;
                }
                smin = sminpr;
                smax = smaxpr;
                ++rk;
            }
        }
        if (lane == 0) {
            s_rank = rk;
            info[0] = rk;
        }
    } else if (!small && t == 0) {
        double* xmin = vwork;
        double* xmax = vwork + n;
        double smax = fabs(W[0]);
        double smin = smax;
        int rk = 0;
        if (kq > 0 && smax != 0.0) {
            rk = 1;
            xmin[0] = 1.0;
            xmax[0] = 1.0;
            while (rk < kq) {
                const int i = rk;
                double amin = 0.0, amax = 0.0;
                for (int k = 0; k < i; ++k) {
                    amin += xmin[k] * W[k + ld * i];
                    amax += xmax[k] * W[k + ld * i];
                }
                const double gamma = W[i + ld * i];
                double sminpr, s1, c1, smaxpr, s2, c2;
                laic1(2, amin, smin, gamma, &sminpr, &s1, &c1);
                laic1(1, amax, smax, gamma, &smaxpr, &s2, &c2);
                if (smaxpr * rcond > sminpr) break;
                for (int k = 0; k < i; ++k) { xmin[k] *= s1; xmax[k] *= s2; }
                xmin[i] = c1;
                xmax[i] = c2;
                smin = sminpr;
                smax = smaxpr;
                ++rk;
            }
        }
        s_rank = rk;
        info[0] = rk;
    }
    __syncthreads();
    const int rk = s_rank;

    // RZ factorisation of the rk x n trapezoid [R11 R12] (xTZRZF / xLATRZ)
    if (rk > 0 && rk < n) {
        const int L = n - rk;
        for (int i = rk - 1; i >= 0; --i) {
            double xs = 0.0;
            for (int q = t; q < L; q += NT) xs += W[i + ld * (rk + q)] * W[i + ld * (rk + q)];
            const double xnorm2 = block_sum<NT>(xs, redv);
            const double alpha = W[i + ld * i];
            double tz = 0.0, beta = alpha, scal = 0.0;
            if (xnorm2 > 0.0) {
                beta = -copysign(hypot(alpha, sqrt(xnorm2)), alpha);
                tz = (beta - alpha) / beta;
                scal = 1.0 / (alpha - beta);
            }
            __syncthreads();
            if (xnorm2 > 0.0)
                for (int q = t; q < L; q += NT) W[i + ld * (rk + q)] *= scal;
            if (t == 0) { W[i + ld * i] = beta; ztau[i] = tz; }
            __syncthreads();
            if (tz != 0.0) {
                for (int k = t >> 6; k < i; k += NT / 64) {
                    const int ln = t & 63;
                    double sdot = (ln == 0) ? W[k + ld * i] : 0.0;
                    for (int q = ln; q < L; q += 64) sdot += W[k + ld * (rk + q)] * W[i + ld * (rk + q)];
                    const double f = tz * wave_sum(sdot);
                    if (ln == 0) W[k + ld * i] -= f;
                    for (int q = ln; q < L; q += 64) W[k + ld * (rk + q)] -= f * W[i + ld * (rk + q)];
                }
            }
            __syncthreads();
        }
    }
}

// dgelsy's solution for one right-hand side per wave (column c of B, m x nrhs, ld m):
// b <- Q^T b, y = T11^-1 b(0:rk), zero beyond rk, y <- Z^T y (rank < n), and
// X(c, jpvt(k)) = y(k) (X: nrhs x n, ld nrhs).  Lane l owns the rows r = l (mod 64)
// of b, so no lane reads another lane's store to global memory; y (n entries per
// wave) lives in LDS, and every hand-over between lanes waits for the LDS writes.
__global__ __launch_bounds__(256) void k_lsq_qr_apply(const double* __restrict__ W, int m, int n,
                                                      double* __restrict__ B, int64_t nrhs,
                                                      double* __restrict__ X,
                                                      const double* __restrict__ tau,
                                                      const double* __restrict__ ztau,
                                                      const int* __restrict__ jpvt, const int* __restrict__ info,
                                                      const DevCheck* __restrict__ chk) {
    if (chk->done) return;
    extern __shared__ double ylds[];
    const int wave = threadIdx.x >> 6, ln = threadIdx.x & 63;
    const int64_t c = (int64_t)blockIdx.x * 4 + wave;
    if (c >= nrhs) return;
    const int64_t ld = m;
    const int kq = m < n ? m : n;
    const int rk = info[0];
    double* b = B + ld * c;
    for (int i = 0; i < kq; ++i) {
        const double ti = tau[i];
        if (ti == 0.0) continue;
        double s = 0.0;
        for (int r = ln; r < m; r += 64)
            if (r >= i) s += (r == i ? 1.0 : W[r + ld * i]) * b[r];
        const double f = ti * wave_sum(s);
        for (int r = ln; r < m; r += 64)
            if (r >= i) b[r] -= f * (r == i ? 1.0 : W[r + ld * i]);
    }
    double* y = ylds + (size_t)wave * n;
    for (int k = ln; k < n; k += 64) y[k] = (k < rk) ? b[k] : 0.0;
    __threadfence_block();
    for (int j = rk - 1; j >= 0; --j) {
        double s = 0.0;
        for (int k = j + 1 + ln; k < rk; k += 64) s += W[j + ld * k] * y[k];
        s = wave_sum(s);
        if (ln == 0) y[j] = (y[j] - s) / W[j + ld * j];
        __threadfence_block();
    }
    if (rk < n) {
        for (int tq = 0; tq < rk; ++tq) {
            const double tz = ztau[tq];
            if (tz == 0.0) continue;
            double part = 0.0;
            for (int k = rk + ln; k < n; k += 64) part += W[tq + ld * k] * y[k];
            const double f = tz * (wave_sum(part) + y[tq]);
            __threadfence_block();
            if (ln == 0) y[tq] -= f;
            for (int k = rk + ln; k < n; k += 64) y[k] -= f * W[tq + ld * k];
            __threadfence_block();
        }
    }
    for (int k = ln; k < n; k += 64) X[c + nrhs * jpvt[k]] = y[k];
}

// The same with the right-hand side in registers for m <= 64 NQ (lane l holds rows
// l + 64 q): Q^T b touches global memory only for the reflectors, which every wave
// reads alike.  The arithmetic and its order are k_lsq_qr_apply's.
template <int NQ>
__global__ __launch_bounds__(256) void k_lsq_qr_apply_reg(const double* __restrict__ W, int m, int n,
                                                          const double* __restrict__ B, int64_t nrhs,
                                                          double* __restrict__ X,
                                                          const double* __restrict__ tau,
                                                          const double* __restrict__ ztau,
                                                          const int* __restrict__ jpvt, const int* __restrict__ info,
                                                          const DevCheck* __restrict__ chk) {
    if (chk->done) return;
    extern __shared__ double ylds[];
    const int wave = threadIdx.x >> 6, ln = threadIdx.x & 63;
    const int64_t c = (int64_t)blockIdx.x * 4 + wave;
    if (c >= nrhs) return;
    const int64_t ld = m;
    const int kq = m < n ? m : n;
    const int rk = info[0];
    const double* b = B + ld * c;
    double bv[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int r = ln + 64 * q;
        bv[q] = r < m ? b[r] : 0.0;
    }
    for (int i = 0; i < kq; ++i) {
        const double ti = tau[i];
        if (ti == 0.0) continue;
        const double* v = W + ld * i;
        double vr[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int r = ln + 64 * q;
            vr[q] = (r < m && r > i) ? v[r] : (r == i ? 1.0 : 0.0);
        }
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int r = ln + 64 * q;
            if (r < m && r >= i) s += vr[q] * bv[q];
        }
        const double f = ti * wave_sum(s);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int r = ln + 64 * q;
            if (r < m && r >= i) bv[q] -= f * vr[q];
        }
    }
    double* y = ylds + (size_t)wave * n;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int k = ln + 64 * q;
        if (k < n) y[k] = (k < rk) ? bv[q] : 0.0;
    }
    for (int k = 64 * NQ + ln; k < n; k += 64) y[k] = 0.0;
    __threadfence_block();
    for (int j = rk - 1; j >= 0; --j) {
        double s = 0.0;
        for (int k = j + 1 + ln; k < rk; k += 64) s += W[j + ld * k] * y[k];
        s = wave_sum(s);
        if (ln == 0) y[j] = (y[j] - s) / W[j + ld * j];
        __threadfence_block();
    }
    if (rk < n) {
        for (int tq = 0; tq < rk; ++tq) {
            const double tz = ztau[tq];
            if (tz == 0.0) continue;
            double part = 0.0;
            for (int k = rk + ln; k < n; k += 64) part += W[tq + ld * k] * y[k];
            const double f = tz * (wave_sum(part) + y[tq]);
            __threadfence_block();
            if (ln == 0) y[tq] -= f;
            for (int k = rk + ln; k < n; k += 64) y[k] -= f * W[tq + ld * k];
            __threadfence_block();
        }
    }
    for (int k = ln; k < n; k += 64) X[c + nrhs * jpvt[k]] = y[k];
}

// compute_leverage_score_probabilitiy (probability.jl:3-10): Q = the thin Q of the
// unpivoted Householder QR of A (m x n), p(i) = sum_j Q(i, j)^2 / min(m, n).  W is
// an m x n scratch (ld m); Q is formed in place as LAPACK xORG2R does.  Runs only
// where the Gram form below cannot (need != 0, or need null).
template <int NT>
__global__ __launch_bounds__(NT) void k_lev_scores(const double* __restrict__ A, int m, int n,
                                                   double* __restrict__ W, double* __restrict__ tau,
                                                   double* __restrict__ vwork, int* __restrict__ jpvt,
                                                   double* __restrict__ probs, const int* __restrict__ need,
                                                   const DevCheck* __restrict__ chk) {
    if (chk->done || (need && *need == 0)) return;
    __shared__ double redv[NT];
    __shared__ int redi[NT];
    const int t = threadIdx.x;
    const int64_t ld = m;
    for (int64_t x = t; x < (int64_t)m * n; x += NT) W[x] = A[x];
    __syncthreads();
    geqp3<NT>(W, m, n, ld, false, tau, jpvt, vwork, vwork + n, redv, redi);
    const int kq = m < n ? m : n;
    for (int i = kq - 1; i >= 0; --i) {
        if (i < kq - 1) house_left<NT>(W + i + ld * i, m - i, tau[i], W + i + ld * (i + 1), ld, kq - 1 - i);
        const double ti = tau[i];
        for (int k = i + 1 + t; k < m; k += NT) W[k + ld * i] *= -ti;
        for (int k = t; k < i; k += NT) W[k + ld * i] = 0.0;
        if (t == 0) W[i + ld * i] = 1.0 - ti;
        __syncthreads();
    }
    for (int i = t; i < m; i += NT) {
        double s = 0.0;
        for (int j = 0; j < kq; ++j) s += W[i + ld * j] * W[i + ld * j];
        probs[i] = s / (double)kq;
    }
}

// Leverage scores of a full-column-rank A (m > n) through its Gram G = A^T A:
// sum_j Q(i, j)^2 = a_i^T G^-1 a_i, the diagonal of the projector onto range(A).
// k_gram_chol_inv (one workgroup): G = U^T U (unpivoted Cholesky) and G^-1 =
// U^-1 U^-T into Gi; need = 1 when a pivot falls below n eps max(diag G) (the
// Householder kernel then runs instead).  G (n x n) is overwritten.
template <int NT>
__global__ __launch_bounds__(NT) void k_gram_chol_inv(double* __restrict__ G, int n, double* __restrict__ Ui,
                                                      double* __restrict__ Gi, int* __restrict__ need,
                                                      const DevCheck* __restrict__ chk) {
    if (chk->done) return;
    __shared__ double redv[NT];
    __shared__ int s_bad;
    const int t = threadIdx.x;
    double dmax = 0.0;
    for (int j = t; j < n; j += NT) dmax = fmax(dmax, G[j + (int64_t)n * j]);
    redv[t] = dmax;
    if (t == 0) s_bad = 0;
    __syncthreads();
    for (int o = NT / 2; o > 0; o >>= 1) {
        if (t < o) redv[t] = fmax(redv[t], redv[t + o]);
        __syncthreads();
    }
    const double thr = (double)n * EPS64 * redv[0];
    // right-looking: row j of U in the upper triangle of G (column-major, G(j, k) at j + n k)
    for (int j = 0; j < n; ++j) {
        const double d = G[j + (int64_t)n * j];
        if (!(d > thr)) {
            if (t == 0) s_bad = 1;
            __syncthreads();
            break;
        }
        const double ujj = sqrt(d), inv = 1.0 / ujj;
        __syncthreads();
        for (int k = j + 1 + t; k < n; k += NT) G[j + (int64_t)n * k] *= inv;
        if (t == 0) G[j + (int64_t)n * j] = ujj;
        __syncthreads();
        const int r = n - j - 1;
        for (int x = t; x < r * r; x += NT) {
            const int a = j + 1 + x % r, b = j + 1 + x / r;
            if (a <= b) G[a + (int64_t)n * b] -= G[j + (int64_t)n * a] * G[j + (int64_t)n * b];
        }
        __syncthreads();
    }
    if (s_bad) {
        if (t == 0) *need = 1;
        return;
    }
    // Ui = U^-1 (upper), one column per thread: U x = e_c
    for (int cidx = t; cidx < n; cidx += NT) {
        for (int i = n - 1; i >= 0; --i) {
            double v = (i == cidx) ? 1.0 : 0.0;
            if (i <= cidx) {
                for (int k = i + 1; k <= cidx; ++k) v -= G[i + (int64_t)n * k] * Ui[k + (int64_t)n * cidx];
                v /= G[i + (int64_t)n * i];
            }
            Ui[i + (int64_t)n * cidx] = (i <= cidx) ? v : 0.0;
        }
    }
    __syncthreads();
    // Gi = Ui Ui^T
    for (int x = t; x < n * n; x += NT) {
        const int a = x % n, b = x / n;
        const int k0 = a > b ? a : b;
        double v = 0.0;
        for (int k = k0; k < n; ++k) v += Ui[a + (int64_t)n * k] * Ui[b + (int64_t)n * k];
        Gi[x] = v;
    }
    if (t == 0) *need = 0;
}

// p(i) = a_i^T Gi a_i / n, one thread per row (skipped when the Householder kernel runs)
__global__ __launch_bounds__(256) void k_lev_rows(const double* __restrict__ A, int m, int n,
                                                  const double* __restrict__ Gi, const int* __restrict__ need,
                                                  double* __restrict__ probs, const DevCheck* __restrict__ chk) {
    if (chk->done || *need != 0) return;
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= m) return;
    double s = 0.0;
    for (int j = 0; j < n; ++j) {
        const double aj = A[i + (int64_t)m * j];
        double u = 0.0;
        for (int k = 0; k < n; ++k) u += Gi[k + (int64_t)n * j] * A[i + (int64_t)m * k];
        s += aj * u;
    }
    probs[i] = s / (double)n;
}

// The same for n <= 64: k_gram_chol64 factors G = U^T U with the Schur complement in
// registers and writes U; k_lev_rows64 solves U^T y = a_i and p(i) = ||y||^2 / n, the
// same a_i^T G^-1 a_i / n without forming G^-1.
constexpr int LEV64_LD = 65;
// One workgroup of 256 threads, the Schur complement in registers: thread (w, l)
// holds rows 16w..16w+15 of column l.  Step j: the wave owning row j hands it over
// through LDS (one barrier), u_l = S(j, l) / sqrt(S(j, j)) and every thread applies
// the rank-1 update to its 16 entries; the pivot test is k_gram_chol_inv's (stop when
// S(j, j) <= n eps max(diag G)).  Writes U (column-major, zero below the diagonal).
__global__ __launch_bounds__(256) void k_gram_chol64(const double* __restrict__ G, int n, double* __restrict__ U,
                                                     int* __restrict__ need, const DevCheck* __restrict__ chk) {
    if (chk->done) return;
    __shared__ double rowb[2][64];
    __shared__ double redv[256];
    const int t = threadIdx.x, l = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    d16 sr;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int m = 16 * w + i;
        sr[i] = (m < n && l < n) ? G[m + (int64_t)n * l] : 0.0;
    }
    double dmax = 0.0;
    for (int j = t; j < n; j += 256) dmax = fmax(dmax, G[j + (int64_t)n * j]);
    redv[t] = dmax;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (t < o) redv[t] = fmax(redv[t], redv[t + o]);
        __syncthreads();
    }
    const double thr = (double)n * EPS64 * redv[0];
    bool bad = false;
    for (int j = 0; j < n; ++j) {
        double* rb = rowb[j & 1];
        if (w == (j >> 4)) rb[l] = sr[j & 15];
        __syncthreads();
        const double d = rb[j];
        if (!(d > thr)) {
            bad = true;
            break;
        }
        // 1/sqrt(d) from the hardware estimate (relative error < 2^-22) and two Newton steps
        const double dc = fmax(d, 0x1p-1020), h = 0.5 * dc;
        double inv = __builtin_amdgcn_rsq(dc);
        inv = fma(inv, fma(-h * inv, inv, 0.5), inv);
        inv = fma(inv, fma(-h * inv, inv, 0.5), inv);
        const double ujj = dc * inv;
        const double ul = rb[l] * inv;
        if (w == 0 && l < n) U[j + (int64_t)n * l] = l > j ? ul : (l == j ? ujj : 0.0);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int m = 16 * w + i;
            const double um = rb[m] * inv;
            if (m > j && l > j) sr[i] -= um * ul;
        }
    }
    // row j of U (with its zeros left of the diagonal) was written at step j
    if (t == 0) *need = bad ? 1 : 0;
}

// p(i) = ||U^-T a_i||^2 / n by blocks of 16 on MFMA, transposed: Y_j = D_j^T (A_j^T - sum_{k<j}
// U_kj^T Y_k), D_j the inverse of the diagonal block (wave j, lane c: column c by substitution).
// A wave takes 16 rows of A; its finished block of Y is the next ones' operand as it stands.
// 256 rows, n = 32: 6.4 us (35.3 with a lane per row, whose chain of n^2 / 2 steps was code
// that ran once).
__global__ __launch_bounds__(256) void k_lev_rows64(const double* __restrict__ A, int m, int n,
                                                   const double* __restrict__ U, const int* __restrict__ need,
                                                   double* __restrict__ probs, const DevCheck* __restrict__ chk) {
    if (chk->done || *need != 0) return;
    __shared__ double S[64 * LEV64_LD];       // U by rows, the identity beyond n
    __shared__ double Di[4][16 * 17];
    const int t = threadIdx.x, l = t & 63, c = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int nt = (n + 15) / 16, np = 16 * nt;
    const int i = (int)blockIdx.x * 64 + 16 * w + c, ic = i < m ? i : m - 1;
    d4 y[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int k = 16 * j + g + 4 * v;
            const double a = A[ic + (int64_t)m * (k < n ? k : 0)];
            y[j][v] = k < n ? a : 0.0;
        }
    for (int x = t; x < np * np; x += 256) {
        const int r = x % np, q = x / np;
        S[r * LEV64_LD + q] = r < n && q < n ? U[r + n * q] : (r == q ? 1.0 : 0.0);
    }
    __syncthreads();
    if (w < nt && l < 16) {
        double xv[16];
        const double* D = S + 16 * w * (LEV64_LD + 1);
#pragma unroll
        for (int r = 15; r >= 0; --r) {
            double acc = r == l ? 1.0 : 0.0;
#pragma unroll
            for (int k = r + 1; k < 16; ++k) acc -= D[r * LEV64_LD + k] * xv[k];
            xv[r] = acc / D[r * LEV64_LD + r];
            Di[w][r * 17 + l] = xv[r];
        }
    }
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (j >= nt) break;
#pragma unroll
        for (int k = 0; k < j; ++k)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                y[j] = mfma_f64(-S[(16 * k + g + 4 * v) * LEV64_LD + 16 * j + c], y[k][v], y[j]);
        d4 o = (d4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int v = 0; v < 4; ++v) o = mfma_f64(Di[j][(g + 4 * v) * 17 + c], y[j][v], o);
        y[j] = o;
#pragma unroll
        for (int v = 0; v < 4; ++v) s = fma(o[v], o[v], s);
    }
    s += __shfl_xor(s, 16);
    s += __shfl_xor(s, 32);
    if (g == 0 && i < m) probs[i] = s / (double)n;
}

// p(i) = 1 / m for m <= n (Q is square and orthogonal: every row has norm 1)
__global__ __launch_bounds__(256) void k_fill_value(double* __restrict__ out, int m, double v,
                                                    const DevCheck* __restrict__ chk) {
    if (chk->done) return;
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < m) out[i] = v;
}

// ------------------------------------------------------------ pivot projections
// QRPivProjected / SEQRCSPivProjected (qr_lev_score_sampled.jl): the pivots come
// from column-pivoted QRs of the mode-n unfolding T_(n) (or of a column subset of it,
// or of its sparse sketch T_(n) Omega^T), computed once before the sweeps.  Column c
// of T_(n) enumerates the other modes with the first one fastest (Julia's reshape of
// array(T, (i, others...))).

// W(i, q) = T_(n)(i, cols[q]) (cols null: column q), I_n x ncols column-major.
template <typename TT>
__global__ __launch_bounds__(256) void k_unfold_cols(const TT* __restrict__ T, OtherModes om,
                                                     int64_t mstride, int64_t In,
                                                     const int64_t* __restrict__ cols, int64_t ncols,
                                                     double* __restrict__ W) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= In * ncols) return;
    const int64_t q = idx / In, i = idx - q * In;
    int64_t c = cols ? cols[q] : q;
    int64_t off = i * mstride;
    for (int k = 0; k < om.n; ++k) {
        off += (c % om.dim[k]) * om.tstride[k];
        c /= om.dim[k];
    }
    W[idx] = (double)T[off];
}

// A_sk(i, j) = sum over the nonzeros e of row j of Omega (increasing column) of
// vals[e] T_(n)(i, colidx[e])   (sketched_matricization, pivot_mapping.jl:103-139),
// I_n x l column-major.  rowptr / colidx / vals: Omega by rows.
template <typename TT>
__global__ __launch_bounds__(256) void k_sketch(const TT* __restrict__ T, OtherModes om, int64_t mstride,
                                                int64_t In, const int64_t* __restrict__ rowptr,
                                                const int64_t* __restrict__ colidx,
                                                const double* __restrict__ vals, int64_t l,
                                                double* __restrict__ W) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= In * l) return;
    const int64_t j = idx / In, i = idx - j * In;
    double acc = 0.0;
    for (int64_t e = rowptr[j]; e < rowptr[j + 1]; ++e) {
        int64_t c = colidx[e];
        int64_t off = i * mstride;
        for (int k = 0; k < om.n; ++k) {
            off += (c % om.dim[k]) * om.tstride[k];
            c /= om.dim[k];
        }
        acc += vals[e] * (double)T[off];
    }
    W[idx] = acc;
}

// The transposed Khatri-Rao product of the other modes' factors as the source (the
// KSEQRCS pivots, qr_lev_score_sampled.jl:250-262): KRP^T(r, c) = prod_k A_k(i_k(c), r),
// R rows.  W(r, q) = KRP^T(r, cols[q]) (cols null: column q), R x ncols.
__global__ __launch_bounds__(256) void k_krp_cols(OtherModes om, int R, const int64_t* __restrict__ cols,
                                                  int64_t ncols, double* __restrict__ W) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (int64_t)R * ncols) return;
    const int64_t q = idx / R;
    const int r = (int)(idx - q * R);
    int64_t c = cols ? cols[q] : q;
    double v = 1.0;
    for (int k = 0; k < om.n; ++k) {
        v *= om.A[k][(c % om.dim[k]) + om.dim[k] * r];
        c /= om.dim[k];
    }
    W[idx] = v;
}

// (Omega KRP)^T (omega_hadamard, had_contract.jl:300-329, transposed as SEQRCS.jl:199
// takes it): W(r, j) = sum over the nonzeros e of row j of Omega (increasing column)
// of vals[e] KRP(colidx[e], r), R x l.
__global__ __launch_bounds__(256) void k_sketch_krp(OtherModes om, int R, const int64_t* __restrict__ rowptr,
                                                    const int64_t* __restrict__ colidx,
                                                    const double* __restrict__ vals, int64_t l,
                                                    double* __restrict__ W) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (int64_t)R * l) return;
    const int64_t j = idx / R;
    const int r = (int)(idx - j * R);
    double acc = 0.0;
    for (int64_t e = rowptr[j]; e < rowptr[j + 1]; ++e) {
        int64_t c = colidx[e];
        double v = 1.0;
        for (int k = 0; k < om.n; ++k) {
            v *= om.A[k][(c % om.dim[k]) + om.dim[k] * r];
            c /= om.dim[k];
        }
        acc += vals[e] * v;
    }
    W[idx] = acc;
}

// Column-pivoted QR of W (m x n, ld m) in one workgroup (xGEQP3 / xLAQP2 pivots);
// jpvt (n) = the column order, rdiag (min(m, n)) = the diagonal of R.
template <int NT>
__global__ __launch_bounds__(NT) void k_qrcp(double* __restrict__ W, int m, int n, double* __restrict__ tau,
                                             double* __restrict__ vwork, int* __restrict__ jpvt,
                                             double* __restrict__ rdiag) {
    __shared__ double redv[NT];
    __shared__ int redi[NT];
    geqp3<NT>(W, m, n, m, true, tau, jpvt, vwork, vwork + n, redv, redi);
    const int kq = m < n ? m : n;
    for (int j = threadIdx.x; j < kq; j += NT) rdiag[j] = W[j + (int64_t)m * j];
}

// The same column-pivoted QR for wide matrices, one step per three launches over the
// whole chip.  Every per-column operation is the one-workgroup form's (a wave per
// column, lanes over rows, wave_sum; the reflector through house<SNT>); the pivot
// choices are the same, the last bits may differ with the compiler's contractions.
__global__ __launch_bounds__(256) void k_qrcp_norms(const double* __restrict__ W, int m, int n,
                                                    double* __restrict__ vn1, double* __restrict__ vn2,
                                                    int* __restrict__ jpvt) {
    const int64_t j = ((int64_t)blockIdx.x * 256 + threadIdx.x) >> 6;
    const int ln = threadIdx.x & 63;
    if (j >= n) return;
    const double* c = W + (int64_t)m * j;
    double ss = 0.0;
    for (int k = ln; k < m; k += 64) ss += c[k] * c[k];
    ss = wave_sum(ss);
    if (ln == 0) {
        vn1[j] = sqrt(ss);
        vn2[j] = sqrt(ss);
        jpvt[j] = (int)j;
    }
}

// first position of the largest |vn1| among [lo, n) within each block's chunk
__global__ __launch_bounds__(256) void k_qrcp_argmax_part(const double* __restrict__ vn1, int lo, int n,
                                                          int per_block, double* __restrict__ part_v,
                                                          int* __restrict__ part_i) {
    __shared__ double redv[256];
    __shared__ int redi[256];
    const int b0 = lo + blockIdx.x * per_block;
    const int b1 = min(n, b0 + per_block);
    const int r = block_argmax<256>(b0, b1, [&](int j) { return fabs(vn1[j]); }, redv, redi);
    if (threadIdx.x == 0) {
        part_v[blockIdx.x] = r < b1 ? fabs(vn1[r]) : -__builtin_inf();
        part_i[blockIdx.x] = r < b1 ? r : n;
    }
}

// step i, one workgroup: the pivot from the block partials (first index on ties), the
// swap, and the reflector of column i (rows i..m-1)
__global__ __launch_bounds__(SNT) void k_qrcp_pivot(double* __restrict__ W, int m, int n, int i,
                                                    const double* __restrict__ part_v,
                                                    const int* __restrict__ part_i, int nparts,
                                                    double* __restrict__ vn1, double* __restrict__ vn2,
                                                    int* __restrict__ jpvt, double* __restrict__ tau,
                                                    double* __restrict__ rdiag) {
    __shared__ double redv[SNT];
    __shared__ int redi[SNT];
    const int t = threadIdx.x;
    const int64_t ld = m;
    // nparts == 0: the columns are few enough to scan here; else among equal maxima the
    // partial with the smallest position wins (blocks cover increasing ranges, so the
    // first block holding the maximum has it)
    int p;
    if (nparts == 0) {
        p = block_argmax<SNT>(i, n, [&](int j) { return fabs(vn1[j]); }, redv, redi);
    } else {
        const int q = block_argmax<SNT>(0, nparts, [&](int b) { return part_v[b]; }, redv, redi);
        p = (q < nparts) ? part_i[q] : n;
    }
    const int pvt = (p < n) ? p : i;
    if (pvt != i) {
        for (int k = t; k < m; k += SNT) {
            const double a = W[k + ld * pvt];
            W[k + ld * pvt] = W[k + ld * i];
            W[k + ld * i] = a;
        }
        if (t == 0) {
            const int x = jpvt[pvt]; jpvt[pvt] = jpvt[i]; jpvt[i] = x;
            vn1[pvt] = vn1[i];
            vn2[pvt] = vn2[i];
        }
    }
    __syncthreads();
    double* col = W + i + ld * i;
    const double ti = house<SNT>(col, m - i, redv);
    if (t == 0) {
        tau[i] = ti;
        if (rdiag) rdiag[i] = col[0];
    }
}

// step i: (I - tau v v^T) on every column j > i and its partial-norm update
// (xLAQP2's downdate, recomputed below sqrt(eps)); a wave per column.  The arithmetic
// is geqp3's (the one-workgroup form) step for step: the dot product with lane ln
// summing rows ln, ln + 64, ... of the column (rows relative to i), the update
// c - f v, and the recomputed norm with lane ln summing rows 1 + ln, 65 + ln, ...
// before the wave sum, so both forms give the same bits.
template <int NQ>
__global__ __launch_bounds__(256) void k_qrcp_apply(double* __restrict__ W, int m, int n, int i,
                                                    const double* __restrict__ tau, double* __restrict__ vn1,
                                                    double* __restrict__ vn2) {
    const int64_t j = i + 1 + (((int64_t)blockIdx.x * 256 + threadIdx.x) >> 6);
    const int ln = threadIdx.x & 63;
    if (j >= n) return;
    const int64_t ld = m;
    const int len = m - i;
    const double* v = W + i + ld * i;
    double* c = W + i + ld * j;
    const double ti = tau[i];
    // ci: row i's new value; ssq: this lane's share (rows 1 + ln + 64 q) of the squared
    // norm of rows i+1 .. m-1
    double ci = 0.0, ssq = 0.0;
    if (ti != 0.0 && len <= 64 * NQ) {
        // the column's rows of this lane stay in registers between the two passes; the
        // norm terms reach their geqp3 lane by a shuffle (row 1 + ln + 64 q is held by
        // lane ln + 1 at q, or by lane 0 at q + 1 for ln = 63), so no lane reads another
        // lane's store
        double cr[NQ], vr[NQ];
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int k = ln + 64 * q;
            cr[q] = k < len ? c[k] : 0.0;
            vr[q] = k < len ? (k == 0 ? 1.0 : v[k]) : 0.0;
            if (k < len) s += vr[q] * cr[q];
        }
        const double f = ti * wave_sum(s);
        double nv[NQ + 1];
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int k = ln + 64 * q;
            nv[q] = cr[q] - f * vr[q];
            if (k < len) c[k] = nv[q];
        }
        nv[NQ] = 0.0;
        ci = nv[0];
        double y[NQ + 1];
#pragma unroll
        for (int q = 0; q < NQ; ++q) y[q] = __shfl(nv[q], (ln + 1) & 63);
        y[NQ] = 0.0;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int k = 1 + ln + 64 * q;
            const double x = ln < 63 ? y[q] : y[q + 1];
            if (k < len) ssq += x * x;
        }
    } else if (ti != 0.0) {
        double s = 0.0;
        for (int k = ln; k < len; k += 64) s += (k == 0 ? 1.0 : v[k]) * c[k];
        const double f = ti * wave_sum(s);
        // reads first: the new values of this lane's norm rows (the same c - f v the
        // writes below store), consumed before any store is issued
        for (int k = 1 + ln; k < len; k += 64) {
            const double x = c[k] - f * v[k];
            ssq += x * x;
        }
        if (ln == 0) ci = c[0] - f;
        for (int k = ln; k < len; k += 64) c[k] = c[k] - f * (k == 0 ? 1.0 : v[k]);
    } else {
        for (int k = 1 + ln; k < len; k += 64) ssq += c[k] * c[k];
        if (ln == 0) ci = c[0];
    }
    ci = __shfl(ci, 0);
    const double tol3z = 1.0536712127723509e-08;   // sqrt(eps)
    const double v1 = vn1[j];
    if (v1 != 0.0) {
        double temp = fabs(ci) / v1;
        temp = fmax(1.0 - temp * temp, 0.0);
        const double q = v1 / vn2[j];
        if (temp * q * q <= tol3z) {
            const double ss = wave_sum(ssq);
            if (ln == 0) { vn1[j] = sqrt(ss); vn2[j] = vn1[j]; }
        } else if (ln == 0) {
            vn1[j] = v1 * sqrt(temp);
        }
    }
}

// splitmix64 (Steele, Lea, Flood 2014): the stream of the sparse sign generator.
__device__ __forceinline__ uint64_t splitmix_next(uint64_t& s) {
    uint64_t z = (s += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// Uniform in [0, n): the 2^64 mod n lowest draws are rejected (at most 2^-33 of them
// for n < 2^31), so r % n is unbiased; the retry count is bounded.
__device__ __forceinline__ int64_t uniform_below(uint64_t& s, int64_t n) {
    const uint64_t un = (uint64_t)n;
    const uint64_t rej = (0ull - un) % un;
    uint64_t r = splitmix_next(s);
    for (int a = 0; a < 64 && r < rej; ++a) r = splitmix_next(s);
    return (int64_t)(r % un);
}

// Sparse sign embedding, d x m with zeta nonzeros per column (sparse_sign.c:25-69:
// distinct rows by rejection; sparsestack.c:24-78 (injective): entry q in block q of
// the near-equal split of 0..d-1), values +-1/sqrt(zeta), one thread per column, each
// column its own stream of the seed.  rows / vals: zeta per column, column-major.
__global__ __launch_bounds__(256) void k_sparse_sign(int d, int64_t m, int zeta, int injective, uint64_t seed,
                                                     double* __restrict__ vals, int* __restrict__ rows) {
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (c >= m) return;
    uint64_t st = seed ^ (0xD1B54A32D192ED03ull * (uint64_t)(c + 1));
    const double a = 1.0 / sqrt((double)zeta);
    int* rc = rows + c * zeta;
    double* vc = vals + c * zeta;
    const int qb = d / zeta, rb = d % zeta;
    for (int q = 0; q < zeta; ++q) {
        int row;
        if (injective) {
            const int size = q < rb ? qb + 1 : qb;
            const int start = q < rb ? q * (qb + 1) : rb * (qb + 1) + (q - rb) * qb;
            row = start + (int)uniform_below(st, size);
        } else {
            // redraw on a repeat; after 4096 repeats (never expected: zeta <= d) the
            // smallest unused row is taken, so the loop always ends
            row = -1;
            for (int a2 = 0; a2 < 4096 && row < 0; ++a2) {
                const int cand = (int)uniform_below(st, d);
                bool dup = false;
                for (int k = 0; k < q; ++k) dup = dup || rc[k] == cand;
                if (!dup) row = cand;
            }
            for (int cand = 0; row < 0 && cand < d; ++cand) {
                bool dup = false;
                for (int k = 0; k < q; ++k) dup = dup || rc[k] == cand;
                if (!dup) row = cand;
            }
        }
        rc[q] = row;
        vc[q] = (splitmix_next(st) & 1ull) ? a : -a;
    }
}

// The grid-wide column-pivoted QR of W (m x n, ld m): tau (min(m, n)), jpvt (n), vwork
// (2 n: the partial norms), rdiag (nullable), part_v / part_i (cdiv(n, 4096) each).
hipError_t launch_grid_geqp3(double* W, int m, int n, double* tau, double* vwork, int* jpvt, double* rdiag,
                             double* part_v, int* part_i, hipStream_t st) {
    constexpr int per_block = 4096;
    double* vn1 = vwork;
    double* vn2 = vwork + n;
    hipLaunchKernelGGL(k_qrcp_norms, dim3((unsigned)cdiv(n, 4)), dim3(256), 0, st, W, m, n, vn1, vn2, jpvt);
    hipError_t e = hipGetLastError();
    const int kq = m < n ? m : n;
    for (int i = 0; i < kq && e == hipSuccess; ++i) {
        // up to one block of columns the pivot kernel scans them itself
        const int np = n <= per_block ? 0 : (int)cdiv(n - i, per_block);
        if (np > 0)
            hipLaunchKernelGGL(k_qrcp_argmax_part, dim3((unsigned)np), dim3(256), 0, st, vn1, i, n, per_block,
                               part_v, part_i);
        hipLaunchKernelGGL(k_qrcp_pivot, dim3(1), dim3(SNT), 0, st, W, m, n, i, part_v, part_i, np, vn1, vn2, jpvt,
                           tau, rdiag);
        // rows per lane kept in registers between the reflector's two passes: 8 up to 512
        // rows, 32 up to 2048; taller columns take both passes from memory
        if (i + 1 < n) {
            const dim3 g((unsigned)cdiv(n - i - 1, 4));
            if (m <= 512)
                hipLaunchKernelGGL(k_qrcp_apply<8>, g, dim3(256), 0, st, W, m, n, i, tau, vn1, vn2);
            else
                hipLaunchKernelGGL(k_qrcp_apply<32>, g, dim3(256), 0, st, W, m, n, i, tau, vn1, vn2);
        }
        e = hipGetLastError();
    }
    return e;
}

OtherModes other_modes(const itcpd_plan* p, int mode) {
    OtherModes om{};
    int64_t stride = 1;
    int q = 0;
    for (int m = 0; m < p->N; ++m) {
        if (m != mode) {
            om.A[q] = p->A[m];
            om.dim[q] = p->dims[m];
            om.tstride[q] = stride;
            ++q;
        }
        stride *= p->dims[m];
    }
    om.n = q;
    return om;
}

int64_t tensor_stride(const itcpd_plan* p, int mode) {
    int64_t s = 1;
    for (int m = 0; m < mode; ++m) s *= p->dims[m];
    return s;
}

// grow-only workspaces of the sampled path
int ensure_sampled_ws(itcpd_plan* p, size_t doubles, size_t ints) {
    int rc;
    if (p->smp_ws_cap < doubles) {
        ITCPD_HIP(hipStreamSynchronize(p->stream));
        dfree(p->smp_ws);
        p->smp_ws = nullptr;
        p->smp_ws_cap = 0;
        if ((rc = dmalloc(&p->smp_ws, doubles))) return rc;
        p->smp_ws_cap = doubles;
    }
    if (p->smp_iws_cap < ints) {
        ITCPD_HIP(hipStreamSynchronize(p->stream));
        dfree(p->smp_iws);
        p->smp_iws = nullptr;
        p->smp_iws_cap = 0;
        if ((rc = dmalloc(&p->smp_iws, ints))) return rc;
        p->smp_iws_cap = ints;
    }
    return ITCPD_OK;
}

}  // namespace

// probs_dev: a device buffer of I_n doubles, or null for the workspace's (returned in
// *probs_used; valid until the next sampled-path call)
int launch_leverage_scores(itcpd_plan* p, int mode, double* probs_dev, double** probs_used) {
    const int m = (int)p->dims[mode], n = (int)p->R;
    int rc;
    // W (m n) | tau (n) | vwork (2n) | probs (m) | G, Ui, Gi (3 n^2)
    if ((rc = ensure_sampled_ws(p, (size_t)m * n + 3 * (size_t)n + (size_t)m + 3 * (size_t)n * n, (size_t)n + 4)))
        return rc;
    double* W = p->smp_ws;
    double* tau = W + (size_t)m * n;
    double* vwork = tau + n;
    double* probs = probs_dev ? probs_dev : vwork + 2 * n;
    double* G = vwork + 2 * n + m;
    double* Ui = G + (size_t)n * n;
    double* Gi = Ui + (size_t)n * n;
    int* need = p->smp_iws + n;
    *probs_used = probs;
    if (m <= n) {
        hipLaunchKernelGGL(k_fill_value, dim3((unsigned)cdiv(m, 256)), dim3(256), 0, p->stream, probs, m,
                           1.0 / (double)m, p->chk);
        ITCPD_HIP(hipGetLastError());
        return ITCPD_OK;
    }
    hipLaunchKernelGGL(k_gemm_tn, dim3((unsigned)cdiv((int64_t)n * n * 64, 256)), dim3(256), 0, p->stream,
                       p->A[mode], p->A[mode], (int64_t)m, n, n, G, p->chk);
    ITCPD_HIP(hipGetLastError());
    if (n <= 64) {
        hipLaunchKernelGGL(k_gram_chol64, dim3(1), dim3(256), 0, p->stream, G, n, Ui, need, p->chk);
        ITCPD_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_lev_rows64, dim3((unsigned)cdiv(m, 64)), dim3(256), 0, p->stream, p->A[mode], m, n, Ui,
                           need, probs, p->chk);
    } else {
        hipLaunchKernelGGL(k_gram_chol_inv<256>, dim3(1), dim3(256), 0, p->stream, G, n, Ui, Gi, need, p->chk);
        ITCPD_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_lev_rows, dim3((unsigned)cdiv(m, 256)), dim3(256), 0, p->stream, p->A[mode], m, n, Gi,
                           need, probs, p->chk);
    }
    ITCPD_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_lev_scores<SNT>, dim3(1), dim3(SNT), 0, p->stream, p->A[mode], m, n, W, tau, vwork,
                       p->smp_iws, probs, need, p->chk);
    ITCPD_HIP(hipGetLastError());
    return ITCPD_OK;
}

namespace {

// Views of the sampled step's workspace.
struct SampledWs {
    double *Ks, *B, *W, *Vs, *tau, *ztau, *vwork;
    int *jpvt, *info;
};
SampledWs sampled_ws(const itcpd_plan* p, int mode, int64_t ns) {
    const size_t R = (size_t)p->R;
    SampledWs w;
    w.Ks = p->smp_ws;                                   // ns x R
    w.B = w.Ks + (size_t)ns * R;                        // ns x In
    w.W = w.B + (size_t)ns * (size_t)p->dims[mode];     // ns x R (QR form)
    w.Vs = w.W + (size_t)ns * R;                        // R x R
    w.tau = w.Vs + R * R;                               // R
    w.ztau = w.tau + R;                                 // R
    w.vwork = w.ztau + R;                               // 2 R
    w.jpvt = p->smp_iws + (size_t)ns * (p->N - 1);
    w.info = w.jpvt + R;
    return w;
}

}  // namespace

bool sampled_corrected_ok(const itcpd_plan* p, int64_t ns) { return p->R <= 64 && ns >= p->R; }

// samples: device, ns x (N-1) column-major.  K_s and the sampled fibers, into the workspace.
int launch_sampled_gather(itcpd_plan* p, int mode, int64_t ns, const int* samples) {
    const int R = (int)p->R;
    const int64_t In = p->dims[mode];
    const OtherModes om = other_modes(p, mode);
    const SampledWs w = sampled_ws(p, mode, ns);
    const int64_t nk = ns * R, nb = ns * In;
    hipLaunchKernelGGL(k_pivot_hadamard, dim3((unsigned)cdiv(nk, 256)), dim3(256), 0, p->stream, om, samples,
                       ns, R, w.Ks, p->chk);
    ITCPD_HIP(hipGetLastError());
    const int64_t ms = tensor_stride(p, mode);
    if (p->elt_bytes == 8)
        hipLaunchKernelGGL(k_sample_fibers<double>, dim3((unsigned)cdiv(nb, 256)), dim3(256), 0, p->stream,
                           (const double*)p->T, om, ms, In, samples, ns, w.B, p->chk);
    else
        hipLaunchKernelGGL(k_sample_fibers<float>, dim3((unsigned)cdiv(nb, 256)), dim3(256), 0, p->stream,
                           (const float*)p->T, om, ms, In, samples, ns, w.B, p->chk);
    ITCPD_HIP(hipGetLastError());
    return ITCPD_OK;
}

// The solve on the gathered samples: X (I_n x R) is left in p->X (with the normal equations
// also row-normed).  info[0] = rank of K_s and, for the corrected form, info[1] != 0 when it
// is not certified and X is not set; or the factorisation's finfo (normal form).
int launch_sampled_solve(itcpd_plan* p, int mode, int64_t ns, int form) {
    const int R = (int)p->R;
    const int64_t In = p->dims[mode];
    const SampledWs ws = sampled_ws(p, mode, ns);
    double *const Ks = ws.Ks, *const B = ws.B, *const W = ws.W, *const Vs = ws.Vs, *const tau = ws.tau,
           *const ztau = ws.ztau, *const vwork = ws.vwork;
    int *const jpvt = ws.jpvt, *const info = ws.info;
    const int64_t nk = ns * R;
    if (form != SAMPLED_QR) {   // V = K_s^T K_s, M = B^T K_s
        const unsigned nt = (unsigned)cdiv(R, 16);
        hipLaunchKernelGGL(k_sampled_products, dim3((unsigned)(nt * (nt + 1) / 2 + cdiv(In, 16) * nt)), dim3(512), 0,
                           p->stream, Ks, B, ns, R, In, Vs, p->M, p->chk);
        ITCPD_HIP(hipGetLastError());
    }
    if (form == SAMPLED_NORMAL) {   // the plan's factorisation and update on V
        p->v_override = Vs;
        int rc = launch_factor(p, mode);
        p->v_override = nullptr;
        if (rc) return rc;
        return launch_solve(p, mode, p->M, 1, In * R, true, false);
    }
    if (form == SAMPLED_CORRECTED) {
        GramSet gs{};
        gs.G[0] = gs.G[1] = Vs;
        gs.N = 2;
        hipLaunchKernelGGL(k_sampled_inverse, dim3(1), dim3(256), 0, p->stream, gs, R, p->Upad, info, p->chk);
        ITCPD_HIP(hipGetLastError());
        auto run = [&](auto kern, int threads) {
            hipLaunchKernelGGL(kern, dim3((unsigned)cdiv(In, 16)), dim3(threads), 0, p->stream, Ks, B, ns, R, In, p->M,
                               p->Upad, info, p->X, p->chk);
        };
        if (R <= 16) run(k_sampled_correct<16>, correct_threads(16));
        else if (R <= 32) run(k_sampled_correct<32>, correct_threads(32));
        else run(k_sampled_correct<64>, correct_threads(64));
        ITCPD_HIP(hipGetLastError());
        return ITCPD_OK;
    }
    ITCPD_HIP(hipMemcpyAsync(W, Ks, (size_t)nk * 8, hipMemcpyDeviceToDevice, p->stream));
    // tall samples: the column-pivoted QR as grid-wide steps (a wave per column instead
    // of eight waves for all of them), then rank estimate and RZ in one workgroup
    const bool grid = ns >= p->qr_grid_min_rows;
    if (grid) {
        double* part_v = vwork + 2 * R;
        int* part_i = info + 4;
        ITCPD_HIP(launch_grid_geqp3(W, (int)ns, R, tau, vwork, jpvt, nullptr, part_v, part_i, p->stream));
    }
    hipLaunchKernelGGL(k_lsq_qr_factor<SNT>, dim3(1), dim3(SNT), 0, p->stream, W, (int)ns, R, tau, ztau, vwork,
                       jpvt, info, grid ? 1 : 0, p->chk);
    ITCPD_HIP(hipGetLastError());
    if (ns <= 64 * 32)
        hipLaunchKernelGGL(k_lsq_qr_apply_reg<32>, dim3((unsigned)cdiv(In, 4)), dim3(256), (size_t)4 * R * 8,
                           p->stream, W, (int)ns, R, B, In, p->X, tau, ztau, jpvt, info, p->chk);
    else
        hipLaunchKernelGGL(k_lsq_qr_apply, dim3((unsigned)cdiv(In, 4)), dim3(256), (size_t)4 * R * 8, p->stream, W,
                           (int)ns, R, B, In, p->X, tau, ztau, jpvt, info, p->chk);
    ITCPD_HIP(hipGetLastError());
    return ITCPD_OK;
}

int sampled_ws_prepare(itcpd_plan* p, int mode, int64_t ns) {
    const int64_t R = p->R, In = p->dims[mode];
    // + the argmax partials of the grid-wide QR (one per 4096 columns; R <= 2048 here)
    const size_t doubles = (size_t)(2 * ns * R + ns * In + R * R + 4 * R + 8);
    const size_t ints = (size_t)(ns * (p->N - 1) + R + 4 + 8);
    return ensure_sampled_ws(p, doubles, ints);
}

// Column-pivoted QR of T_(mode) (krp: of the transposed Khatri-Rao product of the
// other modes' factors, R rows) restricted to the columns `cols` (device, ncols of
// them; null: every column) or, with `omega_rowptr` given, of the sketch T_(mode)
// Omega^T (krp: (Omega KRP)^T) with Omega (l x ncols_all) by rows (omega_rowptr /
// omega_cols / omega_vals, device).  Scratch is allocated here and freed after (a set-up step before the
// sweeps); jpvt_dev (n ints) and rdiag_dev (min(I_n, n)) receive the result, with n
// = ncols or l.  The call synchronises the plan stream.
int launch_qr_pivots(itcpd_plan* p, int mode, bool krp, const int64_t* cols, int64_t ncols,
                     const int64_t* omega_rowptr, const int64_t* omega_cols, const double* omega_vals, int64_t l,
                     int* jpvt_dev, double* rdiag_dev) {
    const int64_t In = krp ? p->R : p->dims[mode];   // rows of the source
    const int64_t n = omega_rowptr ? l : ncols;
    const OtherModes om = other_modes(p, mode);
    const int64_t ms = tensor_stride(p, mode);
    double* W = nullptr;
    int rc;
    // W (I_n x n) | tau (min) | vn1, vn2 (2 n)
    if ((rc = dmalloc(&W, (size_t)(In * n + std::min(In, n) + 2 * n)))) return rc;
    double* tau = W + In * n;
    double* vwork = tau + std::min(In, n);
    const unsigned grid = (unsigned)cdiv(In * n, 256);
    if (krp && omega_rowptr) {
        hipLaunchKernelGGL(k_sketch_krp, dim3(grid), dim3(256), 0, p->stream, om, (int)In, omega_rowptr,
                           omega_cols, omega_vals, l, W);
    } else if (krp) {
        hipLaunchKernelGGL(k_krp_cols, dim3(grid), dim3(256), 0, p->stream, om, (int)In, cols, ncols, W);
    } else if (omega_rowptr) {
        if (p->elt_bytes == 8)
            hipLaunchKernelGGL(k_sketch<double>, dim3(grid), dim3(256), 0, p->stream, (const double*)p->T, om, ms,
                               In, omega_rowptr, omega_cols, omega_vals, l, W);
        else
            hipLaunchKernelGGL(k_sketch<float>, dim3(grid), dim3(256), 0, p->stream, (const float*)p->T, om, ms,
                               In, omega_rowptr, omega_cols, omega_vals, l, W);
    } else {
        if (p->elt_bytes == 8)
            hipLaunchKernelGGL(k_unfold_cols<double>, dim3(grid), dim3(256), 0, p->stream, (const double*)p->T, om,
                               ms, In, cols, ncols, W);
        else
            hipLaunchKernelGGL(k_unfold_cols<float>, dim3(grid), dim3(256), 0, p->stream, (const float*)p->T, om,
                               ms, In, cols, ncols, W);
    }
    hipError_t e = hipGetLastError();
    if (e == hipSuccess && n <= p->qr_one_wg_max) {
        hipLaunchKernelGGL(k_qrcp<SNT>, dim3(1), dim3(SNT), 0, p->stream, W, (int)In, (int)n, tau, vwork, jpvt_dev,
                           rdiag_dev);
        e = hipGetLastError();
    } else if (e == hipSuccess) {
        // wide: a step per three launches
        const int nparts = (int)cdiv(n, 4096);
        double* part_v = nullptr;
        int* part_i = nullptr;
        if ((rc = dmalloc(&part_v, (size_t)nparts)) || (rc = dmalloc(&part_i, (size_t)nparts))) {
            dfree(part_v);
            dfree(part_i);
            dfree(W);
            return rc;
        }
        e = launch_grid_geqp3(W, (int)In, (int)n, tau, vwork, jpvt_dev, rdiag_dev, part_v, part_i, p->stream);
        const hipError_t e3 = hipStreamSynchronize(p->stream);
        dfree(part_v);
        dfree(part_i);
        if (e == hipSuccess) e = e3;
    }
    const hipError_t e2 = hipStreamSynchronize(p->stream);
    dfree(W);
    if (e != hipSuccess) return hip_fail(e, "qr pivots launch");
    if (e2 != hipSuccess) return hip_fail(e2, "qr pivots");
    return ITCPD_OK;
}

int launch_sparse_sign(int d, int64_t m, int zeta, bool injective, uint64_t seed, double* vals_dev, int* rows_dev,
                       hipStream_t st) {
    hipLaunchKernelGGL(k_sparse_sign, dim3((unsigned)cdiv(m, 256)), dim3(256), 0, st, d, m, zeta,
                       injective ? 1 : 0, seed, vals_dev, rows_dev);
    ITCPD_HIP(hipGetLastError());
    return ITCPD_OK;
}

}  // namespace itcpd
