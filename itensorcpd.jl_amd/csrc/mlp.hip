// The warm-start network: a fully connected MLP (ReLU hidden layers, linear
// output) trained and evaluated with the kernels below, FP32 throughout.
//   forward  : H_{l+1} = act(H_l W_l + b_l)        (row-major: batch x width)
//   backward : dH_l = (dH_{l+1} .* act'(H_{l+1})) W_l^T,  dW_l = H_l^T dZ_l,  db_l = 1^T dZ_l
//   loss     : 0.5 * sum(mask .* (Y - Y*)^2) / batch
//   update   : Adam (beta1 0.9, beta2 0.999, eps 1e-8)
// No reference counterpart: the reference initialises from random_CPD only
// (cpd.jl:63-82).  The network is what the learned warm start proposes from the
// mode sketches; the ALS fit decides whether its proposal or random_CPD is used.
#include "internal.h"

#include <algorithm>
#include <cmath>
#include <vector>

namespace itcpd {
namespace {

typedef float mf4 __attribute__((ext_vector_type(4)));
typedef float mfu4 __attribute__((ext_vector_type(4), aligned(4)));

// One product of the network, C(M x N) = op(A)(M x K) op(B)(K x N), row-major, and what is
// done to it on the way out.
struct MlpProduct {
    const float *A, *B;
    float* C;
    int M, N, K, lda, ldb;      // C has leading dimension N
    const float* bias;          // added to every row (null: none)
    int relu;                   // then negative values are set to 0
    const float* gate;          // M x N: the result is 0 where the gate is not > 0 (null: none)
    float* colsum;              // N column sums of op(B) (null: none)
};

// A wave's 16 T x 16 T tile (tile row tm, column tn) of a product on v_mfma_f32_16x16x4_f32,
// operands straight from global memory (a network's matrices live in L2).  A stage is 16
// reduction indices, lane (c, g) taking 4 g .. 4 g + 3: one 16-byte run where the index is
// contiguous, else four rows of which the 16 lanes read 64 bytes each.  Eight stages (T = 1;
// four for T = 2) are in flight together: these products are bound by latency, 256 x 256 x 256
// having one tile per CU, so every round trip to L2 shows.  Rows past the end read the last
// one, stages past the last whole one are zeroed after the load.
template <bool TA, bool TB, int T>
__device__ __forceinline__ void mlp_tile(const MlpProduct& q, int tm, int tn) {
    constexpr int U = T == 1 ? 8 : 4;
    const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
    int m[T], n[T];
#pragma unroll
    for (int i = 0; i < T; ++i) {
        const int mm = 16 * (T * tm + i) + c, nn = 16 * (T * tn + i) + c;
        m[i] = mm < q.M ? mm : q.M - 1;
        n[i] = nn < q.N ? nn : q.N - 1;
    }
    auto loadA = [&](int i, int k, float (&x)[4]) {   // op(A)(m[i], k .. k + 3)
        if constexpr (TA) {
#pragma unroll
            for (int s = 0; s < 4; ++s) x[s] = q.A[(size_t)(k + s) * q.lda + m[i]];
        } else {
            const mfu4 v = *reinterpret_cast<const mfu4*>(q.A + (size_t)m[i] * q.lda + k);
            x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
        }
    };
    auto loadB = [&](int j, int k, float (&x)[4]) {   // op(B)(k .. k + 3, n[j])
        if constexpr (!TB) {
#pragma unroll
            for (int s = 0; s < 4; ++s) x[s] = q.B[(size_t)(k + s) * q.ldb + n[j]];
        } else {
            const mfu4 v = *reinterpret_cast<const mfu4*>(q.B + (size_t)n[j] * q.ldb + k);
            x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
        }
    };
    mf4 acc[T][T];
    float cs[T];
#pragma unroll
    for (int i = 0; i < T; ++i) {
        cs[i] = 0.f;
#pragma unroll
        for (int j = 0; j < T; ++j) acc[i][j] = (mf4){0.f, 0.f, 0.f, 0.f};
    }
    const int full = q.K / 16;
    for (int s0 = 0; s0 < full; s0 += U) {
        float a[U][T][4], b[U][T][4];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = 16 * (s0 + u < full ? s0 + u : full - 1) + 4 * g;
#pragma unroll
            for (int i = 0; i < T; ++i) loadA(i, k, a[u][i]);
#pragma unroll
            for (int j = 0; j < T; ++j) loadB(j, k, b[u][j]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool in = s0 + u < full;
#pragma unroll
            for (int s = 0; s < 4; ++s) {
#pragma unroll
                for (int j = 0; j < T; ++j) {
                    const float bv = in ? b[u][j][s] : 0.f;
                    cs[j] += bv;
#pragma unroll
                    for (int i = 0; i < T; ++i)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? a[u][i][s] : 0.f, bv, acc[i][j], 0, 0, 0);
                }
            }
        }
    }
    if (16 * full < q.K) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int k = 16 * full + 4 * g + s, kc = k < q.K ? k : q.K - 1;
            float a[T], b[T];
#pragma unroll
            for (int i = 0; i < T; ++i) {
                a[i] = TA ? q.A[(size_t)kc * q.lda + m[i]] : q.A[(size_t)m[i] * q.lda + kc];
                b[i] = TB ? q.B[(size_t)n[i] * q.ldb + kc] : q.B[(size_t)kc * q.ldb + n[i]];
                if (k >= q.K) a[i] = b[i] = 0.f;
                cs[i] += b[i];
            }
#pragma unroll
            for (int i = 0; i < T; ++i)
#pragma unroll
                for (int j = 0; j < T; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    }
    // result: lane (c, g), register v holds row 4 g + v, column c
#pragma unroll
    for (int j = 0; j < T; ++j) {
        const int col = 16 * (T * tn + j) + c;
        if (q.colsum && tm == 0) {
            float s = cs[j];
            s += __shfl_xor(s, 16);
            s += __shfl_xor(s, 32);
            if (g == 0 && col < q.N) q.colsum[col] = s;
        }
        if (col >= q.N) continue;
        const float bias = q.bias ? q.bias[col] : 0.f;
#pragma unroll
        for (int i = 0; i < T; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = 16 * (T * tm + i) + 4 * g + v;
                if (row >= q.M) continue;
                float x = acc[i][j][v] + bias;
                if (q.relu && x < 0.f) x = 0.f;
                if (q.gate && !(q.gate[(size_t)row * q.N + col] > 0.f)) x = 0.f;
                q.C[(size_t)row * q.N + col] = x;
            }
    }
}

// H = act(X W + b): wave w of a block takes tile 4 blockIdx.x + w, row by row of tiles.
template <int T>
__global__ __launch_bounds__(256) void k_mlp_forward(MlpProduct q) {
    const int tiles_n = (q.N + 16 * T - 1) / (16 * T);
    const int64_t tile = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int tm = (int)(tile / tiles_n);
    if (tm * 16 * T >= q.M) return;
    mlp_tile<false, false, T>(q, tm, (int)(tile % tiles_n));
}

// A layer's two backward products in one launch: blocks below nw the weight gradient
// dW = H^T dZ (and db, the column sums of dZ), the others dH = dZ W^T gated by H > 0.
template <int T>
__global__ __launch_bounds__(256) void k_mlp_backward(MlpProduct dw, MlpProduct dh, unsigned nw) {
    const bool weight = blockIdx.x < nw;
    const MlpProduct& q = weight ? dw : dh;
    const int tiles_n = (q.N + 16 * T - 1) / (16 * T);
    const int64_t tile = (int64_t)(weight ? blockIdx.x : blockIdx.x - nw) * 4 + (threadIdx.x >> 6);
    const int tm = (int)(tile / tiles_n), tn = (int)(tile % tiles_n);
    if (tm * 16 * T >= q.M) return;
    if (weight) mlp_tile<true, false, T>(q, tm, tn);
    else mlp_tile<false, true, T>(q, tm, tn);
}

// dZ = mask .* (Y - Y*) / batch (output layer), and the per-block loss partials
__global__ __launch_bounds__(256) void k_mse_grad(const float* __restrict__ Y, const float* __restrict__ Yt,
                                                  const float* __restrict__ mask, int64_t n, float inv_batch,
                                                  float* __restrict__ dZ, double* __restrict__ loss_part) {
    __shared__ double red[256];
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    double l = 0.0;
    if (i < n) {
        const float mk = mask ? mask[i] : 1.f;
        const float d = mk * (Y[i] - Yt[i]);
        dZ[i] = d * inv_batch;
        l = 0.5 * (double)d * (double)d * (double)inv_batch;
    }
    red[threadIdx.x] = l;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) loss_part[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(256) void k_adam(float* __restrict__ p, const float* __restrict__ g,
                                              float* __restrict__ m, float* __restrict__ v, int64_t n,
                                              float lr, float c1, float c2) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = 0.9f * m[i] + 0.1f * gi;
    const float vi = 0.999f * v[i] + 0.001f * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + 1e-8f);
}

__global__ __launch_bounds__(256) void k_sum_loss(const double* __restrict__ part, int n, double* __restrict__ out) {
    __shared__ double red[256];
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) s += part[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = red[0];
}

// Candidate factor columns of one mode from its sketch S (D x K, column-major),
// one workgroup per sketch: `ncand` rounds of successive projection -- take the
// row of largest norm, d = that row / its norm, candidate c = S d (positive at
// the chosen row), deflate S <- S - c d^T.  Rounds pick components in order of
// sketch energy (lambda_r^2 up to the sketch's random scaling), the same order in
// every mode.  Output rows: candidate k of sketch s at out[(s * ncand + k) * D],
// scaled to unit maximum magnitude.  D <= 256, K <= 64 (the sketch in LDS).
__global__ __launch_bounds__(256) void k_spa_candidates(const double* __restrict__ S, int D, int K,
                                                        int ncand, float* __restrict__ out) {
    __shared__ double Sl[256 * 65];
    __shared__ double d[64];
    __shared__ double redv[256];
    __shared__ int redi[256];
    __shared__ double cmax[256];
    const int t = threadIdx.x;
    const double* Sg = S + (size_t)blockIdx.x * D * K;
    for (int x = t; x < D * K; x += 256) {
        const int i = x % D, c = x / D;
        Sl[i * 65 + c] = Sg[x];
    }
    __syncthreads();
    for (int k = 0; k < ncand; ++k) {
        double nr = -1.0;
        if (t < D) {
            nr = 0.0;
            for (int c = 0; c < K; ++c) nr += Sl[t * 65 + c] * Sl[t * 65 + c];
        }
        redv[t] = nr;
        redi[t] = t;
        __syncthreads();
        for (int o = 128; o > 0; o >>= 1) {
            if (t < o) {
                const double v2 = redv[t + o];
                const int i2 = redi[t + o];
                if (v2 > redv[t] || (v2 == redv[t] && i2 < redi[t])) { redv[t] = v2; redi[t] = i2; }
            }
            __syncthreads();
        }
        const int istar = redi[0];
        const double nrm = sqrt(redv[0]);
        __syncthreads();
        if (t < K) d[t] = nrm > 0.0 ? Sl[istar * 65 + t] / nrm : 0.0;
        __syncthreads();
        double cv = 0.0;
        if (t < D) {
            for (int c = 0; c < K; ++c) cv += Sl[t * 65 + c] * d[c];
            for (int c = 0; c < K; ++c) Sl[t * 65 + c] -= cv * d[c];
        }
        cmax[t] = fabs(cv);
        __syncthreads();
        for (int o = 128; o > 0; o >>= 1) {
            if (t < o) cmax[t] = fmax(cmax[t], cmax[t + o]);
            __syncthreads();
        }
        const double scale = cmax[0] > 0.0 ? 1.0 / cmax[0] : 0.0;
        if (t < D) out[((size_t)blockIdx.x * ncand + k) * D + t] = (float)(cv * scale);
        __syncthreads();
    }
}

unsigned nblk(int64_t n) { return (unsigned)((n + 255) / 256); }

// Gaussian sketch of one unfolding: S(i, c) = sum_m T_(n)(i, m) Omega(m, c), the
// columns m of the unfolding enumerating the other modes with the first fastest, so
// T_(n)(i, m) = T[(m mod A) + A In (m div A) + A i] with A = prod of the dims before
// mode n.  Omega(m, c) is the N(0,1) draw of the Philox stream of `seed` at element
// e = m + M c (tag OMEGA_TAG), generated on the fly and never stored.  Block b takes
// the 32-column chunks b, b + gridDim.x, ...: the chunk of T (In x 32, loaded along
// the contiguous index) and of Omega (32 x K) go to LDS, thread (row lane, column
// group) accumulates rows l, l + 64, l + 128, l + 192 and columns g, g + 4, ...; the
// block's partial sum goes to part[b] (In x K column-major).  In <= 256, K <= 64.
template <typename TT>
__global__ __launch_bounds__(256) void k_gauss_sketch(const TT* __restrict__ T, int64_t In, int64_t A,
                                                      int64_t M, int K, uint64_t seed,
                                                      double* __restrict__ part) {
    __shared__ double Tt[SK_CH][257];
    __shared__ double Om[SK_CH][65];
    const int t = threadIdx.x;
    const int l = t & 63, g = t >> 6;
    double acc[4][16];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[q][j] = 0.0;
    const int64_t nch = (M + SK_CH - 1) / SK_CH;
    for (int64_t ch = blockIdx.x; ch < nch; ch += gridDim.x) {
        const int64_t m0 = ch * SK_CH;
        __syncthreads();
        const int64_t tile = In * SK_CH;
        for (int64_t x = t; x < tile; x += 256) {
            int64_t i, mm;
            if (A == 1) { i = x % In; mm = x / In; }        // mode 0: rows contiguous
            else { mm = x % SK_CH; i = x / SK_CH; }          // columns contiguous in runs of A
            const int64_t m = m0 + mm;
            double v = 0.0;
            if (m < M) v = (double)T[(m % A) + A * In * (m / A) + A * i];
            Tt[mm][i] = v;
        }
        for (int x = t; x < SK_CH * K; x += 256) {
            const int mm = x % SK_CH, c = x / SK_CH;
            const int64_t m = m0 + mm;
            Om[mm][c] = m < M ? philox_normal((uint64_t)(m + M * (int64_t)c), OMEGA_TAG, seed) : 0.0;
        }
        __syncthreads();
        for (int mm = 0; mm < SK_CH; ++mm) {
            double tv[4], ov[16];
#pragma unroll
            for (int q = 0; q < 4; ++q) tv[q] = Tt[mm][l + 64 * q];
#pragma unroll
            for (int j = 0; j < 16; ++j) ov[j] = Om[mm][g + 4 * j];
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int j = 0; j < 16; ++j) acc[q][j] = fma(tv[q], ov[j], acc[q][j]);
        }
    }
    double* P = part + (size_t)blockIdx.x * In * K;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int64_t i = l + 64 * q;
        if (i >= In) continue;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int c = g + 4 * j;
            if (c < K) P[i + In * c] = acc[q][j];
        }
    }
}

// out[x] = sum_{b < nb} part[b * n + x] in increasing b
__global__ __launch_bounds__(256) void k_sum_blocks(const double* __restrict__ part, int nb, int64_t n,
                                                    double* __restrict__ out) {
    const int64_t x = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (x >= n) return;
    double s = 0.0;
    for (int b = 0; b < nb; ++b) s += part[(int64_t)b * n + x];
    out[x] = s;
}

}  // namespace

// The Gaussian sketch's launch geometry: element offset stride A (prod of the dims
// before `mode`) and column count M of the unfolding.
void sketch_geometry(int order, const int64_t* dims, int mode, int64_t* A, int64_t* M) {
    *A = 1;
    *M = 1;
    for (int q = 0; q < order; ++q) {
        if (q < mode) *A *= dims[q];
        if (q != mode) *M *= dims[q];
    }
}

// The sketch kernel over nb blocks (partials in `part`, nb x In x K doubles) and the
// fixed-order sum of the partials into S_dev, enqueued on `st`.
hipError_t enqueue_gauss_sketch(const void* T, int elt_bytes, int64_t In, int64_t A, int64_t M, int K,
                                       uint64_t seed, int nb, double* part, double* S_dev, hipStream_t st) {
    if (elt_bytes == 8)
        hipLaunchKernelGGL(k_gauss_sketch<double>, dim3((unsigned)nb), dim3(256), 0, st, (const double*)T, In, A,
                           M, K, seed, part);
    else
        hipLaunchKernelGGL(k_gauss_sketch<float>, dim3((unsigned)nb), dim3(256), 0, st, (const float*)T, In, A, M,
                           K, seed, part);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_sum_blocks, dim3(nblk(In * K)), dim3(256), 0, st, (const double*)part, nb, In * K,
                       S_dev);
    return hipGetLastError();
}

int launch_gauss_sketch(itcpd_plan* p, int mode, int K, uint64_t seed, double* S_dev) {
    const int64_t In = p->dims[mode];
    int64_t A, M;
    sketch_geometry(p->N, p->dims, mode, &A, &M);
    const int64_t nch = (M + SK_CH - 1) / SK_CH;
    const int nb = (int)std::min<int64_t>(nch, 512);
    const size_t need = (size_t)nb * (size_t)(In * K);
    if (p->sk_ws_cap < need) {
        ITCPD_HIP(hipStreamSynchronize(p->stream));
        dfree(p->sk_ws);
        p->sk_ws = nullptr;
        p->sk_ws_cap = 0;
        int rc;
        if ((rc = dmalloc(&p->sk_ws, need))) return rc;
        p->sk_ws_cap = need;
    }
    ITCPD_HIP(enqueue_gauss_sketch(p->T, p->elt_bytes, In, A, M, K, seed, nb, p->sk_ws, S_dev, p->stream));
    return ITCPD_OK;
}


// ---------------------------------------------------------------- network
namespace {
int64_t mlp_tiles(const MlpProduct& q, int T) {
    return (int64_t)((q.M + 16 * T - 1) / (16 * T)) * ((q.N + 16 * T - 1) / (16 * T));
}
// 32 x 32 tiles (half the operand loads per flop) once 16 x 16 ones would give every SIMD
// four waves; below that more, smaller tiles hide the latency better.
bool mlp_wide(const MlpProduct& q) { return mlp_tiles(q, 1) >= 4096; }
unsigned mlp_blocks(const MlpProduct& q, int T) { return (unsigned)((mlp_tiles(q, T) + 3) / 4); }
}  // namespace

// Network 200 -> 256 -> 256 -> 200, batch 256: forward 3 launches of 9.8 us (6 of 30 before,
// 64 x 64 VALU tiles on 16 workgroups), backward 3 of 7.4 us beside the loss (10 of 30).
int mlp_forward(const MlpDev& m, int batch, const float* X, hipStream_t st) {
    const float* in = X;
    for (int l = 0; l < m.nlayers; ++l) {
        const int K = m.widths[l], N = m.widths[l + 1];
        float* H = m.act[l];
        const MlpProduct q{in, m.W[l], H, batch, N, K, K, N, m.b[l], l + 1 < m.nlayers ? 1 : 0, nullptr, nullptr};
        if (mlp_wide(q)) hipLaunchKernelGGL(k_mlp_forward<2>, dim3(mlp_blocks(q, 2)), dim3(256), 0, st, q);
        else hipLaunchKernelGGL(k_mlp_forward<1>, dim3(mlp_blocks(q, 1)), dim3(256), 0, st, q);
        ITCPD_HIP(hipGetLastError());
        in = H;
    }
    return ITCPD_OK;
}

// Gradients of the loss for one batch into m.gW / m.gb; loss -> *loss_dev (double)
int mlp_backward(const MlpDev& m, int batch, const float* X, const float* Yt, const float* mask,
                 double* loss_dev, hipStream_t st) {
    const int L = m.nlayers;
    const int Nout = m.widths[L];
    const int64_t nout = (int64_t)batch * Nout;
    float* dZ = m.dA;
    hipLaunchKernelGGL(k_mse_grad, dim3(nblk(nout)), dim3(256), 0, st, m.act[L - 1], Yt, mask, nout,
                       1.f / (float)batch, dZ, m.loss_part);
    ITCPD_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_sum_loss, dim3(1), dim3(256), 0, st, m.loss_part, (int)nblk(nout), loss_dev);
    ITCPD_HIP(hipGetLastError());
    for (int l = L - 1; l >= 0; --l) {
        const int K = m.widths[l], N = m.widths[l + 1];
        const float* in = l == 0 ? X : m.act[l - 1];
        float* dPrev = (dZ == m.dA) ? m.dB : m.dA;
        // dW_l = in^T dZ, db_l = colsum(dZ); dZ_{l-1} = (dZ W_l^T) .* relu'(act[l-1])
        const MlpProduct dw{in, dZ, m.gW[l], K, N, batch, K, N, nullptr, 0, nullptr, m.gb[l]};
        const MlpProduct dh{dZ, m.W[l], dPrev, batch, K, N, N, N, nullptr, 0, l > 0 ? m.act[l - 1] : nullptr, nullptr};
        const int T = mlp_wide(dw) && (l == 0 || mlp_wide(dh)) ? 2 : 1;
        const unsigned nw = mlp_blocks(dw, T), nh = l > 0 ? mlp_blocks(dh, T) : 0;
        if (T == 2) hipLaunchKernelGGL(k_mlp_backward<2>, dim3(nw + nh), dim3(256), 0, st, dw, dh, nw);
        else hipLaunchKernelGGL(k_mlp_backward<1>, dim3(nw + nh), dim3(256), 0, st, dw, dh, nw);
        ITCPD_HIP(hipGetLastError());
        dZ = dPrev;
    }
    return ITCPD_OK;
}

int launch_spa_candidates(int nsk, int D, int K, int ncand, const double* S, float* out, hipStream_t st) {
    hipLaunchKernelGGL(k_spa_candidates, dim3((unsigned)nsk), dim3(256), 0, st, S, D, K, ncand, out);
    ITCPD_HIP(hipGetLastError());
    return ITCPD_OK;
}

int mlp_adam(MlpDev& m, float lr, hipStream_t st) {
    m.step += 1;
    const float c1 = 1.f - powf(0.9f, (float)m.step);
    const float c2 = 1.f - powf(0.999f, (float)m.step);
    hipLaunchKernelGGL(k_adam, dim3(nblk(m.nparams)), dim3(256), 0, st, m.params, m.grads, m.adam_m,
                       m.adam_v, m.nparams, lr, c1, c2);
    ITCPD_HIP(hipGetLastError());
    return ITCPD_OK;
}

}  // namespace itcpd
