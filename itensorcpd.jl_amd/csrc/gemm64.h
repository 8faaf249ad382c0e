// The MTTKRP GEMMs on FP64 MFMA for any tensor shape (included by mttkrp.hip).
//
//   left:  out(m, r) = sum_k T(m + M k) KRP(k, r)   (output rows contiguous in T)
//   right: out(n, r) = sum_k T(k + K n) KRP(k, r)   (reduction contiguous in T)
//
// with KRP(i + I0 j, r) = At0[i][r] W[j][r] formed on the way into the MFMA (NM = 2) or
// At0[k][r] alone (NM = 1, a side of one mode).  At0 is the rank-fastest factor of the
// side's first mode, W the rank-fastest factor of its second mode or, for a side of three
// modes and more, the rest weights that k_krp64 forms.  A Khatri-Rao product that is small
// beside the tensor is formed whole by k_krp64 instead, and the GEMM takes NM = 1.
//
// Both kernels are bound by the tensor's stream at low ranks and by the FP64 matrix cores
// above about 10 flops per byte (R ~ 40 for FP64 storage).  Each tensor element is used by
// one wave only, so it goes from global memory straight to the wave's registers: no LDS, no
// barrier in the loop, and any row length works, since a lane's addresses need no more than
// the element's own alignment.  A wave covers 16 MB outputs x 16 RB ranks; the loads of the
// next stage are issued before the MFMAs of the current one, from addresses that are always
// valid (rows and columns past the end read the last one, their results are not stored;
// reduction indices past the end are replaced by zeros after the load), so no branch stands
// between a load and its use.  With KW = 4 the four waves of a workgroup share one tile and
// split its reduction, adding up through LDS; with KW = 1 each has a tile of its own.
//
// Measured per launch (left / right, us), against the LDS ring and register-staged kernels
// that these replace, on tensors streamed at 6.06 TB/s by a plain sum and FP64 products at
// 72 TFLOP/s: 512^3 rank 16 205 / 251 (218 / 333), rank 32 212 / 287 (253 / 362), rank 48
// 262 / - (314), rank 64 344 / - (364); 301 x 257 x 199 rank 37 44 / 45 (115 / 97);
// 96 x 88 x 80 x 72 rank 16 74 / 79 (155 / 102); 23 x 21 x 20 x 19 x 18 rank 24 16 / 18
// (57 / 78); 200^3 FP32-stored rank 16 17 / 18 (40 / 31); 200^3 rank 150 77 / 86 (171 / 221).
// The right form is slower than the left one where columns lie a power of two apart (its 16
// columns meet in the same HBM channels: 512^3 rank 16 263 us, 171 us at a 240000-element
// column); above two rank blocks the FP64 matrix cores bound both.
//
// MFMA 16x16x4 f64: A lane (c, g) = A[c][g] (c = rank), B lane (c, g) = B[g][c] (c = output
// row or column), result v = D[g + 4 v][c].
#pragma once
#include "internal.h"

namespace itcpd {

typedef double dvu2 __attribute__((ext_vector_type(2), aligned(8)));
typedef float fvu2 __attribute__((ext_vector_type(2), aligned(4)));
typedef float fvu4 __attribute__((ext_vector_type(4), aligned(4)));

struct Krp64 {
    const double* At0;   // [I0][Rp]
    const double* W;     // [K / I0][Rp] (NM = 2)
    int64_t I0;
    int Rp;
};

// W[j][r] = prod_{q >= q0} At_q[digit_q(j)][r]: a side's whole Khatri-Rao product (q0 = 0)
// or the rest weights of its GEMM (q0 = 1), as one rank-fastest array.
static __global__ __launch_bounds__(256) void k_krp64(Side sd, int q0, int64_t n, int Rp, double* __restrict__ W,
                                               const DevCheck* __restrict__ chk) {
    const int64_t x = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (x >= n * Rp) return;
    const int64_t j = x / Rp;
    const int r = (int)(x - j * Rp);
    double w = 1.0;
    int64_t t = j;
    for (int q = q0; q < sd.nm; ++q) {
        const int64_t d = t % sd.dim[q];
        t /= sd.dim[q];
        w *= sd.fac[q][d * Rp + r];
    }
    if (chk->done) return;
    W[x] = w;
}

// Adds the KW waves' accumulators through LDS, in wave order pairs (2,3) -> (0,1), 1 -> 0;
// true in the wave that holds the sum.
template <int N>
__device__ __forceinline__ bool sum_waves(d4 (&acc)[N], d4 (*red)[64], int wave, int lane) {
    // red: N rows of 64, reused by every step
    if (wave == 3) {
#pragma unroll
        for (int a = 0; a < N; ++a) red[a][lane] = acc[a];
    }
    __syncthreads();
    if (wave == 2) {
#pragma unroll
        for (int a = 0; a < N; ++a) acc[a] += red[a][lane];
    }
    __syncthreads();
    if (wave == 1) {
#pragma unroll
        for (int a = 0; a < N; ++a) red[a][lane] = acc[a];
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
        for (int a = 0; a < N; ++a) acc[a] += red[a][lane];
    }
    __syncthreads();
    if (wave == 2) {
#pragma unroll
        for (int a = 0; a < N; ++a) red[a][lane] = acc[a];
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
        for (int a = 0; a < N; ++a) acc[a] += red[a][lane];
    }
    return wave == 0;
}

// VEC consecutive elements, in the element's own alignment.
template <typename TT, int VEC>
__device__ __forceinline__ void ld_vec(const TT* __restrict__ p, double* x) {
    if constexpr (VEC == 1) {
        x[0] = (double)p[0];
    } else if constexpr (sizeof(TT) == 8) {
        const dvu2 v = *reinterpret_cast<const dvu2*>(p);
        x[0] = v.x;
        x[1] = v.y;
    } else {
        const fvu2 v = *reinterpret_cast<const fvu2*>(p);
        x[0] = (double)v.x;
        x[1] = (double)v.y;
    }
}

// Left GEMM.  U 4-steps per stage; lane (c, g) reads its rows at k = 4 step + g.  ny rank
// blocks along grid y, times the slabs of a batch: slab q is the M x K matrix at T + q M K,
// its output rows q M .. + M - 1.
template <typename TT, int NM, int RB, int MB, int U, int KW, int VEC, int OCC>
__global__ __launch_bounds__(256, OCC) void k_left(const TT* __restrict__ T, int64_t M, int64_t K, Krp64 kp,
                                                 int64_t steps_per_split, int ny, int R, double* __restrict__ out,
                                                 int64_t out_ld, int64_t split_stride,
                                                 const DevCheck* __restrict__ chk) {
    if (chk->done) return;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int64_t m0 = (KW == 1 ? (int64_t)blockIdx.x * 4 + wave : (int64_t)blockIdx.x) * (16 * MB);
    if (KW == 1 && m0 >= M) return;
    const int r0 = (int)(blockIdx.y % (unsigned)ny) * (16 * RB);
    const int64_t slab = blockIdx.y / (unsigned)ny;
    T += slab * M * K;
    out += slab * M;
    const int64_t nsteps = (K + 3) / 4;
    int64_t s0 = (int64_t)blockIdx.z * steps_per_split;
    int64_t s1 = s0 + steps_per_split < nsteps ? s0 + steps_per_split : nsteps;
    if (KW > 1) {
        const int64_t per = (s1 - s0 + KW - 1) / KW;
        s0 = s0 + wave * per < s1 ? s0 + wave * per : s1;
        s1 = s0 + per < s1 ? s0 + per : s1;
    }
    // this lane's rows: VEC = 2, the pairs mt + 32 b + 2 c, + 1 of a tile moved back to end at
    // the last row (M >= 16 MB); VEC = 1, rows m0 + 16 b + c, past the end the last one
    constexpr int NB = MB / VEC;
    const int64_t mt = VEC == 1 || m0 + 16 * MB <= M ? m0 : M - 16 * MB;
    int64_t row[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int64_t r = mt + 16 * VEC * b + VEC * c;
        row[b] = VEC == 2 || r < M ? r : M - 1;
    }
    const int Rp = kp.Rp;
    const double* __restrict__ Ak = kp.At0 + r0 + c;
    const double* __restrict__ Wk = kp.W + r0 + c;
    // (i, j) of this lane's reduction index, advanced by 4 per step
    int64_t kl = 4 * s0 + g;
    const uint32_t I0u = (uint32_t)kp.I0;
    uint32_t i = (uint32_t)kl, j = 0;
    if (NM == 2) {
        j = (uint32_t)(kl / kp.I0);
        i = (uint32_t)(kl - j * kp.I0);
    }
    auto advance = [&]() {
        kl += 4;
        i += 4;
        if (NM == 2) {
            const bool over = i >= I0u;
            i -= over ? I0u : 0;
            j += over ? 1 : 0;
            if (I0u < 4)
                while (i >= I0u) { i -= I0u; ++j; }
        }
    };

    d4 acc[RB * MB];
#pragma unroll
    for (int a = 0; a < RB * MB; ++a) acc[a] = (d4){0.0, 0.0, 0.0, 0.0};

    double ta[2][U][MB], ka[2][U][RB], wa[NM == 2 ? 2 : 1][U][RB];
    // requests a stage: U steps from this lane's position (all of them below s1)
    auto load = [&](int buf) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const TT* __restrict__ Tk = T + kl * M;
#pragma unroll
            for (int b = 0; b < NB; ++b) ld_vec<TT, VEC>(Tk + row[b], &ta[buf][u][VEC * b]);
#pragma unroll
            for (int a = 0; a < RB; ++a) ka[buf][u][a] = Ak[(int64_t)i * Rp + 16 * a];
            if (NM == 2) {
#pragma unroll
                for (int a = 0; a < RB; ++a) wa[buf][u][a] = Wk[(int64_t)j * Rp + 16 * a];
            }
            advance();
        }
    };
    auto compute = [&](int buf) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            double kv[RB];
#pragma unroll
            for (int a = 0; a < RB; ++a) kv[a] = NM == 2 ? ka[buf][u][a] * wa[buf][u][a] : ka[buf][u][a];
#pragma unroll
            for (int a = 0; a < RB; ++a)
#pragma unroll
                for (int b = 0; b < MB; ++b)
                    acc[a * MB + b] = mfma_f64(kv[a], ta[buf][u][b], acc[a * MB + b]);
        }
    };
    // whole stages of in-range indices, two register buffers
    const int64_t full = K / 4 < s1 ? K / 4 : s1;   // steps below `full` have all four indices
    int64_t nst = full > s0 ? (full - s0) / U : 0;
    int64_t done = s0 + nst * U;
    if (nst > 0) {
        load(0);
        while (true) {
            if (nst > 1) load(1);
            compute(0);
            if (--nst == 0) break;
            if (nst > 1) load(0);
            compute(1);
            if (--nst == 0) break;
        }
    }
    // the remaining steps one at a time, indices past the end zeroed
    for (; done < s1; ++done) {
        const bool ok = kl < K;
        const int64_t kc = ok ? kl : K - 1, ic = ok ? i : 0, jc = ok ? j : 0;
        double tv[MB], kv[RB];
#pragma unroll
        for (int b = 0; b < NB; ++b) ld_vec<TT, VEC>(T + kc * M + row[b], &tv[VEC * b]);
#pragma unroll
        for (int a = 0; a < RB; ++a) {
            kv[a] = Ak[ic * Rp + 16 * a];
            if (NM == 2) kv[a] *= Wk[jc * Rp + 16 * a];
        }
#pragma unroll
        for (int b = 0; b < MB; ++b) tv[b] = ok ? tv[b] : 0.0;
#pragma unroll
        for (int a = 0; a < RB; ++a) kv[a] = ok ? kv[a] : 0.0;
#pragma unroll
        for (int a = 0; a < RB; ++a)
#pragma unroll
            for (int b = 0; b < MB; ++b) acc[a * MB + b] = mfma_f64(kv[a], tv[b], acc[a * MB + b]);
        advance();
    }

    if constexpr (KW > 1) {
        __shared__ d4 red[RB * MB][64];
        if (!sum_waves<RB * MB>(acc, red, wave, lane)) return;
    }
    double* o = out + (int64_t)blockIdx.z * split_stride;
#pragma unroll
    for (int a = 0; a < RB; ++a)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = r0 + 16 * a + g + 4 * v;
            if (r >= R) continue;
#pragma unroll
            for (int b = 0; b < MB; ++b) {
                const int64_t m = mt + 16 * VEC * (b / VEC) + VEC * c + b % VEC;
                if (VEC == 2 ? m >= m0 : m < M) o[m + out_ld * r] = acc[a * MB + b][v];
            }
        }
}

// The four elements of a column that a lane takes of a stage, in the element's own
// alignment: RUN = 4 consecutive ones, or RUN = 2 pairs eight apart.
template <typename TT, int RUN>
__device__ __forceinline__ void ld_run4(const TT* __restrict__ p, double (&x)[4]) {
    if constexpr (sizeof(TT) == 4 && RUN == 4) {
        const fvu4 a = *reinterpret_cast<const fvu4*>(p);
        x[0] = (double)a.x; x[1] = (double)a.y; x[2] = (double)a.z; x[3] = (double)a.w;
    } else {
        ld_vec<TT, 2>(p, x);
        ld_vec<TT, 2>(p + (RUN == 4 ? 2 : 8), x + 2);
    }
}

// Right GEMM.  A stage is 16 consecutive reduction indices; lane (c, g) reads four of them,
// k = k0 + RUN g + koff(s), of columns n0 + 16 b + c (the four g's of one load together a
// whole run of 16 RUN or 8 RUN bytes of each column) for MFMA s = 0..3.  REST: 0 one mode; 1 two modes with I0 % 16 == 0 (a stage
// lies in one j); 2 two modes, any I0.
template <typename TT, int REST, int RB, int MB, int KW, int RUN, int OCC>
__global__ __launch_bounds__(256, OCC) void k_right(const TT* __restrict__ T, int64_t N, int64_t K, Krp64 kp,
                                                  int64_t stages_per_split, int R, double* __restrict__ out,
                                                  int64_t split_stride, const DevCheck* __restrict__ chk) {
    if (chk->done) return;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int64_t n0 = (KW == 1 ? (int64_t)blockIdx.x * 4 + wave : (int64_t)blockIdx.x) * (16 * MB);
    if (KW == 1 && n0 >= N) return;
    const int r0 = blockIdx.y * (16 * RB);
    const int64_t nstages = (K + 15) / 16;
    int64_t s0 = (int64_t)blockIdx.z * stages_per_split;
    int64_t s1 = s0 + stages_per_split < nstages ? s0 + stages_per_split : nstages;
    if (KW > 1) {
        const int64_t per = (s1 - s0 + KW - 1) / KW;
        s0 = s0 + wave * per < s1 ? s0 + wave * per : s1;
        s1 = s0 + per < s1 ? s0 + per : s1;
    }
    const TT* __restrict__ col[MB];
#pragma unroll
    for (int b = 0; b < MB; ++b) {
        const int64_t n = n0 + 16 * b + c;
        col[b] = T + K * (n < N ? n : N - 1);
    }
    const int Rp = kp.Rp;
    const int64_t I0 = kp.I0;
    const uint32_t I0u = (uint32_t)I0;
    const double* __restrict__ Ak = kp.At0 + r0 + c;
    const double* __restrict__ Wk = kp.W + r0 + c;
    auto koff = [](int s) { return RUN == 4 ? s : 8 * (s >> 1) + (s & 1); };
    int64_t kl = 16 * s0 + RUN * g;   // this lane's first index of the next stage
    uint32_t i = (uint32_t)kl, j = 0;
    if (REST) {
        j = (uint32_t)(kl / I0);
        i = (uint32_t)(kl - j * I0);
    }
    // (i, j) of an index at most 16 past one with i < I0
    auto wrap = [&](uint32_t& ii, uint32_t& jj) {
        const bool over = ii >= I0u;
        ii -= over ? I0u : 0;
        jj += over ? 1 : 0;
        if (I0u < 16)
            while (ii >= I0u) { ii -= I0u; ++jj; }
    };
    auto advance = [&]() {
        kl += 16;
        i += 16;
        if (REST) wrap(i, j);
    };

    d4 acc[RB * MB];
#pragma unroll
    for (int a = 0; a < RB * MB; ++a) acc[a] = (d4){0.0, 0.0, 0.0, 0.0};

    constexpr int WS = REST == 2 ? 4 : 1;   // weight rows per stage and lane
    double ta[2][MB][4], ka[2][4][RB], wa[REST ? 2 : 1][WS][RB];
    auto load = [&](int buf) {
#pragma unroll
        for (int b = 0; b < MB; ++b) ld_run4<TT, RUN>(col[b] + kl, ta[buf][b]);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            uint32_t is = i + koff(s), js = j;
            if (REST == 2) wrap(is, js);
#pragma unroll
            for (int a = 0; a < RB; ++a) ka[buf][s][a] = Ak[(int64_t)is * Rp + 16 * a];
            if (REST == 2 || (REST == 1 && s == 0)) {
#pragma unroll
                for (int a = 0; a < RB; ++a) wa[buf][s % WS][a] = Wk[(int64_t)js * Rp + 16 * a];
            }
        }
        advance();
    };
    auto compute = [&](int buf) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            double kv[RB];
#pragma unroll
            for (int a = 0; a < RB; ++a) kv[a] = REST ? ka[buf][s][a] * wa[buf][s % WS][a] : ka[buf][s][a];
#pragma unroll
            for (int a = 0; a < RB; ++a)
#pragma unroll
                for (int b = 0; b < MB; ++b)
                    acc[a * MB + b] = mfma_f64(kv[a], ta[buf][b][s], acc[a * MB + b]);
        }
    };
    const int64_t full = K / 16 < s1 ? K / 16 : s1;
    int64_t nst = full > s0 ? full - s0 : 0;
    int64_t done = s0 + nst;
    if (nst > 0) {
        load(0);
        while (true) {
            if (nst > 1) load(1);
            compute(0);
            if (--nst == 0) break;
            if (nst > 1) load(0);
            compute(1);
            if (--nst == 0) break;
        }
    }
    // the last, partial stage: elements one by one, indices past the end zeroed
    for (; done < s1; ++done) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int64_t k = kl + koff(s);
            const bool ok = k < K;
            const int64_t kc = ok ? k : K - 1;
            uint32_t is = ok ? i + koff(s) : 0, js = ok ? j : 0;
            if (REST) wrap(is, js);
            double tv[MB], kv[RB];
#pragma unroll
            for (int b = 0; b < MB; ++b) tv[b] = (double)col[b][kc];
#pragma unroll
            for (int a = 0; a < RB; ++a) {
                kv[a] = Ak[(int64_t)is * Rp + 16 * a];
                if (REST) kv[a] *= Wk[(int64_t)js * Rp + 16 * a];
            }
#pragma unroll
            for (int b = 0; b < MB; ++b) tv[b] = ok ? tv[b] : 0.0;
#pragma unroll
            for (int a = 0; a < RB; ++a) kv[a] = ok ? kv[a] : 0.0;
#pragma unroll
            for (int a = 0; a < RB; ++a)
#pragma unroll
                for (int b = 0; b < MB; ++b) acc[a * MB + b] = mfma_f64(kv[a], tv[b], acc[a * MB + b]);
        }
        advance();
    }

    if constexpr (KW > 1) {
        __shared__ d4 red[RB * MB][64];
        if (!sum_waves<RB * MB>(acc, red, wave, lane)) return;
    }
    double* o = out + (int64_t)blockIdx.z * split_stride;
#pragma unroll
    for (int a = 0; a < RB; ++a)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = r0 + 16 * a + g + 4 * v;
            if (r >= R) continue;
#pragma unroll
            for (int b = 0; b < MB; ++b) {
                const int64_t n = n0 + 16 * b + c;
                if (n < N) o[n + N * r] = acc[a * MB + b][v];
            }
        }
}

}  // namespace itcpd
