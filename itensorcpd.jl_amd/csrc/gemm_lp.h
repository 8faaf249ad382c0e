// The reduced-precision MTTKRP GEMMs for any tensor shape (included by mttkrp.hip):
//
//   left:  out(m, r) = sum_k T(m + M k) Kt(r, k)   (output rows contiguous in T)
//   right: out(n, r) = sum_k T(k + K n) Kt(r, k)   (reduction contiguous in T)
//
// with FP32 MFMA (v_mfma_f32_16x16x4_f32) or BF16x3 (v_mfma_f32_16x16x32_bf16 on hi hi +
// hi lo + lo hi, x = hi + lo, hi = bf16(x), lo = bf16(x - hi)).  Kt is the side's Khatri-Rao
// product from k_krp_lp: rank-major, rows padded with zeros to a multiple of 32 indices, in
// one part (FP32), two (BF16x3: hi, lo) or four.
//
// Four parts: BF16x3 where the factor, not the product, is what is rounded to two parts, x = (a_hi
// + a_lo) w with w the other modes' weight.  Rounding the product instead moves the CPD by a
// factor's rounding times the conditioning of its solves (up to 6.7e-5 over drawn order-4
// problems, of which 6.6e-5 is the factor's rounding against 64 bits).  The parts are h, m, r
// of x with h = bf16(a_hi w), and l = bf16(a_hi w - h): T_hi (h + m + r) + T_lo (h + l), the
// tensor's lo part meeting a_hi alone.
//
// As in gemm64.h each tensor element goes from global memory to the registers of the one
// wave that uses it, from addresses that are always valid, with the next stage's loads issued
// before the current one's MFMAs.  A stage is 16 reduction indices (FP32) or 32 (BF16x3);
// lane (c, g) takes the E = 4 or 8 consecutive ones from E g on, a 16-byte run of each of
// its rows of Kt.  The left form reads VEC consecutive output rows at each index, the right
// form an E-element run of each of its columns.  The FP32 accumulators are added into FP64
// ones every stage (FP32) or every 128 indices (BF16x3, whose parts round at 2^-18).  FP32, the
// relative error of M on Gaussian data and the GEMMs' times below: 16 indices 7.8e-8, 243 / 281;
// 8 indices 5.9e-8, 279 / 306; 32 1.05e-7, 250 / 301; 128 2.0e-7, 253 / 298 (the LDS ring form's
// sums still run over 128).  MFMA 16x16x4
// step s takes k = k0 + 4 g + s; result: lane (c, g), register v holds rank 4 g + v, output c.
//
// Measured per launch (left / right, us) on 150 x 130 x 110 x 90 FP32-stored, rank 48: FP32
// 243 / 281, BF16x3 in four parts 397 / 429 (280 / 306 in two, where the fourfold operand is not
// read) against 741 / 994 and 1128 / 1534 for the masked register-staged kernels that these
// replace; 301 x 257 x 199 rank 40, FP32 35 / 40 (97 / 78).  Bound by the
// tensor's stream (0.77 GB, 127 us at 6.06 TB/s) and, in FP32, the matrix cores (122 us at 152
// TFLOP/s).
#pragma once
#include "gemm64.h"

namespace itcpd {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

// x = hi + lo with hi = bf16(x), lo = bf16(x - hi), for the 8 k-values of a lane.
__device__ __forceinline__ void split8(const float (&x)[8], bf8& hi, bf8& lo) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        hi[e] = (__bf16)x[e];
        lo[e] = (__bf16)(x[e] - (float)hi[e]);
    }
}

// N consecutive elements as floats, in the element's own alignment.
template <typename TT, int N>
__device__ __forceinline__ void ld_float(const TT* __restrict__ p, float* x) {
    if constexpr (N == 1) {
        x[0] = (float)p[0];
    } else if constexpr (sizeof(TT) == 8) {
#pragma unroll
        for (int q = 0; q < N / 2; ++q) {
            const dvu2 v = *reinterpret_cast<const dvu2*>(p + 2 * q);
            x[2 * q] = (float)v.x;
            x[2 * q + 1] = (float)v.y;
        }
    } else if constexpr (N == 2) {
        const fvu2 v = *reinterpret_cast<const fvu2*>(p);
        x[0] = v.x;
        x[1] = v.y;
    } else {
#pragma unroll
        for (int q = 0; q < N / 4; ++q) {
            const fvu4 v = *reinterpret_cast<const fvu4*>(p + 4 * q);
            x[4 * q] = v.x; x[4 * q + 1] = v.y; x[4 * q + 2] = v.z; x[4 * q + 3] = v.w;
        }
    }
}

// The Khatri-Rao operand of one rank row and stage, in KP parts.
template <int KP>
struct KrpRun {
    bf8 hi, lo, r, l;   // r, l: of four parts (h, m, r, l)
    __device__ __forceinline__ void load(const void* row, int64_t part, int64_t k) {
        const __bf16* p = reinterpret_cast<const __bf16*>(row) + k;
        hi = *reinterpret_cast<const bf8*>(p);
        lo = *reinterpret_cast<const bf8*>(p + part);
        if constexpr (KP == 4) {
            r = *reinterpret_cast<const bf8*>(p + 2 * part);
            l = *reinterpret_cast<const bf8*>(p + 3 * part);
        }
    }
};
template <>
struct KrpRun<1> {
    float v[4];
    __device__ __forceinline__ void load(const void* row, int64_t, int64_t k) {
        const f4 x = *reinterpret_cast<const f4*>(reinterpret_cast<const float*>(row) + k);
        v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
    }
};

template <int N>
__device__ __forceinline__ void lp_flush(f4 (&acc)[N], d4 (&tot)[N]) {
#pragma unroll
    for (int a = 0; a < N; ++a) {
#pragma unroll
        for (int v = 0; v < 4; ++v) tot[a][v] += (double)acc[a][v];
        acc[a] = (f4){0.f, 0.f, 0.f, 0.f};
    }
}

// One stage of Kt-rows x T, x[b] the lane's E values of output tile b: BF16x3 into acc, FP32
// through acc into tot.
template <int KP, int RB, int MB, int E>
__device__ __forceinline__ void lp_stage(const KrpRun<KP> (&kr)[RB], const float (&x)[MB][E], f4 (&acc)[RB * MB],
                                         d4 (&tot)[RB * MB]) {
    if constexpr (KP > 1) {
#pragma unroll
        for (int b = 0; b < MB; ++b) {
            bf8 bh, bl;
            split8(x[b], bh, bl);
#pragma unroll
            for (int a = 0; a < RB; ++a) {
                f4 s = acc[a * MB + b];
                if constexpr (KP == 4) {
                    s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kr[a].r, bh, s, 0, 0, 0);
                    s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kr[a].l, bl, s, 0, 0, 0);
                }
                s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kr[a].lo, bh, s, 0, 0, 0);
                s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kr[a].hi, bl, s, 0, 0, 0);
                acc[a * MB + b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kr[a].hi, bh, s, 0, 0, 0);
            }
        }
    } else {
#pragma unroll
        for (int s = 0; s < E; ++s)
#pragma unroll
            for (int a = 0; a < RB; ++a)
#pragma unroll
                for (int b = 0; b < MB; ++b)
                    acc[a * MB + b] = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[a].v[s], x[b][s], acc[a * MB + b], 0, 0, 0);
        lp_flush<RB * MB>(acc, tot);
    }
}

// LEFT: outputs are rows (VEC of them consecutive per lane, the tile moved back to end at the
// last row when VEC > 1, which then needs outs >= 16 MB); else columns.  Grid: x rank blocks
// (the workgroups that share a tensor tile run together) times tiles, z reduction splits.
template <bool LEFT, typename TT, int KP, int RB, int MB, int KW, int VEC, int D, int OCC>
__global__ __launch_bounds__(256, OCC) void k_gemm_lp(const TT* __restrict__ T, int64_t outs, int64_t K,
                                                    const void* __restrict__ Kt, int64_t Kp, int64_t part,
                                                    int64_t stages_per_split, int ny, int R,
                                                    double* __restrict__ out, int64_t split_stride,
                                                    const DevCheck* __restrict__ chk) {
    constexpr bool BF = KP > 1;
    constexpr int E = BF ? 8 : 4, ST = 4 * E, FLUSH = 128 / ST;
    constexpr int NB = MB / VEC;
    if (chk->done) return;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int64_t tile = blockIdx.x / (unsigned)ny;
    const int r0 = (int)(blockIdx.x % (unsigned)ny) * (16 * RB);
    const int64_t m0 = (KW == 1 ? tile * 4 + wave : tile) * (16 * MB);
    if (KW == 1 && m0 >= outs) return;
    const int64_t nstages = (K + ST - 1) / ST;
    int64_t s0 = (int64_t)blockIdx.z * stages_per_split;
    int64_t s1 = s0 + stages_per_split < nstages ? s0 + stages_per_split : nstages;
    if (KW > 1) {
        const int64_t per = (s1 - s0 + KW - 1) / KW;
        s0 = s0 + wave * per < s1 ? s0 + wave * per : s1;
        s1 = s0 + per < s1 ? s0 + per : s1;
    }
    const int64_t mt = VEC == 1 || m0 + 16 * MB <= outs ? m0 : outs - 16 * MB;
    const TT* __restrict__ base[NB];   // LEFT: this lane's rows; else its columns
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int64_t m = mt + 16 * VEC * b + VEC * c;
        const int64_t mc = VEC > 1 || m < outs ? m : outs - 1;
        base[b] = T + (LEFT ? mc : K * mc);
    }
    const size_t esz = BF ? 2 : 4;
    const unsigned char* __restrict__ krow[RB];
#pragma unroll
    for (int a = 0; a < RB; ++a)
        krow[a] = reinterpret_cast<const unsigned char*>(Kt) + (size_t)(r0 + 16 * a + c) * (size_t)Kp * esz;

    f4 acc[RB * MB];
    d4 tot[RB * MB];
#pragma unroll
    for (int a = 0; a < RB * MB; ++a) {
        acc[a] = (f4){0.f, 0.f, 0.f, 0.f};
        tot[a] = (d4){0.0, 0.0, 0.0, 0.0};
    }
    KrpRun<KP> kr[D][RB];
    float x[D][MB][E];
    auto load = [&](int buf, int64_t st) {
        const int64_t k = st * ST + E * g;
        if constexpr (LEFT) {
#pragma unroll
            for (int e = 0; e < E; ++e)
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    float v[VEC];
                    ld_float<TT, VEC>(base[b] + (k + e) * outs, v);
#pragma unroll
                    for (int j = 0; j < VEC; ++j) x[buf][VEC * b + j][e] = v[j];
                }
        } else {
#pragma unroll
            for (int b = 0; b < NB; ++b) ld_float<TT, E>(base[b] + k, x[buf][b]);
        }
#pragma unroll
        for (int a = 0; a < RB; ++a) kr[buf][a].load(krow[a], part, k);
    };
    int flush = 0;
    auto compute = [&](int buf) {
        lp_stage<KP, RB, MB, E>(kr[buf], x[buf], acc, tot);
        if (BF && ++flush == FLUSH) {
            lp_flush<RB * MB>(acc, tot);
            flush = 0;
        }
    };
    const int64_t full = K / ST < s1 ? K / ST : s1;
    int64_t st = s0;
#pragma unroll
    for (int d = 0; d < D - 1; ++d)
        if (st + d < full) load(d, st + d);
    while (st < full) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (st >= full) break;
            if (st + D - 1 < full) load((d + D - 1) % D, st + D - 1);
            compute(d);
            ++st;
        }
    }
    // the last, partial stage: indices past the end read the last one and become zeros
    if (st < s1) {
        const int64_t k = st * ST + E * g;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const bool ok = k + e < K;
            const int64_t kc = ok ? k + e : K - 1;
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int j = 0; j < VEC; ++j) {
                    const float v = (float)(LEFT ? base[b][kc * outs + j] : base[b][kc]);
                    x[0][VEC * b + j][e] = ok ? v : 0.f;
                }
        }
#pragma unroll
        for (int a = 0; a < RB; ++a) kr[0][a].load(krow[a], part, k);
        lp_stage<KP, RB, MB, E>(kr[0], x[0], acc, tot);
    }
    if (BF) lp_flush<RB * MB>(acc, tot);

    if constexpr (KW > 1) {
        __shared__ d4 red[RB * MB][64];
        if (!sum_waves<RB * MB>(tot, red, wave, lane)) return;
    }
    double* o = out + (int64_t)blockIdx.z * split_stride;
#pragma unroll
    for (int a = 0; a < RB; ++a)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = r0 + 16 * a + 4 * g + v;
            if (r >= R) continue;
#pragma unroll
            for (int b = 0; b < MB; ++b) {
                const int64_t m = mt + 16 * VEC * (b / VEC) + VEC * c + b % VEC;
                if (VEC > 1 ? m >= m0 : m < outs) o[m + outs * r] = tot[a * MB + b][v];
            }
        }
}

}  // namespace itcpd
