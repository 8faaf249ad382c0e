// MTTKRP as a dimension tree on FP64 MFMA (gfx950).
//
// The reference computes each M_n = T_(n) (KRP of the other factors) separately,
// one full contraction of T per rank slice (algebra/had_contract.jl:111-121).
// Here the modes are split into a left side [0, s) and a right side [s, N):
//   left  GEMM  P_L(mL, r) = sum_mR T(mL, mR) KRP_right(mR, r)   (output rows contiguous in T)
//   right GEMM  P_R(mR, r) = sum_mL T(mL, mR) KRP_left(mL, r)    (reduction contiguous in T)
// with T viewed as an ML x MR column-major matrix (mL = left multi-index, mode 0
// fastest).  The KRP operand is generated on the fly from the factors (gemm64.h).  A side
// with one mode yields its M directly; a side with several modes gets each M_n
// from its partial by a Hadamard-reduce against the side's other (current)
// factors.  T is read twice per sweep; at order 3 three times per two sweeps where the
// partials are shared across sweeps (launch_tree3_gemm).
#include "internal.h"
#include "factor64.h"
#include "gemm64.h"
#include "gemm_lp.h"

namespace itcpd {

typedef double dv2 __attribute__((ext_vector_type(2)));

// A mode's R <= 64 factorisation riding along with another launch: block x = 0 of
// the grid runs factor64_dev (block (0, 0, 0)) or exits; the launch's own work
// uses blockIdx.x - 1.  The factorisation reads only Grams, which the launches it
// rides do not touch.  Along the right GEMM only the unpivoted form rides (in the
// GEMM's LDS budget; finfo[3] = 1 when it certified the result); the partial-sum
// launch after it then runs the pivoted form only when finfo[3] is 0
// (fallback_only).
struct FactorJob {
    GramSet gs;
    int on, mode, R, fallback_only;
    double tol;
    double *Uperm, *Vinv, *invdiag, *W, *qtau, *ztau, *vwork;
    int *piv, *finfo, *jpvt;
};
// The factorisation block runs without testing the done flag: it writes only the
// row solves' inputs (V^-1, pivots, status), which the later kernels of a finished
// run ignore, and the test's round trip would precede its Gram loads.
__device__ __forceinline__ bool factor_block(const FactorJob& fj) {
    if (!fj.on || blockIdx.x != 0) return false;
    if (blockIdx.y == 0 && blockIdx.z == 0 && !(fj.fallback_only && fj.finfo[3] == 1))
        factor64_dev(fj.gs, fj.mode, fj.R, fj.tol, fj.Uperm, fj.Vinv, fj.invdiag, fj.piv, fj.finfo, fj.W,
                     fj.qtau, fj.ztau, fj.jpvt, fj.vwork, !fj.fallback_only);
    return true;
}

// ---- direct global->LDS loads: lane l of a wave writes 16 bytes at dst + 16 l
typedef __attribute__((address_space(3))) void lds_void_t;

__device__ __forceinline__ void lds_dma16(const void* src, unsigned char* dst) {
    __builtin_amdgcn_global_load_lds(src, (lds_void_t*)dst, 16, 0, 0);
}
// s_waitcnt: vmcnt <= n (n < 16), lgkmcnt = 0, expcnt not waited for
#define VM_WAIT(n) __builtin_amdgcn_s_waitcnt(0x0000 | ((n) & 0xf) | (0x7 << 4) | (0x0 << 8))

// ------------------------------------ reduced-precision GEMMs, LDS ring form
// For an FP32-stored tensor whose GEMM dimensions fit 256-row tiles and 32-index
// stages.  The side's Khatri-Rao product is formed once per GEMM by k_krp_lp:
// Kt(r, m) = prod_q A_q(digit_q(m), r) for m over the reduction side and r over
// the rank padded to 128, rank-major (m fastest), FP32 or BF16 hi followed by
// BF16 lo.  The GEMM is then plain:
//   left:  out(mL, r) = sum_mR T(mL, mR) Kt(r, mR)   (tile: 256 rows mL)
//   right: out(mR, r) = sum_mL T(mL, mR) Kt(r, mL)   (tile: 256 columns mR)
// A workgroup of 8 waves covers 256 rows / columns x 128 ranks; wave w owns the
// 64 rows / columns 64 (w & 3) .. and the 64 ranks 64 (w >> 2) ..: 4 x 4 MFMA
// tiles.  A stage is 32 consecutive reduction indices: the T tile (32 KB) and the
// Kt tile (128 ranks x 128 bytes) arrive in an LDS slot by direct global->LDS
// loads (lane l of a wave writes 16 bytes at slot offset + 16 l); stages q+1 and
// q+2 are in flight while stage q is computed.
//
// LDS layouts.  Rows of 128 bytes (a Kt rank row, or 32 indices of one T column
// in the right GEMM) are stored in pairs, 256-byte lines of 16 chunks: chunk q of
// row j sits at line j >> 1, position (8 (j & 1) + q) ^ ((j >> 1) & 15), so the
// 16 lanes that read chunk q of 16 consecutive rows hit 16 distinct bank groups.
// The left GEMM's T tile is 32 columns of 256 rows (1 KB each, unswizzled: 16
// lanes read 256 contiguous bytes).
//
// Lane (c, g) takes reduction indices 8g .. 8g+7 of a stage: for BF16x3 the 8
// k-values of one 16x16x32 MFMA, for FP32 eight 16x16x4 MFMAs (MFMA e takes
// k = 8g + e).  The right GEMM reads two 16-byte chunks of each of its rows; the
// left GEMM reads rows 4c .. 4c+3 of columns 8g .. 8g+7 (one 16-byte read per
// column), so its MFMA column c of tile b is row 4c + b.
constexpr int LPR_NS = 3;
constexpr int LPR_TBYTES = 32 * 1024;
constexpr int LPR_KBYTES = 128 * 128;
constexpr int LPR_SLOT = LPR_TBYTES + LPR_KBYTES;
constexpr int LPR_LDS = LPR_NS * LPR_SLOT;
constexpr int LPR_FLUSH = 4;

// byte offset of chunk q (16 bytes) of 128-byte row j in a paired-line region
__device__ __forceinline__ int lpr_chunk(int j, int q) {
    return (j >> 1) * 256 + 16 * ((((j & 1) << 3) | q) ^ ((j >> 1) & 15));
}

// KP parts of Mp x Rk: the value in FP32 (1), BF16 hi and lo (2), or h, m, r, l of gemm_lp.h (4).
template <int KP>
__global__ __launch_bounds__(256) void k_krp_lp(Side sd, int64_t M, int64_t Mp, int R, int Rk,
                                                void* __restrict__ Kt,
                                                const DevCheck* __restrict__ chk) {
    if (chk->done) return;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t part = Mp * Rk;
    if (idx >= part) return;
    const int r = (int)(idx / Mp);
    const int64_t m = idx - (int64_t)r * Mp;
    double a = 0.0, w = 1.0;   // the product; of four parts, the fastest mode's factor and the others' weight
    if (r < R && m < M) {
        int64_t t = m / sd.dim[0];
        a = sd.fac[0][m - t * sd.dim[0] + sd.dim[0] * r];
        for (int q = 1; q < sd.nm; ++q) {
            const int64_t d = t % sd.dim[q];
            t /= sd.dim[q];
            (KP == 4 ? w : a) *= sd.fac[q][d + sd.dim[q] * r];
        }
    }
    if constexpr (KP == 1) {
        reinterpret_cast<float*>(Kt)[idx] = (float)a;
    } else if constexpr (KP == 2) {
        __bf16* o = reinterpret_cast<__bf16*>(Kt);
        const float x = (float)a;
        const __bf16 hi = (__bf16)x;
        o[idx] = hi;
        o[part + idx] = (__bf16)(x - (float)hi);
    } else {
        __bf16* o = reinterpret_cast<__bf16*>(Kt);
        const float af = (float)a;
        const __bf16 ah = (__bf16)af, al = (__bf16)(af - (float)ah);
        const double wf = (double)(float)w, xh = (double)(float)ah * wf;
        const __bf16 h = (__bf16)(float)xh;
        const double rest = fma((double)(float)al, wf, xh) - (double)(float)h;
        const __bf16 mid = (__bf16)(float)rest;
        o[idx] = h;
        o[part + idx] = mid;
        o[2 * part + idx] = (__bf16)(float)(rest - (double)(float)mid);
        o[3 * part + idx] = (__bf16)(float)(xh - (double)(float)h);
    }
}

template <bool LEFT, bool BF>
__global__ __launch_bounds__(512, 1) void k_lp_ring(const float* __restrict__ T, int64_t ML,
                                                    const void* __restrict__ Kt, int64_t Mk,
                                                    int64_t kt_lo_off, int64_t kper, int64_t nstages,
                                                    int R, double* __restrict__ out, int64_t out_ld,
                                                    int64_t split_stride,
                                                    const DevCheck* __restrict__ chk) {
    if (chk->done) return;
    extern __shared__ __attribute__((aligned(16))) unsigned char ring[];
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int wq = wave & 3, wr = wave >> 2;
    const int64_t n0 = (int64_t)blockIdx.x * 256;
    const int r0 = blockIdx.y * 128;
    const int64_t s0 = (int64_t)blockIdx.z * kper;
    const int64_t s1 = s0 + kper < nstages ? s0 + kper : nstages;
    const int nst = (int)(s1 - s0);

    // lane's (row, chunk) in a 1 KB paired-line block: line 4 ins + (l >> 4), position l & 15
    const int lline = lane >> 4, lpos = lane & 15;
    // stage q into slot q % LPR_NS: wave w loads 4 KB of T and 2 KB of Kt
    auto issue = [&](int q) {
        const int64_t k0 = (s0 + q) * 32;
        unsigned char* slot = ring + (q % LPR_NS) * LPR_SLOT;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int ins = 4 * wave + u;
            if constexpr (LEFT) {
                lds_dma16(T + (k0 + ins) * ML + n0 + 4 * lane, slot + ins * 1024);
            } else {
                const int L = 4 * ins + lline, P = lpos ^ (L & 15);
                const int j = 2 * L + (P >> 3), qc = P & 7;
                lds_dma16(T + (n0 + j) * ML + k0 + 4 * qc, slot + ins * 1024);
            }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int ins = 2 * wave + u;
            const int L = 4 * ins + lline, P = lpos ^ (L & 15);
            const int j = 2 * L + (P >> 3), qc = P & 7;
            const void* src;
            if constexpr (BF)
                src = reinterpret_cast<const __bf16*>(Kt) + (qc >= 4 ? kt_lo_off : 0) +
                      (int64_t)(r0 + j) * Mk + k0 + 8 * (qc & 3);
            else
                src = reinterpret_cast<const float*>(Kt) + (int64_t)(r0 + j) * Mk + k0 + 4 * qc;
            lds_dma16(src, slot + LPR_TBYTES + ins * 1024);
        }
    };

    // FP32: the FP32 accumulators are added into FP64 ones every LPR_FLUSH stages, so
    // no FP32 sum runs over more than 128 reduction indices (32 MFMA accumulations)
    f4 acc[4][4];
    double tot[4][4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            acc[a][b] = (f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int v = 0; v < 4; ++v) tot[a][b][v] = 0.0;
        }

    for (int q = 0; q < LPR_NS - 1 && q < nst; ++q) issue(q);
    for (int q = 0; q < nst; ++q) {
        // this wave's loads of stage q are done once at most the 6 of stage q+1 pend
        if (q + 1 < nst) VM_WAIT(6);
        else VM_WAIT(0);
        __asm__ volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __asm__ volatile("" ::: "memory");
        if (q + LPR_NS - 1 < nst) issue(q + LPR_NS - 1);
        const unsigned char* slot = ring + (q % LPR_NS) * LPR_SLOT;
        const unsigned char* kb = slot + LPR_TBYTES;
        float tv[4][8];
        if constexpr (LEFT) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const f4 x = *reinterpret_cast<const f4*>(slot + (8 * g + e) * 1024 + (64 * wq + 4 * c) * 4);
                tv[0][e] = x.x; tv[1][e] = x.y; tv[2][e] = x.z; tv[3][e] = x.w;
            }
        } else {
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int j = 64 * wq + 16 * b + c;
                const f4 x0 = *reinterpret_cast<const f4*>(slot + lpr_chunk(j, 2 * g));
                const f4 x1 = *reinterpret_cast<const f4*>(slot + lpr_chunk(j, 2 * g + 1));
                tv[b][0] = x0.x; tv[b][1] = x0.y; tv[b][2] = x0.z; tv[b][3] = x0.w;
                tv[b][4] = x1.x; tv[b][5] = x1.y; tv[b][6] = x1.z; tv[b][7] = x1.w;
            }
        }
        if constexpr (BF) {
            bf8 khi[4], klo[4];
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const int j = 64 * wr + 16 * a + c;
                khi[a] = *reinterpret_cast<const bf8*>(kb + lpr_chunk(j, g));
                klo[a] = *reinterpret_cast<const bf8*>(kb + lpr_chunk(j, 4 + g));
            }
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                bf8 bh, bl;
                split8(tv[b], bh, bl);
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(klo[a], bh, acc[a][b], 0, 0, 0);
                    acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(khi[a], bl, acc[a][b], 0, 0, 0);
                    acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(khi[a], bh, acc[a][b], 0, 0, 0);
                }
            }
        } else {
            float kv[4][8];
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const int j = 64 * wr + 16 * a + c;
                const f4 x0 = *reinterpret_cast<const f4*>(kb + lpr_chunk(j, 2 * g));
                const f4 x1 = *reinterpret_cast<const f4*>(kb + lpr_chunk(j, 2 * g + 1));
                kv[a][0] = x0.x; kv[a][1] = x0.y; kv[a][2] = x0.z; kv[a][3] = x0.w;
                kv[a][4] = x1.x; kv[a][5] = x1.y; kv[a][6] = x1.z; kv[a][7] = x1.w;
            }
#pragma unroll
            for (int e = 0; e < 8; ++e)
#pragma unroll
                for (int a = 0; a < 4; ++a)
#pragma unroll
                    for (int b = 0; b < 4; ++b)
                        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[a][e], tv[b][e], acc[a][b], 0, 0, 0);
            if ((q & (LPR_FLUSH - 1)) == LPR_FLUSH - 1 || q + 1 == nst) {
#pragma unroll
                for (int a = 0; a < 4; ++a)
#pragma unroll
                    for (int b = 0; b < 4; ++b) {
#pragma unroll
                        for (int v = 0; v < 4; ++v) tot[a][b][v] += (double)acc[a][b][v];
                        acc[a][b] = (f4){0.f, 0.f, 0.f, 0.f};
                    }
            }
        }
    }

    double* o = out + (int64_t)blockIdx.z * split_stride;
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = r0 + 64 * wr + 16 * a + 4 * g + v;
            if (r >= R) continue;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int64_t row = LEFT ? n0 + 64 * wq + 4 * c + b : n0 + 64 * wq + 16 * b + c;
                o[row + out_ld * r] = BF ? (double)acc[a][b][v] : tot[a][b][v];
            }
        }
}

// ------------------------------------------------------- Hadamard-reduce (ttv)
// Two waves a SIMD are asked for: the factorisation that rides along wants a register more than
// they leave, and with one wave the reduces of 200 x 200 x 150 take 21 us instead of 14.
//
// M(i, r) = sum_{a<A, b<B} P(a + A*i + A*In*b, r) * Wa(a, r) * Wb(b, r)
// Wa = product over the side's modes before `pos`, Wb over the modes after it
// (column-major factors).  P has leading dimension MS and is the sum of np partials, pstride
// apart, when its GEMM left them (added in increasing order, as k_sum_parts).
// w[k] *= the product over the side's modes [q0, q1) at the flattened index x[k] (x is used
// up), mode by mode so that the U loads of one are in flight together.
template <int U, typename I>
__device__ __forceinline__ void side_weights(const Side& sd, int q0, int q1, int r, I (&x)[U], double (&w)[U]) {
    for (int q = q0; q < q1; ++q) {
        const I d = (I)sd.dim[q];
        const double* __restrict__ f = sd.fac[q] + sd.dim[q] * r;
        double fv[U];
#pragma unroll
        for (int k = 0; k < U; ++k) {
            const I t = q + 1 < q1 ? x[k] / d : (I)0;
            fv[k] = f[x[k] - t * d];
            x[k] = t;
        }
#pragma unroll
        for (int k = 0; k < U; ++k) w[k] *= fv[k];
    }
}

// The side's fastest mode: thread per (i, r), split over b; 8 steps of b in flight.  Bound by
// HBM when large (512 x 512 x 64: 32 us, 4.2 TB/s).  When small, by the factorisation in the
// same launch: In = 20, B = 342, R = 24 takes 14.0 us.
template <bool PARTS, typename I>
__global__ __launch_bounds__(256, 2) void k_ttv_lead(const double* __restrict__ P, int np, int64_t pstride,
                                                  int64_t MS, int64_t In, int R, Side sd, I B, I b_per_split,
                                                  double* __restrict__ out, int64_t split_stride,
                                                  FactorJob fj, const DevCheck* __restrict__ chk) {
    if (factor_block(fj)) return;
    if (chk->done) return;
    const int64_t idx = ((int64_t)blockIdx.x - (fj.on ? 1 : 0)) * 256 + threadIdx.x;
    if (idx >= In * R) return;
    const int64_t i = idx % In;
    const int r = (int)(idx / In);
    const I b0 = (I)blockIdx.y * b_per_split;
    const I b1 = b0 + b_per_split < B ? b0 + b_per_split : B;
    const double* __restrict__ Pc = P + MS * r + i;
    double sum = 0.0;
    for (I b = b0; b < b1; b += 8) {
        I x[8];
        double pv[8], w[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {   // past the end: a valid element, not added
            x[k] = b + k < b1 ? b + k : b1 - 1;
            pv[k] = Pc[In * x[k]];
            w[k] = 1.0;
        }
        if constexpr (PARTS)
#pragma unroll 2
            for (int z = 1; z < np; ++z)
#pragma unroll
                for (int k = 0; k < 8; ++k) pv[k] += Pc[z * pstride + In * x[k]];
        side_weights<8, I>(sd, 1, sd.nm, r, x, w);
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (b + k < b1) sum += pv[k] * w[k];
    }
    out[(int64_t)blockIdx.y * split_stride + i + In * r] = sum;
}

// The other modes: one wave per JW consecutive i of one r; lanes stride over the flattened
// (a, b) with U steps and the JW rows' loads in flight together, and share the weights over
// the rows.  Bound as k_ttv_lead (512 x 512 x 64: 30 us).  Lanes over a alone, b one by one,
// left most lanes idle behind one load at a time where A is short: A = 20, In = 19, B = 18,
// R = 24 took 18.6 us, now 13.1 with its factorisation.
template <bool PARTS, int JW, int U, typename I>
__global__ __launch_bounds__(256, 2) void k_ttv_inner(const double* __restrict__ P, int np, int64_t pstride,
                                                   int64_t MS, int64_t In, int R, Side sd, int pos, I A, I B,
                                                   double* __restrict__ out, FactorJob fj,
                                                   const DevCheck* __restrict__ chk) {
    if (factor_block(fj)) return;
    if (chk->done) return;
    const int lane = threadIdx.x & 63;
    const int64_t wid = ((int64_t)blockIdx.x - (fj.on ? 1 : 0)) * 4 + (threadIdx.x >> 6);
    const int64_t ngi = (In + JW - 1) / JW;
    if (wid >= ngi * R) return;
    const int64_t i0 = (wid % ngi) * JW;
    const int r = (int)(wid / ngi);
    const double* __restrict__ Pr[JW];   // rows past the end read the last one
    double sum[JW];
#pragma unroll
    for (int j = 0; j < JW; ++j) {
        Pr[j] = P + MS * r + (int64_t)A * (i0 + j < In ? i0 + j : In - 1);
        sum[j] = 0.0;
    }
    const I n = A * B;
    const int64_t skip = (int64_t)A * (In - 1);   // x = a + A b is at x + skip b
    for (I x0 = lane; x0 < n; x0 += 64 * U) {
        I xa[U], xb[U];
        int64_t off[U];
        double w[U], pv[JW][U];
#pragma unroll
        for (int k = 0; k < U; ++k) {
            const I x = x0 + 64 * k < n ? x0 + 64 * k : n - 1;
            xb[k] = B > 1 ? x / A : (I)0;
            xa[k] = x - xb[k] * A;
            off[k] = x + skip * xb[k];
#pragma unroll
            for (int j = 0; j < JW; ++j) pv[j][k] = Pr[j][off[k]];
            w[k] = 1.0;
        }
        if constexpr (PARTS)
#pragma unroll 2
            for (int z = 1; z < np; ++z)
#pragma unroll
                for (int k = 0; k < U; ++k)
#pragma unroll
                    for (int j = 0; j < JW; ++j) pv[j][k] += Pr[j][off[k] + z * pstride];
        side_weights<U, I>(sd, 0, pos, r, xa, w);
        side_weights<U, I>(sd, pos + 1, sd.nm, r, xb, w);
#pragma unroll
        for (int k = 0; k < U; ++k)
            if (x0 + 64 * k < n) {
#pragma unroll
                for (int j = 0; j < JW; ++j) sum[j] += pv[j][k] * w[k];
            }
    }
#pragma unroll
    for (int j = 0; j < JW; ++j) {
        const double v = wave_sum_dpp(sum[j]);
        if (lane == 0 && i0 + j < In) out[i0 + j + In * r] = v;
    }
}

// out[x] = sum_{z < nz} parts[z*stride + x] (fixed order); with fj on, block 0
// runs that factorisation instead
__global__ __launch_bounds__(256, 2) void k_sum_parts(const double* __restrict__ parts, int nz,
                                                   int64_t stride, int64_t n,
                                                   double* __restrict__ out, FactorJob fj,
                                                   const DevCheck* __restrict__ chk) {
    if (factor_block(fj)) return;
    if (chk && chk->done) return;
    const int64_t x = ((int64_t)blockIdx.x - (fj.on ? 1 : 0)) * 256 + threadIdx.x;
    if (x >= n) return;
    out[x] = sum_parts_at(parts, stride, nz, x);
}

// Sum of squares of T: per-block partials, then one block in fixed order.
template <typename TT>
__global__ __launch_bounds__(256) void k_sumsq_part(const TT* __restrict__ T, int64_t n,
                                                    double* __restrict__ part) {
    __shared__ double red[256];
    double s = 0.0;
    const int64_t st = (int64_t)gridDim.x * 256;
    int64_t x = (int64_t)blockIdx.x * 256 + threadIdx.x;
    for (; x + 7 * st < n; x += 8 * st) {
        double v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = (double)T[x + k * st];
#pragma unroll
        for (int k = 0; k < 8; ++k) s += v[k] * v[k];
    }
    for (; x < n; x += st) {
        const double v = (double)T[x];
        s += v * v;
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}
__global__ void k_sum_small(const double* __restrict__ part, int n, double* __restrict__ out) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        double s = 0.0;
        for (int i = 0; i < n; ++i) s += part[i];
        out[0] = s;
    }
}

// ----------------------------------------------------------------- launchers
// A side's Khatri-Rao product (K rows) is formed whole when writing and reading it costs at
// most 1/16 of the tensor's bytes: the GEMM then has one operand load per rank block and
// step instead of two.
bool krp64_whole(const itcpd_plan* p, int64_t K) {
    return (double)K * (double)p->Rp * 8.0 * 16.0 <= (double)p->ML * (double)p->MR * (double)p->elt_bytes;
}
int64_t krp64_elems(const itcpd_plan* p) {
    int64_t rows = 0;
    for (int left = 0; left < 2; ++left) {   // the left GEMM reduces over the right side
        const int nm = left ? p->N - p->s : p->s;
        const int64_t K = left ? p->MR : p->ML, d0 = left ? p->dims[p->s] : p->dims[0];
        if (nm > 1 && krp64_whole(p, K)) rows = std::max(rows, K);
        else if (nm > 2) rows = std::max(rows, K / d0);
    }
    return rows * p->Rp;
}

namespace {

// ------------------------------------------- right GEMM, LDS ring form
// out(mR, r) = sum_{mL} T(mL, mR) KRP(mL, r) for a left side of one or two modes,
// mL = i + I0 rest, KRP(mL, r) = A0(i, r) w(rest, r) with w = 1 (one mode) or
// At1(rest, r) (two modes).  FP64 T, 64-column x 64-rank tiles.  A stage is SI
// (16 or 32) consecutive i of one rest: T (64 columns x SI i), A0 (64 ranks x SI
// i) -- an 8 SI-byte run per column / rank -- and the 64 weights of the rest land in
// an LDS slot through global_load_lds_dwordx4.  The 16-byte chunk q of run j is
// stored at chunk position q ^ (j mod SI/2), so the lanes that read chunk q of
// consecutive runs hit distinct banks.  Workgroup z takes stages [z kk_per,
// (z+1) kk_per) of the (rest, i) range.  Wave w computes rank block w & 3 for its
// share of the 16-column tiles; over a stage lane (c, g) covers i = (SI/4) g ..
// (SI/4) (g+1) - 1 (k-step s takes i = (SI/4) g + s for all four g).  Measured at
// 512^3, rank 64: four waves and two 32-index slots with two workgroups per CU
// (340 us) beat eight waves and four slots with one (389 us) -- a workgroup waiting
// at its barrier leaves the matrix cores to the other one.
template <int SI>
struct TrrGeom {
    static constexpr int RUN = SI * 8;             // bytes per column / rank run
    static constexpr int NCH = SI / 2;             // 16-byte chunks per run
    static constexpr int HALF = 64 * RUN;          // the T (or A0) part of a slot
    // + the 64 weights of the rest (the weight load's 64 lanes write 1 KB)
    static constexpr int SLOT = 2 * HALF + 1024;
};

// s_waitcnt vmcnt <= n (0 <= n < 16), lgkmcnt = 0
__device__ __forceinline__ void wait_vm(int n) {
    switch (n) {
        case 0: VM_WAIT(0); break;   case 1: VM_WAIT(1); break;   case 2: VM_WAIT(2); break;
        case 3: VM_WAIT(3); break;   case 4: VM_WAIT(4); break;   case 5: VM_WAIT(5); break;
        case 6: VM_WAIT(6); break;   case 7: VM_WAIT(7); break;   case 8: VM_WAIT(8); break;
        case 9: VM_WAIT(9); break;   case 10: VM_WAIT(10); break; case 11: VM_WAIT(11); break;
        case 12: VM_WAIT(12); break; case 13: VM_WAIT(13); break; case 14: VM_WAIT(14); break;
        default: VM_WAIT(15); break;
    }
}

// NW waves (8: two 16-column tiles per wave, 4: four), NS slots, SI-index stages
template <int NW, int NS, int SI>
__global__ __launch_bounds__(NW * 64, 4) void k_tr_ring(const double* __restrict__ T, int64_t ML,
                                                     int64_t MR, int64_t I0,
                                                     const double* __restrict__ A0,
                                                     const double* __restrict__ At1, int Rp,
                                                     int64_t kk_per, int64_t kk_total, int R,
                                                     double* __restrict__ out, int64_t split_stride,
                                                     int ntx, int ngy, FactorJob fj,
                                                     const DevCheck* __restrict__ chk) {
    using Gm = TrrGeom<SI>;
    constexpr int RPW = 64 / NW;          // runs of T (and of A0) loaded per wave
    constexpr int NCT = 16 / NW;          // 16-column tiles per wave
    constexpr int LPR = Gm::NCH;          // lanes per run in a load instruction
    constexpr int RPI = 64 / LPR;         // runs per load instruction
    constexpr int KS = SI / 4;            // MFMA k-steps per stage
    constexpr int CPL = KS / 2;           // 16-byte chunks a lane reads per run
    extern __shared__ __attribute__((aligned(16))) unsigned char ring[];
    if (fj.on && blockIdx.x == 0) {
        // the unpivoted factorisation of mode fj.mode (R > 32: whole 64-rank tiles) in this
        // launch's LDS (no done test, as factor_block)
        const bool ok = factor64_unpivoted<false>(fj.gs, fj.mode, fj.R, fj.tol, fj.Vinv, fj.finfo, reinterpret_cast<double*>(ring));
        if (threadIdx.x == 0) fj.finfo[3] = ok ? 1 : 0;
        return;
    }
    if (chk->done) return;
    // tile (x, y) and split z of this workgroup: 1D grid, x fastest
    const int64_t lin = (int64_t)blockIdx.x - fj.on;
    const int64_t bxl = lin % ntx;
    const int byl = (int)((lin / ntx) % ngy);
    const int64_t bzl = lin / ((int64_t)ntx * ngy);
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int rb = wave & 3, ch = wave >> 2;
    const int64_t n0 = bxl * 64;
    const int r0 = byl * 64;
    const int64_t nstg = I0 / SI;
    const int64_t q0 = bzl * kk_per;
    const int64_t q1 = q0 + kk_per < kk_total ? q0 + kk_per : kk_total;
    const int nst = (int)(q1 - q0);
    const bool weighted = At1 != nullptr;
    const int nper = 2 * (RPW / RPI) + ((weighted && wave == 0) ? 1 : 0);

    // (rest, SI-index chunk) of the next stage to request, advanced without divisions
    int64_t rest_is = q0 / nstg, ic_is = q0 - rest_is * nstg;
    // stage q into slot q % NS: wave w loads runs RPW w .. RPW (w+1) - 1 of T
    // (columns) and of A0 (ranks), RPI runs per instruction; wave 0 also the weights
    auto issue = [&](int q) {
        const int64_t rest = rest_is;
        const int64_t i0 = ic_is * SI;
        if (++ic_is == nstg) { ic_is = 0; ++rest_is; }
        unsigned char* slot = ring + (q % NS) * Gm::SLOT;
        const int jj = lane / LPR, pos = lane % LPR;
#pragma unroll
        for (int k = 0; k < RPW / RPI; ++k) {
            const int j0 = RPW * wave + RPI * k, j = j0 + jj;
            const int qc = pos ^ (j % LPR);
            lds_dma16(T + (n0 + j) * ML + I0 * rest + i0 + 2 * qc, slot + j0 * Gm::RUN);
            lds_dma16(A0 + (int64_t)(r0 + j) * I0 + i0 + 2 * qc, slot + Gm::HALF + j0 * Gm::RUN);
        }
        if (weighted && wave == 0)
            lds_dma16(At1 + rest * Rp + r0 + 2 * (lane & 31), slot + 2 * Gm::HALF);
    };

    // the operands of stage q from its slot: the A0 run of rank 16 rb + c (times the
    // rest weight) and the T runs of the wave's columns
    auto read_stage = [&](int q, double (&kv)[KS], double (&tv)[NCT][KS]) {
        const unsigned char* slot = ring + (q % NS) * Gm::SLOT;
        const double wr = weighted ? reinterpret_cast<const double*>(slot + 2 * Gm::HALF)[16 * rb + c] : 1.0;
        const unsigned char* kr = slot + Gm::HALF + (16 * rb + c) * Gm::RUN;
#pragma unroll
        for (int h = 0; h < CPL; ++h) {
            const dv2 x = *reinterpret_cast<const dv2*>(kr + 16 * ((CPL * g + h) ^ (c % LPR)));
            kv[2 * h] = x.x * wr;
            kv[2 * h + 1] = x.y * wr;
        }
#pragma unroll
        for (int b = 0; b < NCT; ++b) {
            const unsigned char* tr = slot + (16 * NCT * ch + 16 * b + c) * Gm::RUN;
#pragma unroll
            for (int h = 0; h < CPL; ++h) {
                const dv2 x = *reinterpret_cast<const dv2*>(tr + 16 * ((CPL * g + h) ^ (c % LPR)));
                tv[b][2 * h] = x.x;
                tv[b][2 * h + 1] = x.y;
            }
        }
    };
    // waits until this wave's loads of stage q have landed (at most those of the
    // stages requested after it pending, issued up to `last`), then the barrier
    auto arrive = [&](int q, int last) {
        wait_vm((last - q) * nper);
        __asm__ volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __asm__ volatile("" ::: "memory");
    };
    d4 acc[NCT];
#pragma unroll
    for (int b = 0; b < NCT; ++b) acc[b] = (d4){0.0, 0.0, 0.0, 0.0};
    auto mfmas = [&](const double (&kv)[KS], const double (&tv)[NCT][KS]) {
#pragma unroll
        for (int sk = 0; sk < KS; ++sk)
#pragma unroll
            for (int b = 0; b < NCT; ++b) acc[b] = mfma_f64(kv[sk], tv[b][sk], acc[b]);
    };
    for (int q = 0; q < NS - 1 && q < nst; ++q) issue(q);
    for (int q = 0; q < nst; ++q) {
        // this wave's loads of stage q are done once at most those of the later
        // stages already requested are pending
        const int later = (nst - 1 - q) < (NS - 2) ? (nst - 1 - q) : (NS - 2);
        arrive(q, q + later);
        if (q + NS - 1 < nst) issue(q + NS - 1);
        double kv[KS], tv[NCT][KS];
        read_stage(q, kv, tv);
        mfmas(kv, tv);
    }
    double* o = out + bzl * split_stride;
#pragma unroll
    for (int b = 0; b < NCT; ++b) {
        const int64_t col = n0 + 16 * NCT * ch + 16 * b + c;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = r0 + 16 * rb + g + 4 * v;
            if (r < R) o[col + MR * r] = acc[b][v];
        }
    }
}
// the configuration in use: waves per workgroup, LDS slots, indices per stage.
// Measured at 512^3 rank 64 (right GEMM per launch): 16-index stages in two slots,
// four workgroups per CU, 308 us; 32-index stages in two slots (two per CU) 312 us;
// 16 x 3 slots (three per CU) 317 us; 16 x 4 slots (two per CU) 334 us.  Register
// double buffering of the operands (the LDS reads of stage q+1 in flight under
// stage q's MFMAs) was slower in every form (+9 to +46 us).
constexpr int TRR_NW = 4, TRR_NS = 2, TRR_SI = 16;
constexpr int TRR_LDS = TRR_NS * TrrGeom<TRR_SI>::SLOT;
constexpr int TRR_WG_PER_CU = (160 * 1024) / TRR_LDS < 4 ? (160 * 1024) / TRR_LDS : 4;

struct Timed {
    itcpd_plan* p;
    hipEvent_t e1 = nullptr;
    Timed(itcpd_plan* pp, int kind, double flops, double bytes) : p(pp) {
        if (!p->profiling || (p->profile_only >= 0 && p->profile_only != kind)) return;
        if (p->profile_seen[kind]++ % p->profile_every != 0) return;
        hipEvent_t e0;
        if (hipEventCreate(&e0) != hipSuccess) return;
        if (hipEventCreate(&e1) != hipSuccess) { (void)hipEventDestroy(e0); e1 = nullptr; return; }
        (void)hipEventRecord(e0, p->stream);
        p->timer.ev.push_back(e0);
        p->timer.pending_flops.push_back(flops);
        p->timer.pending_bytes.push_back(bytes);
        p->timer.pending_kind.push_back(kind);
    }
    ~Timed() {
        if (!e1) return;
        (void)hipEventRecord(e1, p->stream);
        p->timer.ev.push_back(e1);
    }
};

Side make_side(itcpd_plan* p, int first, int nm, bool rank_fast) {
    Side sd{};
    sd.nm = nm;
    sd.first = first;
    for (int q = 0; q < nm; ++q) {
        sd.dim[q] = p->dims[first + q];
        sd.fac[q] = rank_fast ? p->At[first + q] : p->A[first + q];
    }
    return sd;
}

// Chooses the split-K factor so the grid has roughly `target` workgroups.
int64_t pick_split(int64_t base_wgs, int64_t kk_total, int64_t target, int64_t min_kk) {
    int64_t nz = 1;
    while (base_wgs * nz < target && kk_total / (nz * 2) >= min_kk) nz *= 2;
    return nz;
}

// The factorisation of `mode` as a job for one extra workgroup of another launch
// (off for R > 64, which takes the larger factor kernels, and for a V override).
FactorJob factor_job_for(itcpd_plan* p, int mode) {
    FactorJob fj{};
    fj.on = 0;
    if (mode < 0 || p->R > 64 || p->v_override) return fj;
    const int R = (int)p->R;
    fj.on = 1;
    fj.mode = mode;
    fj.R = R;
    fj.tol = 1e-6;
    fj.gs.N = p->N;
    for (int m = 0; m < p->N; ++m) fj.gs.G[m] = p->G[m];
    fj.Uperm = p->U;
    fj.Vinv = p->Upad;
    fj.invdiag = p->invdiag;
    fj.piv = p->piv;
    fj.finfo = p->finfo;
    fj.W = p->qr_aux;
    fj.qtau = fj.W + (size_t)R * R;
    fj.ztau = fj.qtau + R;
    fj.vwork = fj.ztau + R;
    fj.jpvt = p->piv + R;
    return fj;
}

// ---- the direct FP64 GEMMs (gemm64.h): configuration and launch
// Rank blocks of 16 per wave: the fewest blocks in all (padding included; within the Rp
// columns of the rank-fastest factors), weighed against the passes over T.
int gemm64_rb(int64_t R, int64_t Rp) {
    const int64_t nb = cdiv(R, 16);
    int best = 1;
    int64_t bestc = INT64_MAX;
    for (int rb = 5; rb >= 1; --rb) {
        const int64_t ny = cdiv(nb, rb), c = 2 * rb * ny + ny;
        if (16 * rb * ny <= Rp && c < bestc) { bestc = c; best = rb; }
    }
    return best;
}

// Split-K partials (n elements each) of a GEMM whose output side has nout modes that need no
// launch to sum them.  One mode: what the row solves sum as they read M.  More: what its
// Hadamard-reduces sum as they read the side, when a factorisation runs in their launch and
// hides it (R <= 64): at most 8, at most 32 MB in all.  Per sweep of
// 96x88x80x72 rank 16: one sum launch of 5.0 us instead of two of 6.6.
int64_t unsummed_parts(const itcpd_plan* p, int nout, int64_t n, int factor_mode) {
    if (nout == 1) return p->RT ? SOLVE_MAX_PARTS : 1;
    if (p->R > 64 || p->v_override || factor_mode >= 0) return 1;
    return std::max<int64_t>(1, std::min<int64_t>(8, ((int64_t)1 << 22) / n));
}

struct Gemm64Cfg {
    int MB, KW;
    int64_t per, nz;    // reduction units (4-steps / 16-index stages) per split, splits
};
// Tiles of 16 MB outputs.  With at least three workgroups of four such tiles per CU every
// wave takes its own tile and no reduction is split (KW = 1).  Otherwise the four waves of a
// workgroup split one tile's reduction, and so do nz workgroups, for the fewest rounds of
// two workgroups per CU per unit of work plus a charge for the partials' traffic and, above
// `unsummed` of them, 6 us (30 MB of the tensor's stream) for the launch that sums them; a wave
// keeps at least `min_units`.  16-output tiles are taken when the large ones cannot give
// every CU a workgroup, or when a slab has fewer rows than one (the large left tile is moved
// back to end at the slab's last row).  Measured, us (KW = 1 / KW = 4): 301 x (257) x 199
// rank 37, 398 workgroups, 60 / 42; 512 x (512) x 512 rank 64, 1024 workgroups, 338 / 347.
Gemm64Cfg gemm64_cfg(const itcpd_plan* p, int64_t M, int64_t slabs, int64_t units, int64_t min_units, int ny,
                     int big, int64_t unsummed) {
    Gemm64Cfg c{};
    const int64_t slots = 2 * (int64_t)p->num_cu;
    const int64_t out_elems = M * slabs * p->R;
    const bool fits = M >= 16 * big;
    if (fits && cdiv(cdiv(M, 16 * big), 4) * slabs * ny >= 3 * (int64_t)p->num_cu) return Gemm64Cfg{big, 1, units, 1};
    const double tbytes = (double)p->ML * (double)p->MR * (double)p->elt_bytes;
    for (int mb : {big, 1}) {
        if (mb == big && !fits) continue;
        const int64_t base = cdiv(M, 16 * mb) * slabs * ny;
        double best = 1e300;
        int64_t nz = 1;
        for (int64_t z = 1; z <= 512; ++z) {
            if (z > 1 && (units < 4 * min_units * z || (size_t)(z * out_elems) > p->parts_elems)) break;
            const double cost = (double)cdiv(base * z, slots) * (double)slots / (double)(base * z) +
                                (z > 1 ? 16.0 * (double)(z * out_elems) / tbytes : 0.0) + (z > unsummed ? 3e7 / tbytes : 0.0);
            if (cost < best - 1e-9) { best = cost; nz = z; }
        }
        c = Gemm64Cfg{mb, 4, cdiv(units, nz), nz};
        c.nz = cdiv(units, c.per);
        if (base * c.nz >= p->num_cu) break;
    }
    return c;
}

// The rank-fastest factors of a side as the kernels' Khatri-Rao operand; *nm = 1 or 2.
int krp64_of(itcpd_plan* p, const Side& sd, int64_t K, Krp64* kp, int* nm) {
    kp->At0 = sd.fac[0];
    kp->W = sd.fac[0];
    kp->I0 = sd.dim[0];
    kp->Rp = (int)p->Rp;
    *nm = sd.nm < 2 ? 1 : 2;
    if (sd.nm < 2) return ITCPD_OK;
    const bool whole = krp64_whole(p, K);
    if (!whole && sd.nm == 2) {
        kp->W = sd.fac[1];
        return ITCPD_OK;
    }
    const int64_t n = whole ? K : K / sd.dim[0];
    hipLaunchKernelGGL(k_krp64, dim3((unsigned)cdiv(n * p->Rp, 256)), dim3(256), 0, p->stream, sd, whole ? 0 : 1, n,
                       (int)p->Rp, p->Wrest, p->chk);
    ITCPD_HIP(hipGetLastError());
    kp->W = p->Wrest;
    if (whole) {
        kp->At0 = p->Wrest;
        kp->I0 = K;
        *nm = 1;
    }
    return ITCPD_OK;
}

// One direct GEMM: outs x R outputs (a batch of slabs of M rows for the left form),
// reduction length K over the operand kp.
struct Gemm64 {
    bool left;
    int64_t M, slabs, K;   // outputs per slab, slabs (1 for the right form)
    Krp64 kp;
    int nm, rb, ny;
    int64_t unsummed;      // splits whose partials no launch sums
    Gemm64Cfg c;
    double* out;
};

template <typename TT, int RB, int MB, int U, int KW, int VEC, int OCC>
void launch_left64(itcpd_plan* p, const Gemm64& q) {
    const int64_t nt = cdiv(q.M, 16 * MB);
    const dim3 grid((unsigned)(KW == 1 ? cdiv(nt, 4) : nt), (unsigned)(q.ny * q.slabs), (unsigned)q.c.nz);
    const int64_t ld = q.M * q.slabs;
    if (q.nm == 1)
        hipLaunchKernelGGL((k_left<TT, 1, RB, MB, U, KW, VEC, OCC>), grid, dim3(256), 0, p->stream,
                           (const TT*)p->T, q.M, q.K, q.kp, q.c.per, q.ny, (int)p->R, q.out, ld, ld * p->R, p->chk);
    else
        hipLaunchKernelGGL((k_left<TT, 2, RB, MB, U, KW, VEC, 2>), grid, dim3(256), 0, p->stream,
                           (const TT*)p->T, q.M, q.K, q.kp, q.c.per, q.ny, (int)p->R, q.out, ld, ld * p->R, p->chk);
}
template <typename TT, int RB, int MB, int KW>
void launch_right64(itcpd_plan* p, const Gemm64& q) {
    const int64_t nt = cdiv(q.M, 16 * MB);
    const dim3 grid((unsigned)(KW == 1 ? cdiv(nt, 4) : nt), (unsigned)q.ny, (unsigned)q.c.nz);
    const int64_t elems = q.M * p->R;
    if (q.nm == 1)
        hipLaunchKernelGGL((k_right<TT, 0, RB, MB, KW, 4, 2>), grid, dim3(256), 0, p->stream, (const TT*)p->T, q.M,
                           q.K, q.kp, q.c.per, (int)p->R, q.out, elems, p->chk);
    else if (q.kp.I0 % 16 == 0)
        hipLaunchKernelGGL((k_right<TT, 1, RB, MB, KW, 4, 2>), grid, dim3(256), 0, p->stream, (const TT*)p->T, q.M,
                           q.K, q.kp, q.c.per, (int)p->R, q.out, elems, p->chk);
    else
        hipLaunchKernelGGL((k_right<TT, 2, RB, MB, KW, 4, 2>), grid, dim3(256), 0, p->stream, (const TT*)p->T, q.M,
                           q.K, q.kp, q.c.per, (int)p->R, q.out, elems, p->chk);
}

// Tile heights (16-output tiles per wave) by rank blocks: what the accumulators and two
// stages of operands leave of the registers of two (RB >= 3) or four waves per SIMD.
constexpr int left64_big(int rb) { return rb <= 4 ? 4 : 2; }
constexpr int right64_big(int rb) { return rb <= 2 ? 4 : 2; }

template <typename TT, int RB>
void run_left64(itcpd_plan* p, const Gemm64& q) {
    constexpr int B = left64_big(RB), OCC = RB <= 2 ? 4 : 2;
    if (q.c.KW == 1) launch_left64<TT, RB, B, 2, 1, 2, OCC>(p, q);
    else if (q.c.MB == B) launch_left64<TT, RB, B, 2, 4, 2, OCC>(p, q);
    else launch_left64<TT, RB, 1, 4, 4, 1, 2>(p, q);
}
template <typename TT, int RB>
void run_right64(itcpd_plan* p, const Gemm64& q) {
    constexpr int B = right64_big(RB);
    if (q.c.KW == 1) launch_right64<TT, RB, B, 1>(p, q);
    else if (q.c.MB == B) launch_right64<TT, RB, B, 4>(p, q);
    else launch_right64<TT, RB, 1, 4>(p, q);
}
template <typename TT>
void dispatch_gemm64(itcpd_plan* p, const Gemm64& q) {
    if (q.left) {
        switch (q.rb) {
            case 1: return run_left64<TT, 1>(p, q);
            case 2: return run_left64<TT, 2>(p, q);
            case 3: return run_left64<TT, 3>(p, q);
            case 4: return run_left64<TT, 4>(p, q);
            default: return run_left64<TT, 5>(p, q);
        }
    }
    switch (q.rb) {
        case 1: return run_right64<TT, 1>(p, q);
        case 2: return run_right64<TT, 2>(p, q);
        case 3: return run_right64<TT, 3>(p, q);
        case 4: return run_right64<TT, 4>(p, q);
        default: return run_right64<TT, 5>(p, q);
    }
}
// Configures and launches q (M, slabs, K, kp, nm set): into dst, or into the split partials
// (q.c.nz > 1).
int run_gemm64(itcpd_plan* p, Gemm64& q, double* dst) {
    q.rb = gemm64_rb(p->R, p->Rp);
    q.ny = (int)cdiv(cdiv(p->R, 16), q.rb);
    q.c = q.left ? gemm64_cfg(p, q.M, q.slabs, cdiv(q.K, 4), 4, q.ny, left64_big(q.rb), q.unsummed)
                 : gemm64_cfg(p, q.M, 1, cdiv(q.K, 16), 2, q.ny, right64_big(q.rb), q.unsummed);
    q.out = q.c.nz > 1 ? p->parts : dst;
    Timed tm(p, q.left ? 0 : 1, 2.0 * (double)p->ML * (double)p->MR * (double)p->R,
             (double)p->ML * (double)p->MR * p->elt_bytes);
    if (p->elt_bytes == 8) dispatch_gemm64<double>(p, q);
    else dispatch_gemm64<float>(p, q);
    ITCPD_HIP(hipGetLastError());
    return ITCPD_OK;
}

// ---- the direct reduced-precision GEMMs (gemm_lp.h)
// Rank blocks of 16 per wave (at most 4, or 3 with four parts: FP32 sums, their FP64 totals and
// two stages of operands share 256 registers) and tile heights, as gemm64_rb / left64_big.
int lp_rb(int64_t R, int kp) {
    const int64_t nb = cdiv(R, 16);
    int best = 1;
    int64_t bestc = INT64_MAX;
    for (int rb = kp == 4 ? 3 : 4; rb >= 1; --rb) {
        const int64_t ny = cdiv(nb, rb), c = 2 * rb * ny + ny;
        if (c < bestc) { bestc = c; best = rb; }
    }
    return best;
}
constexpr int lp_big(int kp, int rb) { return rb <= (kp > 1 ? 2 : 3) ? 4 : 2; }

// Register stages: three where they fit (160^4-like shapes, FP32, us with two / three: rank 32
// 231 / 208, rank 64 397 / 360); at rank 48 the third costs more than it hides (252 / 263).
constexpr int lp_depth(int kp, int rb) { return kp == 1 && (rb == 2 || rb == 4) ? 3 : 2; }

struct GemmLp {
    bool left;
    int64_t outs, K, Kp, part;
    int kp, rb, ny;
    Gemm64Cfg c;
    double* out;
};
template <bool LEFT, typename TT, int KP, int RB, int MB, int KW, int VEC>
void launch_lp(itcpd_plan* p, const GemmLp& q) {
    const int64_t nt = cdiv(q.outs, 16 * MB);
    const dim3 grid((unsigned)((KW == 1 ? cdiv(nt, 4) : nt) * q.ny), 1, (unsigned)q.c.nz);
    hipLaunchKernelGGL((k_gemm_lp<LEFT, TT, KP, RB, MB, KW, VEC, lp_depth(KP, RB), 2>), grid, dim3(256), 0, p->stream, (const TT*)p->T,
                       q.outs, q.K, (const void*)p->Kt, q.Kp, q.part, q.c.per, q.ny, (int)p->R, q.out, q.outs * p->R,
                       p->chk);
}
template <bool LEFT, typename TT, int KP, int RB>
void run_lp(itcpd_plan* p, const GemmLp& q) {
    constexpr int B = lp_big(KP, RB), V = LEFT ? B : 1;
    if (q.c.KW == 1) launch_lp<LEFT, TT, KP, RB, B, 1, V>(p, q);
    else if (q.c.MB == B) launch_lp<LEFT, TT, KP, RB, B, 4, V>(p, q);
    else launch_lp<LEFT, TT, KP, RB, 1, 4, 1>(p, q);
}
template <bool LEFT, typename TT, int KP>
void dispatch_lp(itcpd_plan* p, const GemmLp& q) {
    switch (q.rb) {
        case 1: return run_lp<LEFT, TT, KP, 1>(p, q);
        case 2: return run_lp<LEFT, TT, KP, 2>(p, q);
        case 3: return run_lp<LEFT, TT, KP, 3>(p, q);
        default:
            if constexpr (KP < 4) run_lp<LEFT, TT, KP, 4>(p, q);
    }
}
template <bool LEFT, typename TT>
void dispatch_lp(itcpd_plan* p, const GemmLp& q) {
    if (q.kp == 1) dispatch_lp<LEFT, TT, 1>(p, q);
    else if (q.kp == 2) dispatch_lp<LEFT, TT, 2>(p, q);
    else dispatch_lp<LEFT, TT, 4>(p, q);
}
template <bool LEFT>
void dispatch_lp(itcpd_plan* p, const GemmLp& q) {
    p->elt_bytes == 4 ? dispatch_lp<LEFT, float>(p, q) : dispatch_lp<LEFT, double>(p, q);
}

}  // namespace

// Parts with at most this many partials are summed by the consumer (the solve).
static constexpr int MAX_CONSUMER_PARTS = 16;

int launch_sum_parts(itcpd_plan* p, const MSrc& ms, int64_t n, double* out, int factor_mode,
                     bool fallback_only) {
    FactorJob fj = factor_job_for(p, factor_mode);
    fj.fallback_only = fallback_only ? 1 : 0;
    hipLaunchKernelGGL(k_sum_parts, dim3((unsigned)(cdiv(n, 256) + fj.on)), dim3(256),
                       fj.on ? FACTOR64_LDS : 0, p->stream, ms.ptr, ms.nparts, ms.stride, n, out, fj, p->chk);
    ITCPD_HIP(hipGetLastError());
    if (factor_mode >= 0 && !fj.on) return launch_factor(p, factor_mode);
    return ITCPD_OK;
}

namespace {
// Hands split partials to the consumer, or sums them into dst when there are many.
// factor_mode >= 0: that mode's factorisation rides the partial-sum launch, else
// (no sum launched, R > 64) runs as its own launch after the producer.
//
// The partials of a side with more modes (consumer_sums false) stay as they are up to
// unsummed_parts.
int finish_parts(itcpd_plan* p, double* parts, int64_t nz, int64_t n, double* dst, MSrc* ms,
                 bool consumer_sums, int factor_mode = -1, bool fallback_only = false) {
    MSrc pm{parts, (int)nz, n};
    if (!consumer_sums) {
        const bool keep = nz > 1 && nz <= unsummed_parts(p, 2, n, factor_mode);
        p->side = keep ? pm : MSrc{dst, 1, n};
        if (keep) {
            *ms = pm;
            return ITCPD_OK;
        }
    }
    if (nz == 1 || (consumer_sums && nz <= MAX_CONSUMER_PARTS)) {
        *ms = nz == 1 ? MSrc{dst, 1, n} : pm;
        return factor_mode >= 0 ? launch_factor(p, factor_mode) : ITCPD_OK;
    }
    *ms = MSrc{dst, 1, n};
    return launch_sum_parts(p, pm, n, dst, factor_mode, fallback_only);
}
}  // namespace

// Left GEMM: rows = left multi-index (ML), reduction = right side.  Produces PL
// (s > 1) or the M of mode 0 (s == 1).
static int launch_ttv(itcpd_plan* p, const MSrc& P, int64_t MS, const Side& sd, int pos, MSrc* ms,
                      int factor_mode);
int launch_left_gemm_lp(itcpd_plan* p, MSrc* ms);
int launch_right_gemm_lp(itcpd_plan* p, MSrc* ms);

int launch_left_gemm_impl(itcpd_plan* p, MSrc* ms);
int launch_right_gemm_impl(itcpd_plan* p, MSrc* ms, int factor_mode);

// A GEMM launch, then (factor_mode >= 0) that mode's factorisation on the same
// stream: after the left GEMM as its own launch; with the FP64 right GEMM in an
// extra workgroup of the launch that sums its split-K partials, when there is one.
int launch_left_gemm(itcpd_plan* p, MSrc* ms, int factor_mode) {
    const int rc = launch_left_gemm_impl(p, ms);
    if (rc || factor_mode < 0) return rc;
    return launch_factor(p, factor_mode);
}
int launch_right_gemm(itcpd_plan* p, MSrc* ms, int factor_mode) {
    if (p->prec == ITCPD_FP64) return launch_right_gemm_impl(p, ms, factor_mode);
    const int rc = launch_right_gemm_lp(p, ms);
    if (rc || factor_mode < 0) return rc;
    return launch_factor(p, factor_mode);
}

// The direct FP64 GEMM of a side (gemm64.h), any shape.
static int launch_gemm64(itcpd_plan* p, MSrc* ms, bool left, int factor_mode) {
    const Side sd = left ? make_side(p, p->s, p->N - p->s, /*rank_fast=*/true)
                         : make_side(p, 0, p->s, /*rank_fast=*/true);
    const int nout = left ? p->s : p->N - p->s;   // modes on the output side
    Gemm64 q{};
    q.left = left;
    q.M = left ? p->ML : p->MR;
    q.slabs = 1;
    q.K = left ? p->MR : p->ML;
    int rc;
    if ((rc = krp64_of(p, sd, q.K, &q.kp, &q.nm))) return rc;
    q.unsummed = unsummed_parts(p, nout, q.M * p->R, factor_mode);
    double* dst = nout > 1 ? (left ? p->PL : p->PR) : p->M;
    if ((rc = run_gemm64(p, q, dst))) return rc;
    return finish_parts(p, p->parts, q.c.nz, q.M * p->R, dst, ms, nout == 1, factor_mode);
}

// ---- order 3, across sweeps: one contraction of T per two mode updates
// P_c(a, b, r) = sum over mode c of T A_c gives M of both other modes by Hadamard-reduces,
// and the updates cycle 0, 1, 2, 0, ..., so the partial formed for update u (contracting the
// mode updated last) also serves update u + 1: 3 passes over T per two sweeps instead of 4.
// Contracting mode 2 or mode 1 is a left GEMM (mode 1: a batch of K slabs), mode 0 a right
// one, each against one factor.  The price is one and a half partials written and three read
// per sweep instead of one and two: taken when half a pass over T (the tensor's read or
// 2 n R flops, at the rates the GEMMs reach) costs more than that.  A sweep with and
// without, us: 512^3 rank 64 653 / 759; 301 x 257 x 199 rank 37 178 / 201.
bool tree3_pays(const itcpd_plan* p) {
    if (p->N != 3 || p->prec != ITCPD_FP64) return false;
    const double n = (double)p->ML * (double)p->MR;
    const double pair = ((double)p->dims[0] * p->dims[1] + (double)p->dims[0] * p->dims[2] +
                         (double)p->dims[1] * p->dims[2]) / 3.0;
    const double gemm = std::max(n * p->elt_bytes / 5.2e12, 2.0 * n * 16.0 * (double)cdiv(p->R, 16) / 5.0e13);
    // the batched left GEMM has one grid row per slab and rank block
    if (p->dims[2] * cdiv(p->R, 16) > 65535) return false;
    return 0.5 * gemm > 1.5 * 8.0 * pair * (double)p->R / 4.5e12;
}
int64_t tree3_elems(const itcpd_plan* p) {
    return std::max(p->dims[0] * std::max(p->dims[1], p->dims[2]), p->dims[1] * p->dims[2]) * p->R;
}
int launch_tree3_gemm(itcpd_plan* p, int c) {
    Gemm64 q{};
    q.left = c != 0;
    q.slabs = c == 1 ? p->dims[2] : 1;
    q.M = c == 2 ? p->dims[0] * p->dims[1] : (c == 1 ? p->dims[0] : p->dims[1] * p->dims[2]);
    q.K = p->dims[c];
    q.kp = Krp64{p->At[c], p->At[c], p->dims[c], (int)p->Rp};
    q.nm = 1;
    q.unsummed = 1;
    int rc;
    if ((rc = run_gemm64(p, q, p->P3))) return rc;
    if (q.c.nz == 1) return ITCPD_OK;
    const int64_t n = q.M * q.slabs * p->R;
    return launch_sum_parts(p, MSrc{p->parts, (int)q.c.nz, n}, n, p->P3);
}
int launch_tree3_ttv(itcpd_plan* p, int mode, int c, MSrc* ms, int factor_mode) {
    Side sd{};
    sd.nm = 2;
    int pos = 0;
    for (int m = 0, q = 0; m < 3; ++m) {
        if (m == c) continue;
        if (m == mode) pos = q;
        sd.dim[q] = p->dims[m];
        sd.fac[q] = p->A[m];
        ++q;
    }
    return launch_ttv(p, MSrc{p->P3, 1, 0}, sd.dim[0] * sd.dim[1], sd, pos, ms, factor_mode);
}

int launch_left_gemm_impl(itcpd_plan* p, MSrc* ms) {
    if (p->prec != ITCPD_FP64) return launch_left_gemm_lp(p, ms);
    return launch_gemm64(p, ms, true, -1);
}

// Right GEMM: rows = right multi-index (MR), reduction = left side.  Produces PR
// (N-s > 1) or the M of mode N-1 (N-s == 1).
int launch_right_gemm_impl(itcpd_plan* p, MSrc* ms, int factor_mode) {
    const Side sd = make_side(p, 0, p->s, /*rank_fast=*/false);
    if (p->s <= 2 && p->elt_bytes == 8 && sd.dim[0] % TRR_SI == 0 && p->MR % 64 == 0 && p->Rp % 64 == 0) {
        // left side of one or two modes: the LDS ring form (TRR_WG_PER_CU workgroups
        // per CU), split over the (rest, i) stages to fill the chip
        const int64_t ntx = p->MR / 64;
        const int gy = (int)(p->Rp / 64);
        const int64_t kk_total = (sd.dim[0] / TRR_SI) * (p->ML / sd.dim[0]);
        const int64_t out_elems = p->MR * p->R;
        const bool consumer_sums = p->N - p->s == 1;
        // Split: one round of resident workgroups (a multiple of the tile count
        // when that fills the slots exactly), else the power-of-two split; with the
        // factorisation along, one slot's worth of tiles fewer.
        const int64_t tiles = ntx * gy;
        auto split_for = [&](int64_t slots) {
            int64_t nz = (slots % tiles == 0 && kk_total / (slots / tiles) >= 8)
                             ? slots / tiles
                             : pick_split(tiles, kk_total, slots, 8);
            if (nz > 1 && (size_t)(nz * out_elems) > p->parts_elems) nz = (int64_t)(p->parts_elems / out_elems);
            if (nz < 1) nz = 1;
            return cdiv(kk_total, cdiv(kk_total, nz));
        };
        const int64_t slots = (int64_t)p->num_cu * TRR_WG_PER_CU;   // workgroups resident at once
        // Mode s's unpivoted factorisation rides in workgroup 0 (in the GEMM's LDS
        // budget, all workgroups resident at once) when a partial-sum launch follows
        // to run the pivoted fallback.  Its dependent steps then overlap the GEMM.
        // With tiles for every slot nothing is split and no such launch follows.
        FactorJob fj = factor_job_for(p, factor_mode);
        if (slots <= tiles) fj.on = 0;
        int64_t nz = split_for(fj.on ? slots - tiles : slots);
        if (fj.on && !(nz > 1 && !(consumer_sums && nz <= MAX_CONSUMER_PARTS) && slots - tiles * nz >= 1)) {
            fj.on = 0;
            nz = split_for(slots);
        }
        const int64_t kk_per = cdiv(kk_total, nz);
        double* dst = (p->N - p->s > 1) ? p->PR : p->M;
        double* out = nz > 1 ? p->parts : dst;
        const size_t lds = fj.on ? std::max<size_t>((size_t)TRR_LDS, FACTOR64_UNPIV_LDS) : (size_t)TRR_LDS;
        {
            Timed tm(p, 1, 2.0 * (double)p->ML * (double)p->MR * (double)p->R,
                     (double)p->ML * (double)p->MR * p->elt_bytes);
            hipLaunchKernelGGL((k_tr_ring<TRR_NW, TRR_NS, TRR_SI>), dim3((unsigned)(fj.on + tiles * nz)),
                               dim3(TRR_NW * 64), lds,
                               p->stream, (const double*)p->T, p->ML, p->MR, sd.dim[0],
                               (const double*)sd.fac[0], p->s == 2 ? (const double*)p->At[1] : nullptr,
                               (int)p->Rp, kk_per, kk_total, (int)p->R, out, out_elems, (int)ntx, gy, fj,
                               p->chk);
            ITCPD_HIP(hipGetLastError());
        }
        return finish_parts(p, p->parts, nz, out_elems, dst, ms, consumer_sums, factor_mode, fj.on != 0);
    }
    return launch_gemm64(p, ms, false, factor_mode);
}

// The LDS ring form of a reduced-precision GEMM applies: FP32-stored T, 256-row
// (left) / 256-column (right) tiles, 32-index stages of the reduction, tiles for every CU
// within 8 splits, and a rank that is worth its 128-rank tiles, whose cost does not depend on
// the rank in them while the direct form's grows with every 16 ranks.  In FP32 it sums 128
// products before they go to FP64, the direct form 16.  Measured at 160^4,
// left GEMM, us (ring / direct): FP32 rank 32 1342 / 581, rank 64 1346 / 1169, rank 128 1372 /
// 2160; BF16x3 rank 16 530 / 491, rank 32 543 / 548, rank 64 545 / 1055.  512^3 rank 64, right
// GEMM (2 tiles): FP32 4268 / 276, BF16x3 1597 / 231.
static bool lp_ring_ok(const itcpd_plan* p, bool left, int prec) {
    const int64_t M = left ? p->ML : p->MR, K = left ? p->MR : p->ML;
    const int64_t nb = cdiv(p->R, 16), ny = cdiv(p->R, 128);
    return p->elt_bytes == 4 && M % 256 == 0 && K % 32 == 0 && M / 256 * ny * 8 >= p->num_cu &&
           nb >= (prec == ITCPD_BF16X3 ? 3 : 5) * ny;
}

// A side's Khatri-Rao product in Kt: kp parts of Rk rows (ranks, padded to the GEMM's blocks)
// of Kp elements (a multiple of 32).  Four parts (the factor is rounded, gemm_lp.h) unless the
// side is one mode, whose product is the factor, or the tensor is whole tiles of the ring form,
// which rounds the product: each shape keeps the rounding that its BF16x3 results have had.
struct LpKrp {
    int kp, Rk;
    int64_t Kp;
};
static LpKrp lp_krp(const itcpd_plan* p, bool left, int prec) {
    const int64_t M = left ? p->ML : p->MR, K = left ? p->MR : p->ML;
    const bool one = (left ? p->N - p->s : p->s) == 1, whole = p->elt_bytes == 4 && M % 256 == 0 && K % 32 == 0;
    LpKrp k;
    k.kp = prec != ITCPD_BF16X3 ? 1 : (one || whole ? 2 : 4);
    const int rb = lp_rb(p->R, k.kp);
    k.Rk = lp_ring_ok(p, left, prec) ? 128 * (int)cdiv(p->R, 128) : 16 * rb * (int)cdiv(cdiv(p->R, 16), rb);
    k.Kp = cdiv(K, 32) * 32;
    return k;
}
// for either precision: a plan keeps the buffer when it changes between them
int64_t lp_krp_elems(const itcpd_plan* p) {
    int64_t n = 0;
    for (int prec : {ITCPD_FP32, ITCPD_BF16X3})
        for (int left = 0; left < 2; ++left) {
            const LpKrp k = lp_krp(p, left != 0, prec);
            n = std::max(n, k.Kp * k.Rk * (k.kp == 4 ? 2 : 1));
        }
    return n;
}
static int launch_krp_lp(itcpd_plan* p, bool left, const LpKrp& k) {
    const Side sd = left ? make_side(p, p->s, p->N - p->s, /*rank_fast=*/false)
                         : make_side(p, 0, p->s, /*rank_fast=*/false);
    auto run = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3((unsigned)cdiv(k.Kp * k.Rk, 256)), dim3(256), 0, p->stream, sd,
                           left ? p->MR : p->ML, k.Kp, (int)p->R, k.Rk, (void*)p->Kt, p->chk);
    };
    if (k.kp == 1) run(k_krp_lp<1>);
    else if (k.kp == 2) run(k_krp_lp<2>);
    else run(k_krp_lp<4>);
    ITCPD_HIP(hipGetLastError());
    return ITCPD_OK;
}

static int launch_lp_ring(itcpd_plan* p, MSrc* ms, bool left) {
    const bool bf = p->prec == ITCPD_BF16X3;
    const int64_t M = left ? p->ML : p->MR;    // output rows
    const int64_t Mk = left ? p->MR : p->ML;   // reduction length
    const int ny = (int)cdiv(p->R, 128);
    const LpKrp kr = lp_krp(p, left, p->prec);
    const int64_t lo = kr.Kp * kr.Rk;   // hi to lo
    if (int rc = launch_krp_lp(p, left, kr)) return rc;

    // split-K factor: one workgroup per CU, so the fewest rounds per unit of work,
    // plus a small charge per partial for summing them
    const int64_t nstages = Mk / 32;
    const int64_t base = (M / 256) * ny;
    const int64_t out_elems = M * p->R;
    int64_t nz = 1;
    double best = 1e30;
    for (int64_t z = 1; z <= 8; ++z) {
        if (z > 1 && ((size_t)(z * out_elems) > p->parts_elems || nstages / z < 8)) break;
        const double cost = (double)cdiv(base * z, p->num_cu) / (double)z + (z > 1 ? 0.005 * (double)z : 0.0);
        if (cost < best - 1e-9) { best = cost; nz = z; }
    }
    const int64_t kper = cdiv(nstages, nz);
    nz = cdiv(nstages, kper);
    double* dst = left ? (p->s > 1 ? p->PL : p->M) : (p->N - p->s > 1 ? p->PR : p->M);
    double* out = nz > 1 ? p->parts : dst;
    {
        Timed tm(p, left ? 0 : 1, 2.0 * (double)p->ML * (double)p->MR * (double)p->R,
                 (double)p->ML * (double)p->MR * p->elt_bytes);
        const dim3 grid((unsigned)(M / 256), (unsigned)ny, (unsigned)nz);
        const float* T = (const float*)p->T;
        if (left && bf)
            hipLaunchKernelGGL((k_lp_ring<true, true>), grid, dim3(512), LPR_LDS, p->stream, T, p->ML,
                               (const void*)p->Kt, Mk, lo, kper, nstages, (int)p->R, out, M, out_elems, p->chk);
        else if (left)
            hipLaunchKernelGGL((k_lp_ring<true, false>), grid, dim3(512), LPR_LDS, p->stream, T, p->ML,
                               (const void*)p->Kt, Mk, lo, kper, nstages, (int)p->R, out, M, out_elems, p->chk);
        else if (bf)
            hipLaunchKernelGGL((k_lp_ring<false, true>), grid, dim3(512), LPR_LDS, p->stream, T, p->ML,
                               (const void*)p->Kt, Mk, lo, kper, nstages, (int)p->R, out, M, out_elems, p->chk);
        else
            hipLaunchKernelGGL((k_lp_ring<false, false>), grid, dim3(512), LPR_LDS, p->stream, T, p->ML,
                               (const void*)p->Kt, Mk, lo, kper, nstages, (int)p->R, out, M, out_elems, p->chk);
        ITCPD_HIP(hipGetLastError());
    }
    return finish_parts(p, p->parts, nz, out_elems, dst, ms, left ? p->s == 1 : p->N - p->s == 1);
}

// Reduced-precision forms of the two GEMMs (FP32 or BF16x3 arithmetic, FP64 output).
static int launch_gemm_lp(itcpd_plan* p, MSrc* ms, bool left) {
    if (lp_ring_ok(p, left, p->prec)) return launch_lp_ring(p, ms, left);
    GemmLp q{};
    q.left = left;
    q.outs = left ? p->ML : p->MR;
    q.K = left ? p->MR : p->ML;
    const LpKrp kr = lp_krp(p, left, p->prec);
    if (int rc = launch_krp_lp(p, left, kr)) return rc;
    q.kp = kr.kp;
    q.Kp = kr.Kp;
    q.part = kr.Kp * kr.Rk;
    const int nout = left ? p->s : p->N - p->s;
    q.rb = lp_rb(p->R, q.kp);
    q.ny = (int)cdiv(cdiv(p->R, 16), q.rb);
    q.c = gemm64_cfg(p, q.outs, 1, cdiv(q.K, q.kp > 1 ? 32 : 16), 2, q.ny, lp_big(q.kp, q.rb),
                     unsummed_parts(p, nout, q.outs * p->R, -1));
    double* dst = nout > 1 ? (left ? p->PL : p->PR) : p->M;
    q.out = q.c.nz > 1 ? p->parts : dst;
    {
        Timed tm(p, left ? 0 : 1, 2.0 * (double)p->ML * (double)p->MR * (double)p->R,
                 (double)p->ML * (double)p->MR * p->elt_bytes);
        left ? dispatch_lp<true>(p, q) : dispatch_lp<false>(p, q);
        ITCPD_HIP(hipGetLastError());
    }
    return finish_parts(p, p->parts, q.c.nz, q.outs * p->R, dst, ms, nout == 1);
}
int launch_left_gemm_lp(itcpd_plan* p, MSrc* ms) { return launch_gemm_lp(p, ms, true); }
int launch_right_gemm_lp(itcpd_plan* p, MSrc* ms) { return launch_gemm_lp(p, ms, false); }

int launch_side_ttv(itcpd_plan* p, int mode, MSrc* ms, int factor_mode) {
    const bool left = mode < p->s;
    const int first = left ? 0 : p->s;
    const Side sd = make_side(p, first, left ? p->s : p->N - p->s, /*rank_fast=*/false);
    return launch_ttv(p, p->side, left ? p->ML : p->MR, sd, mode - first, ms, factor_mode);
}

// M of the side's mode `pos` from the partial P (leading dimension MS) by a
// Hadamard-reduce.  With factor_mode >= 0 that mode's factorisation runs in an extra
// workgroup of the same launch when it can (R <= 64), else it is launched right after.
static int launch_ttv(itcpd_plan* p, const MSrc& P, int64_t MS, const Side& sd, int pos, MSrc* ms,
                      int factor_mode) {
    const int nm = sd.nm;
    int64_t A = 1, B = 1;
    for (int q = 0; q < pos; ++q) A *= sd.dim[q];
    for (int q = pos + 1; q < nm; ++q) B *= sd.dim[q];
    const int64_t In = sd.dim[pos];
    const int64_t nout = In * p->R;
    const FactorJob fj = factor_job_for(p, factor_mode);
    const size_t lds = fj.on ? FACTOR64_LDS : 0;
    const bool small = A * B < ((int64_t)1 << 30);   // 32-bit digits
    int rc = ITCPD_OK;
    if (pos == 0) {
        int64_t nz = 1;
        const int64_t blocks = cdiv(nout, 256);
        // behind the side's own partials, which the next modes still read
        const int64_t taken = P.nparts > 1 ? P.nparts * P.stride : 0;
        double* const parts = p->parts + taken;
        while (blocks * nz < 2048 && B / (nz * 2) >= 16 && (size_t)(taken + nz * 2 * nout) <= p->parts_elems &&
               nz * 2 <= MAX_CONSUMER_PARTS)
            nz *= 2;
        const int64_t bper = cdiv(B, nz);
        nz = cdiv(B, bper);
        double* out = nz > 1 ? parts : p->M;
        const dim3 grid((unsigned)(blocks + fj.on), (unsigned)nz);
        auto run = [&](auto kern, auto b, auto per) {
            hipLaunchKernelGGL(kern, grid, dim3(256), lds, p->stream, P.ptr, P.nparts, P.stride, MS, In, (int)p->R, sd,
                               b, per, out, nout, fj, p->chk);
        };
        if (!small) run(k_ttv_lead<true, int64_t>, B, bper);
        else if (P.nparts > 1) run(k_ttv_lead<true, int>, (int)B, (int)bper);
        else run(k_ttv_lead<false, int>, (int)B, (int)bper);
        ITCPD_HIP(hipGetLastError());
        rc = finish_parts(p, parts, nz, nout, p->M, ms, true);
    } else {
        auto run = [&](auto kern, int jw, auto a, auto b) {
            hipLaunchKernelGGL(kern, dim3((unsigned)(cdiv(cdiv(In, jw) * p->R, 4) + fj.on)), dim3(256), lds,
                               p->stream, P.ptr, P.nparts, P.stride, MS, In, (int)p->R, sd, pos, a, b, p->M, fj, p->chk);
        };
        const bool shrt = A * B <= 128, parts = P.nparts > 1;
        if (!small) run(k_ttv_inner<true, 4, 4, int64_t>, 4, A, B);
        else if (shrt && parts) run(k_ttv_inner<true, 4, 2, int>, 4, (int)A, (int)B);
        else if (shrt) run(k_ttv_inner<false, 4, 2, int>, 4, (int)A, (int)B);
        else if (parts) run(k_ttv_inner<true, 4, 4, int>, 4, (int)A, (int)B);
        else run(k_ttv_inner<false, 4, 4, int>, 4, (int)A, (int)B);
        ITCPD_HIP(hipGetLastError());
        *ms = MSrc{p->M, 1, nout};
    }
    if (rc) return rc;
    if (factor_mode >= 0 && !fj.on) return launch_factor(p, factor_mode);
    return ITCPD_OK;
}

// Full MTTKRP of one mode from the current factors, summed into p->M (hook).
int mttkrp_mode(itcpd_plan* p, int mode) {
    int rc;
    MSrc ms{};
    const int64_t n = p->dims[mode] * p->R;
    if (mode < p->s) {
        if ((rc = launch_left_gemm(p, &ms))) return rc;
        if (p->s > 1 && (rc = launch_side_ttv(p, mode, &ms))) return rc;
    } else {
        if ((rc = launch_right_gemm(p, &ms))) return rc;
        if (p->N - p->s > 1 && (rc = launch_side_ttv(p, mode, &ms))) return rc;
    }
    if (ms.nparts > 1) return launch_sum_parts(p, ms, n, p->M);
    return ITCPD_OK;
}

int launch_tensor_norm(itcpd_plan* p) {
    int64_t n = 1;
    for (int q = 0; q < p->N; ++q) n *= p->dims[q];
    const int nb = 1024;
    if (p->elt_bytes == 8)
        hipLaunchKernelGGL(k_sumsq_part<double>, dim3(nb), dim3(256), 0, p->stream,
                           (const double*)p->T, n, p->parts);
    else
        hipLaunchKernelGGL(k_sumsq_part<float>, dim3(nb), dim3(256), 0, p->stream,
                           (const float*)p->T, n, p->parts);
    ITCPD_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_sum_small, dim3(1), dim3(64), 0, p->stream, p->parts, nb, p->scal + 3);
    ITCPD_HIP(hipGetLastError());
    return ITCPD_OK;
}

}  // namespace itcpd
