// C ABI of libitcpd_hip.so (declared in include/itcpd.h).
#include <cstdio>
#include <algorithm>
#include <cstring>
#include <new>
#include <vector>

#include "internal.h"

namespace itcpd {

static thread_local std::string g_last_error;

void set_error(const std::string& msg) { g_last_error = msg; }
int fail(int code, const std::string& msg) {
    g_last_error = msg;
    return code;
}
int hip_fail(hipError_t e, const char* what) {
    g_last_error = std::string("HIP error '") + hipGetErrorString(e) + "' in " + what;
    return e == hipErrorOutOfMemory ? ITCPD_E_OOM : ITCPD_E_HIP;
}

namespace {

int choose_rb(int64_t R) {
    if (R <= 16) return 1;
    if (R <= 32) return 2;
    if (R <= 64) return 4;
    return 8;
}

// Dimension-tree split: minimise ML + MR (the partial sizes); ties -> larger s.
int choose_split(int N, const int64_t* dims) {
    int best = 1;
    double bestc = -1;
    for (int s = 1; s < N; ++s) {
        double ml = 1, mr = 1;
        for (int q = 0; q < s; ++q) ml *= (double)dims[q];
        for (int q = s; q < N; ++q) mr *= (double)dims[q];
        const double c = ml + mr;
        if (bestc < 0 || c <= bestc) {
            bestc = c;
            best = s;
        }
    }
    return best;
}

// Copies an I x R column-major block into an I x Rp column-major device array.
int put_factor(itcpd_plan* p, int m, const double* src, int mem) {
    const int64_t In = p->dims[m];
    return copy_in(p->A[m], src, (size_t)In * p->R * 8, mem, p->stream);
}

// Clears done / nan so that hook calls after a converged run execute.
int reset_check_flags(itcpd_plan* p) { return launch_reset_flags(p); }

// Folds finished begin/end event pairs into the per-kernel totals.  With
// wait == false only pairs whose end event has already completed are taken
// (the sweep loop calls it that way so the host never stalls the queue).
int collect_timer(itcpd_plan* p, bool wait) {
    KernelTimer& tm = p->timer;
    const size_t npair = tm.ev.size() / 2;
    size_t k = 0;
    for (; k < npair; ++k) {
        if (!wait) {
            const hipError_t q = hipEventQuery(tm.ev[2 * k + 1]);
            if (q == hipErrorNotReady) break;
            ITCPD_HIP(q);
        }
        float ms = 0.f;
        ITCPD_HIP(hipEventSynchronize(tm.ev[2 * k + 1]));
        ITCPD_HIP(hipEventElapsedTime(&ms, tm.ev[2 * k], tm.ev[2 * k + 1]));
        KernelTimer::Acc& a = tm.acc[tm.pending_kind[k]];
        a.total_ms += ms;
        a.flops += tm.pending_flops[k];
        a.bytes += tm.pending_bytes[k];
        a.launches += 1;
        (void)hipEventDestroy(tm.ev[2 * k]);
        (void)hipEventDestroy(tm.ev[2 * k + 1]);
    }
    tm.ev.erase(tm.ev.begin(), tm.ev.begin() + 2 * k);
    tm.pending_flops.erase(tm.pending_flops.begin(), tm.pending_flops.begin() + k);
    tm.pending_bytes.erase(tm.pending_bytes.begin(), tm.pending_bytes.begin() + k);
    tm.pending_kind.erase(tm.pending_kind.begin(), tm.pending_kind.begin() + k);
    return ITCPD_OK;
}

// Main and side streams, both at the default priority.
hipError_t create_streams(itcpd_plan* p) {
    return hipStreamCreateWithFlags(&p->stream, hipStreamNonBlocking);
}

// Buffers of the reduced-precision GEMMs, allocated on the first switch away from
// FP64: a side's Khatri-Rao product (4 bytes per element); for an FP32-stored tensor
// also room for 8 split-K partials of the larger side's output.
size_t lp_parts(const itcpd_plan* p) {
    if (p->elt_bytes != 4) return 0;
    return std::min<size_t>((size_t)8 * (size_t)(std::max(p->ML, p->MR) * p->R), (size_t)1 << 27);
}
int ensure_lp_buffers(itcpd_plan* p) {
    int rc;
    if (!p->Kt && (rc = dmalloc(&p->Kt, (size_t)lp_krp_elems(p)))) return rc;
    const size_t want = lp_parts(p);
    if (p->parts_elems < want) {
        ITCPD_HIP(hipStreamSynchronize(p->stream));
        dfree(p->parts);
        p->parts = nullptr;
        p->parts_elems = 0;
        if ((rc = dmalloc(&p->parts, want))) return rc;
        p->parts_elems = want;
    }
    return ITCPD_OK;
}

// A plan's device buffers come from one allocation: requests are collected, then laid out in
// order at 256-byte steps (about 25 hipMalloc / hipFree pairs a plan otherwise, most of a
// short als_optimize call).
struct Arena {
    std::vector<std::pair<void**, size_t>> req;
    size_t bytes = 0;
    template <typename T>
    void add(T** ptr, size_t count) {
        *ptr = nullptr;
        req.emplace_back((void**)ptr, bytes);
        bytes += (std::max<size_t>(count, 1) * sizeof(T) + 255) / 256 * 256;
    }
    int alloc(char** base) {
        const int rc = dmalloc(base, bytes);
        if (rc) return rc;
        for (auto& r : req) *r.first = *base + r.second;
        return ITCPD_OK;
    }
};

// Per-mode factor state shared by plans and the plan-free random init.  The factors and
// lambda come first, then the other buffers that start at zero: p->cpd_bytes covers the CPD
// (what set_cpd and get_cpd move in one copy), p->zero_bytes all that is cleared.
void factor_state(itcpd_plan* p, Arena& ar) {
    const int64_t R = p->R, Rp = p->Rp, maxI = p->maxI;
    for (int q = 0; q < p->N; ++q) ar.add(&p->A[q], (size_t)(p->dims[q] * Rp));
    ar.add(&p->lam, (size_t)Rp);
    p->cpd_bytes = ar.bytes;
    for (int q = 0; q < p->N; ++q) ar.add(&p->At[q], (size_t)(p->dims[q] * Rp));
    ar.add(&p->counters, 64);
    ar.add(&p->chk, 1);
    p->zero_bytes = ar.bytes;
    for (int q = 0; q < p->N; ++q) ar.add(&p->G[q], (size_t)(R * R));
    ar.add(&p->X, (size_t)(maxI * Rp));
    ar.add(&p->M, (size_t)(maxI * Rp));
    ar.add(&p->Msum, (size_t)(maxI * Rp));
    ar.add(&p->sumsq_part, (size_t)(128 * R));
    // Gram partials: one per 16-row tile of the R <= 64 row solves (at most 256), else per
    // row range of the Gram or normalisation kernels (at most 64); at most 2^25 doubles
    const int64_t most = R <= 64 ? std::min<int64_t>(256, std::max<int64_t>(64, cdiv(maxI, 16))) : 64;
    const int64_t nb = std::min<int64_t>(most, std::max<int64_t>(1, ((int64_t)1 << 25) / (R * R)));
    ar.add(&p->gram_part, (size_t)(nb * R * R));
    ar.add(&p->inner_part, 256);
    ar.add(&p->scal, 8);
}
int alloc_arena(itcpd_plan* p, Arena& ar) {
    const int rc = ar.alloc(&p->arena);
    if (rc) return rc;
    ITCPD_HIP(hipMemsetAsync(p->arena, 0, p->zero_bytes, p->stream));
    return ITCPD_OK;
}

// Pinned mirror of the CPD region for host factors (up to 8 MiB): one copy instead of N + 1
// from pageable memory.  Null where there is none; its padding columns stay zero.
char* cpd_stage(itcpd_plan* p) {
    if (!p->stage && !p->stage_failed) {
        p->stage_failed = p->cpd_bytes > ((size_t)8 << 20) ||
                          hipHostMalloc((void**)&p->stage, p->cpd_bytes, hipHostMallocDefault) != hipSuccess;
        if (p->stage_failed) {
            (void)hipGetLastError();
            p->stage = nullptr;
        } else {
            std::memset(p->stage, 0, p->cpd_bytes);
        }
    }
    return p->stage;
}

// One ALS sweep (optimize.jl:17-30), every launch on the plan's stream.  Mode n's
// V_n depends only on the other modes' Grams, which are final once mode n-1's update
// has run.  M of the first mode of each side comes from a GEMM launch, the others'
// from a short Hadamard-reduce of the side's partial; then solve, row_norm, Gram
// refresh (and the fit after the last mode).  For R <= 64 the factorisation of a
// mode with a Hadamard-reduce rides in one extra workgroup of that launch (mode
// 0's too: its V_0 is final once the previous sweep ended), and that of the right
// GEMM's own mode in one of the launch that sums the GEMM's split-K partials; the
// others (R > 64) run as their own launch right after mode n-1's update.
//
// Order 3 with shared partials (tree3): update u (counted from the run's start) with u even
// contracts T over the mode updated last, and that partial serves updates u and u + 1.  When
// only one update is left for a partial (the last of an odd number of sweeps), M_2 comes
// from the right GEMM, as in the plain tree.
int sweep3(itcpd_plan* p, int64_t k, bool last) {
    int rc;
    MSrc ms{};
    const bool rides = p->R <= 64 && !p->v_override;
    if (!rides && (rc = launch_factor(p, 0))) return rc;
    for (int n = 0; n < 3; ++n) {
        const int64_t u = 3 * k + n;
        if (u % 2 == 0 && n == 2 && last && p->s == 2) {
            if ((rc = launch_right_gemm(p, &ms, rides ? n : -1))) return rc;
        } else {
            const int c = u % 2 == 0 ? (n + 2) % 3 : (n + 1) % 3;
            if (u % 2 == 0 && (rc = launch_tree3_gemm(p, c))) return rc;
            if ((rc = launch_tree3_ttv(p, n, c, &ms, rides ? n : -1))) return rc;
        }
        const int next = n + 1 < 3 && !rides ? n + 1 : -1;
        if ((rc = launch_solve(p, n, ms.ptr, ms.nparts, ms.stride, true, n == 2, next))) return rc;
    }
    if (p->profiling && p->timer.ev.size() >= 64) return collect_timer(p, false);
    return ITCPD_OK;
}

int sweep(itcpd_plan* p, int64_t k, bool last) {
    if (p->tree3) return sweep3(p, k, last);
    int rc;
    const int N = p->N;
    MSrc ms{};
    auto has_ttv = [&](int n) { return n < p->s ? p->s > 1 : N - p->s > 1; };
    auto rides_ttv = [&](int n) { return has_ttv(n) && p->R <= 64 && !p->v_override; };
    auto with_right = [&](int n) { return n == p->s && !has_ttv(n); };
    if ((rc = launch_left_gemm(p, &ms, rides_ttv(0) ? -1 : 0))) return rc;
    for (int n = 0; n < N; ++n) {
        if (n == p->s && (rc = launch_right_gemm(p, &ms, with_right(n) ? n : -1))) return rc;
        if (has_ttv(n) && (rc = launch_side_ttv(p, n, &ms, rides_ttv(n) ? n : -1))) return rc;
        const int next = n + 1 < N && !rides_ttv(n + 1) && !with_right(n + 1) ? n + 1 : -1;
        if ((rc = launch_solve(p, n, ms.ptr, ms.nparts, ms.stride, true, n == N - 1, next))) return rc;
    }
    if (p->profiling && p->timer.ev.size() >= 64) return collect_timer(p, false);
    return ITCPD_OK;
}

}  // namespace
}  // namespace itcpd

using namespace itcpd;

extern "C" {

const char* itcpd_last_error(void) { return g_last_error.c_str(); }

const char* itcpd_version(void) { return "itcpd-hip 0.1 (gfx950)"; }

int itcpd_plan_create(itcpd_plan** out, int32_t order, const int64_t* dims, int64_t rank,
                      int32_t elt_bytes, const void* tensor, int32_t tensor_mem, int32_t prec,
                      int32_t alg, int32_t device) {
    if (!out) return fail(ITCPD_E_ARG, "plan pointer is null");
    *out = nullptr;
    if (order < 2 || order > ITCPD_MAX_ORDER)
        return fail(ITCPD_E_ARG, "tensor order must be between 2 and 8");
    if (!dims || !tensor) return fail(ITCPD_E_ARG, "dims or tensor pointer is null");
    if (rank < 1 || rank > ITCPD_MAX_RANK) return fail(ITCPD_E_ARG, "rank must be in [1, 1024]");
    if (elt_bytes != 8 && elt_bytes != 4) return fail(ITCPD_E_ARG, "elt_bytes must be 8 or 4");
    if (tensor_mem != ITCPD_MEM_HOST && tensor_mem != ITCPD_MEM_DEVICE)
        return fail(ITCPD_E_ARG, "tensor_mem must be ITCPD_MEM_HOST or ITCPD_MEM_DEVICE");
    if (prec != ITCPD_FP64 && prec != ITCPD_FP32 && prec != ITCPD_BF16X3)
        return fail(ITCPD_E_UNSUPPORTED, "prec must be ITCPD_FP64, ITCPD_FP32 or ITCPD_BF16X3");
    if (alg != ITCPD_ALG_KRP_FREE_NORMAL && alg != ITCPD_ALG_KRP_NORMAL)
        return fail(ITCPD_E_ARG, "alg must be KRPFreeNormal or KRPNormal");
    for (int q = 0; q < order; ++q)
        if (dims[q] < 1) return fail(ITCPD_E_ARG, "every dimension must be >= 1");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
        return fail(ITCPD_E_HIP, "no HIP device available");
    if (device < 0 || device >= ndev) return fail(ITCPD_E_ARG, "device index out of range");

    itcpd_plan* p = new (std::nothrow) itcpd_plan();
    if (!p) return fail(ITCPD_E_OOM, "host allocation failed");
    DeviceGuard dg(device);
    p->device = device;
    if (hipDeviceGetAttribute(&p->num_cu, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess ||
        p->num_cu < 1)
        p->num_cu = 256;
    p->N = order;
    for (int q = 0; q < order; ++q) p->dims[q] = dims[q];
    p->R = rank;
    p->RB = choose_rb(rank);
    p->Rp = cdiv(rank, 16 * p->RB) * 16 * p->RB;
    p->elt_bytes = elt_bytes;
    p->prec = prec;
    p->alg = alg;
    p->s = choose_split(order, dims);
    p->ML = 1;
    p->MR = 1;
    for (int q = 0; q < p->s; ++q) p->ML *= dims[q];
    for (int q = p->s; q < order; ++q) p->MR *= dims[q];
    p->maxI = 0;
    for (int q = 0; q < order; ++q) p->maxI = dims[q] > p->maxI ? dims[q] : p->maxI;

    int rc = ITCPD_OK;
    auto bail = [&](int code) {
        itcpd_plan_destroy(p);
        return code;
    };
    hipError_t e = create_streams(p);
    if (e != hipSuccess) return bail(hip_fail(e, "hipStreamCreate"));
    for (int q = 0; q < ITCPD_POLL_SLOTS; ++q) {
        e = hipEventCreateWithFlags(&p->ev_poll[q], hipEventDisableTiming);
        if (e != hipSuccess) return bail(hip_fail(e, "hipEventCreate"));
    }

    const int64_t R = p->R, Rp = p->Rp, maxI = p->maxI;
    const size_t nel = (size_t)(p->ML * p->MR);
    if (tensor_mem == ITCPD_MEM_HOST) {
        if ((rc = dmalloc((char**)&p->T_owned, nel * elt_bytes))) return bail(rc);
        e = hipMemcpy(p->T_owned, tensor, nel * elt_bytes, hipMemcpyHostToDevice);
        if (e != hipSuccess) return bail(hip_fail(e, "hipMemcpy(tensor)"));
        p->T = p->T_owned;
    } else {
        e = hipDeviceSynchronize();   // the tensor may have been produced on another stream
        if (e != hipSuccess) return bail(hip_fail(e, "hipDeviceSynchronize"));
        if (((uintptr_t)tensor) % 16 != 0) return bail(fail(ITCPD_E_ARG, "device tensor must be 16-byte aligned"));
        p->T = tensor;
    }
    Arena ar;
    factor_state(p, ar);
    ar.add(&p->U, (size_t)(R * R));
    if (R <= 64) {
        p->RT = R <= 16 ? 16 : (R <= 32 ? 32 : 64);
        ar.add(&p->Upad, (size_t)(R * R));   // V^-1
    } else {
        const int64_t nb = cdiv(R, 64);
        ar.add(&p->inv_buf, (size_t)(2 * 4096 * nb * nb));
        ar.add(&p->inv_stat, inv_stat_elems(R));
    }
    ar.add(&p->invdiag, (size_t)R);
    ar.add(&p->qr_aux, (size_t)(R * R + 4 * R));
    ar.add(&p->piv, (size_t)(2 * R));
    ar.add(&p->finfo, 4);
    if (const int64_t n = krp64_elems(p)) ar.add(&p->Wrest, (size_t)n);
    if (p->s > 1) ar.add(&p->PL, (size_t)(p->ML * R));
    if (order - p->s > 1) ar.add(&p->PR, (size_t)(p->MR * R));
    p->trace_cap = 1024;
    ar.add(&p->fit_trace, (size_t)p->trace_cap);
    if ((rc = alloc_arena(p, ar))) return bail(rc);
    {
        // split-K partials: what 512 splits of the larger side could use, up to half of the
        // tensor's elements (their traffic is weighed against the tensor's) and 128 MiB, and
        // the 16 partials of the longest mode's Hadamard-reduce
        const size_t outmax = (size_t)std::max<int64_t>(std::max(p->ML, p->MR), maxI) * R;
        size_t want = std::min<size_t>((size_t)1 << 24, outmax * 512);
        want = std::min<size_t>(want, std::max<size_t>(nel / 2, (size_t)(16 * maxI * R)));
        want = std::max<size_t>(want, 1024 * 4);
        if (prec != ITCPD_FP64) want = std::max(want, lp_parts(p));
        p->parts_elems = want;
        if ((rc = dmalloc(&p->parts, want))) return bail(rc);
    }
    if (prec != ITCPD_FP64 && (rc = ensure_lp_buffers(p))) return bail(rc);
    e = hipHostMalloc((void**)&p->chk_host, sizeof(DevCheck) * (1 + ITCPD_POLL_SLOTS),
                      hipHostMallocDefault);
    if (e != hipSuccess) return bail(hip_fail(e, "hipHostMalloc"));
    std::memset(p->chk_host, 0, sizeof(DevCheck) * (1 + ITCPD_POLL_SLOTS));
    e = hipStreamSynchronize(p->stream);
    if (e != hipSuccess) return bail(hip_fail(e, "hipStreamSynchronize"));
    *out = p;
    return ITCPD_OK;
}

int itcpd_plan_destroy(itcpd_plan* p) {
    if (!p) return ITCPD_OK;
    DeviceGuard dg(p->device);
    if (p->stream) (void)hipStreamSynchronize(p->stream);
    for (hipEvent_t e : p->timer.ev) (void)hipEventDestroy(e);
    dfree(p->T_owned);
    dfree(p->arena);
    dfree(p->Kt);
    dfree(p->parts);
    dfree(p->trace_owned);
    for (int q = 0; q < ITCPD_MAX_ORDER; ++q) dfree(p->Atprev[q]);
    dfree(p->lamprev);
    dfree(p->smp_ws);
    dfree(p->sk_ws);
    dfree(p->P3_owned);
    dfree(p->smp_iws);
    dfree(p->xg_part);
    if (p->chk_host) (void)hipHostFree(p->chk_host);
    if (p->stage) (void)hipHostFree(p->stage);
    for (int q = 0; q < ITCPD_POLL_SLOTS; ++q)
        if (p->ev_poll[q]) (void)hipEventDestroy(p->ev_poll[q]);
    if (p->stream) (void)hipStreamDestroy(p->stream);
    delete p;
    return ITCPD_OK;
}

int itcpd_set_cpd(itcpd_plan* p, const double* const* factors, const double* lambda, int32_t mem) {
    if (!p || !factors) return fail(ITCPD_E_ARG, "null argument");
    DeviceGuard dg(p->device);
    int rc;
    for (int m = 0; m < p->N; ++m)
        if (!factors[m]) return fail(ITCPD_E_ARG, "null factor pointer");
    char* const stage = mem == ITCPD_MEM_HOST && lambda ? cpd_stage(p) : nullptr;
    if (stage) {
        for (int m = 0; m < p->N; ++m)
            std::memcpy(stage + ((char*)p->A[m] - p->arena), factors[m], (size_t)(p->dims[m] * p->R) * 8);
        std::memcpy(stage + ((char*)p->lam - p->arena), lambda, (size_t)p->R * 8);
        if ((rc = copy_in(p->arena, stage, p->cpd_bytes, mem, p->stream))) return rc;
    } else {
        for (int m = 0; m < p->N; ++m)
            if ((rc = put_factor(p, m, factors[m], mem))) return rc;
        if (lambda && (rc = copy_in(p->lam, lambda, (size_t)p->R * 8, mem, p->stream))) return rc;
    }
    if ((rc = reset_check_flags(p))) return rc;
    if ((rc = launch_seed_grams(p))) return rc;
    ITCPD_HIP(hipStreamSynchronize(p->stream));
    p->have_cpd = true;
    return ITCPD_OK;
}

int itcpd_random_cpd(itcpd_plan* p, uint64_t seed) {
    if (!p) return fail(ITCPD_E_ARG, "null plan");
    DeviceGuard dg(p->device);
    int rc;
    if ((rc = reset_check_flags(p))) return rc;
    if ((rc = launch_random_init(p, seed))) return rc;
    ITCPD_HIP(hipStreamSynchronize(p->stream));
    p->have_cpd = true;
    return ITCPD_OK;
}

int itcpd_random_factors(int32_t order, const int64_t* dims, int64_t rank, uint64_t seed,
                         double* const* factors, double* lambda, int32_t mem, int32_t device) {
    if (order < 1 || order > ITCPD_MAX_ORDER) return fail(ITCPD_E_ARG, "order must be in [1, 8]");
    if (!dims || !factors) return fail(ITCPD_E_ARG, "null argument");
    if (rank < 1 || rank > ITCPD_MAX_RANK) return fail(ITCPD_E_ARG, "rank must be in [1, 1024]");
    for (int q = 0; q < order; ++q)
        if (dims[q] < 1 || !factors[q]) return fail(ITCPD_E_ARG, "bad dims or factor pointer");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
        return fail(ITCPD_E_HIP, "no HIP device available");
    if (device < 0 || device >= ndev) return fail(ITCPD_E_ARG, "device index out of range");
    // a plan without a tensor: only the factor state is allocated
    itcpd_plan* p = new (std::nothrow) itcpd_plan();
    if (!p) return fail(ITCPD_E_OOM, "host allocation failed");
    DeviceGuard dg(device);
    auto bail = [&](int code) {
        itcpd_plan_destroy(p);
        return code;
    };
    p->device = device;
    p->N = order;
    p->R = rank;
    p->RB = choose_rb(rank);
    p->Rp = cdiv(rank, 16 * p->RB) * 16 * p->RB;
    for (int q = 0; q < order; ++q) {
        p->dims[q] = dims[q];
        p->maxI = dims[q] > p->maxI ? dims[q] : p->maxI;
    }
    int rc;
    hipError_t e = hipStreamCreateWithFlags(&p->stream, hipStreamNonBlocking);
    if (e != hipSuccess) return bail(hip_fail(e, "hipStreamCreate"));
    p->stage_failed = true;   // one transfer: a pinned mirror costs more than it saves
    Arena ar;
    factor_state(p, ar);
    if ((rc = alloc_arena(p, ar))) return bail(rc);
    if ((rc = launch_random_init(p, seed))) return bail(rc);
    p->have_cpd = true;
    rc = itcpd_get_cpd(p, factors, lambda, mem);
    return bail(rc);
}

int itcpd_get_cpd(itcpd_plan* p, double* const* factors, double* lambda, int32_t mem) {
    if (!p) return fail(ITCPD_E_ARG, "null plan");
    if (!p->have_cpd) return fail(ITCPD_E_STATE, "no CPD set on this plan");
    DeviceGuard dg(p->device);
    int rc;
    if (char* const stage = mem == ITCPD_MEM_HOST && factors ? cpd_stage(p) : nullptr) {
        if ((rc = copy_out(stage, p->arena, p->cpd_bytes, mem, p->stream))) return rc;
        ITCPD_HIP(hipStreamSynchronize(p->stream));
        for (int m = 0; m < p->N; ++m)
            if (factors[m])
                std::memcpy(factors[m], stage + ((char*)p->A[m] - p->arena), (size_t)(p->dims[m] * p->R) * 8);
        if (lambda) std::memcpy(lambda, stage + ((char*)p->lam - p->arena), (size_t)p->R * 8);
        return ITCPD_OK;
    }
    for (int m = 0; factors && m < p->N; ++m) {
        if (!factors[m]) continue;
        if ((rc = copy_out(factors[m], p->A[m], (size_t)p->dims[m] * p->R * 8, mem, p->stream)))
            return rc;
    }
    if (lambda && (rc = copy_out(lambda, p->lam, (size_t)p->R * 8, mem, p->stream))) return rc;
    ITCPD_HIP(hipStreamSynchronize(p->stream));
    return ITCPD_OK;
}

// PrevCP storage of the CP checks and their cross-Gram partials (row chunks bounded
// so that the partials stay within 2^24 doubles), allocated on first use.
static int ensure_prevcp(itcpd_plan* p) {
    if (p->lamprev) return ITCPD_OK;
    int rc;
    for (int q = 0; q < p->N; ++q)
        if ((rc = dmalloc(&p->Atprev[q], (size_t)(p->dims[q] * p->Rp)))) return rc;
    if ((rc = dmalloc(&p->lamprev, (size_t)p->Rp))) return rc;
    const int64_t RR = p->R * p->R;
    int64_t ch = ((int64_t)1 << 24) / (p->N * RR);
    ch = std::max<int64_t>(1, std::min<int64_t>(ch, 16));
    p->xg_chunks = (int)ch;
    return dmalloc(&p->xg_part, (size_t)(p->N * ch * RR));
}

int itcpd_run(itcpd_plan* p, itcpd_check* c, double* fit_trace) {
    if (!p || !c) return fail(ITCPD_E_ARG, "null argument");
    if (!p->have_cpd) return fail(ITCPD_E_STATE, "itcpd_run before itcpd_set_cpd / itcpd_random_cpd");
    if (c->kind != ITCPD_CHECK_NONE && c->kind != ITCPD_CHECK_FIT && c->kind != ITCPD_CHECK_CPDIFF &&
        c->kind != ITCPD_CHECK_CPANGLE)
        return fail(ITCPD_E_ARG, "unknown check kind");
    const bool cp_check = c->kind == ITCPD_CHECK_CPDIFF || c->kind == ITCPD_CHECK_CPANGLE;
    if (cp_check && c->has_prev && !p->prev_valid)
        return fail(ITCPD_E_STATE, "check holds a previous CPD that this plan does not have");
    DeviceGuard dg(p->device);
    if (cp_check) {
        const int rc = ensure_prevcp(p);
        if (rc) return rc;
    }
    // optimize.jl:8: the sweep loop runs while the local counter (starting at
    // check.iter) is below check.max_counter
    const int64_t nsweeps = (int64_t)c->max_counter - c->iter;
    c->sweeps_run = 0;
    c->converged = 0;
    if (nsweeps <= 0) return ITCPD_OK;
    p->tree3 = nsweeps > 1 && tree3_pays(p);
    if (p->tree3 && !p->P3) {
        // the plain tree's partial, which a shared run does not use, where it is large enough
        double* const side = p->s > 1 ? p->PL : p->PR;
        if (tree3_elems(p) <= (p->s > 1 ? p->ML : p->MR) * p->R) {
            p->P3 = side;
        } else if (hipMalloc((void**)&p->P3_owned, (size_t)tree3_elems(p) * 8) == hipSuccess) {
            p->P3 = p->P3_owned;
        } else {
            (void)hipGetLastError();   // no memory for it: the plain tree
            p->P3_owned = nullptr;
            p->tree3 = false;
        }
    }
    if (nsweeps > p->trace_cap) {
        dfree(p->trace_owned);
        p->trace_owned = nullptr;
        const int rc = dmalloc(&p->trace_owned, (size_t)nsweeps);
        if (rc) {
            p->trace_cap = 0;
            p->fit_trace = nullptr;
            return rc;
        }
        p->fit_trace = p->trace_owned;
        p->trace_cap = (int)nsweeps;
    }
    DevCheck* h = p->chk_host;
    std::memset(h, 0, sizeof(DevCheck));
    h->kind = c->kind;
    h->iter = c->iter;
    h->counter = c->counter;
    h->max_counter = c->max_counter;
    h->total_iter = c->total_iter;
    h->tolerance = c->tolerance;
    h->ref_norm = c->ref_norm;
    h->lastfit = c->lastfit;
    h->final_fit = c->final_fit;
    if (cp_check) {
        h->ref_norm = 0.0;
        h->norm_prev = c->ref_norm;
        h->has_prev = c->has_prev ? 1 : 0;
    }
    p->check_kind = c->kind;
    // h is written again only by the copy back at the run's end, behind this one on the stream
    ITCPD_HIP(hipMemcpyAsync(p->chk, h, sizeof(DevCheck), hipMemcpyHostToDevice, p->stream));

    // FitCheck: every POLL_EVERY sweeps a snapshot of the device check state is
    // copied to a pinned slot behind an event.  The host keeps enqueueing and
    // only waits once two snapshots are outstanding, so the queue never drains;
    // sweeps enqueued after convergence return at their first instruction (each
    // kernel tests chk->done).
    constexpr int64_t POLL_EVERY = 4;
    const int64_t batch = (c->kind != ITCPD_CHECK_NONE) ? POLL_EVERY : nsweeps;
    DevCheck* slots = p->chk_host + 1;
    int64_t polls_issued = 0, polls_seen = 0;
    int rc = ITCPD_OK;
    for (int64_t k = 0; k < nsweeps;) {
        const int64_t nb = std::min<int64_t>(batch, nsweeps - k);
        for (int64_t b = 0; b < nb; ++b)
            if ((rc = sweep(p, k + b, k + b == nsweeps - 1))) return rc;
        k += nb;
        if (c->kind == ITCPD_CHECK_NONE || k >= nsweeps) continue;
        const int slot = (int)(polls_issued % ITCPD_POLL_SLOTS);
        ITCPD_HIP(hipMemcpyAsync(&slots[slot], p->chk, sizeof(DevCheck), hipMemcpyDeviceToHost,
                                 p->stream));
        ITCPD_HIP(hipEventRecord(p->ev_poll[slot], p->stream));
        ++polls_issued;
        bool stop = false;
        while (polls_seen < polls_issued) {
            const int os = (int)(polls_seen % ITCPD_POLL_SLOTS);
            if (polls_issued - polls_seen >= 2) {
                ITCPD_HIP(hipEventSynchronize(p->ev_poll[os]));
            } else {
                const hipError_t q = hipEventQuery(p->ev_poll[os]);
                if (q == hipErrorNotReady) break;
                ITCPD_HIP(q);
            }
            ++polls_seen;
            if (slots[os].done) { stop = true; break; }
        }
        if (stop) break;
    }
    ITCPD_HIP(hipMemcpyAsync(h, p->chk, sizeof(DevCheck), hipMemcpyDeviceToHost, p->stream));
    ITCPD_HIP(hipStreamSynchronize(p->stream));
    p->check_kind = 0;
    if (p->profiling && (rc = collect_timer(p, true))) return rc;
    if (cp_check) {
        c->ref_norm = h->norm_prev;
        c->has_prev = h->has_prev;
        p->prev_valid = h->has_prev != 0;
    }
    c->iter = h->iter;
    c->counter = h->counter;
    c->total_iter = h->total_iter;
    c->lastfit = h->lastfit;
    c->final_fit = h->final_fit;
    c->sweeps_run = h->sweeps > 0 ? h->sweeps : (int)std::min<int64_t>(nsweeps, INT32_MAX);
    c->converged = (h->done && !h->nan_flag) ? 1 : 0;
    if (c->kind == ITCPD_CHECK_NONE) c->sweeps_run = h->sweeps;
    if (fit_trace && c->kind != ITCPD_CHECK_NONE && h->sweeps > 0)
        ITCPD_HIP(hipMemcpy(fit_trace, p->fit_trace, (size_t)std::min(h->sweeps, p->trace_cap) * 8,
                            hipMemcpyDeviceToHost));
    if (h->nan_flag) return fail(ITCPD_E_NAN, "Error NAN");
    return ITCPD_OK;
}

int itcpd_compute_krp(itcpd_plan* p, int32_t mode, double* V_out, int32_t mem) {
    if (!p || !V_out) return fail(ITCPD_E_ARG, "null argument");
    if (mode < 0 || mode >= p->N) return fail(ITCPD_E_ARG, "mode out of range");
    if (!p->have_cpd) return fail(ITCPD_E_STATE, "no CPD set");
    DeviceGuard dg(p->device);
    int rc;
    if ((rc = launch_hadamard(p, mode, p->U))) return rc;
    if ((rc = copy_out(V_out, p->U, (size_t)(p->R * p->R) * 8, mem, p->stream))) return rc;
    ITCPD_HIP(hipStreamSynchronize(p->stream));
    return ITCPD_OK;
}

int itcpd_mttkrp(itcpd_plan* p, int32_t mode, double* M_out, int32_t mem) {
    if (!p || !M_out) return fail(ITCPD_E_ARG, "null argument");
    if (mode < 0 || mode >= p->N) return fail(ITCPD_E_ARG, "mode out of range");
    if (!p->have_cpd) return fail(ITCPD_E_STATE, "no CPD set");
    DeviceGuard dg(p->device);
    int rc;
    if ((rc = reset_check_flags(p))) return rc;
    if ((rc = mttkrp_mode(p, mode))) return rc;
    if ((rc = copy_out(M_out, p->M, (size_t)p->dims[mode] * p->R * 8, mem, p->stream))) return rc;
    ITCPD_HIP(hipStreamSynchronize(p->stream));
    return ITCPD_OK;
}

int itcpd_solve_ls(itcpd_plan* p, int32_t mode, const double* M, double* X_out, int32_t mem,
                   int32_t* used_fallback) {
    if (!p || !M || !X_out) return fail(ITCPD_E_ARG, "null argument");
    if (mode < 0 || mode >= p->N) return fail(ITCPD_E_ARG, "mode out of range");
    if (!p->have_cpd) return fail(ITCPD_E_STATE, "no CPD set");
    DeviceGuard dg(p->device);
    int rc;
    if ((rc = reset_check_flags(p))) return rc;
    const size_t bytes = (size_t)p->dims[mode] * p->R * 8;
    if ((rc = copy_in(p->M, M, bytes, mem, p->stream))) return rc;
    if ((rc = launch_factor(p, mode))) return rc;
    if ((rc = launch_solve(p, mode, p->M, 1, (int64_t)p->dims[mode] * p->R, false, false))) return rc;
    if ((rc = copy_out(X_out, p->X, bytes, mem, p->stream))) return rc;
    int info[4];
    ITCPD_HIP(hipMemcpyAsync(info, p->finfo, sizeof(info), hipMemcpyDeviceToHost, p->stream));
    ITCPD_HIP(hipStreamSynchronize(p->stream));
    if (used_fallback) *used_fallback = info[1];
    return ITCPD_OK;
}

int itcpd_row_norm_post_solve(itcpd_plan* p, int32_t mode, const double* X, int32_t mem) {
    if (!p || !X) return fail(ITCPD_E_ARG, "null argument");
    if (mode < 0 || mode >= p->N) return fail(ITCPD_E_ARG, "mode out of range");
    if (!p->have_cpd) return fail(ITCPD_E_STATE, "no CPD set");
    DeviceGuard dg(p->device);
    int rc;
    if ((rc = reset_check_flags(p))) return rc;
    const int64_t In = p->dims[mode];
    if ((rc = copy_in(p->X, X, (size_t)In * p->R * 8, mem, p->stream))) return rc;
    if ((rc = launch_col_sumsq(p, mode, p->X))) return rc;
    if ((rc = launch_normalize(p, mode, p->X, false))) return rc;
    ITCPD_HIP(hipStreamSynchronize(p->stream));
    return ITCPD_OK;
}

int itcpd_fit(itcpd_plan* p, const double* M_last, int32_t mem, double ref_norm, double* inner,
              double* fact_square, double* fit) {
    if (!p || !M_last) return fail(ITCPD_E_ARG, "null argument");
    if (!p->have_cpd) return fail(ITCPD_E_STATE, "no CPD set");
    DeviceGuard dg(p->device);
    int rc;
    const int N = p->N;
    if ((rc = copy_in(p->M, M_last, (size_t)p->dims[N - 1] * p->R * 8, mem, p->stream))) return rc;
    if ((rc = launch_fit_only(p, p->M, ref_norm))) return rc;
    double sc[3];
    ITCPD_HIP(hipMemcpyAsync(sc, p->scal, sizeof(sc), hipMemcpyDeviceToHost, p->stream));
    ITCPD_HIP(hipStreamSynchronize(p->stream));
    if (inner) *inner = sc[0];
    if (fact_square) *fact_square = sc[1];
    if (fit) *fit = sc[2];
    return ITCPD_OK;
}

int itcpd_leverage_scores(itcpd_plan* p, int32_t mode, double* probs, int32_t mem) {
    if (!p || !probs) return fail(ITCPD_E_ARG, "null argument");
    if (mode < 0 || mode >= p->N) return fail(ITCPD_E_ARG, "mode out of range");
    if (!p->have_cpd) return fail(ITCPD_E_STATE, "no CPD set");
    DeviceGuard dg(p->device);
    int rc;
    if ((rc = reset_check_flags(p))) return rc;
    double* used = nullptr;
    if ((rc = launch_leverage_scores(p, mode, mem == ITCPD_MEM_DEVICE ? probs : nullptr, &used))) return rc;
    if (mem != ITCPD_MEM_DEVICE && (rc = copy_out(probs, used, (size_t)p->dims[mode] * 8, mem, p->stream)))
        return rc;
    ITCPD_HIP(hipStreamSynchronize(p->stream));
    return ITCPD_OK;
}

int itcpd_sampled_solve(itcpd_plan* p, int32_t mode, int64_t nsamps, const int32_t* samples, int32_t mem,
                        int32_t normal, int32_t* info) {
    if (!p || !samples) return fail(ITCPD_E_ARG, "null argument");
    if (mode < 0 || mode >= p->N) return fail(ITCPD_E_ARG, "mode out of range");
    if (p->N < 2) return fail(ITCPD_E_ARG, "sampling needs at least two modes");
    if (nsamps < 1 || nsamps > ((int64_t)1 << 31) / p->N) return fail(ITCPD_E_ARG, "nsamps out of range");
    if (!p->have_cpd) return fail(ITCPD_E_STATE, "no CPD set");
    if (!normal && p->R > 2048) return fail(ITCPD_E_UNSUPPORTED, "the QR form takes rank <= 2048");
    DeviceGuard dg(p->device);
    int rc;
    if ((rc = reset_check_flags(p))) return rc;
    if ((rc = sampled_ws_prepare(p, mode, nsamps))) return rc;
    // the indices address the factors and T: check every one on the host
    const size_t nidx = (size_t)nsamps * (size_t)(p->N - 1);
    std::vector<int32_t> h(nidx);
    if (mem == ITCPD_MEM_DEVICE) {
        ITCPD_HIP(hipMemcpyAsync(h.data(), samples, nidx * 4, hipMemcpyDeviceToHost, p->stream));
        ITCPD_HIP(hipStreamSynchronize(p->stream));
    } else {
        std::memcpy(h.data(), samples, nidx * 4);
    }
    int q = 0;
    for (int m = 0; m < p->N; ++m) {
        if (m == mode) continue;
        const int32_t* col = h.data() + (size_t)nsamps * q;
        for (int64_t s = 0; s < nsamps; ++s)
            if (col[s] < 0 || col[s] >= p->dims[m]) return fail(ITCPD_E_ARG, "sample index out of range");
        ++q;
    }
    ITCPD_HIP(hipMemcpyAsync(p->smp_iws, h.data(), nidx * 4, hipMemcpyHostToDevice, p->stream));
    if ((rc = launch_sampled_gather(p, mode, nsamps, p->smp_iws))) return rc;
    int form = normal ? SAMPLED_NORMAL : (sampled_corrected_ok(p, nsamps) ? SAMPLED_CORRECTED : SAMPLED_QR);
    int fi[4] = {0, 0, 0, 0};
    const int* const status = p->smp_iws + nidx + p->R;
    for (;;) {
        if ((rc = launch_sampled_solve(p, mode, nsamps, form))) return rc;
        // the CPD takes no X that the corrected form has not certified
        if (!normal && (rc = launch_row_norm(p, mode, form == SAMPLED_CORRECTED ? status + 1 : nullptr))) return rc;
        ITCPD_HIP(hipMemcpyAsync(fi, normal ? p->finfo : status, sizeof(fi), hipMemcpyDeviceToHost,
                                 p->stream));
        ITCPD_HIP(hipStreamSynchronize(p->stream));
        if (form != SAMPLED_CORRECTED || fi[1] == 0) break;
        form = SAMPLED_QR;   // not certified: the update is made again from the QR
    }
    if (info) {
        info[0] = normal ? fi[1] : 0;            // the Cholesky fell back to the QR solve
        info[1] = normal ? fi[2] : fi[0];        // rank of the solve
    }
    return ITCPD_OK;
}

// Column-pivoted QR of the unfolding (or a column subset) or of its sparse sketch;
// the results come back to the host.
static int qr_pivots_common(itcpd_plan* p, int32_t mode, bool krp, const std::vector<int64_t>* cols, int64_t n,
                            const std::vector<int64_t>* rowptr, const std::vector<int64_t>* colidx,
                            const std::vector<double>* ovals, int64_t* jpvt, double* rdiag) {
    const int64_t In = krp ? p->R : p->dims[mode];
    int rc;
    int64_t* d_cols = nullptr;
    int64_t* d_rowptr = nullptr;
    int64_t* d_colidx = nullptr;
    double* d_vals = nullptr;
    int* d_jpvt = nullptr;
    double* d_rdiag = nullptr;
    auto cleanup = [&]() {
        dfree(d_cols);
        dfree(d_rowptr);
        dfree(d_colidx);
        dfree(d_vals);
        dfree(d_jpvt);
        dfree(d_rdiag);
    };
    const int64_t kq = std::min(In, n);
    rc = dmalloc(&d_jpvt, (size_t)n);
    if (!rc) rc = dmalloc(&d_rdiag, (size_t)kq);
    if (!rc && cols) {
        rc = dmalloc(&d_cols, cols->size());
        if (!rc) rc = copy_in(d_cols, cols->data(), cols->size() * 8, ITCPD_MEM_HOST, p->stream);
    }
    if (!rc && rowptr) {
        rc = dmalloc(&d_rowptr, rowptr->size());
        if (!rc) rc = dmalloc(&d_colidx, std::max<size_t>(1, colidx->size()));
        if (!rc) rc = dmalloc(&d_vals, std::max<size_t>(1, ovals->size()));
        if (!rc) rc = copy_in(d_rowptr, rowptr->data(), rowptr->size() * 8, ITCPD_MEM_HOST, p->stream);
        if (!rc && !colidx->empty())
            rc = copy_in(d_colidx, colidx->data(), colidx->size() * 8, ITCPD_MEM_HOST, p->stream);
        if (!rc && !ovals->empty()) rc = copy_in(d_vals, ovals->data(), ovals->size() * 8, ITCPD_MEM_HOST, p->stream);
    }
    if (!rc)
        rc = launch_qr_pivots(p, mode, krp, d_cols, cols ? (int64_t)cols->size() : n, d_rowptr, d_colidx, d_vals,
                              rowptr ? n : 0, d_jpvt, d_rdiag);
    std::vector<int32_t> hj((size_t)n);
    if (!rc) {
        const hipError_t e1 = hipMemcpy(hj.data(), d_jpvt, (size_t)n * 4, hipMemcpyDeviceToHost);
        const hipError_t e2 = hipMemcpy(rdiag, d_rdiag, (size_t)kq * 8, hipMemcpyDeviceToHost);
        if (e1 != hipSuccess) rc = hip_fail(e1, "hipMemcpy(jpvt)");
        else if (e2 != hipSuccess) rc = hip_fail(e2, "hipMemcpy(rdiag)");
    }
    cleanup();
    if (rc) return rc;
    for (int64_t q = 0; q < n; ++q) jpvt[q] = hj[(size_t)q];
    return ITCPD_OK;
}

static int64_t other_columns(const itcpd_plan* p, int mode) {
    int64_t c = 1;
    for (int m = 0; m < p->N; ++m)
        if (m != mode) c *= p->dims[m];
    return c;
}

static int check_source(const itcpd_plan* p, int32_t source) {
    if (source != ITCPD_PIVOT_TENSOR && source != ITCPD_PIVOT_KRP) return fail(ITCPD_E_ARG, "unknown pivot source");
    if (source == ITCPD_PIVOT_KRP && !p->have_cpd) return fail(ITCPD_E_STATE, "no CPD set");
    return ITCPD_OK;
}

int itcpd_qr_pivots(itcpd_plan* p, int32_t mode, int32_t source, const int64_t* cols, int64_t ncols,
                    int64_t* jpvt, double* rdiag) {
    if (!p || !jpvt || !rdiag) return fail(ITCPD_E_ARG, "null argument");
    if (mode < 0 || mode >= p->N) return fail(ITCPD_E_ARG, "mode out of range");
    if (int rc = check_source(p, source)) return rc;
    const int64_t nall = other_columns(p, mode);
    if (ncols < 1 || ncols > (int64_t)INT32_MAX) return fail(ITCPD_E_ARG, "ncols out of range");
    if (!cols && ncols != nall) return fail(ITCPD_E_ARG, "without a column list ncols must be every column");
    if ((p->dims[mode] > (int64_t)INT32_MAX)) return fail(ITCPD_E_UNSUPPORTED, "mode too long");
    DeviceGuard dg(p->device);
    std::vector<int64_t> hc;
    if (cols) {
        hc.assign(cols, cols + ncols);
        for (int64_t c : hc)
            if (c < 0 || c >= nall) return fail(ITCPD_E_ARG, "column index out of range");
    }
    return qr_pivots_common(p, mode, source == ITCPD_PIVOT_KRP, cols ? &hc : nullptr, ncols, nullptr, nullptr,
                            nullptr, jpvt, rdiag);
}

int itcpd_sketch_qr_pivots(itcpd_plan* p, int32_t mode, int32_t source, int64_t l, int32_t s, const int32_t* rows,
                           const double* vals, int64_t* jpvt, double* rdiag) {
    if (!p || !rows || !vals || !jpvt || !rdiag) return fail(ITCPD_E_ARG, "null argument");
    if (mode < 0 || mode >= p->N) return fail(ITCPD_E_ARG, "mode out of range");
    if (int rc = check_source(p, source)) return rc;
    if (l < 1 || l > (int64_t)INT32_MAX || s < 1) return fail(ITCPD_E_ARG, "embedding size out of range");
    if ((p->dims[mode] > (int64_t)INT32_MAX)) return fail(ITCPD_E_UNSUPPORTED, "mode too long");
    const int64_t nall = other_columns(p, mode);
    const int64_t nnz = nall * s;
    // Omega by rows: for row j the columns with a nonzero there, increasing
    std::vector<int64_t> rowptr((size_t)l + 1, 0);
    for (int64_t e = 0; e < nnz; ++e) {
        const int32_t r = rows[e];
        if (r < 0 || r >= l) return fail(ITCPD_E_ARG, "embedding row out of range");
        ++rowptr[(size_t)r + 1];
    }
    for (int64_t j = 0; j < l; ++j) rowptr[(size_t)j + 1] += rowptr[(size_t)j];
    std::vector<int64_t> fillp(rowptr.begin(), rowptr.end() - 1);
    std::vector<int64_t> colidx((size_t)nnz);
    std::vector<double> ov((size_t)nnz);
    for (int64_t c = 0; c < nall; ++c)
        for (int q = 0; q < s; ++q) {
            const int64_t e = c * s + q;
            const int64_t at = fillp[(size_t)rows[e]]++;
            colidx[(size_t)at] = c;
            ov[(size_t)at] = vals[e];
        }
    DeviceGuard dg(p->device);
    return qr_pivots_common(p, mode, source == ITCPD_PIVOT_KRP, nullptr, l, &rowptr, &colidx, &ov, jpvt, rdiag);
}

int itcpd_sparse_sign(int32_t d, int64_t m, int32_t zeta, int32_t injective, uint64_t seed, double* vals,
                      int32_t* rows, int32_t* colstarts, int32_t device) {
    if (!vals || !rows) return fail(ITCPD_E_ARG, "null argument");
    if (d < 1 || m < 1 || zeta < 1) return fail(ITCPD_E_ARG, "sizes must be positive");
    if (zeta > d) zeta = d;
    if (m > ((int64_t)1 << 40) / zeta) return fail(ITCPD_E_ARG, "embedding too large");
    if (colstarts && m * zeta > (int64_t)INT32_MAX)
        return fail(ITCPD_E_ARG, "column starts exceed 32-bit offsets (pass colstarts = NULL)");
    DeviceGuard dg(device);
    const size_t nnz = (size_t)m * (size_t)zeta;
    double* dv = nullptr;
    int* dr = nullptr;
    int rc = dmalloc(&dv, nnz);
    if (!rc) rc = dmalloc(&dr, nnz);
    if (!rc) rc = launch_sparse_sign(d, m, zeta, injective != 0, seed, dv, dr, nullptr);
    if (!rc) {
        const hipError_t e1 = hipMemcpy(vals, dv, nnz * 8, hipMemcpyDeviceToHost);
        const hipError_t e2 = hipMemcpy(rows, dr, nnz * 4, hipMemcpyDeviceToHost);
        if (e1 != hipSuccess) rc = hip_fail(e1, "hipMemcpy(vals)");
        else if (e2 != hipSuccess) rc = hip_fail(e2, "hipMemcpy(rows)");
    }
    dfree(dv);
    dfree(dr);
    if (rc) return rc;
    if (colstarts)
        for (int64_t c = 0; c <= m; ++c) colstarts[c] = (int32_t)(c * zeta);
    return ITCPD_OK;
}

int itcpd_check_cpd(itcpd_plan* p, itcpd_check* c) {
    if (!p || !c) return fail(ITCPD_E_ARG, "null argument");
    if (c->kind != ITCPD_CHECK_CPDIFF && c->kind != ITCPD_CHECK_CPANGLE)
        return fail(ITCPD_E_ARG, "itcpd_check_cpd takes a CPDiffCheck or CPAngleCheck");
    if (!p->have_cpd) return fail(ITCPD_E_STATE, "no CPD set");
    if (c->has_prev && !p->prev_valid)
        return fail(ITCPD_E_STATE, "check holds a previous CPD that this plan does not have");
    DeviceGuard dg(p->device);
    int rc;
    if ((rc = ensure_prevcp(p))) return rc;
    DevCheck* h = p->chk_host;
    std::memset(h, 0, sizeof(DevCheck));
    h->kind = c->kind;
    h->iter = c->iter;
    h->counter = c->counter;
    h->max_counter = c->max_counter;
    h->total_iter = c->total_iter;
    h->tolerance = c->tolerance;
    h->lastfit = c->lastfit;
    h->final_fit = c->final_fit;
    h->norm_prev = c->ref_norm;
    h->has_prev = c->has_prev ? 1 : 0;
    p->check_kind = c->kind;
    ITCPD_HIP(hipMemcpyAsync(p->chk, h, sizeof(DevCheck), hipMemcpyHostToDevice, p->stream));
    rc = launch_cp_check(p);
    p->check_kind = 0;
    if (rc) return rc;
    ITCPD_HIP(hipMemcpyAsync(h, p->chk, sizeof(DevCheck), hipMemcpyDeviceToHost, p->stream));
    ITCPD_HIP(hipStreamSynchronize(p->stream));
    c->ref_norm = h->norm_prev;
    c->has_prev = h->has_prev;
    p->prev_valid = h->has_prev != 0;
    c->iter = h->iter;
    c->counter = h->counter;
    c->total_iter = h->total_iter;
    c->lastfit = h->lastfit;
    c->final_fit = h->final_fit;
    c->sweeps_run = 1;
    c->converged = (h->done && !h->nan_flag) ? 1 : 0;
    if (h->nan_flag) return fail(ITCPD_E_NAN, "Error NAN");
    return ITCPD_OK;
}

int itcpd_tensor_norm(itcpd_plan* p, double* norm_out) {
    if (!p || !norm_out) return fail(ITCPD_E_ARG, "null argument");
    DeviceGuard dg(p->device);
    int rc;
    if ((rc = launch_tensor_norm(p))) return rc;
    double ss = 0.0;
    ITCPD_HIP(hipMemcpyAsync(&ss, p->scal + 3, 8, hipMemcpyDeviceToHost, p->stream));
    ITCPD_HIP(hipStreamSynchronize(p->stream));
    *norm_out = std::sqrt(ss);
    return ITCPD_OK;
}

int itcpd_plan_set_precision(itcpd_plan* p, int32_t prec) {
    if (!p) return fail(ITCPD_E_ARG, "null plan");
    if (prec != ITCPD_FP64 && prec != ITCPD_FP32 && prec != ITCPD_BF16X3)
        return fail(ITCPD_E_UNSUPPORTED, "prec must be ITCPD_FP64, ITCPD_FP32 or ITCPD_BF16X3");
    DeviceGuard dg(p->device);
    ITCPD_HIP(hipStreamSynchronize(p->stream));
    if (prec != ITCPD_FP64) {
        int rc;
        if ((rc = ensure_lp_buffers(p))) return rc;
    }
    p->prec = prec;
    return ITCPD_OK;
}

int itcpd_gaussian_sketch(itcpd_plan* p, int32_t mode, int32_t K, uint64_t seed, double* S_out, int32_t mem) {
    if (!p || !S_out) return fail(ITCPD_E_ARG, "null argument");
    if (mode < 0 || mode >= p->N) return fail(ITCPD_E_ARG, "mode out of range");
    if (K < 1 || K > 64) return fail(ITCPD_E_ARG, "sketch width K must be in [1, 64]");
    if (p->dims[mode] > 256) return fail(ITCPD_E_UNSUPPORTED, "the Gaussian sketch takes modes of at most 256 rows");
    DeviceGuard dg(p->device);
    const int64_t n = p->dims[mode] * K;
    double* dst = S_out;
    int rc;
    if (mem == ITCPD_MEM_HOST) {
        if (p->smp_ws_cap < (size_t)n) {
            ITCPD_HIP(hipStreamSynchronize(p->stream));
            dfree(p->smp_ws);
            p->smp_ws = nullptr;
            p->smp_ws_cap = 0;
            if ((rc = dmalloc(&p->smp_ws, (size_t)n))) return rc;
            p->smp_ws_cap = (size_t)n;
        }
        dst = p->smp_ws;
    }
    if ((rc = launch_gauss_sketch(p, mode, K, seed, dst))) return rc;
    if (mem == ITCPD_MEM_HOST) {
        if ((rc = copy_out(S_out, dst, (size_t)n * 8, mem, p->stream))) return rc;
    }
    ITCPD_HIP(hipStreamSynchronize(p->stream));
    return ITCPD_OK;
}

int itcpd_plan_set_qr_forms(itcpd_plan* p, int64_t one_wg_max_cols, int64_t grid_min_rows) {
    if (!p) return fail(ITCPD_E_ARG, "null plan");
    if (one_wg_max_cols < 0 || grid_min_rows < 0) return fail(ITCPD_E_ARG, "thresholds must be >= 0");
    p->qr_one_wg_max = one_wg_max_cols;
    p->qr_grid_min_rows = grid_min_rows;
    return ITCPD_OK;
}

int itcpd_plan_set_profiling(itcpd_plan* p, int32_t on) {
    if (!p) return fail(ITCPD_E_ARG, "null plan");
    DeviceGuard dg(p->device);
    int rc;
    if ((rc = collect_timer(p, true))) return rc;   // retire outstanding events
    if (on < 0 || on > 3) return fail(ITCPD_E_ARG, "profiling must be 0 (off), 1 (both GEMMs), 2 (left) or 3 (right)");
    p->profiling = on != 0;
    p->profile_only = on == 2 ? ITCPD_KERNEL_GEMM_LEFT : (on == 3 ? ITCPD_KERNEL_GEMM_RIGHT : -1);
    p->profile_seen[0] = p->profile_seen[1] = 0;
    p->timer = KernelTimer();
    return ITCPD_OK;
}

int itcpd_plan_set_profiling_period(itcpd_plan* p, int32_t every) {
    if (!p) return fail(ITCPD_E_ARG, "null plan");
    if (every < 1) return fail(ITCPD_E_ARG, "the profiling period must be >= 1");
    p->profile_every = every;
    p->profile_seen[0] = p->profile_seen[1] = 0;
    return ITCPD_OK;
}

int itcpd_get_kernel_stats(itcpd_plan* p, int32_t kernel, itcpd_kernel_stats* st) {
    if (!p || !st) return fail(ITCPD_E_ARG, "null argument");
    if (kernel < ITCPD_KERNEL_GEMM_LEFT || kernel > ITCPD_KERNEL_GEMM_ALL)
        return fail(ITCPD_E_ARG, "unknown kernel id");
    DeviceGuard dg(p->device);
    int rc;
    if ((rc = collect_timer(p, true))) return rc;
    *st = itcpd_kernel_stats{0, 0.0, 0.0, 0.0};
    for (int k = 0; k < 2; ++k) {
        if (kernel != ITCPD_KERNEL_GEMM_ALL && kernel != k) continue;
        const KernelTimer::Acc& a = p->timer.acc[k];
        st->launches += a.launches;
        st->total_ms += a.total_ms;
        st->flops += a.flops;
        st->bytes += a.bytes;
    }
    return ITCPD_OK;
}

int itcpd_synchronize(itcpd_plan* p) {
    if (!p) return fail(ITCPD_E_ARG, "null plan");
    DeviceGuard dg(p->device);
    ITCPD_HIP(hipStreamSynchronize(p->stream));
    return ITCPD_OK;
}

}  // extern "C"

// ------------------------------------------------------------------ batches
struct itcpd_batch {
    int device = 0;
    hipStream_t stream = nullptr;
    itcpd::BatchDev d{};
    itcpd::BatchProblem* probs = nullptr;   // device
    int* order = nullptr;                   // device
    int* order_run = nullptr;               // device: the full run's group order
    std::vector<int> ord_host;              // the class order
    std::vector<double> work_host;          // per problem: I J K R
    double* T = nullptr;                    // device (owned copy or borrowed)
    bool T_owned = false;
    double* Tp = nullptr;                   // the mode-1 and mode-2 copies (owned; null without memory)
    double* factors = nullptr;
    double* backup = nullptr;               // factors saved across tuning runs
    double* lambdas = nullptr;
    double* fits = nullptr;
    int* counters = nullptr;                // one queue counter per class
    int64_t nfac = 0, nlam = 0, nel = 0;
    int nprob = 0;
    bool have_cpd = false;
    // one instantiated graph (every class's reset + persistent kernel) for the last
    // configuration and sweep count
    hipGraphExec_t gexec = nullptr;
    hipGraph_t graph = nullptr;
    uint64_t g_key = 0;
    int g_sweeps = -1;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    // classes 1.. run on their own streams inside the graph (fork/join events)
    itcpd::BatchFork fk{};
};

namespace itcpd {
namespace {

void batch_free(itcpd_batch* b) {
    if (!b) return;
    DeviceGuard dg(b->device);
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    if (b->gexec) (void)hipGraphExecDestroy(b->gexec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    if (b->ev0) (void)hipEventDestroy(b->ev0);
    if (b->ev1) (void)hipEventDestroy(b->ev1);
    if (b->fk.fork) (void)hipEventDestroy(b->fk.fork);
    for (int c = 0; c < BATCH_MAX_CLASSES - 1; ++c) {
        if (b->fk.join[c]) (void)hipEventDestroy(b->fk.join[c]);
        if (b->fk.side[c]) (void)hipStreamDestroy(b->fk.side[c]);
    }
    dfree(b->probs);
    dfree(b->order);
    dfree(b->order_run);
    if (b->T_owned) dfree(b->T);
    dfree(b->Tp);
    dfree(b->factors);
    dfree(b->backup);
    dfree(b->lambdas);
    dfree(b->fits);
    dfree(b->counters);
    if (b->stream) (void)hipStreamDestroy(b->stream);
    delete b;
}

// The launch configuration as a key: a graph is rebuilt when it (or the sweep
// count) changes.
uint64_t batch_key(const itcpd_batch* b) {
    uint64_t k = 0;
    for (int c = 0; c < b->d.nclass; ++c)
        k = k * 128 + (uint64_t)((b->d.cls[c].nt / 256) * 16 + b->d.cls[c].wpc);
    return k;
}

// The graph replays every class's reset + persistent kernel.
int batch_graph(itcpd_batch* b, int sweeps) {
    const uint64_t key = batch_key(b);
    if (b->gexec && b->g_key == key && b->g_sweeps == sweeps) return ITCPD_OK;
    if (b->gexec) { (void)hipGraphExecDestroy(b->gexec); b->gexec = nullptr; }
    if (b->graph) { (void)hipGraphDestroy(b->graph); b->graph = nullptr; }
    if (b->g_key != key) {
        std::vector<int> run((size_t)b->nprob);
        batch_groups(b->d, b->ord_host, b->work_host, run);
        ITCPD_HIP(hipStreamSynchronize(b->stream));
        ITCPD_HIP(hipMemcpy(b->order_run, run.data(), sizeof(int) * (size_t)b->nprob, hipMemcpyHostToDevice));
    }
    ITCPD_HIP(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
    const int rc = launch_batch(b->d, sweeps, b->stream, -1, &b->fk);
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(b->stream, &g);
    if (rc) { if (g) (void)hipGraphDestroy(g); return rc; }
    if (e != hipSuccess) return hip_fail(e, "hipStreamEndCapture");
    b->graph = g;
    ITCPD_HIP(hipGraphInstantiate(&b->gexec, g, nullptr, nullptr, 0));
    b->g_key = key;
    b->g_sweeps = sweeps;
    return ITCPD_OK;
}

int batch_launch_timed(itcpd_batch* b, int sweeps, double* ms) {
    int rc;
    if ((rc = batch_graph(b, sweeps))) return rc;
    ITCPD_HIP(hipEventRecord(b->ev0, b->stream));
    ITCPD_HIP(hipGraphLaunch(b->gexec, b->stream));
    ITCPD_HIP(hipEventRecord(b->ev1, b->stream));
    ITCPD_HIP(hipEventSynchronize(b->ev1));
    float f = 0.f;
    ITCPD_HIP(hipEventElapsedTime(&f, b->ev0, b->ev1));
    if (ms) *ms = f;
    return ITCPD_OK;
}

// One class alone, launched directly (the tuner's trial runs).
int batch_class_timed(itcpd_batch* b, int c, int sweeps, double* ms) {
    ITCPD_HIP(hipEventRecord(b->ev0, b->stream));
    int rc;
    if ((rc = launch_batch(b->d, sweeps, b->stream, c))) return rc;
    ITCPD_HIP(hipEventRecord(b->ev1, b->stream));
    ITCPD_HIP(hipEventSynchronize(b->ev1));
    float f = 0.f;
    ITCPD_HIP(hipEventElapsedTime(&f, b->ev0, b->ev1));
    if (ms) *ms = f;
    return ITCPD_OK;
}

constexpr size_t BATCH_LDS_CU = 160 * 1024;   // LDS of one CU

}  // namespace
}  // namespace itcpd

extern "C" {

int itcpd_batch_create(itcpd_batch** out, int32_t nprob, const int64_t* dims, const int32_t* ranks,
                       const double* tensors, int32_t tensor_mem, int32_t device) {
    if (!out) return fail(ITCPD_E_ARG, "batch pointer is null");
    *out = nullptr;
    if (nprob < 1 || !dims || !ranks || !tensors) return fail(ITCPD_E_ARG, "empty batch or null input");
    if (tensor_mem != ITCPD_MEM_HOST && tensor_mem != ITCPD_MEM_DEVICE)
        return fail(ITCPD_E_ARG, "tensor_mem must be ITCPD_MEM_HOST or ITCPD_MEM_DEVICE");
    std::vector<BatchProblem> hp((size_t)nprob);
    int64_t toff = 0, foff = 0, loff = 0;
    for (int b = 0; b < nprob; ++b) {
        const int64_t I = dims[3 * b], J = dims[3 * b + 1], K = dims[3 * b + 2];
        const int R = ranks[b];
        if (I < 1 || J < 1 || K < 1 || I > BATCH_MAXD || J > BATCH_MAXD || K > BATCH_MAXD)
            return fail(ITCPD_E_UNSUPPORTED, "batched problems need every dimension in [1, 96]");
        if (R < 1 || R > BATCH_MAXR) return fail(ITCPD_E_UNSUPPORTED, "batched problems need rank in [1, 32]");
        hp[b] = BatchProblem{toff, foff, (int)I, (int)J, (int)K, R, (int)loff, b};
        toff += I * J * K;
        foff += (I + J + K) * R;
        loff += R;
    }
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return fail(ITCPD_E_HIP, "no HIP device available");
    if (device < 0 || device >= ndev) return fail(ITCPD_E_ARG, "device index out of range");
    itcpd_batch* b = new (std::nothrow) itcpd_batch();
    if (!b) return fail(ITCPD_E_OOM, "host allocation failed");
    DeviceGuard dg(device);
    b->device = device;
    b->nprob = nprob;
    b->nel = toff;
    b->nfac = foff;
    b->nlam = loff;
    auto bail = [&](int code) { batch_free(b); return code; };
    hipError_t e = hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking);
    if (e != hipSuccess) return bail(hip_fail(e, "hipStreamCreate"));
    if ((e = hipEventCreate(&b->ev0)) != hipSuccess || (e = hipEventCreate(&b->ev1)) != hipSuccess)
        return bail(hip_fail(e, "hipEventCreate"));
    if ((e = hipEventCreateWithFlags(&b->fk.fork, hipEventDisableTiming)) != hipSuccess)
        return bail(hip_fail(e, "hipEventCreate"));
    for (int c = 0; c < BATCH_MAX_CLASSES - 1; ++c) {
        if ((e = hipStreamCreateWithFlags(&b->fk.side[c], hipStreamNonBlocking)) != hipSuccess)
            return bail(hip_fail(e, "hipStreamCreate"));
        if ((e = hipEventCreateWithFlags(&b->fk.join[c], hipEventDisableTiming)) != hipSuccess)
            return bail(hip_fail(e, "hipEventCreate"));
    }
    int rc;
    // classes by how many workgroups of the class's LDS fit on a CU (1, 2, 3, 4+),
    // the LDS taken at 512 threads; inside a class the most work first
    // (longest-processing-time order)
    std::vector<size_t> need((size_t)nprob);
    std::vector<int> cls_of((size_t)nprob);
    for (int q = 0; q < nprob; ++q) {
        need[q] = batch_problem_lds(hp[q].I, hp[q].J, hp[q].K, hp[q].R, 512);
        const size_t fit = BATCH_LDS_CU / need[q];
        cls_of[q] = (int)std::min<size_t>(fit, 4) - 1;   // 0: one per CU ... 3: four or more
    }
    std::vector<int> ord((size_t)nprob);
    for (int q = 0; q < nprob; ++q) ord[q] = q;
    std::stable_sort(ord.begin(), ord.end(), [&](int x, int y) {
        if (cls_of[x] != cls_of[y]) return cls_of[x] < cls_of[y];
        const double wx = (double)hp[x].I * hp[x].J * hp[x].K * hp[x].R;
        const double wy = (double)hp[y].I * hp[y].J * hp[y].K * hp[y].R;
        return wx > wy;
    });
    hipDeviceProp_t prop;
    e = hipGetDeviceProperties(&prop, device);
    if (e != hipSuccess) return bail(hip_fail(e, "hipGetDeviceProperties"));
    BatchDev d{};
    d.nclass = 0;
    for (int q = 0; q < nprob;) {
        const int c = cls_of[ord[q]];
        BatchClass cl{};
        cl.first = q;
        size_t mx = 0;
        int maxd = 0;
        while (q < nprob && cls_of[ord[q]] == c) {
            const BatchProblem& pb = hp[ord[q]];
            maxd = std::max(maxd, std::max(pb.I, std::max(pb.J, pb.K)));
            mx = std::max(mx, need[ord[q++]]);
        }
        cl.maxd = maxd;
        cl.count = q - cl.first;
        cl.lds = mx;
        cl.fit = (int)std::min<size_t>(BATCH_LDS_CU / mx, 4);
        cl.nt = 256;
        cl.wpc = cl.fit;
        d.cls[d.nclass++] = cl;
    }
    if ((rc = dmalloc(&b->probs, (size_t)nprob))) return bail(rc);
    if ((rc = dmalloc(&b->order, (size_t)nprob))) return bail(rc);
    if ((rc = dmalloc(&b->order_run, (size_t)nprob))) return bail(rc);
    if ((rc = dmalloc(&b->factors, (size_t)foff))) return bail(rc);
    if ((rc = dmalloc(&b->backup, (size_t)foff))) return bail(rc);
    if ((rc = dmalloc(&b->lambdas, (size_t)loff))) return bail(rc);
    if ((rc = dmalloc(&b->fits, (size_t)nprob))) return bail(rc);
    if ((rc = dmalloc(&b->counters, BATCH_MAX_CLASSES))) return bail(rc);
    e = hipMemcpy(b->probs, hp.data(), sizeof(BatchProblem) * nprob, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(b->order, ord.data(), sizeof(int) * nprob, hipMemcpyHostToDevice);
    if (e != hipSuccess) return bail(hip_fail(e, "hipMemcpy(batch descriptors)"));
    if (tensor_mem == ITCPD_MEM_HOST) {
        if ((rc = dmalloc(&b->T, (size_t)toff))) return bail(rc);
        b->T_owned = true;
        e = hipMemcpy(b->T, tensors, (size_t)toff * 8, hipMemcpyHostToDevice);
        if (e != hipSuccess) return bail(hip_fail(e, "hipMemcpy(tensors)"));
    } else {
        e = hipDeviceSynchronize();
        if (e != hipSuccess) return bail(hip_fail(e, "hipDeviceSynchronize"));
        b->T = const_cast<double*>(tensors);
    }
    d.probs = b->probs;
    d.order = b->order;
    d.order_run = b->order_run;
    d.ngroup = 0;
    b->ord_host = ord;
    b->work_host.resize((size_t)nprob);
    for (int q = 0; q < nprob; ++q)
        b->work_host[(size_t)q] = (double)hp[q].I * hp[q].J * hp[q].K * hp[q].R;
    d.nprob = nprob;
    d.T = b->T;
    // each mode's own copy of the tensors for the MTTKRPs of modes 1 and 2 (their loads
    // then read consecutive elements); without the memory those modes read T strided
    d.T1 = d.T2 = nullptr;
    if (hipMalloc((void**)&b->Tp, (size_t)(2 * toff) * 8) == hipSuccess) {
        d.T1 = b->Tp;
        d.T2 = b->Tp + toff;
        if ((rc = launch_batch_permute(d, b->Tp, b->Tp + toff, b->stream))) return bail(rc);
        e = hipStreamSynchronize(b->stream);
        if (e != hipSuccess) return bail(hip_fail(e, "batch tensor copies"));
    } else {
        (void)hipGetLastError();
        b->Tp = nullptr;
    }
    d.factors = b->factors;
    d.lambdas = b->lambdas;
    d.fits = b->fits;
    d.counters = b->counters;
    d.num_cu = prop.multiProcessorCount;
    b->d = d;
    *out = b;
    return ITCPD_OK;
}

int itcpd_batch_destroy(itcpd_batch* b) {
    batch_free(b);
    return ITCPD_OK;
}

int itcpd_batch_set_cpd(itcpd_batch* b, const double* factors, int32_t mem) {
    if (!b || !factors) return fail(ITCPD_E_ARG, "null argument");
    DeviceGuard dg(b->device);
    int rc;
    if ((rc = copy_in(b->factors, factors, (size_t)b->nfac * 8, mem, b->stream))) return rc;
    ITCPD_HIP(hipStreamSynchronize(b->stream));
    b->have_cpd = true;
    return ITCPD_OK;
}

int itcpd_batch_get_cpd(itcpd_batch* b, double* factors, double* lambdas, int32_t mem) {
    if (!b) return fail(ITCPD_E_ARG, "null batch");
    DeviceGuard dg(b->device);
    int rc;
    if (factors && (rc = copy_out(factors, b->factors, (size_t)b->nfac * 8, mem, b->stream))) return rc;
    if (lambdas && (rc = copy_out(lambdas, b->lambdas, (size_t)b->nlam * 8, mem, b->stream))) return rc;
    ITCPD_HIP(hipStreamSynchronize(b->stream));
    return ITCPD_OK;
}

int itcpd_batch_set_threads(itcpd_batch* b, int32_t threads) {
    if (!b) return fail(ITCPD_E_ARG, "null batch");
    if (threads != 256 && threads != 512 && threads != 1024)
        return fail(ITCPD_E_ARG, "threads must be 256, 512 or 1024");
    for (int c = 0; c < b->d.nclass; ++c) {
        BatchClass probe = b->d.cls[c];
        probe.nt = threads;
        if (threads == 1024 && batch_class_lds(probe) > BATCH_LDS_CU)
            return fail(ITCPD_E_ARG, "a class's LDS does not fit 1024 threads per workgroup");
    }
    for (int c = 0; c < b->d.nclass; ++c) {
        b->d.cls[c].nt = threads;
        if (threads == 1024) b->d.cls[c].wpc = 1;   // 16 waves of at most 128 registers: one per CU
    }
    return ITCPD_OK;
}

int itcpd_batch_run(itcpd_batch* b, int32_t sweeps, double* fits, double* elapsed_ms) {
    if (!b) return fail(ITCPD_E_ARG, "null batch");
    if (sweeps < 1) return fail(ITCPD_E_ARG, "sweeps must be >= 1");
    if (!b->have_cpd) return fail(ITCPD_E_STATE, "itcpd_batch_run before itcpd_batch_set_cpd");
    DeviceGuard dg(b->device);
    int rc;
    if ((rc = batch_launch_timed(b, sweeps, elapsed_ms))) return rc;
    if (fits) ITCPD_HIP(hipMemcpy(fits, b->fits, (size_t)b->nprob * 8, hipMemcpyDeviceToHost));
    return ITCPD_OK;
}

int itcpd_batch_tune(itcpd_batch* b, int32_t sweeps, int32_t* threads_chosen, double* ms_per_config) {
    if (!b) return fail(ITCPD_E_ARG, "null batch");
    if (sweeps < 1) return fail(ITCPD_E_ARG, "sweeps must be >= 1");
    if (!b->have_cpd) return fail(ITCPD_E_STATE, "itcpd_batch_tune before itcpd_batch_set_cpd");
    DeviceGuard dg(b->device);
    ITCPD_HIP(hipMemcpyAsync(b->backup, b->factors, (size_t)b->nfac * 8, hipMemcpyDeviceToDevice, b->stream));
    // per class: every (threads, workgroups per CU) the LDS allows, timed on the class
    // alone from the same factors; the fastest is kept.  1024 threads (16 waves, at most
    // 128 registers each): one workgroup per CU, when its LDS fits
    for (int c = 0; c < b->d.nclass; ++c) {
        BatchClass& cl = b->d.cls[c];
        double best = 1e300;
        int best_nt = cl.nt, best_wpc = cl.wpc;
        int k = 0;
        for (int nt : {256, 512, 1024}) {
            BatchClass probe = cl;
            probe.nt = nt;
            const int fit = nt == 1024 ? (batch_class_lds(probe) <= BATCH_LDS_CU ? 1 : 0) : cl.fit;
            for (int wpc = 1; wpc <= 4; ++wpc, ++k) {
                if (wpc > fit) {
                    if (ms_per_config) ms_per_config[BATCH_TUNE_SLOTS * c + k] = -1.0;
                    continue;
                }
                cl.nt = nt;
                cl.wpc = wpc;
                double ms = 0.0;
                int rc;
                if ((rc = batch_class_timed(b, c, sweeps, &ms))) return rc;
                if (ms_per_config) ms_per_config[BATCH_TUNE_SLOTS * c + k] = ms;
                if (ms < best) { best = ms; best_nt = nt; best_wpc = wpc; }
                ITCPD_HIP(hipMemcpyAsync(b->factors, b->backup, (size_t)b->nfac * 8, hipMemcpyDeviceToDevice,
                                         b->stream));
            }
        }
        cl.nt = best_nt;
        cl.wpc = best_wpc;
    }
    for (int c = b->d.nclass; c < BATCH_MAX_CLASSES; ++c)
        for (int k = 0; k < BATCH_TUNE_SLOTS; ++k)
            if (ms_per_config) ms_per_config[BATCH_TUNE_SLOTS * c + k] = -1.0;
    ITCPD_HIP(hipStreamSynchronize(b->stream));
    if (threads_chosen) *threads_chosen = b->d.cls[0].nt;
    return ITCPD_OK;
}

int itcpd_batch_get_config(itcpd_batch* b, int32_t* nclass, int32_t* counts, int32_t* threads, int32_t* wgs_per_cu,
                           int64_t* lds_bytes) {
    if (!b || !nclass) return fail(ITCPD_E_ARG, "null argument");
    *nclass = b->d.nclass;
    for (int c = 0; c < b->d.nclass; ++c) {
        if (counts) counts[c] = b->d.cls[c].count;
        if (threads) threads[c] = b->d.cls[c].nt;
        if (wgs_per_cu) wgs_per_cu[c] = b->d.cls[c].wpc;
        if (lds_bytes) lds_bytes[c] = (int64_t)batch_class_lds(b->d.cls[c]);
    }
    return ITCPD_OK;
}

}  // extern "C"

// ------------------------------------------------------ device utilities
extern "C" {

int itcpd_device_alloc(void** ptr, uint64_t bytes, int32_t device) {
    if (!ptr) return fail(ITCPD_E_ARG, "null pointer argument");
    *ptr = nullptr;
    DeviceGuard dg(device);
    const hipError_t e = hipMalloc(ptr, bytes ? bytes : 1);
    if (e != hipSuccess) return hip_fail(e, "hipMalloc");
    return ITCPD_OK;
}

int itcpd_device_free(void* ptr, int32_t device) {
    DeviceGuard dg(device);
    if (ptr) ITCPD_HIP(hipFree(ptr));
    return ITCPD_OK;
}

int itcpd_memcpy(void* dst, const void* src, uint64_t bytes, int32_t kind, int32_t device) {
    if ((!dst || !src) && bytes) return fail(ITCPD_E_ARG, "null pointer argument");
    const hipMemcpyKind k = kind == 0 ? hipMemcpyHostToDevice
                          : kind == 1 ? hipMemcpyDeviceToHost : hipMemcpyDeviceToDevice;
    if (kind < 0 || kind > 2) return fail(ITCPD_E_ARG, "kind must be 0 (to device), 1 (to host) or 2");
    DeviceGuard dg(device);
    ITCPD_HIP(hipMemcpy(dst, src, bytes, k));
    return ITCPD_OK;
}

int itcpd_reconstruct(int32_t order, const int64_t* dims, int64_t rank, const double* const* factors,
                      const double* lambda, int32_t mem, void* out, int32_t out_elt_bytes,
                      double noise_sigma, uint64_t seed, int32_t device) {
    if (order < 1 || order > ITCPD_MAX_ORDER) return fail(ITCPD_E_ARG, "order must be between 1 and 8");
    if (!dims || !factors || !lambda || !out) return fail(ITCPD_E_ARG, "null argument");
    if (rank < 1) return fail(ITCPD_E_ARG, "rank must be >= 1");
    if (out_elt_bytes != 8 && out_elt_bytes != 4) return fail(ITCPD_E_ARG, "out_elt_bytes must be 8 or 4");
    for (int n = 0; n < order; ++n)
        if (dims[n] < 1) return fail(ITCPD_E_ARG, "every dimension must be >= 1");
    DeviceGuard dg(device);
    hipStream_t st;
    ITCPD_HIP(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
    int64_t nfac = 0;
    for (int n = 0; n < order; ++n) nfac += dims[n] * rank;
    double* buf = nullptr;
    int rc = dmalloc(&buf, (size_t)(nfac + rank));
    const double* fdev[ITCPD_MAX_ORDER];
    int64_t off = 0;
    for (int n = 0; n < order && !rc; ++n) {
        rc = copy_in(buf + off, factors[n], (size_t)(dims[n] * rank) * 8, mem, st);
        fdev[n] = buf + off;
        off += dims[n] * rank;
    }
    if (!rc) rc = copy_in(buf + off, lambda, (size_t)rank * 8, mem, st);
    if (!rc) rc = launch_reconstruct(order, dims, rank, fdev, buf + off, out, out_elt_bytes, noise_sigma, seed, st);
    const hipError_t e = hipStreamSynchronize(st);
    dfree(buf);
    (void)hipStreamDestroy(st);
    if (rc) return rc;
    if (e != hipSuccess) return hip_fail(e, "hipStreamSynchronize");
    return ITCPD_OK;
}

}  // extern "C"

// ------------------------------------------------------------- the MLP
struct itcpd_mlp {
    int device = 0;
    hipStream_t stream = nullptr;
    itcpd::MlpDev m;
    float* xs = nullptr;   // host-input staging: batch_cap x in
    float* ys = nullptr;   // batch_cap x out (targets)
    float* ms = nullptr;   // batch_cap x out (mask)
};

namespace itcpd {
namespace {
void mlp_free(itcpd_mlp* q) {
    if (!q) return;
    DeviceGuard dg(q->device);
    if (q->stream) (void)hipStreamSynchronize(q->stream);
    MlpDev& m = q->m;
    dfree(m.params); dfree(m.grads); dfree(m.adam_m); dfree(m.adam_v);
    for (int l = 0; l < MLP_MAX_LAYERS; ++l) dfree(m.act[l]);
    dfree(m.dA); dfree(m.dB); dfree(m.loss_part); dfree(m.loss);
    dfree(q->xs); dfree(q->ys); dfree(q->ms);
    if (q->stream) (void)hipStreamDestroy(q->stream);
    delete q;
}

// stage host inputs (mem == HOST) into the network's buffers
int mlp_stage(itcpd_mlp* q, int batch, const float* X, const float* Yt, const float* mask, int mem,
              const float** Xd, const float** Yd, const float** Md) {
    const MlpDev& m = q->m;
    const size_t nin = (size_t)batch * m.widths[0], nout = (size_t)batch * m.widths[m.nlayers];
    if (mem == ITCPD_MEM_DEVICE) {
        *Xd = X; if (Yd) *Yd = Yt; if (Md) *Md = mask;
        return ITCPD_OK;
    }
    int rc;
    if ((rc = copy_in(q->xs, X, nin * 4, ITCPD_MEM_HOST, q->stream))) return rc;
    *Xd = q->xs;
    if (Yd) {
        if ((rc = copy_in(q->ys, Yt, nout * 4, ITCPD_MEM_HOST, q->stream))) return rc;
        *Yd = q->ys;
    }
    if (Md) {
        if (mask && (rc = copy_in(q->ms, mask, nout * 4, ITCPD_MEM_HOST, q->stream))) return rc;
        *Md = mask ? q->ms : nullptr;
    }
    return ITCPD_OK;
}

int mlp_check(itcpd_mlp* q, int batch, const void* X) {
    if (!q || !X) return fail(ITCPD_E_ARG, "null argument");
    if (batch < 1 || batch > q->m.batch_cap) return fail(ITCPD_E_ARG, "batch must be in [1, batch_cap]");
    return ITCPD_OK;
}
}  // namespace
}  // namespace itcpd

extern "C" {

int itcpd_mlp_create(itcpd_mlp** out, int32_t nlayers, const int32_t* widths, int32_t batch_cap,
                     uint64_t seed, int32_t device) {
    if (!out || !widths) return fail(ITCPD_E_ARG, "null argument");
    *out = nullptr;
    if (nlayers < 1 || nlayers > MLP_MAX_LAYERS) return fail(ITCPD_E_ARG, "nlayers must be in [1, 6]");
    if (batch_cap < 1) return fail(ITCPD_E_ARG, "batch_cap must be >= 1");
    for (int l = 0; l <= nlayers; ++l)
        if (widths[l] < 1) return fail(ITCPD_E_ARG, "every width must be >= 1");
    itcpd_mlp* q = new (std::nothrow) itcpd_mlp();
    if (!q) return fail(ITCPD_E_OOM, "host allocation failed");
    DeviceGuard dg(device);
    q->device = device;
    MlpDev& m = q->m;
    m.nlayers = nlayers;
    m.batch_cap = batch_cap;
    int maxw = 0;
    for (int l = 0; l <= nlayers; ++l) { m.widths[l] = widths[l]; maxw = std::max(maxw, widths[l]); }
    int64_t np = 0;
    for (int l = 0; l < nlayers; ++l) np += (int64_t)widths[l] * widths[l + 1] + widths[l + 1];
    m.nparams = np;
    auto bail = [&](int code) { mlp_free(q); return code; };
    hipError_t e = hipStreamCreateWithFlags(&q->stream, hipStreamNonBlocking);
    if (e != hipSuccess) return bail(hip_fail(e, "hipStreamCreate"));
    int rc;
    if ((rc = dmalloc(&m.params, (size_t)np))) return bail(rc);
    if ((rc = dmalloc(&m.grads, (size_t)np))) return bail(rc);
    if ((rc = dmalloc(&m.adam_m, (size_t)np))) return bail(rc);
    if ((rc = dmalloc(&m.adam_v, (size_t)np))) return bail(rc);
    for (int l = 0; l < nlayers; ++l)
        if ((rc = dmalloc(&m.act[l], (size_t)batch_cap * widths[l + 1]))) return bail(rc);
    if ((rc = dmalloc(&m.dA, (size_t)batch_cap * maxw))) return bail(rc);
    if ((rc = dmalloc(&m.dB, (size_t)batch_cap * maxw))) return bail(rc);
    if ((rc = dmalloc(&m.loss_part, (size_t)((int64_t)batch_cap * widths[nlayers] / 256 + 2)))) return bail(rc);
    if ((rc = dmalloc(&m.loss, 1))) return bail(rc);
    if ((rc = dmalloc(&q->xs, (size_t)batch_cap * widths[0]))) return bail(rc);
    if ((rc = dmalloc(&q->ys, (size_t)batch_cap * widths[nlayers]))) return bail(rc);
    if ((rc = dmalloc(&q->ms, (size_t)batch_cap * widths[nlayers]))) return bail(rc);
    // He-uniform weights (bound sqrt(6 / fan_in)), zero biases; host stream seeded by `seed`
    std::vector<float> h((size_t)np);
    uint64_t s = seed * 0x9E3779B97F4A7C15ull + 0x632BE59BD9B4E019ull;
    auto next = [&]() {   // splitmix64
        s += 0x9E3779B97F4A7C15ull;
        uint64_t z = s;
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return z ^ (z >> 31);
    };
    int64_t off = 0;
    for (int l = 0; l < nlayers; ++l) {
        const int64_t nw = (int64_t)widths[l] * widths[l + 1];
        const float bound = std::sqrt(6.0f / (float)widths[l]);
        for (int64_t i = 0; i < nw; ++i) {
            const double u = (double)(next() >> 11) * (1.0 / 9007199254740992.0);
            h[off + i] = (float)((2.0 * u - 1.0) * bound);
        }
        m.W[l] = m.params + off;
        m.gW[l] = m.grads + off;
        off += nw;
        for (int j = 0; j < widths[l + 1]; ++j) h[off + j] = 0.f;
        m.b[l] = m.params + off;
        m.gb[l] = m.grads + off;
        off += widths[l + 1];
    }
    e = hipMemcpy(m.params, h.data(), (size_t)np * 4, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemset(m.adam_m, 0, (size_t)np * 4);
    if (e == hipSuccess) e = hipMemset(m.adam_v, 0, (size_t)np * 4);
    if (e != hipSuccess) return bail(hip_fail(e, "hipMemcpy(mlp init)"));
    *out = q;
    return ITCPD_OK;
}

int itcpd_mlp_destroy(itcpd_mlp* q) {
    mlp_free(q);
    return ITCPD_OK;
}

int itcpd_mlp_num_params(itcpd_mlp* q, int64_t* n) {
    if (!q || !n) return fail(ITCPD_E_ARG, "null argument");
    *n = q->m.nparams;
    return ITCPD_OK;
}

int itcpd_mlp_get_params(itcpd_mlp* q, float* out, int32_t mem) {
    if (!q || !out) return fail(ITCPD_E_ARG, "null argument");
    DeviceGuard dg(q->device);
    int rc;
    if ((rc = copy_out(out, q->m.params, (size_t)q->m.nparams * 4, mem, q->stream))) return rc;
    ITCPD_HIP(hipStreamSynchronize(q->stream));
    return ITCPD_OK;
}

int itcpd_mlp_set_params(itcpd_mlp* q, const float* in, int32_t mem) {
    if (!q || !in) return fail(ITCPD_E_ARG, "null argument");
    DeviceGuard dg(q->device);
    int rc;
    if ((rc = copy_in(q->m.params, in, (size_t)q->m.nparams * 4, mem, q->stream))) return rc;
    ITCPD_HIP(hipStreamSynchronize(q->stream));
    return ITCPD_OK;
}

int itcpd_mlp_forward(itcpd_mlp* q, int32_t batch, const float* X, int32_t mem, float* Y) {
    int rc;
    if ((rc = mlp_check(q, batch, X))) return rc;
    if (!Y) return fail(ITCPD_E_ARG, "null output");
    DeviceGuard dg(q->device);
    const float* Xd;
    if ((rc = mlp_stage(q, batch, X, nullptr, nullptr, mem, &Xd, nullptr, nullptr))) return rc;
    if ((rc = mlp_forward(q->m, batch, Xd, q->stream))) return rc;
    const MlpDev& m = q->m;
    if ((rc = copy_out(Y, m.act[m.nlayers - 1], (size_t)batch * m.widths[m.nlayers] * 4, mem, q->stream))) return rc;
    ITCPD_HIP(hipStreamSynchronize(q->stream));
    return ITCPD_OK;
}

int itcpd_mlp_gradients(itcpd_mlp* q, int32_t batch, const float* X, const float* Yt, const float* mask,
                        int32_t mem, float* grads, double* loss) {
    int rc;
    if ((rc = mlp_check(q, batch, X))) return rc;
    if (!Yt) return fail(ITCPD_E_ARG, "null target");
    DeviceGuard dg(q->device);
    const float *Xd, *Yd, *Md;
    if ((rc = mlp_stage(q, batch, X, Yt, mask, mem, &Xd, &Yd, &Md))) return rc;
    if ((rc = mlp_forward(q->m, batch, Xd, q->stream))) return rc;
    if ((rc = mlp_backward(q->m, batch, Xd, Yd, Md, q->m.loss, q->stream))) return rc;
    if (grads && (rc = copy_out(grads, q->m.grads, (size_t)q->m.nparams * 4, mem, q->stream))) return rc;
    if (loss) ITCPD_HIP(hipMemcpyAsync(loss, q->m.loss, 8, hipMemcpyDeviceToHost, q->stream));
    ITCPD_HIP(hipStreamSynchronize(q->stream));
    return ITCPD_OK;
}

int itcpd_mlp_train_step(itcpd_mlp* q, int32_t batch, const float* X, const float* Yt, const float* mask,
                         int32_t mem, float lr, double* loss) {
    int rc;
    if ((rc = mlp_check(q, batch, X))) return rc;
    if (!Yt) return fail(ITCPD_E_ARG, "null target");
    DeviceGuard dg(q->device);
    const float *Xd, *Yd, *Md;
    if ((rc = mlp_stage(q, batch, X, Yt, mask, mem, &Xd, &Yd, &Md))) return rc;
    if ((rc = mlp_forward(q->m, batch, Xd, q->stream))) return rc;
    if ((rc = mlp_backward(q->m, batch, Xd, Yd, Md, q->m.loss, q->stream))) return rc;
    if ((rc = mlp_adam(q->m, lr, q->stream))) return rc;
    if (loss) ITCPD_HIP(hipMemcpyAsync(loss, q->m.loss, 8, hipMemcpyDeviceToHost, q->stream));
    ITCPD_HIP(hipStreamSynchronize(q->stream));   // host inputs may be reused by the caller
    return ITCPD_OK;
}

}  // extern "C"

extern "C" {

int itcpd_sketch_candidates(int32_t nsk, int32_t D, int32_t K, int32_t ncand, const double* S,
                            int32_t mem, float* out, int32_t device) {
    if (!S || !out) return fail(ITCPD_E_ARG, "null argument");
    if (nsk < 1 || D < 1 || D > 256 || K < 1 || K > 64 || ncand < 1 || ncand > K)
        return fail(ITCPD_E_ARG, "need nsk >= 1, 1 <= D <= 256, 1 <= ncand <= K <= 64");
    DeviceGuard dg(device);
    hipStream_t st;
    ITCPD_HIP(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
    double* Sd = nullptr;
    float* od = nullptr;
    const size_t ns = (size_t)nsk * D * K, no = (size_t)nsk * ncand * D;
    int rc = ITCPD_OK;
    if (mem == ITCPD_MEM_HOST) {
        rc = dmalloc(&Sd, ns);
        if (!rc) rc = dmalloc(&od, no);
        if (!rc) rc = copy_in(Sd, S, ns * 8, ITCPD_MEM_HOST, st);
    }
    if (!rc) rc = launch_spa_candidates(nsk, D, K, ncand, Sd ? Sd : S, od ? od : out, st);
    if (!rc && od) rc = copy_out(out, od, no * 4, ITCPD_MEM_HOST, st);
    const hipError_t e = hipStreamSynchronize(st);
    dfree(Sd);
    dfree(od);
    (void)hipStreamDestroy(st);
    if (rc) return rc;
    if (e != hipSuccess) return hip_fail(e, "hipStreamSynchronize");
    return ITCPD_OK;
}

}  // extern "C"
