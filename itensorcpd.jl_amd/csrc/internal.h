// Internal declarations shared by the engine's translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "itcpd.h"

#define ITCPD_MAX_ORDER 8
#define ITCPD_MAX_RANK 1024
#define ITCPD_POLL_SLOTS 4       // in-flight FitCheck state snapshots per run
#define SOLVE_MAX_PARTS 16       // M partials the R <= 64 row solves sum while loading

namespace itcpd {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d16 __attribute__((ext_vector_type(16)));

// v_mfma_f64_16x16x4f64 on gfx950 (layout measured on the device):
//   A operand: lane l holds A[l & 15][l >> 4]
//   B operand: lane l holds B[l >> 4][l & 15]
//   result   : lane l, register v holds D[(l >> 4) + 4 v][l & 15]
__device__ __forceinline__ d4 mfma_f64(double a, double b, d4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Philox-4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11), ten rounds on the counter c
// with key (k0, k1).  The engine's streams use counter = (element lo, element hi,
// stream tag, 0) and key = (seed lo, seed hi), and one N(0,1) value per counter by
// Box-Muller on two 53-bit uniforms (u1 in (0, 1], u2 in [0, 1)).
__device__ __forceinline__ void philox4x32_10(uint32_t c[4], uint32_t k0, uint32_t k1) {
    for (int r = 0; r < 10; ++r) {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c[0];
        const uint64_t p1 = (uint64_t)0xCD9E8D57u * c[2];
        const uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0;
        const uint32_t hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
        const uint32_t n0 = hi1 ^ c[1] ^ k0, n2 = hi0 ^ c[3] ^ k1;
        c[0] = n0; c[1] = lo1; c[2] = n2; c[3] = lo0;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
}
__device__ __forceinline__ double philox_normal(uint64_t e, uint32_t tag, uint64_t seed) {
    uint32_t c[4] = {(uint32_t)e, (uint32_t)(e >> 32), tag, 0u};
    philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
    const uint64_t a = ((uint64_t)c[0] << 32) | c[1];
    const uint64_t b = ((uint64_t)c[2] << 32) | c[3];
    const double u1 = (double)((a >> 11) + 1) * 1.1102230246251565e-16;
    const double u2 = (double)(b >> 11) * 1.1102230246251565e-16;
    return sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
}

// Device-side copy of the convergence-check state (FitCheck / NoCheck fields).
struct DevCheck {
    int kind;
    int iter;
    int counter;
    int max_counter;
    int total_iter;
    int done;        // check_converge returned true, or NaN: later sweeps are no-ops
    int nan_flag;
    int sweeps;      // sweeps executed since the last reset
    double tolerance;
    double ref_norm;
    double lastfit;
    double final_fit;
    int has_prev;    // CPDiff / CPAngle: the previous sweep's CPD is held
    int pad_;
    double norm_prev;  // CPDiff: ||X_prev||^2, CPAngle: ||X_prev||
};

// One side of the dimension tree: the modes a GEMM contracts against T.
struct Side {
    int nm;                              // number of modes on this side
    int first;                           // index of the first mode of the side
    int64_t dim[ITCPD_MAX_ORDER];        // dims of the side's modes (first is fastest)
    const double* fac[ITCPD_MAX_ORDER];  // factor pointers, layout set by the consumer
};

struct KernelTimer {
    struct Acc {
        int64_t launches = 0;
        double total_ms = 0, flops = 0, bytes = 0;
    };
    std::vector<hipEvent_t> ev;          // begin/end pairs recorded this run
    Acc acc[2];                          // 0: left GEMM, 1: right GEMM
    std::vector<double> pending_flops, pending_bytes;
    std::vector<int> pending_kind;
};

}  // namespace itcpd

namespace itcpd {
// An MTTKRP result: M(i, r) = sum_{z < nparts} ptr[z * stride + i + I_n * r].
struct MSrc {
    const double* ptr;
    int nparts;
    int64_t stride;
};
}  // namespace itcpd

struct itcpd_plan {
    int device = 0;
    int num_cu = 256;                          // compute units of the device
    hipStream_t stream = nullptr;
    int N = 0;
    int64_t dims[ITCPD_MAX_ORDER] = {0};
    int64_t R = 0, Rp = 0;   // rank and padded rank (multiple of 16 * RB)
    int RB = 4;              // rank blocks of 16 per wave in the GEMMs
    int elt_bytes = 8;
    const void* T = nullptr;
    void* T_owned = nullptr;
    int prec = ITCPD_FP64;
    int alg = ITCPD_ALG_KRP_FREE_NORMAL;
    int s = 1;               // dimension-tree split: left = modes [0, s), right = [s, N)
    int64_t ML = 1, MR = 1;  // products of left / right dims
    int64_t maxI = 0;
    bool have_cpd = false;

    // device state: one allocation (arena), the CPD (factors, lambda) at its start
    char* arena = nullptr;
    size_t cpd_bytes = 0, zero_bytes = 0;
    char* stage = nullptr;                     // pinned mirror of the CPD region (made on first use)
    bool stage_failed = false;
    double* trace_owned = nullptr;             // fit trace of a run longer than the arena's
    double* A[ITCPD_MAX_ORDER] = {nullptr};    // I_n x Rp column-major (zero beyond R)
    double* At[ITCPD_MAX_ORDER] = {nullptr};   // Rp x I_n (rank fastest, zero beyond R)
    double* G[ITCPD_MAX_ORDER] = {nullptr};    // R x R
    double* lam = nullptr;                     // Rp
    double* X = nullptr;                       // maxI x R column-major (unnormalised solution)
    double* M = nullptr;                       // maxI x R column-major (summed MTTKRP)
    double* U = nullptr;                       // R x R factor workspace (Cholesky / QR)
    double* qr_aux = nullptr;                  // QR fallback workspace (tau, Z reflectors)
    double* invdiag = nullptr;                 // R: 1 / U(j,j) of the pivoted Cholesky
    double* Upad = nullptr;                    // R <= 64: V^-1 (R x R) from the factor kernel
    double* inv_buf = nullptr;                 // R > 64: two (64 nb)^2 buffers of the blocked inverse
    double* inv_stat = nullptr;                // norms and flags of the certificate
    int RT = 0;                                // 16, 32 or 64 for R <= 64, else 0
    double* Msum = nullptr;                    // maxI x R: summed MTTKRP of the last mode (fit)
    unsigned* counters = nullptr;              // arrival counters of last-block reductions
    int* piv = nullptr;                        // R
    int* finfo = nullptr;                      // [0] = rank, [1] = used fallback, [2] = QR rank
    itcpd::MSrc side{};                        // the current side's partial: PL, PR or its GEMM's parts
    double* PL = nullptr;                      // ML x Rp partial of the left side (if s > 1)
    float* Kt = nullptr;                       // reduced precision: a side's Khatri-Rao product, rank-major
    double* Wrest = nullptr;                   // a side's Khatri-Rao product or rest weights (rank fastest)
    double* P3 = nullptr;                      // order 3: the partial that serves two mode updates (tree3):
    double* P3_owned = nullptr;                // PL or PR, or this where neither is large enough
    bool tree3 = false;                        // order 3: partials shared across sweeps
    double* PR = nullptr;                      // MR x Rp partial of the right side (if N-s > 1)
    double* parts = nullptr;                   // split-K partial buffer
    size_t parts_elems = 0;
    double* sumsq_part = nullptr;              // [nb][Rp]
    double* gram_part = nullptr;               // [nb][R*R]
    double* inner_part = nullptr;              // [nb]
    double* scal = nullptr;                    // [0]=inner [1]=fact_square [2]=fit [3]=tensor norm^2
    itcpd::DevCheck* chk = nullptr;
    double* fit_trace = nullptr;               // device, length trace_cap
    int trace_cap = 0;
    itcpd::DevCheck* chk_host = nullptr;       // pinned mirror, then ITCPD_POLL_SLOTS poll slots
    hipEvent_t ev_poll[ITCPD_POLL_SLOTS] = {nullptr};
    bool profiling = false;
    int profile_only = -1;                     // >= 0: time only this GEMM kind (0 left, 1 right)
    int profile_every = 1;                     // time every n-th launch of a timed kind
    int64_t profile_seen[2] = {0, 0};          // launches of each kind since profiling was set
    itcpd::KernelTimer timer;
    // CPDiffCheck / CPAngleCheck: the previous sweep's CPD (rank-fastest factors and
    // lambda), cross-Gram partials A_prev^T A per mode and row chunk
    int check_kind = 0;
    double* Atprev[ITCPD_MAX_ORDER] = {nullptr};
    double* lamprev = nullptr;
    double* xg_part = nullptr;
    int xg_chunks = 0;
    bool prev_valid = false;
    // leverage-score-sampled steps: grow-only workspaces, and the V the factorisation
    // takes instead of the Hadamard of the Grams (when set)
    double* smp_ws = nullptr;
    size_t smp_ws_cap = 0;
    int* smp_iws = nullptr;
    size_t smp_iws_cap = 0;
    const double* v_override = nullptr;
    // column-pivoted QR forms: the widest matrix whose QR runs in one workgroup (wider
    // ones take a step per three grid-wide launches), and the shortest sampled block
    // whose QR takes the grid-wide steps; both forms give the same bits
    double* sk_ws = nullptr;                   // Gaussian sketch partials (grow-only)
    size_t sk_ws_cap = 0;
    int64_t qr_one_wg_max = 4096;
    int64_t qr_grid_min_rows = 1024;
};

namespace itcpd {

// error plumbing (api.hip)
void set_error(const std::string& msg);
int fail(int code, const std::string& msg);
int hip_fail(hipError_t e, const char* what);

// launchers (mttkrp.hip)
// PL (or M of mode 0 when s == 1) / PR (or M of mode N-1 when N-s == 1).  With
// factor_mode >= 0 the launch may also run that mode's R <= 64 factorisation in an
// extra workgroup; *fused says whether it did (otherwise the caller launches it).
int launch_left_gemm(itcpd_plan* p, MSrc* ms, int factor_mode = -1);
int launch_right_gemm(itcpd_plan* p, MSrc* ms, int factor_mode = -1);
// M of `mode` from PL / PR; with factor_mode >= 0 also that mode's factorisation
int launch_side_ttv(itcpd_plan* p, int mode, MSrc* ms, int factor_mode = -1);
// order 3 across sweeps: the partial of T contracted over mode c, and a mode's M from it
bool tree3_pays(const itcpd_plan* p);
int64_t tree3_elems(const itcpd_plan* p);
int launch_tree3_gemm(itcpd_plan* p, int c);
int launch_tree3_ttv(itcpd_plan* p, int mode, int c, MSrc* ms, int factor_mode);
int64_t lp_krp_elems(const itcpd_plan* p);     // 4-byte elements of p->Kt
int64_t krp64_elems(const itcpd_plan* p);      // doubles of p->Wrest
int mttkrp_mode(itcpd_plan* p, int mode);      // full M_mode into p->M from the current factors
// out = the sum of ms's partials; factor_mode >= 0: that mode's factorisation too
// (in an extra workgroup for R <= 64, else as its own launch after the sum);
// fallback_only: only its pivoted form, when the unpivoted one (along the right
// GEMM) did not certify its result
int launch_sum_parts(itcpd_plan* p, const MSrc& ms, int64_t n, double* out, int factor_mode = -1,
                     bool fallback_only = false);
int launch_tensor_norm(itcpd_plan* p);

// launchers (solve.hip)
int launch_update_mode(itcpd_plan* p, int mode, bool fit_after, const double* Msrc, int nparts,
                       int64_t stride);  // factor + solve + row_norm + post_solve (+ fit)
int launch_factor(itcpd_plan* p, int mode);
int launch_factor_on(itcpd_plan* p, int mode, hipStream_t st);
size_t inv_stat_elems(int64_t R);              // doubles of p->inv_stat
int launch_cp_check(itcpd_plan* p);
// solve + row_norm + Gram refresh of `mode` (finalize), the fit after the last mode
// (fit_after), then next_factor's factorisation (>= 0), all on the plan's stream
int launch_solve(itcpd_plan* p, int mode, const double* Msrc, int nparts, int64_t stride,
                 bool finalize, bool fit_after, int next_factor = -1);
int launch_normalize(itcpd_plan* p, int mode, const double* Xsrc, bool fit_after);
// (A_n, lambda) and G_n from p->X, unless *hold (device, nullable) is nonzero
int launch_row_norm(itcpd_plan* p, int mode, const int* hold);
int launch_seed_grams(itcpd_plan* p);
int launch_reset_flags(itcpd_plan* p);         // chk->done = chk->nan_flag = 0
int launch_random_init(itcpd_plan* p, uint64_t seed);
int launch_fit_only(itcpd_plan* p, const double* Mlast, double ref_norm);
int launch_hadamard(itcpd_plan* p, int mode, double* V);
int launch_col_sumsq(itcpd_plan* p, int mode, const double* X);
// leverage-score-sampled ALS (sampled.hip)
int launch_leverage_scores(itcpd_plan* p, int mode, double* probs_dev, double** probs_used);
int sampled_ws_prepare(itcpd_plan* p, int mode, int64_t ns);
// form: the normal equations, the column-pivoted QR, or corrected normal equations in its place
enum { SAMPLED_NORMAL, SAMPLED_QR, SAMPLED_CORRECTED };
bool sampled_corrected_ok(const itcpd_plan* p, int64_t ns);
int launch_sampled_gather(itcpd_plan* p, int mode, int64_t ns, const int* samples);
int launch_sampled_solve(itcpd_plan* p, int mode, int64_t ns, int form);
int launch_qr_pivots(itcpd_plan* p, int mode, bool krp, const int64_t* cols, int64_t ncols,
                     const int64_t* omega_rowptr, const int64_t* omega_cols, const double* omega_vals, int64_t l,
                     int* jpvt_dev, double* rdiag_dev);
int launch_sparse_sign(int d, int64_t m, int zeta, bool injective, uint64_t seed, double* vals_dev, int* rows_dev,
                       hipStream_t st);

inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }


// ------------------------------------------------------------ host helpers
// Makes `dev` current for the scope and restores the caller's device after.
struct DeviceGuard {
    int prev = -1;
    explicit DeviceGuard(int dev) {
        if (hipGetDevice(&prev) != hipSuccess) prev = -1;
        (void)hipSetDevice(dev);
    }
    ~DeviceGuard() {
        if (prev >= 0) (void)hipSetDevice(prev);
    }
};

template <typename T>
inline int dmalloc(T** ptr, size_t count) {
    *ptr = nullptr;
    if (count == 0) count = 1;
    hipError_t e = hipMalloc((void**)ptr, count * sizeof(T));
    if (e != hipSuccess) return hip_fail(e, "hipMalloc");
    return ITCPD_OK;
}

inline void dfree(void* p) {
    if (p) (void)hipFree(p);
}

inline int copy_in(void* dst, const void* src, size_t bytes, int mem, hipStream_t st) {
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, mem == ITCPD_MEM_DEVICE ? hipMemcpyDeviceToDevice
                                                                                 : hipMemcpyHostToDevice, st);
    return e == hipSuccess ? ITCPD_OK : hip_fail(e, "hipMemcpyAsync(in)");
}
inline int copy_out(void* dst, const void* src, size_t bytes, int mem, hipStream_t st) {
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, mem == ITCPD_MEM_DEVICE ? hipMemcpyDeviceToDevice
                                                                                 : hipMemcpyDeviceToHost, st);
    return e == hipSuccess ? ITCPD_OK : hip_fail(e, "hipMemcpyAsync(out)");
}

// ------------------------------------------------------------ warm-start MLP
constexpr int MLP_MAX_LAYERS = 6;

struct MlpDev {
    int nlayers = 0;
    int widths[MLP_MAX_LAYERS + 1] = {0};
    int64_t nparams = 0;
    float* params = nullptr;    // W_0 | b_0 | W_1 | b_1 | ...  (W_l: widths[l] x widths[l+1] row-major)
    float* grads = nullptr;     // same layout
    float* adam_m = nullptr;
    float* adam_v = nullptr;
    float* W[MLP_MAX_LAYERS] = {nullptr};
    float* b[MLP_MAX_LAYERS] = {nullptr};
    float* gW[MLP_MAX_LAYERS] = {nullptr};
    float* gb[MLP_MAX_LAYERS] = {nullptr};
    float* act[MLP_MAX_LAYERS] = {nullptr};   // batch_cap x widths[l+1]
    float* dA = nullptr;                      // batch_cap x max width (two gradient buffers)
    float* dB = nullptr;
    double* loss_part = nullptr;
    double* loss = nullptr;
    int batch_cap = 0;
    int64_t step = 0;
};

int mlp_forward(const MlpDev& m, int batch, const float* X, hipStream_t st);
int mlp_backward(const MlpDev& m, int batch, const float* X, const float* Yt, const float* mask,
                 double* loss_dev, hipStream_t st);
int mlp_adam(MlpDev& m, float lr, hipStream_t st);
int launch_spa_candidates(int nsk, int D, int K, int ncand, const double* S, float* out, hipStream_t st);
// S = T_(mode) Omega with Omega a Gaussian (prod of the other dims) x K matrix drawn on
// the fly from the Philox stream of `seed` (tag OMEGA_TAG); S_dev: I_mode x K
constexpr uint32_t OMEGA_TAG = 0x4F6D6567u;
int launch_gauss_sketch(itcpd_plan* p, int mode, int K, uint64_t seed, double* S_dev);
constexpr int SK_CH = 32;   // unfolding columns per chunk of the sketch kernel
void sketch_geometry(int order, const int64_t* dims, int mode, int64_t* A, int64_t* M);
hipError_t enqueue_gauss_sketch(const void* T, int elt_bytes, int64_t In, int64_t A, int64_t M, int K,
                                uint64_t seed, int nb, double* part, double* S_dev, hipStream_t st);

// reconstruct.jl:2-9 on the device (+ optional N(0, sigma^2) noise, Philox stream)
int launch_reconstruct(int order, const int64_t* dims, int64_t rank, const double* const* factors_dev,
                       const double* lambda_dev, void* out, int out_elt, double sigma, uint64_t seed,
                       hipStream_t st);

// ----------------------------------------------------------------- batches
constexpr int BATCH_MAXD = 96;   // largest mode size of a batched problem
constexpr int BATCH_MAXR = 32;   // largest rank of a batched problem

struct BatchProblem {
    int64_t toff;    // offset of the problem's tensor (elements, column-major)
    int64_t foff;    // offset of its factors (A_0 | A_1 | A_2, each I_n x R column-major)
    int I, J, K, R;
    int loff;        // offset of its lambda
    int index;       // position in the caller's list
};

// Problems sharing one persistent launch: their largest LDS need sets the
// workgroup's LDS; the autotuner picks threads per workgroup and workgroups per CU.
struct BatchClass {
    int first, count;        // range of the class in the queue order
    size_t lds;              // dynamic LDS bytes per workgroup
    int nt;                  // threads per workgroup: 256, 512 or 1024
    int wpc;                 // persistent workgroups per CU
    int fit;                 // most workgroups per CU the LDS allows (<= 4)
    int maxd;                // largest mode size in the class
};
constexpr int BATCH_MAX_CLASSES = 4;
// tuner timings per class: (256, 512, 1024 threads) x (1..4 workgroups per CU)
constexpr int BATCH_TUNE_SLOTS = 12;

struct BatchDev {
    const BatchProblem* probs;
    const int* order;        // queue order: classes one after another, most work first
    int nprob;
    const double* T;
    const double* T1;        // T(j, i, k) and T(k, i, j) per problem (null: modes 1, 2 read T)
    const double* T2;
    double* factors;
    double* lambdas;
    double* fits;
    int* counters;           // one queue counter per class
    int num_cu;
    int nclass;
    BatchClass cls[BATCH_MAX_CLASSES];
    // The launches of a full run: classes that run alike (same threads and tile count,
    // one workgroup per CU) share one queue, re-sorted most work first in order_run
    const int* order_run;
    int ngroup;
    BatchClass grp[BATCH_MAX_CLASSES];
};

// Groups the classes for a full run (d.grp, d.ngroup) and fills `run` (host, nprob) with
// each group's problems, most work first (`work` per problem, `ord` the class order).
void batch_groups(BatchDev& d, const std::vector<int>& ord, const std::vector<double>& work,
                  std::vector<int>& run);

// LDS bytes one problem takes in the batch kernel (threads per workgroup nt)
size_t batch_problem_lds(int I, int J, int K, int R, int nt);
// a class's LDS per workgroup at its thread count
size_t batch_class_lds(const BatchClass& cl);
// Streams and events that let the classes run side by side: class c >= 1 goes on
// side[c - 1], forked from the launching stream after `fork` and joined back by join[c - 1].
struct BatchFork {
    hipStream_t side[BATCH_MAX_CLASSES - 1];
    hipEvent_t fork;
    hipEvent_t join[BATCH_MAX_CLASSES - 1];
};

// Enqueues every class (or only class `only` >= 0): counter reset + persistent kernel.
// With `fk` (and every class), classes 1.. run on the side streams, so the workgroups of a
// class take the CUs that the workgroups of the classes before it leave as their queues
// drain; `st` waits for all of them.
int launch_batch(const BatchDev& b, int sweeps, hipStream_t st, int only = -1, const BatchFork* fk = nullptr);
// Fills the mode-1 and mode-2 copies of every problem's tensor.
int launch_batch_permute(const BatchDev& b, double* T1, double* T2, hipStream_t st);

}  // namespace itcpd

#define ITCPD_HIP(call)                                              \
    do {                                                             \
        hipError_t e_ = (call);                                      \
        if (e_ != hipSuccess) return itcpd::hip_fail(e_, #call);     \
    } while (0)
