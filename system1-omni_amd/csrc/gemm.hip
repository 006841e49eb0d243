// bfloat16 GEMMs of the decoder's projections, float32 accumulation (reference interface
// ops.h:117-124, gemm.cu): the library's own kernel (gemm_mfma.hip) for the shapes that its plan
// takes, hipBLASLt for the others (K not a multiple of 64, N or ldy not of 8, operands not on 16
// bytes, and the shapes where hipBLASLt measured faster).
//
// Through hipBLASLt: row-major y [M, N] (row stride ldy >= N) = x [M, K] * w [N, K]^T. hipBLASLt is
// column-major, so the call computes y^T [N, M] = op(A) * B with A = w seen as the
// column-major [K, N] matrix (transposed) and B = x seen as the column-major [K, M]
// matrix; y^T's leading dimension is ldy, so one GEMM can fill a column slice of a wider
// row-major buffer.
//
// Every shape (M, N, K, ldy) gets one plan, built on first use and then reused, so a given
// shape always runs the same kernel and its float32 summation order is fixed from call to
// call. The own kernel's plan is a function of the shape and the workspace size. cs1_gemm itself
// never waits on the host: a new hipBLASLt plan is its first heuristic
// choice that it accepts at launch (a stream-K kernel can be listed and then refused for the
// handle's workspace) among the kernels that do not accumulate split-K partial sums into the
// output with atomics (the reference excludes in-place split-K reductions for the same reason,
// gemm.cu:63-80), so the plan, and with it every result bit, is the same in every process
// on the same device and library.
//
// cs1_gemm_tune is the additive, explicit alternative for callers that prefer speed over
// cross-process repeatability: it times up to kCandidates heuristic choices on the call's
// own operands (y is overwritten by each trial and finally by the kept kernel) and the own
// kernel's plan where there is one, keeps the fastest unless it beats the default by less than
// kMargin, and synchronises the stream to
// do so, so it must run before any capture. A tuned choice follows measured times and can
// differ between processes. The plans live in the caller-owned handle, which is not safe
// for concurrent use (one model drives it from one thread, as the reference's executor
// does). CS1_GEMM_LOG=1 prints each plan's kernel to stderr.
#include <hip/hip_runtime.h>
#include <hipblaslt/hipblaslt-ext.hpp>
#include <hipblaslt/hipblaslt.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <tuple>
#include <vector>

#include "common.h"
#include "gemm_mfma.h"
#include "qwen3_5_ops.h"

namespace {

constexpr int kCandidates = 16;
constexpr float kMargin = 0.03f;
constexpr int kTrialWarm = 2, kTrialTimed = 5;

struct Plan {
    hipblasLtMatmulDesc_t op = nullptr;
    hipblasLtMatrixLayout_t a = nullptr, b = nullptr, c = nullptr;
    hipblasLtMatmulAlgo_t algo{};
    // Until a launch succeeds, the later heuristic choices (in heuristic order) that replace
    // algo if hipBLASLt rejects it at launch; a host-side rejection depends only on the shape,
    // the workspace size and the library, so the kernel a shape settles on is the same in
    // every process.
    std::vector<hipblasLtMatmulAlgo_t> fallback;
    bool settled = false;
};

using Key = std::tuple<int, int, int, int>;  // M, N, K, ldy

struct Gemm {
    hipblasLtHandle_t handle = nullptr;
    void* workspace = nullptr;
    size_t workspace_bytes = 0;
    std::map<Key, Plan> plans;             // hipBLASLt's
    std::map<Key, q35::MfmaPlan> own;      // the own kernel's (tile -1: hipBLASLt runs the shape)
    bool forced = false;                   // test hook: every shape takes force (tile -1: hipBLASLt)
    q35::MfmaPlan force;
};

const q35::MfmaPlan& own_plan(Gemm& g, int M, int N, int K, int ldy) {
    auto it = g.own.find(Key{M, N, K, ldy});
    if (it == g.own.end())
        it = g.own.emplace(Key{M, N, K, ldy}, q35::mfma_gemm_plan(M, N, K, ldy, g.workspace_bytes, q35::device_cus()))
                 .first;
    return it->second;
}

// the own kernel loads and stores 16 bytes at a time
bool aligned16(const void* x, const void* w, const void* y) {
    return ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(y)) & 15) == 0;
}

// hipBLASLt statuses are reported as 1000 + status, like the reference's cuBLAS codes.
int status(hipblasStatus_t s) { return s == HIPBLAS_STATUS_SUCCESS ? 0 : 1000 + (int)s; }

void release(Plan& p) {
    if (p.a) hipblasLtMatrixLayoutDestroy(p.a);
    if (p.b) hipblasLtMatrixLayoutDestroy(p.b);
    if (p.c) hipblasLtMatrixLayoutDestroy(p.c);
    if (p.op) hipblasLtMatmulDescDestroy(p.op);
    p = Plan{};
}

bool env_flag(const char* name, bool dflt) {
    const char* v = std::getenv(name);
    if (!v || !*v) return dflt;
    return std::strcmp(v, "0") != 0;
}

// Average time in ms of one launch (0 on success), or a negative value if it fails to run.
template <typename F>
float time_launch(F&& launch, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
    for (int i = 0; i < kTrialWarm + kTrialTimed; i++) {
        if (i == kTrialWarm && hipEventRecord(e0, st) != hipSuccess) return -1.f;
        if (launch() != 0) return -1.f;
    }
    float ms = -1.f;
    if (hipEventRecord(e1, st) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
        hipEventElapsedTime(&ms, e0, e1) != hipSuccess)
        return -1.f;
    return ms / kTrialTimed;
}

// Picks by measured time among the heuristic results r[0..n) and, as candidate n, the own kernel's
// plan (own.tile >= 0): the default (the own kernel if own_first, or r[0]) unless another is faster
// by at least kMargin.
int tune(Gemm& g, Plan& p, const hipblasLtMatmulHeuristicResult_t* r, int n, const q35::MfmaPlan& own, bool own_first,
         int M, int N, int K, int ldy, const void* x, const void* w, void* y, hipStream_t st) {
    const int dflt = own_first ? n : 0, total = own.tile >= 0 ? n + 1 : n;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (hipEventCreate(&e0) != hipSuccess) return dflt;
    if (hipEventCreate(&e1) != hipSuccess) {
        (void)hipEventDestroy(e0);
        return dflt;
    }
    // Two rounds over the candidates, each keeping its faster round: the first round also
    // brings the clock up from idle, which would otherwise penalise the first candidate.
    const float alpha = 1.f, beta = 0.f;
    float ms[kCandidates + 1];
    for (int i = 0; i < total; i++) ms[i] = -1.f;
    for (int round = 0; round < 2; round++)
        for (int i = 0; i < total; i++) {
            if (i < n && r[i].state != HIPBLAS_STATUS_SUCCESS) continue;
            const float t = time_launch(
                [&] {
                    if (i == n) return q35::mfma_gemm(own, x, w, y, g.workspace, M, N, K, ldy, st);
                    return status(hipblasLtMatmul(g.handle, p.op, &alpha, w, p.a, x, p.b, &beta, y, p.c, y, p.c,
                                                  &r[i].algo, g.workspace, g.workspace_bytes, st));
                },
                st, e0, e1);
            if (t > 0.f && (ms[i] < 0.f || t < ms[i])) ms[i] = t;
        }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipGetLastError();
    int best = dflt;
    for (int i = 0; i < total; i++)
        if (ms[i] > 0.f && (ms[best] <= 0.f || ms[i] < ms[best])) best = i;
    const int pick = ms[dflt] > 0.f && ms[best] > ms[dflt] * (1.f - kMargin) ? dflt : best;
    if (env_flag("CS1_GEMM_TUNE_LOG", false))
        std::fprintf(stderr, "cs1_gemm tune M=%d N=%d K=%d: %d candidates, default %.1f us, best %.1f us (#%d), kept #%d\n",
                     M, N, K, total, ms[dflt] * 1e3f, ms[best] * 1e3f, best, pick);
    return pick;
}

int describe(int M, int N, int K, int ldy, Plan& p) {
    hipblasStatus_t s = hipblasLtMatmulDescCreate(&p.op, HIPBLAS_COMPUTE_32F, HIP_R_32F);
    if (s != HIPBLAS_STATUS_SUCCESS) return status(s);
    const hipblasOperation_t ta = HIPBLAS_OP_T, tb = HIPBLAS_OP_N;
    if ((s = hipblasLtMatmulDescSetAttribute(p.op, HIPBLASLT_MATMUL_DESC_TRANSA, &ta, sizeof(ta))) !=
        HIPBLAS_STATUS_SUCCESS)
        return status(s);
    if ((s = hipblasLtMatmulDescSetAttribute(p.op, HIPBLASLT_MATMUL_DESC_TRANSB, &tb, sizeof(tb))) !=
        HIPBLAS_STATUS_SUCCESS)
        return status(s);
    if ((s = hipblasLtMatrixLayoutCreate(&p.a, HIP_R_16BF, K, N, K)) != HIPBLAS_STATUS_SUCCESS) return status(s);
    if ((s = hipblasLtMatrixLayoutCreate(&p.b, HIP_R_16BF, K, M, K)) != HIPBLAS_STATUS_SUCCESS) return status(s);
    if ((s = hipblasLtMatrixLayoutCreate(&p.c, HIP_R_16BF, N, M, ldy)) != HIPBLAS_STATUS_SUCCESS) return status(s);
    return 0;
}

// Kernels whose split-K partial sums meet in the output through atomic adds: their
// summation order, and so the rounding, changes from run to run. hipBLASLt names the
// global-split-U algorithm of a kernel in its name ("GSUASB": single buffer, atomic
// accumulation); the multiple-buffer form reduces through the workspace in a fixed order.
// The naming was checked against the hipBLASLt of ROCm 7.2.0 (this image's library); the
// public API exposes no attribute for the split-K accumulation mode. If a later library
// renames these kernels, the cross-process bitwise test of the config-3 decision
// (test_cfg3_decision_is_bitwise_repeatable_across_processes) is the guard that notices.
bool accumulates_atomically(Gemm& g, hipblasLtMatmulAlgo_t& algo) {
    const std::string name = hipblaslt_ext::getKernelNameFromAlgo(g.handle, algo);
    return name.find("GSUASB") != std::string::npos;
}

// Up to want heuristic results for the plan's shape, atomically accumulating kernels removed;
// returns their count in *n.
int candidates(Gemm& g, Plan& p, int want, hipblasLtMatmulHeuristicResult_t* r, int* n) {
    hipblasLtMatmulPreference_t pref = nullptr;
    hipblasStatus_t s = hipblasLtMatmulPreferenceCreate(&pref);
    if (s != HIPBLAS_STATUS_SUCCESS) return status(s);
    const uint64_t ws = g.workspace_bytes;
    hipblasLtMatmulPreferenceSetAttribute(pref, HIPBLASLT_MATMUL_PREF_MAX_WORKSPACE_BYTES, &ws, sizeof(ws));
    hipblasLtMatmulHeuristicResult_t all[kCandidates]{};
    int found = 0;
    s = hipblasLtMatmulAlgoGetHeuristic(g.handle, p.op, p.a, p.b, p.c, p.c, pref, kCandidates, all, &found);
    hipblasLtMatmulPreferenceDestroy(pref);
    if (s != HIPBLAS_STATUS_SUCCESS) return status(s);
    int k = 0;
    for (int i = 0; i < found && k < want; i++) {
        if (all[i].state == HIPBLAS_STATUS_SUCCESS && all[i].workspaceSize <= g.workspace_bytes &&
            !accumulates_atomically(g, all[i].algo))
            r[k++] = all[i];
    }
    *n = k;
    return k == 0 ? status(HIPBLAS_STATUS_NOT_SUPPORTED) : 0;
}

void log_plan(Gemm& g, Plan& p, int M, int N, int K, const char* how) {
    if (!env_flag("CS1_GEMM_LOG", false)) return;
    std::fprintf(stderr, "cs1_gemm plan M=%d N=%d K=%d (%s): %s\n", M, N, K, how,
                 hipblaslt_ext::getKernelNameFromAlgo(g.handle, p.algo).c_str());
}

int new_plan(Gemm& g, int M, int N, int K, int ldy, Plan*& out) {
    Plan p;
    int rc = describe(M, N, K, ldy, p);
    hipblasLtMatmulHeuristicResult_t r[kCandidates]{};
    int n = 0;
    if (rc == 0) rc = candidates(g, p, kCandidates, r, &n);
    if (rc != 0) {
        release(p);
        return rc;
    }
    p.algo = r[0].algo;
    for (int i = 1; i < n; i++) p.fallback.push_back(r[i].algo);
    log_plan(g, p, M, N, K, "first choice");
    out = &g.plans.emplace(Key{M, N, K, ldy}, p).first->second;
    return 0;
}

int plan_for(Gemm& g, int M, int N, int K, int ldy, Plan*& out) {
    auto it = g.plans.find(Key{M, N, K, ldy});
    if (it != g.plans.end()) {
        out = &it->second;
        return 0;
    }
    return new_plan(g, M, N, K, ldy, out);
}

bool valid(const Gemm* g, const void* x, const void* w, const void* y, int M, int N, int K, int ldy) {
    return g && M >= 0 && N > 0 && K > 0 && ldy >= N && (M == 0 || (x && w && y));
}

}  // namespace

extern "C" {

void* cs1_gemm_create(size_t workspace_bytes) {
    Gemm* g = new Gemm();
    if (hipblasLtCreate(&g->handle) != HIPBLAS_STATUS_SUCCESS) {
        delete g;
        return nullptr;
    }
    if (workspace_bytes > 0 && hipMalloc(&g->workspace, workspace_bytes) != hipSuccess) {
        hipblasLtDestroy(g->handle);
        delete g;
        return nullptr;
    }
    g->workspace_bytes = workspace_bytes;
    return g;
}

void cs1_gemm_destroy(void* gemm) {
    Gemm* g = static_cast<Gemm*>(gemm);
    if (!g) return;
    for (auto& kv : g->plans) release(kv.second);
    if (g->workspace) (void)hipFree(g->workspace);
    hipblasLtDestroy(g->handle);
    delete g;
}

int cs1_gemm(void* gemm, const void* x, const void* w, void* y, int M, int N, int K, int ldy, void* stream) {
    Gemm* g = static_cast<Gemm*>(gemm);
    if (!valid(g, x, w, y, M, N, K, ldy)) return hipErrorInvalidValue;
    if (M == 0) return hipSuccess;
    const q35::MfmaPlan& own = g->forced ? g->force : own_plan(*g, M, N, K, ldy);
    if (g->forced && own.tile >= 0 && !q35::mfma_gemm_takes(own, M, N, K, ldy, g->workspace_bytes)) return hipErrorInvalidValue;
    if (own.tile >= 0 && aligned16(x, w, y))
        return q35::mfma_gemm(own, x, w, y, g->workspace, M, N, K, ldy, static_cast<hipStream_t>(stream));
    Plan* p = nullptr;
    const int rc = plan_for(*g, M, N, K, ldy, p);
    if (rc != 0) return rc;
    const float alpha = 1.f, beta = 0.f;
    for (;;) {
        const hipblasStatus_t s = hipblasLtMatmul(g->handle, p->op, &alpha, w, p->a, x, p->b, &beta, y, p->c, y,
                                                  p->c, &p->algo, g->workspace, g->workspace_bytes,
                                                  static_cast<hipStream_t>(stream));
        if (s == HIPBLAS_STATUS_SUCCESS) {
            p->settled = true;
            return 0;
        }
        // Only a launch refused for the kernel itself moves the plan on (the operands were
        // validated above, so these statuses come from the algorithm or its workspace; the
        // stream-K refusal seen for 1217 x 2176 x 5120 with 32 MiB is status 6). Anything else
        // is returned with the plan untouched, so a plan depends only on the shape.
        const bool kernel_refused = s == HIPBLAS_STATUS_NOT_SUPPORTED || s == HIPBLAS_STATUS_INVALID_VALUE ||
                                    s == HIPBLAS_STATUS_INTERNAL_ERROR;
        if (p->settled || p->fallback.empty() || !kernel_refused) return status(s);
        p->algo = p->fallback.front();
        p->fallback.erase(p->fallback.begin());
        log_plan(*g, *p, M, N, K, "next choice after a rejected launch");
    }
}

int cs1_gemm_tune(void* gemm, const void* x, const void* w, void* y, int M, int N, int K, int ldy, void* stream) {
    Gemm* g = static_cast<Gemm*>(gemm);
    if (!valid(g, x, w, y, M, N, K, ldy)) return hipErrorInvalidValue;
    if (M == 0) return hipSuccess;
    hipStream_t st = static_cast<hipStream_t>(stream);
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    hipError_t e = hipStreamIsCapturing(st, &cap);
    if (e != hipSuccess) return e;
    if (cap != hipStreamCaptureStatusNone) return hipErrorStreamCaptureUnsupported;
    Plan* p = nullptr;
    int rc = plan_for(*g, M, N, K, ldy, p);
    if (rc != 0) return rc;
    hipblasLtMatmulHeuristicResult_t r[kCandidates]{};
    int n = 0;
    if ((rc = candidates(*g, *p, kCandidates, r, &n)) != 0) return rc;
    // The own kernel's modelled plan is a candidate whichever side runs the shape by default; operands that
    // it cannot load re-choose hipBLASLt's kernel only, and the shape's plan stays.
    const bool loads = aligned16(x, w, y);
    const int cus = q35::device_cus();
    const q35::MfmaPlan own = loads ? q35::mfma_gemm_model(M, N, K, ldy, g->workspace_bytes, cus) : q35::MfmaPlan{};
    const bool own_first = loads && q35::mfma_gemm_plan(M, N, K, ldy, g->workspace_bytes, cus).tile >= 0;
    const int choice = n > 1 || own.tile >= 0 ? tune(*g, *p, r, n, own, own_first, M, N, K, ldy, x, w, y, st) : 0;
    if (loads) g->own[Key{M, N, K, ldy}] = choice == n ? own : q35::MfmaPlan{};
    const int pick = choice == n ? 0 : choice;  // (kept for operands that the own kernel does not take)
    p->algo = r[pick].algo;
    p->fallback.clear();
    for (int i = 0; i < n; i++)
        if (i != pick) p->fallback.push_back(r[i].algo);
    p->settled = false;
    log_plan(*g, *p, M, N, K, "tuned");
    return cs1_gemm(gemm, x, w, y, M, N, K, ldy, stream);
}

// ---- test hooks, outside the op ABI ----

// The plan (tile form, split; -1: hipBLASLt) that a handle with ws_bytes of workspace gives a shape on
// a device of cus CUs; with modelled != 0 the own kernel's plan, also where hipBLASLt runs the shape.
int q35_gemm_default_plan(int M, int N, int K, int ldy, size_t ws_bytes, int cus, int modelled, int* tile, int* split) {
    const q35::MfmaPlan p = modelled ? q35::mfma_gemm_model(M, N, K, ldy, ws_bytes, cus)
                                     : q35::mfma_gemm_plan(M, N, K, ldy, ws_bytes, cus);
    *tile = p.tile, *split = p.split;
    return hipSuccess;
}

// The plan that this handle's calls on 16-byte operands take now.
int q35_gemm_plan_of(void* gemm, int M, int N, int K, int ldy, int* tile, int* split) {
    const q35::MfmaPlan& p = own_plan(*static_cast<Gemm*>(gemm), M, N, K, ldy);
    *tile = p.tile, *split = p.split;
    return hipSuccess;
}

// From now on the handle's cs1_gemm calls run this form and split (-1: hipBLASLt; -2: by shape again).
// A shape that the form cannot run is refused.
int q35_gemm_force(void* gemm, int tile, int split) {
    Gemm* g = static_cast<Gemm*>(gemm);
    g->forced = tile != -2;
    g->force = q35::MfmaPlan{tile, split};
    return hipSuccess;
}

int q35_gemm_form(int tile, int* bm, int* bn, int* stages) {
    return q35::mfma_gemm_form(tile, bm, bn, stages) ? hipSuccess : hipErrorInvalidValue;
}

}  // extern "C"
