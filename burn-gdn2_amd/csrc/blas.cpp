// The layer's row-major GEMMs: split products and hipBLASLt plans (see blas.hpp).
//
// Row-major C = op(A) op(B) is column-major C^T = op(B)^T op(A)^T, so the
// library's first operand is B's memory and its second is A's; a row-major
// [r, c] matrix with row stride ld is a column-major [c, r] one with leading
// dimension ld.
#include "blas.hpp"

#include "kernels.hpp"

#include <algorithm>
#include <string>

namespace gdn2 {

namespace {
constexpr size_t kMaxWorkspace = size_t(64) << 20;
constexpr int kCandidates = 32;  // heuristic results timed per shape
// Shapes of at most this many rows (a decode step) read mostly weights, which
// the real call finds outside L2 (the step's other kernels stream far more
// than the 8 x 4 MB of L2): each of their timed runs follows a read sweep
// over kFlushBytes, twice the L2s together (reads, so that no write-back
// overlaps the timed run), and a candidate's time is its best of three, so
// that an algorithm that only wins on L2-resident weights is not picked.
constexpr int64_t kColdTimingMaxM = 256;
constexpr size_t kFlushBytes = size_t(64) << 20;

// Whether a product gains more from the f16 matrix cores (about 400 against
// hipBLASLt's 145 TFLOP/s of f32) than splitting its operands costs.  Measured,
// splitting rows: 11 us up to 1024 x 2048, 26 us at 8192 x 2048, 107 us at
// 32768 x 2048 (8 bytes an element, 5 TB/s); splitting columns (two reads of
// the operand): 38 us at 8192 x 2048, 210 us at 8192 x 10496.  Both sides near
// the line, f32 against split + product: 148 x 10496 x 2048 68 and 66 us,
// 8192 x 2048 x 128 50 and 43 us; 148 x 2048 x 2048 23 and 39 us,
// 8192 x 128 x 2048 41 and 61 us and 1024 x 1408 x 256 22 and 28 us stay.
// Below 128 rows a product is bound by reading its weights, not by the cores.
// (Beyond 2^20 elements of a contraction a row's record could overflow.)
bool split_pays(bool ta, bool tb, int64_t M, int64_t N, int64_t Kd, bool b_kept) {
    if (M < 128 || N < 128 || Kd < 64 || Kd > (int64_t(1) << 20)) return false;
    const double gain = 2.0 * (double)M * (double)N * (double)Kd * (1 / 145e12 - 1 / 400e12);
    const auto cost = [](double n, bool trans) { return trans ? 20e-6 + n * 12 / 4.5e12 : 14e-6 + n * 8 / 4.5e12; };
    return gain > cost((double)M * (double)Kd, ta) + (b_kept ? 0.0 : cost((double)N * (double)Kd, !tb));
}
}

gdn2_status Gemm::init() {
    if (hipblasLtCreate(&lt_) != HIPBLAS_STATUS_SUCCESS) return fail(GDN2_EHIP, "hipblasLtCreate failed");
    if (rocblas_create_handle(&rb_) != rocblas_status_success) return fail(GDN2_EHIP, "rocblas_create_handle failed");
    return GDN2_OK;
}

void Gemm::destroy() {
    for (Plan &p : plans_) {
        if (!p.ok) continue;
        hipblasLtMatrixLayoutDestroy(p.la);
        hipblasLtMatrixLayoutDestroy(p.lb);
        hipblasLtMatrixLayoutDestroy(p.lc);
        hipblasLtMatmulDescDestroy(p.desc);
    }
    plans_.clear();
    ws_.destroy();
    sws_.destroy();
    if (lt_) hipblasLtDestroy(lt_);
    lt_ = nullptr;
    if (rb_) rocblas_destroy_handle(rb_);
    rb_ = nullptr;
}

gdn2_status Gemm::plan(bool ta, bool tb, int64_t M, int64_t N, int64_t Kd, const float *A, int64_t lda,
                       const float *B, int64_t ldb, int64_t ldc, hipStream_t s, const Plan **out) {
    for (const Plan &p : plans_)
        if (p.ta == ta && p.tb == tb && p.M == M && p.N == N && p.Kd == Kd && p.lda == lda && p.ldb == ldb &&
            p.ldc == ldc) {
            *out = &p;
            return GDN2_OK;
        }
    Plan p{};
    p.ta = ta; p.tb = tb; p.M = M; p.N = N; p.Kd = Kd; p.lda = lda; p.ldb = ldb; p.ldc = ldc;
    const hipblasOperation_t op1 = tb ? HIPBLAS_OP_T : HIPBLAS_OP_N, op2 = ta ? HIPBLAS_OP_T : HIPBLAS_OP_N;
    bool ok = hipblasLtMatmulDescCreate(&p.desc, HIPBLAS_COMPUTE_32F, HIP_R_32F) == HIPBLAS_STATUS_SUCCESS;
    ok = ok && hipblasLtMatmulDescSetAttribute(p.desc, HIPBLASLT_MATMUL_DESC_TRANSA, &op1, sizeof op1) ==
                   HIPBLAS_STATUS_SUCCESS;
    ok = ok && hipblasLtMatmulDescSetAttribute(p.desc, HIPBLASLT_MATMUL_DESC_TRANSB, &op2, sizeof op2) ==
                   HIPBLAS_STATUS_SUCCESS;
    // first operand: B's memory, column-major [N, Kd] (op N) or [Kd, N] (op T)
    ok = ok && hipblasLtMatrixLayoutCreate(&p.la, HIP_R_32F, tb ? Kd : N, tb ? N : Kd, ldb) == HIPBLAS_STATUS_SUCCESS;
    // second operand: A's memory, column-major [Kd, M] (op N) or [M, Kd] (op T)
    ok = ok && hipblasLtMatrixLayoutCreate(&p.lb, HIP_R_32F, ta ? M : Kd, ta ? Kd : M, lda) == HIPBLAS_STATUS_SUCCESS;
    ok = ok && hipblasLtMatrixLayoutCreate(&p.lc, HIP_R_32F, N, M, ldc) == HIPBLAS_STATUS_SUCCESS;
    if (!ok) {
        if (p.la) hipblasLtMatrixLayoutDestroy(p.la);
        if (p.lb) hipblasLtMatrixLayoutDestroy(p.lb);
        if (p.lc) hipblasLtMatrixLayoutDestroy(p.lc);
        if (p.desc) hipblasLtMatmulDescDestroy(p.desc);
        return fail(GDN2_EHIP, "hipBLASLt descriptor creation failed");
    }
    hipblasLtMatmulPreference_t pref;
    if (hipblasLtMatmulPreferenceCreate(&pref) != HIPBLAS_STATUS_SUCCESS)
        return fail(GDN2_EHIP, "hipblasLtMatmulPreferenceCreate failed");
    const uint64_t maxws = kMaxWorkspace;
    hipblasLtMatmulPreferenceSetAttribute(pref, HIPBLASLT_MATMUL_PREF_MAX_WORKSPACE_BYTES, &maxws, sizeof maxws);
    hipblasLtMatmulHeuristicResult_t res[kCandidates];
    int n = 0;
    const hipblasStatus_t hs =
        hipblasLtMatmulAlgoGetHeuristic(lt_, p.desc, p.la, p.lb, p.lc, p.lc, pref, kCandidates, res, &n);
    hipblasLtMatmulPreferenceDestroy(pref);
    int best = -1;
    if (hs == HIPBLAS_STATUS_SUCCESS)
        for (int i = 0; i < n && best < 0; ++i)
            if (res[i].state == HIPBLAS_STATUS_SUCCESS && res[i].workspaceSize <= kMaxWorkspace) best = i;
    if (best >= 0 && n > 1 && !recording_) {
        // time the candidates on these operands, writing a scratch output
        size_t wsmax = 0;
        for (int i = 0; i < n; ++i)
            if (res[i].state == HIPBLAS_STATUS_SUCCESS && res[i].workspaceSize <= kMaxWorkspace)
                wsmax = std::max(wsmax, res[i].workspaceSize);
        GDN2_HIP_CHECK(ws_.ensure(wsmax, false));
        float *scratch = nullptr, *flush = nullptr;
        hipEvent_t e0 = nullptr, e1 = nullptr;
        if (M <= kColdTimingMaxM && hipMalloc(&flush, kFlushBytes) != hipSuccess) flush = nullptr;
        const int64_t nflush = (int64_t)(kFlushBytes / sizeof(float));
        if (hipMalloc(&scratch, sizeof(float) * (size_t)ldc * M) == hipSuccess && hipEventCreate(&e0) == hipSuccess &&
            hipEventCreate(&e1) == hipSuccess) {
            const float alpha = 1.0f, beta = 0.0f;
            float best_ms = 0.0f;
            for (int i = 0; i < n; ++i) {
                if (res[i].state != HIPBLAS_STATUS_SUCCESS || res[i].workspaceSize > kMaxWorkspace) continue;
                bool ok = true;
                float total = 0.0f;
                for (int r = 0; r < 4 && ok; ++r) {  // one warm-up, then three timed runs
                    if (flush) ok = launch_cache_sweep(flush, nflush, flush, s) == hipSuccess;
                    if (r > 0) ok = ok && hipEventRecord(e0, s) == hipSuccess;
                    ok = ok && hipblasLtMatmul(lt_, p.desc, &alpha, B, p.la, A, p.lb, &beta, scratch, p.lc, scratch,
                                               p.lc, &res[i].algo, res[i].workspaceSize ? ws_.ptr() : nullptr,
                                               res[i].workspaceSize, s) == HIPBLAS_STATUS_SUCCESS;
                    if (r > 0) {
                        float ms = 0.0f;
                        ok = ok && hipEventRecord(e1, s) == hipSuccess && hipEventSynchronize(e1) == hipSuccess &&
                             hipEventElapsedTime(&ms, e0, e1) == hipSuccess;
                        total = (r == 1 || ms < total) ? ms : total;
                    }
                }
                if (ok && (total < best_ms || best_ms == 0.0f)) {
                    best_ms = total;
                    best = i;
                }
            }
        }
        (void)hipGetLastError();  // a failed scratch allocation only skips the timing (or the flush)
        if (e0) (void)hipEventDestroy(e0);
        if (e1) (void)hipEventDestroy(e1);
        if (scratch || flush) (void)hipStreamSynchronize(s);
        if (scratch) (void)hipFree(scratch);
        if (flush) (void)hipFree(flush);
    }
    p.ok = best >= 0;
    if (p.ok) {
        p.algo = res[best].algo;
        p.ws = res[best].workspaceSize;
    } else {
        hipblasLtMatrixLayoutDestroy(p.la);
        hipblasLtMatrixLayoutDestroy(p.lb);
        hipblasLtMatrixLayoutDestroy(p.lc);
        hipblasLtMatmulDescDestroy(p.desc);
    }
    plans_.push_back(p);
    *out = &plans_.back();
    return GDN2_OK;
}

// Runs the product on the f16 matrix cores if that pays and its memory is
// there; false: not run, take the library's product.  Memory grows only while
// the stream is not being captured; a failed allocation is no error.
bool Gemm::run_split(bool ta, bool tb, int64_t M, int64_t N, int64_t Kd, const float *A, int64_t lda, const float *B,
                     int64_t ldb, float *C, int64_t ldc, float beta, hipStream_t s, SplitWeight *w, gdn2_status *st) {
    if (!split_pays(ta, tb, M, N, Kd, w != nullptr)) return false;
    SplitGemmParams p{};
    p.A = A; p.B = B; p.C = C; p.lda = lda; p.ldb = ldb; p.ldc = ldc; p.M = M; p.N = N; p.Kd = Kd;
    p.beta = beta; p.ta = ta; p.tb = tb;
    p.vec_c = reinterpret_cast<uintptr_t>(C) % 16 == 0 && ldc % 4 == 0;
    const size_t sums = (plan_split_gemm(&p) + 255) & ~(size_t)255;
    size_t flags, failed;
    split_redo_bytes(p, &flags, &failed);
    const size_t part = sums + flags + failed;
    const size_t fa = split_frag_bytes(M, Kd), sa = split_stat_bytes(M);
    const size_t fb = split_frag_bytes(N, Kd), sb = split_stat_bytes(N);
    const size_t need = part + fa + sa + (w ? 0 : fb + sb);
    if (recording_ && need > sws_.bytes()) return false;
    if (sws_.ensure(need, recording_) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    const auto check = [&](hipError_t e) {
        if (e != hipSuccess) *st = fail(GDN2_EHIP, std::string("split product: ") + hipGetErrorString(e));
        return e == hipSuccess;
    };
    *st = GDN2_OK;
    if (w) {
        hipError_t e = hipSuccess;
        if (!w->ready(s, recording_, &e)) return false;
        if (!check(e)) return true;
    }
    char *base = static_cast<char *>(sws_.ptr());
    p.part = reinterpret_cast<float *>(base);
    p.redo = reinterpret_cast<unsigned char *>(base + sums);
    p.failed = reinterpret_cast<unsigned short *>(base + sums + flags);
    void *fra = base + part;
    SplitStat *sta = reinterpret_cast<SplitStat *>(base + part + fa);
    if (!check(launch_split(A, lda, ta, M, Kd, fra, sta, s))) return true;
    p.fa = fra;
    p.sa = sta;
    if (w) {
        p.fb = w->frags;
        p.sb = w->stat;
    } else {
        void *frb = base + part + fa + sa;
        SplitStat *stb = reinterpret_cast<SplitStat *>(base + part + fa + sa + fb);
        if (!check(launch_split(B, ldb, !tb, N, Kd, frb, stb, s))) return true;
        p.fb = frb;
        p.sb = stb;
    }
    (void)check(launch_split_gemm(p, s));
    return true;
}

gdn2_status Gemm::run(bool ta, bool tb, int64_t M, int64_t N, int64_t Kd, const float *A, int64_t lda, const float *B,
                      int64_t ldb, float *C, int64_t ldc, float beta, hipStream_t s, SplitWeight *w) {
    if (M == 0 || N == 0) return GDN2_OK;
    gdn2_status st = GDN2_OK;
    if (run_split(ta, tb, M, N, Kd, A, lda, B, ldb, C, ldc, beta, s, w, &st)) return st;
    const float alpha = 1.0f;
    const Plan *p = nullptr;
    st = plan(ta, tb, M, N, Kd, A, lda, B, ldb, ldc, s, &p);
    if (st != GDN2_OK) return st;
    if (p->ok) {
        GDN2_HIP_CHECK(ws_.ensure(p->ws, recording_));
        const hipblasStatus_t hs = hipblasLtMatmul(lt_, p->desc, &alpha, B, p->la, A, p->lb, &beta, C, p->lc, C,
                                                   p->lc, &p->algo, p->ws ? ws_.ptr() : nullptr, p->ws, s);
        if (hs != HIPBLAS_STATUS_SUCCESS)
            return fail(GDN2_EHIP, "hipblasLtMatmul failed with status " + std::to_string((int)hs));
        return GDN2_OK;
    }
    if (rocblas_set_stream(rb_, s) != rocblas_status_success) return fail(GDN2_EHIP, "rocblas_set_stream failed");
    const rocblas_status rs =
        rocblas_sgemm(rb_, tb ? rocblas_operation_transpose : rocblas_operation_none,
                      ta ? rocblas_operation_transpose : rocblas_operation_none, (rocblas_int)N, (rocblas_int)M,
                      (rocblas_int)Kd, &alpha, B, (rocblas_int)ldb, A, (rocblas_int)lda, &beta, C, (rocblas_int)ldc);
    if (rs != rocblas_status_success)
        return fail(GDN2_EHIP, std::string("rocblas_sgemm: ") + rocblas_status_to_string(rs));
    return GDN2_OK;
}

}  // namespace gdn2
