// Direct hipBLASLt GEMM with timed algo autotuning (decode-step GEMMs).
//
// rocBLAS's default tile selection for the skinny decode shapes
// (M = batch, N/K = model dims) measured well below the HBM roofline
// (qkv GEMM at ~1.3 TB/s of ~6.3 achievable — profiles/r01_decode_*).
// This module asks hipBLASLt for its candidate algorithms for each exact
// (M, N, K, bias) shape, TIMES each candidate on the device at warmup, and
// replays the winner from then on. Replay is a plain stream enqueue, so it
// is hipGraph-capturable; a cache miss during capture is a loud error
// (warmup runs every bucket shape before capture).
//
// Mirrors the role of the reference's compiler-side GEMM selection
// (neuronx-cc picks tiles AOT per traced shape): here the
// "compile" step is the timed tune, persisted in-process.

#include <hipblaslt/hipblaslt.h>
#include <torch/extension.h>

#include <ATen/hip/HIPContext.h>
#include <hip/hip_runtime.h>

#include <cstdint>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#define LT_CHECK(expr)                                                        \
    do {                                                                      \
        hipblasStatus_t st_ = (expr);                                         \
        TORCH_CHECK(st_ == HIPBLAS_STATUS_SUCCESS, "hipblaslt error ",        \
                    (int)st_, " at ", #expr);                                 \
    } while (0)

#define HIP_CHECK(expr)                                                       \
    do {                                                                      \
        hipError_t e_ = (expr);                                               \
        TORCH_CHECK(e_ == hipSuccess, "hip error: ", hipGetErrorString(e_));  \
    } while (0)

namespace {

constexpr size_t kWorkspaceBytes = 64ull << 20;
constexpr size_t kMaxFirst = 4096;   // choices kept without timing: a few for each number of rows seen

struct LtCtx {
    hipblasLtHandle_t handle{nullptr};
    void* workspace{nullptr};
    std::mutex mu;
    // key: (M, N, K, has_bias, dtype) -> tuned algo
    std::map<std::tuple<int64_t, int64_t, int64_t, int, int>,
             hipblasLtMatmulAlgo_t>
        algos;
    // same key -> the library's own first choice
    std::map<std::tuple<int64_t, int64_t, int64_t, int, int>,
             hipblasLtMatmulAlgo_t>
        first;
    bool disabled{false};
};

LtCtx& ctx() {
    static LtCtx c;
    static std::once_flag once;
    std::call_once(once, [] {
        if (hipblasLtCreate(&c.handle) != HIPBLAS_STATUS_SUCCESS) {
            c.disabled = true;
            return;
        }
        if (hipMalloc(&c.workspace, kWorkspaceBytes) != hipSuccess) {
            c.disabled = true;
        }
    });
    return c;
}

hipDataType lt_dtype(const torch::Tensor& t) {
    switch (t.scalar_type()) {
        case torch::kBFloat16: return HIP_R_16BF;
        case torch::kHalf: return HIP_R_16F;
        default: TORCH_CHECK(false, "lt_gemm: bf16/f16 only");
    }
}

struct Descs {
    hipblasLtMatmulDesc_t op{nullptr};
    hipblasLtMatrixLayout_t a{nullptr}, b{nullptr}, d{nullptr};
    ~Descs() {
        if (op) hipblasLtMatmulDescDestroy(op);
        if (a) hipblasLtMatrixLayoutDestroy(a);
        if (b) hipblasLtMatrixLayoutDestroy(b);
        if (d) hipblasLtMatrixLayoutDestroy(d);
    }
};

// Row-major y(M,N) = x(M,K) @ w(N,K)^T + bias  ==  column-major
// y'(N,M) = w'(K,N)^T . x'(K,M): opA=T on w, opB=N on x.
void build_descs(Descs& ds, int64_t M, int64_t N, int64_t K, hipDataType dt,
                 const void* bias_ptr) {
    LT_CHECK(hipblasLtMatmulDescCreate(&ds.op, HIPBLAS_COMPUTE_32F, HIP_R_32F));
    hipblasOperation_t opT = HIPBLAS_OP_T, opN = HIPBLAS_OP_N;
    LT_CHECK(hipblasLtMatmulDescSetAttribute(
        ds.op, HIPBLASLT_MATMUL_DESC_TRANSA, &opT, sizeof(opT)));
    LT_CHECK(hipblasLtMatmulDescSetAttribute(
        ds.op, HIPBLASLT_MATMUL_DESC_TRANSB, &opN, sizeof(opN)));
    if (bias_ptr != nullptr) {
        hipblasLtEpilogue_t ep = HIPBLASLT_EPILOGUE_BIAS;
        LT_CHECK(hipblasLtMatmulDescSetAttribute(
            ds.op, HIPBLASLT_MATMUL_DESC_EPILOGUE, &ep, sizeof(ep)));
        LT_CHECK(hipblasLtMatmulDescSetAttribute(
            ds.op, HIPBLASLT_MATMUL_DESC_BIAS_POINTER, &bias_ptr,
            sizeof(bias_ptr)));
    }
    // A = w viewed column-major (K, N), transposed in the op; lda = K
    LT_CHECK(hipblasLtMatrixLayoutCreate(&ds.a, dt, K, N, K));
    // B = x viewed column-major (K, M); ldb = K
    LT_CHECK(hipblasLtMatrixLayoutCreate(&ds.b, dt, K, M, K));
    // D = y viewed column-major (N, M); ldd = N
    LT_CHECK(hipblasLtMatrixLayoutCreate(&ds.d, dt, N, M, N));
}

hipblasStatus_t enqueue(const Descs& ds, const hipblasLtMatmulAlgo_t* algo,
                        const void* w, const void* x, void* y, hipStream_t stream) {
    float alpha = 1.0f, beta = 0.0f;
    return hipblasLtMatmul(ctx().handle, ds.op, &alpha, w, ds.a, x, ds.b,
                           &beta, y, ds.d, y, ds.d, algo, ctx().workspace,
                           kWorkspaceBytes, stream);
}

std::tuple<int64_t, int64_t, int64_t, int, int> make_key(
    int64_t M, int64_t N, int64_t K, bool has_bias, hipDataType dt) {
    return {M, N, K, has_bias ? 1 : 0, (int)dt};
}

// The library's candidates for a product, its first choice first.
int ask(const Descs& ds, int most, std::vector<hipblasLtMatmulHeuristicResult_t>& results) {
    hipblasLtMatmulPreference_t pref;
    LT_CHECK(hipblasLtMatmulPreferenceCreate(&pref));
    size_t ws = kWorkspaceBytes;
    LT_CHECK(hipblasLtMatmulPreferenceSetAttribute(
        pref, HIPBLASLT_MATMUL_PREF_MAX_WORKSPACE_BYTES, &ws, sizeof(ws)));
    results.resize(most);
    int found = 0;
    const hipblasStatus_t st = hipblasLtMatmulAlgoGetHeuristic(
        ctx().handle, ds.op, ds.a, ds.b, ds.d, ds.d, pref, most, results.data(), &found);
    hipblasLtMatmulPreferenceDestroy(pref);
    return st == HIPBLAS_STATUS_SUCCESS ? found : 0;
}

// Timed tune: try the heuristic candidates, keep the fastest. Returns the
// number of candidates that ran, or -1 if none work (caller falls back).
int tune_shape(int64_t M, int64_t N, int64_t K, bool has_bias,
               hipDataType dt, const void* w, const void* x, void* y,
               const void* bias, hipStream_t stream) {
    Descs ds;
    build_descs(ds, M, N, K, dt, has_bias ? bias : nullptr);

    std::vector<hipblasLtMatmulHeuristicResult_t> results;
    const int found = ask(ds, 48, results);
    if (found == 0) return -1;

    hipEvent_t t0, t1;
    HIP_CHECK(hipEventCreate(&t0));
    HIP_CHECK(hipEventCreate(&t1));
    // COLD-WEIGHT timing: the decode regime cycles 10s of GB of weights
    // through the 256 MB MALL every step, so a tune that reps the same
    // cache-hot weight picks tiles that stream badly in production
    // (measured: the hot-tuned qkv tile ran 1.2 TB/s in-bench while other
    // shapes hit 3.3-4.5). Evict the cache with a large memset before
    // every timed rep; events bracket only the matmul.
    void* flush_buf = nullptr;
    const size_t kFlushBytes = 768ull << 20;
    const bool can_flush = hipMalloc(&flush_buf, kFlushBytes) == hipSuccess;
    float best_ms = 1e30f;
    int best = -1, ran = 0;
    for (int i = 0; i < found; ++i) {
        if (results[i].state != HIPBLAS_STATUS_SUCCESS) continue;
        float alpha = 1.0f, beta = 0.0f;
        // probe once (skip algos that fail at launch)
        if (hipblasLtMatmul(ctx().handle, ds.op, &alpha, w, ds.a, x, ds.b,
                            &beta, y, ds.d, y, ds.d, &results[i].algo,
                            ctx().workspace, kWorkspaceBytes,
                            stream) != HIPBLAS_STATUS_SUCCESS)
            continue;
        float total_ms = 0.f;
        for (int r = 0; r < 3; ++r) {
            if (can_flush)
                HIP_CHECK(hipMemsetAsync(flush_buf, r, kFlushBytes, stream));
            HIP_CHECK(hipEventRecord(t0, stream));
            LT_CHECK(hipblasLtMatmul(ctx().handle, ds.op, &alpha, w, ds.a, x,
                                     ds.b, &beta, y, ds.d, y, ds.d,
                                     &results[i].algo, ctx().workspace,
                                     kWorkspaceBytes, stream));
            HIP_CHECK(hipEventRecord(t1, stream));
            HIP_CHECK(hipEventSynchronize(t1));
            float ms = 0.f;
            HIP_CHECK(hipEventElapsedTime(&ms, t0, t1));
            total_ms += ms;
        }
        ++ran;
        if (total_ms < best_ms) { best_ms = total_ms; best = i; }
    }
    if (flush_buf) (void)hipFree(flush_buf);
    HIP_CHECK(hipEventDestroy(t0));
    HIP_CHECK(hipEventDestroy(t1));
    if (best < 0) return -1;
    auto& c = ctx();
    std::lock_guard<std::mutex> lock(c.mu);
    c.algos[make_key(M, N, K, has_bias, dt)] = results[best].algo;
    return ran;
}

}  // namespace

bool lt_available() {
    auto& c = ctx();
    return !c.disabled;
}

// y(M,N) = x(M,K) @ w(N,K)^T [+ bias(N)]; tunes on first sight of a shape
// (loud error if that happens inside hipGraph capture — warmup must cover
// every bucket shape first).
// `timed` false: the library's own first choice for the shape instead of the timed one. Prompts
// without their padding have another number of rows each time: a search takes 25 to 80 ms, the
// question 0.1. What does not run is passed over for the library's next; false, with nothing done,
// where it has none that does. A choice is kept once it has run.
bool lt_linear(torch::Tensor y, torch::Tensor x, torch::Tensor w,
               c10::optional<torch::Tensor> bias_opt, bool timed) {
    auto& c = ctx();
    TORCH_CHECK(!c.disabled, "hipblaslt unavailable");
    TORCH_CHECK(x.is_contiguous() && w.is_contiguous() && y.is_contiguous());
    const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
    TORCH_CHECK(w.size(1) == K && y.size(0) == M && y.size(1) == N);
    hipDataType dt = lt_dtype(x);
    const bool has_bias = bias_opt.has_value();
    const void* bias = has_bias ? bias_opt->data_ptr() : nullptr;
    hipStream_t stream = at::hip::getCurrentHIPStream();

    hipblasLtMatmulAlgo_t algo;
    bool hit = false;
    const auto key = make_key(M, N, K, has_bias, dt);
    {
        std::lock_guard<std::mutex> lock(c.mu);
        auto it = c.algos.find(key);
        if (it != c.algos.end()) { algo = it->second; hit = true; }
        if (!hit && !timed) {
            it = c.first.find(key);
            if (it != c.first.end()) { algo = it->second; hit = true; }
        }
    }
    Descs ds;
    build_descs(ds, M, N, K, dt, has_bias ? bias : nullptr);
    auto run = [&]() { return enqueue(ds, &algo, w.data_ptr(), x.data_ptr(), y.data_ptr(), stream); };
    if (!hit && !timed) {
        std::vector<hipblasLtMatmulHeuristicResult_t> results;
        int found = ask(ds, 1, results);
        for (int at = 0;; ++at) {
            if (at == 1) found = ask(ds, 16, results);       // the first of them is known to fail
            if (at >= found) return false;
            algo = results[at].algo;
            if (results[at].state == HIPBLAS_STATUS_SUCCESS && run() == HIPBLAS_STATUS_SUCCESS) break;
        }
        std::lock_guard<std::mutex> lock(c.mu);
        if (c.first.size() >= kMaxFirst) c.first.clear();
        c.first[key] = algo;
        return true;
    } else if (!hit) {
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        hipStreamIsCapturing(stream, &cap);
        TORCH_CHECK(cap == hipStreamCaptureStatusNone,
                    "lt_linear: untuned GEMM shape (", M, "x", N, "x", K,
                    ") inside graph capture — warmup must run this shape first");
        int ran = tune_shape(M, N, K, has_bias, dt, w.data_ptr(), x.data_ptr(),
                             y.data_ptr(), bias, stream);
        TORCH_CHECK(ran > 0, "lt_linear: no hipblaslt algo for ",
                    M, "x", N, "x", K);
        std::lock_guard<std::mutex> lock(c.mu);
        algo = c.algos[key];
    }
    LT_CHECK(run());
    return true;
}

// Pre-tune one shape with scratch tensors (called from python warmup).
int lt_tune(int64_t M, int64_t N, int64_t K, bool has_bias,
            torch::Tensor scratch_x, torch::Tensor scratch_w,
            torch::Tensor scratch_y, c10::optional<torch::Tensor> bias_opt) {
    auto& c = ctx();
    if (c.disabled) return -1;
    hipDataType dt = lt_dtype(scratch_x);
    {
        std::lock_guard<std::mutex> lock(c.mu);
        if (c.algos.count(make_key(M, N, K, has_bias, dt))) return 0;
    }
    return tune_shape(M, N, K, has_bias, dt, scratch_w.data_ptr(),
                      scratch_x.data_ptr(), scratch_y.data_ptr(),
                      has_bias ? bias_opt->data_ptr() : nullptr,
                      at::hip::getCurrentHIPStream());
}
