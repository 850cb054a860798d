// Largest element, and the k largest in order, of each row of logits. Order as in torch: NaN is
// the largest, equal values (-0 and 0 are) go by index. Elements become 64-bit keys, the value's
// bits in an order that integers compare in above the complement of the index.
//
// row_max: one workgroup of 1024 a row, 16 B loads, one launch. Bound by the instructions an element
// costs: a lane keeps the largest value and the vector it came in, keys are made of that vector
// only. Rows of 128256 in bf16, 1 row 17 -> 8 us, 64 rows 55 -> 8 us (torch's two-step
// reduction before), 256 rows 12.
// row_topk: workgroups sort 4096 keys each in LDS (bitonic) and hand the first k on until one is
// left: 3 launches for 128256 and k = 256 (1 row 84 us, 64 rows 236). Kernels only, so a captured step replays: torch's own
// topk over wide rows records a memset, which replays have not survived.

#include "common.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

namespace {

typedef unsigned long long rk_key;

DEV_INLINE rk_key rk_pack(float v, unsigned idx) {
    unsigned u = __float_as_uint(v + 0.f);       // -0 becomes 0
    u = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
    if (v != v) u = 0xffffffffu;
    return ((rk_key)u << 32) | (0xffffffffu - idx);
}
DEV_INLINE float rk_value(rk_key k) {
    const unsigned u = (unsigned)(k >> 32);
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}
DEV_INLINE unsigned rk_index(rk_key k) { return 0xffffffffu - (unsigned)k; }

DEV_INLINE rk_key rk_wave_max(rk_key v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const rk_key o = __shfl_xor(v, off, WAVE_SIZE);
        v = o > v ? o : v;
    }
    return v;
}

template <typename T>
__global__ void __launch_bounds__(1024)
row_max_kernel(T* __restrict__ val, long* __restrict__ idx, const T* __restrict__ x,
               const long stride, const int n, const int vec) {
    __shared__ rk_key part[16];
    const T* row = x + blockIdx.x * stride;
    rk_key best = 0;
    const int nv = vec ? n / 8 : 0;
    // a thread keeps the largest value (NaN once seen) and the vector it came in
    float top = 0.f;
    int at = -1;
    for (int i = threadIdx.x; i < nv; i += 4096) {
        Vec8<T> v[4];                            // four loads in flight
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = load_vec8(row + min(i + u * 1024, nv - 1) * 8L);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            float m = VecTraits<T>::to_float(v[u].v[0]);
#pragma unroll
            for (int j = 1; j < 8; ++j)
                m = __builtin_elementwise_maximum(m, VecTraits<T>::to_float(v[u].v[j]));
            const bool take = (at < 0) | (m > top) | ((m != m) & (top == top));
            top = take ? m : top;
            at = take ? min(i + u * 1024, nv - 1) : at;
        }
    }
    if (at >= 0) {
        const Vec8<T> v = load_vec8(row + at * 8L);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const rk_key k = rk_pack(VecTraits<T>::to_float(v.v[j]), at * 8 + j);
            best = k > best ? k : best;
        }
    }
    for (int i = nv * 8 + threadIdx.x; i < n; i += 1024) {
        const rk_key k = rk_pack(VecTraits<T>::to_float(row[i]), i);
        best = k > best ? k : best;
    }
    best = rk_wave_max(best);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x < 64) {
        best = rk_wave_max(threadIdx.x < 16 ? part[threadIdx.x] : 0);
        if (threadIdx.x == 0) {
            const unsigned i = rk_index(best);
            idx[blockIdx.x] = i;
            val[blockIdx.x] = row[i];
        }
    }
}

constexpr int RK_N = 4096;                       // keys a workgroup sorts

// keys (rows, n) or x (rows, n) -> the k largest of each 4096, in order: to `out` as keys
// (rows, gridDim.x * k), or with val/idx as the result
template <typename T>
__global__ void __launch_bounds__(1024)
row_topk_kernel(rk_key* __restrict__ out, T* __restrict__ val, long* __restrict__ idx,
                const T* __restrict__ x, const long stride, const rk_key* __restrict__ keys,
                const int n, const int k) {
    __shared__ rk_key s[RK_N];
    const int row = blockIdx.y, base = blockIdx.x * RK_N;
    for (int i = threadIdx.x; i < RK_N; i += 1024) {
        const int at = base + i;
        s[i] = at >= n ? 0 : keys ? keys[(long)row * n + at]
                                  : rk_pack(VecTraits<T>::to_float(x[row * stride + at]), at);
    }
    for (int size = 2; size <= RK_N; size <<= 1)
        for (int step = size >> 1; step > 0; step >>= 1) {
            __syncthreads();
#pragma unroll
            for (int p = 0; p < RK_N / 2; p += 1024) {
                const int t = p + threadIdx.x;
                const int lo = 2 * t - (t & (step - 1)), hi = lo + step;
                const rk_key a = s[lo], b = s[hi];
                // largest first; odd runs of `size` the other way until the last merge
                if ((a < b) == ((lo & size) == 0)) { s[lo] = b; s[hi] = a; }
            }
        }
    __syncthreads();
    for (int i = threadIdx.x; i < k; i += 1024) {
        const rk_key v = s[i];
        if (val) {
            val[(long)row * k + i] = VecTraits<T>::from_float(rk_value(v));
            idx[(long)row * k + i] = rk_index(v);
        } else {
            out[((long)row * gridDim.x + blockIdx.x) * k + i] = v;
        }
    }
}

#define RK_DISPATCH(TYPE, ...)                                                                     \
    do {                                                                                           \
        if (TYPE == at::ScalarType::BFloat16) { using scalar_t = __hip_bfloat16; __VA_ARGS__; }    \
        else if (TYPE == at::ScalarType::Half) { using scalar_t = __half; __VA_ARGS__; }           \
        else if (TYPE == at::ScalarType::Float) { using scalar_t = float; __VA_ARGS__; }           \
        else { TORCH_CHECK(false, "row_topk: unsupported dtype"); }                                \
    } while (0)

void rk_check(const torch::Tensor& x, const torch::Tensor& val, const torch::Tensor& idx, long k) {
    TORCH_CHECK(x.dim() == 2 && x.stride(1) == 1 && x.size(1) >= 1 && x.size(1) < (1L << 31) - RK_N,
                "row_topk: rows of at least one element");
    TORCH_CHECK(val.scalar_type() == x.scalar_type() && idx.scalar_type() == at::ScalarType::Long &&
                val.is_contiguous() && idx.is_contiguous() && val.numel() == x.size(0) * k &&
                idx.numel() == x.size(0) * k, "row_topk: results");
}

}  // namespace

void row_max(torch::Tensor val, torch::Tensor idx, torch::Tensor x) {
    rk_check(x, val, idx, 1);
    if (x.size(0) == 0) return;
    auto st = at::hip::getCurrentHIPStream();
    const long es = x.element_size();
    const int vec = (size_t)x.data_ptr() % 16 == 0 && x.stride(0) * es % 16 == 0;
    RK_DISPATCH(x.scalar_type(), hipLaunchKernelGGL(row_max_kernel<scalar_t>, dim3(x.size(0)),
        dim3(1024), 0, st, (scalar_t*)val.data_ptr(), idx.data_ptr<long>(),
        (const scalar_t*)x.data_ptr(), x.stride(0), (int)x.size(1), vec));
    HIP_CHECK_KERNEL();
}

// ws: int64, room for two passes' keys
void row_topk(torch::Tensor val, torch::Tensor idx, torch::Tensor x, torch::Tensor ws, long k) {
    TORCH_CHECK(k >= 1 && k <= RK_N / 2 && k <= x.size(1), "row_topk: k");
    rk_check(x, val, idx, k);
    const long rows = x.size(0);
    TORCH_CHECK(rows < 65536, "row_topk: rows");
    if (rows == 0) return;
    const long need = rows * k * ((x.size(1) + RK_N - 1) / RK_N);
    TORCH_CHECK(ws.scalar_type() == at::ScalarType::Long && ws.is_contiguous() &&
                ws.numel() >= 2 * need, "row_topk: workspace");
    auto st = at::hip::getCurrentHIPStream();
    rk_key* buf[2] = {(rk_key*)ws.data_ptr(), (rk_key*)ws.data_ptr() + need};
    const rk_key* in = nullptr;
    long n = x.size(1);
    for (int pass = 0;; ++pass) {
        const long nb = (n + RK_N - 1) / RK_N;
        const bool last = nb == 1;
        rk_key* out = last ? nullptr : buf[pass & 1];
        RK_DISPATCH(x.scalar_type(), hipLaunchKernelGGL(row_topk_kernel<scalar_t>, dim3(nb, rows),
            dim3(1024), 0, st, out, last ? (scalar_t*)val.data_ptr() : nullptr,
            last ? idx.data_ptr<long>() : nullptr, (const scalar_t*)x.data_ptr(), x.stride(0), in,
            (int)n, (int)k));
        HIP_CHECK_KERNEL();
        if (last) return;
        in = out;
        n = nb * k;
    }
}
