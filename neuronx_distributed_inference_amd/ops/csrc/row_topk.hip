// Largest element, and the k largest in order, of each row of logits. Order as in torch: NaN is
// the largest, equal values (-0 and 0 are) go by index. Elements become 64-bit keys, the value's
// bits in an order that integers compare in above the complement of the index.
//
// row_max: one workgroup of 1024 a row, 16 B loads, one launch. Bound by the instructions an element
// costs: a lane keeps the largest value and the vector it came in, keys are made of that vector
// only. Rows of 128256 in bf16, 1 row 17 -> 8 us, 64 rows 55 -> 8 us (torch's two-step
// reduction before), 256 rows 12.
// row_topk: a workgroup a row, one launch. The k-th largest of 1024 (k > 512: 4096) maxima of
// disjoint groups is a bound that at least k elements reach, and little more do: a second pass
// (from L2) gathers those into LDS, where they are sorted. Rows of up to 512: a wave each.
// Bound by the chain of two reads of the row and two sorts. us, torch's topk -> before -> now:
//   128256 in bf16, k = 256: 1 row 45 -> 84 -> 37, 64 rows 129 -> 237 -> 37, 256 rows 199 -> 776
//   -> 43; k = 50: 64 rows 127 -> 208 -> 27; k = 2048: 1 row 41 -> 168 -> 92, 64 rows 137 -> 405 ->
//   93; 32000, k = 256: 64 rows 68 -> 77 -> 27; 4096, k = 8: 1 row 34 -> 30 -> 13;
//   fp32 2048 rows of 128, k = 8: 29 -> 141 -> 8; 8192 of 64, k = 6: 39 -> 542 -> 9.
// Kernels only, so a captured step replays: torch's own topk over wide rows records a memset,
// which replays have not survived.

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

constexpr int RK_N = 4096;                       // keys a workgroup holds
constexpr int RK_SMALL = 512;                    // elements of a row that one wave sorts

// s[0 .. N), N a power of two, largest first. Steps of up to 64 keys stay inside the 128 keys of a
// wave's 64 pairs: only the others need a barrier.
template <bool WAVE>
DEV_INLINE void rk_sort(rk_key* s, const int N) {
    const int tid = WAVE ? threadIdx.x & 63 : threadIdx.x, all = WAVE ? 64 : 1024;
    bool wide = true;                            // the step before reached beyond a wave's keys
    for (int size = 2; size <= N; size <<= 1)
        for (int step = size >> 1; step > 0; step >>= 1) {
            if (!WAVE && (wide || step > 64)) __syncthreads();
            else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            wide = step > 64;
            for (int t = tid; t < N / 2; t += all) {
                const int lo = 2 * t - (t & (step - 1)), hi = lo + step;
                const rk_key a = s[lo], b = s[hi];
                // odd runs of `size` the other way until the last merge
                if ((a < b) == ((lo & size) == 0)) { s[lo] = b; s[hi] = a; }
            }
        }
    if (!WAVE) __syncthreads();
    else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// the keys of `s`, sorted, as values and indices
template <typename T>
DEV_INLINE void rk_emit(T* val, long* idx, const T* row, const rk_key* s, const int k,
                        const int first, const int all) {
    for (int i = first; i < k; i += all) {
        const unsigned at = rk_index(s[i]);
        val[i] = row[at];
        idx[i] = at;
    }
}

// rows of few elements: a wave each
template <typename T>
__global__ void __launch_bounds__(256)
row_topk_small_kernel(T* __restrict__ val, long* __restrict__ idx, const T* __restrict__ x,
                      const long stride, const long rows, const int n, const int N, const int k) {
    extern __shared__ rk_key small_keys[];
    const long r = blockIdx.x * 4L + (threadIdx.x >> 6);
    if (r >= rows) return;                       // whole waves; no barrier below
    rk_key* s = small_keys + (threadIdx.x >> 6) * N;
    const T* row = x + r * stride;
    for (int i = threadIdx.x & 63; i < N; i += 64)
        s[i] = i < n ? rk_pack(VecTraits<T>::to_float(row[i]), i) : 0;
    rk_sort<true>(s, N);
    rk_emit(val + r * k, idx + r * k, row, s, k, threadIdx.x & 63, 64);
}

// GP: groups that a thread keeps a maximum of; 1024 * GP of them are at least 2 k
template <typename T, int GP>
__global__ void __launch_bounds__(1024)
row_topk_kernel(T* __restrict__ val, long* __restrict__ idx, const T* __restrict__ x,
                const long stride, const int n, const int k, const int vec) {
    __shared__ rk_key s[RK_N];
    __shared__ int count;
    const long r = blockIdx.x;
    const T* row = x + r * stride;
    const int tid = threadIdx.x, nv = vec ? n / 8 : 0;
    constexpr int U = 4;                         // loads in flight

    // 1. a bound from below: the k-th of the groups' maxima (groups are disjoint)
    {
        float top[GP];
        int at[GP];                              // the vector, or element, it came in
#pragma unroll
        for (int g = 0; g < GP; ++g) { top[g] = 0.f; at[g] = -1; }
        auto take = [&](int g, float m, int from, bool in) {
            const bool t = in & ((at[g] < 0) | (m > top[g]) | ((m != m) & (top[g] == top[g])));
            top[g] = t ? m : top[g];
            at[g] = t ? from : at[g];
        };
        for (int i = tid; i < nv; i += 1024 * U) {
            Vec8<T> v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = load_vec8(row + min(i + u * 1024, nv - 1) * 8L);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                float m = VecTraits<T>::to_float(v[u].v[0]);
#pragma unroll
                for (int j = 1; j < 8; ++j)
                    m = __builtin_elementwise_maximum(m, VecTraits<T>::to_float(v[u].v[j]));
                take(u % GP, m, i + u * 1024, i + u * 1024 < nv);
            }
        }
        if (!vec)
            for (int i = tid; i < n; i += 1024 * U) {
                float v[U];
#pragma unroll
                for (int u = 0; u < U; ++u) v[u] = VecTraits<T>::to_float(row[min(i + u * 1024, n - 1)]);
#pragma unroll
                for (int u = 0; u < U; ++u) take(u % GP, v[u], i + u * 1024, i + u * 1024 < n);
            }
#pragma unroll
        for (int g = 0; g < GP; ++g) {
            rk_key best = 0;
            if (at[g] >= 0) {
                if (vec) {
                    const Vec8<T> v = load_vec8(row + at[g] * 8L);
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const rk_key key = rk_pack(VecTraits<T>::to_float(v.v[j]), at[g] * 8 + j);
                        best = key > best ? key : best;
                    }
                } else {
                    best = rk_pack(top[g], at[g]);
                }
            }
            // the up to 7 elements behind the last vector join the first threads' first groups
            const int rest = nv * 8 + tid;
            if (vec && g == 0 && rest < n) {
                const rk_key key = rk_pack(VecTraits<T>::to_float(row[rest]), rest);
                best = key > best ? key : best;
            }
            s[tid * GP + g] = best;
        }
    }
    rk_sort<false>(s, 1024 * GP);
    rk_key bound = s[k - 1];                     // 0: fewer than k groups have an element

    // 2. what reaches the bound, in any order. More than fits gives a better bound (at least
    // RK_N - k elements drop out each time: it ends)
    for (;;) {
        __syncthreads();
        if (tid == 0) count = 0;
        __syncthreads();
        const float least = bound ? rk_value(bound) : -INFINITY;
        auto put = [&](float v, int i) {
            const rk_key key = rk_pack(v, i);
            if (key < bound) return;
            const int at = atomicAdd(&count, 1);
            if (at < RK_N) s[at] = key;
        };
        for (int i = tid; i < nv; i += 1024 * U) {
            Vec8<T> v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = load_vec8(row + min(i + u * 1024, nv - 1) * 8L);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                float m = VecTraits<T>::to_float(v[u].v[0]);
#pragma unroll
                for (int j = 1; j < 8; ++j)
                    m = __builtin_elementwise_maximum(m, VecTraits<T>::to_float(v[u].v[j]));
                if (i + u * 1024 >= nv || m < least) continue;       // (a NaN is not below)
#pragma unroll
                for (int j = 0; j < 8; ++j) put(VecTraits<T>::to_float(v[u].v[j]), (i + u * 1024) * 8 + j);
            }
        }
        for (int i = nv * 8 + tid; i < n; i += 1024) {
            const float v = VecTraits<T>::to_float(row[i]);
            if (!(v < least)) put(v, i);
        }
        __syncthreads();
        if (count <= RK_N) break;                // uniform
        rk_sort<false>(s, RK_N);
        bound = s[k - 1];
    }

    // 3. those in order
    const int c = count;
    int N = 2;
    while (N < c) N <<= 1;
    for (int i = c + tid; i < N; i += 1024) s[i] = 0;
    rk_sort<false>(s, N);
    rk_emit(val + r * k, idx + r * k, row, s, k, tid, 1024);
}

// rows of few elements: a wave each
template <typename T>
__global__ void __launch_bounds__(256)
row_max_small_kernel(T* __restrict__ val, long* __restrict__ idx, const T* __restrict__ x,
                     const long stride, const long rows, const int n) {
    const long r = blockIdx.x * 4L + (threadIdx.x >> 6);
    if (r >= rows) return;
    const T* row = x + r * stride;
    rk_key best = 0;
    for (int i = threadIdx.x & 63; i < n; i += 64) {
        const rk_key k = rk_pack(VecTraits<T>::to_float(row[i]), i);
        best = k > best ? k : best;
    }
    best = rk_wave_max(best);
    if ((threadIdx.x & 63) == 0) {
        idx[r] = rk_index(best);
        val[r] = row[rk_index(best)];
    }
}

constexpr long RK_ROWS = 1L << 20;               // rows of a launch

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
    auto st = at::hip::getCurrentHIPStream();
    const long es = x.element_size(), n = x.size(1);
    const int vec = (size_t)x.data_ptr() % 16 == 0 && x.stride(0) * es % 16 == 0;
    for (long r = 0; r < x.size(0); r += RK_ROWS) {
        const long rows = std::min(RK_ROWS, x.size(0) - r);
#define RK_MAX_ARGS (scalar_t*)val.data_ptr() + r, idx.data_ptr<long>() + r,                       \
        (const scalar_t*)x.data_ptr() + r * x.stride(0), x.stride(0)
        // a wave for up to 1024 elements: fp32 8192 rows of 64 27 -> 3 us (torch's 6), 2048 of 1000 8.7 -> 5.0
        if (n <= 1024)
            RK_DISPATCH(x.scalar_type(), hipLaunchKernelGGL(row_max_small_kernel<scalar_t>,
                dim3((rows + 3) / 4), dim3(256), 0, st, RK_MAX_ARGS, rows, (int)n));
        else
            RK_DISPATCH(x.scalar_type(), hipLaunchKernelGGL(row_max_kernel<scalar_t>, dim3(rows),
                dim3(1024), 0, st, RK_MAX_ARGS, (int)n, vec));
#undef RK_MAX_ARGS
        HIP_CHECK_KERNEL();
    }
}

void row_topk(torch::Tensor val, torch::Tensor idx, torch::Tensor x, long k) {
    TORCH_CHECK(k >= 1 && k <= RK_N / 2 && k <= x.size(1), "row_topk: k");
    rk_check(x, val, idx, k);
    auto st = at::hip::getCurrentHIPStream();
    const long es = x.element_size(), n = x.size(1);
    // (rows of fewer vectors than threads give each thread an element before a second one)
    const int vec = n >= 8 * 1024 && (size_t)x.data_ptr() % 16 == 0 && x.stride(0) * es % 16 == 0;
    int N = 2;
    while (N < n) N <<= 1;
    for (long r = 0; r < x.size(0); r += RK_ROWS) {
        const long rows = std::min(RK_ROWS, x.size(0) - r);
#define RK_TOPK_ARGS (scalar_t*)val.data_ptr() + r * k, idx.data_ptr<long>() + r * k,              \
        (const scalar_t*)x.data_ptr() + r * x.stride(0), x.stride(0)
        if (n <= RK_SMALL)
            RK_DISPATCH(x.scalar_type(), hipLaunchKernelGGL(row_topk_small_kernel<scalar_t>,
                dim3((rows + 3) / 4), dim3(256), 4 * N * sizeof(rk_key), st, RK_TOPK_ARGS, rows,
                (int)n, N, (int)k));
        else if (k <= 512)
            RK_DISPATCH(x.scalar_type(), hipLaunchKernelGGL((row_topk_kernel<scalar_t, 1>), dim3(rows),
                dim3(1024), 0, st, RK_TOPK_ARGS, (int)n, (int)k, vec));
        else
            RK_DISPATCH(x.scalar_type(), hipLaunchKernelGGL((row_topk_kernel<scalar_t, 4>), dim3(rows),
                dim3(1024), 0, st, RK_TOPK_ARGS, (int)n, (int)k, vec));
#undef RK_TOPK_ARGS
        HIP_CHECK_KERNEL();
    }
}
