// Fused MoE router selection (SURVEY §2.7 router analog): ONE kernel
// replaces the torch topk chain (gatherTopK + bitonicSort + softmax +
// div — measured ~0.9 ms/step of launch latency on Mixtral b256 decode,
// rocprofv3 r02_moe_quant_kernel_stats.md): the top-k (k <= 8) of E
// logits, then the router activation (post-softmax over k | full-E pre-softmax |
// sigmoid) and optional sum-normalization — all in fp32, matching
// modules/moe.py MoERouter semantics.

#include "common.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

namespace {

constexpr int KMAX = 8;

// largest of a wave's values, in every lane; down the rows of 16 lanes and across them by DPP, which
// takes a few cycles a step where a shuffle goes through the LDS
DEV_INLINE float rt_wave_max(float x) {
#define RT_STEP(CTRL, ROWS)                                                                        \
    x = fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(                            \
                     __builtin_bit_cast(int, x), __builtin_bit_cast(int, x), CTRL, ROWS, 0xf, false)))
    RT_STEP(0x111, 0xf);             // row_shr 1, 2, 4, 8
    RT_STEP(0x112, 0xf);
    RT_STEP(0x114, 0xf);
    RT_STEP(0x118, 0xf);
    RT_STEP(0x142, 0xa);             // row_bcast 15, 31
    RT_STEP(0x143, 0xc);
#undef RT_STEP
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), 63));
}

// One wave per token row: k rounds of the wave's largest value, the lowest index first. NE > 0: a
// lane keeps its NE logits in registers; 0: reads them anew each round (more than 512 experts).
// Bound by the rounds' chain of exchanges: 2048 rows of 128 logits, 8 chosen, 14.5 us with 12
// shuffles a round, 6.0 now.
template <int NE>
DEV_INLINE void rt_row(float* vals, long* idx, const float* lr, const int row, const int E,
                       const int k, const int act_sigmoid, const int pre_softmax,
                       const int normalize) {
    const int lane = threadIdx.x & 63;
    float cv[KMAX];
    int ci[KMAX];
#pragma unroll
    for (int j = 0; j < KMAX; ++j) {
        cv[j] = -1e30f;
        ci[j] = -1;
    }
    // what is not chosen at all (below -1e30, NaN) or any more is -inf
    float v[NE ? NE : 1];
    if constexpr (NE > 0) {
#pragma unroll
        for (int n = 0; n < NE; ++n) {
            const float x = n * 64 + lane < E ? lr[n * 64 + lane] : -INFINITY;
            v[n] = x >= -1e30f ? x : -INFINITY;
        }
    }
#pragma unroll
    for (int round = 0; round < KMAX; ++round) {
        if (round >= k) break;
        float m = -INFINITY;
        int li = E;                  // nothing left: an index past the last
        if constexpr (NE > 0) {
#pragma unroll
            for (int n = 0; n < NE; ++n) m = fmaxf(m, v[n]);
            m = rt_wave_max(m);
            if (m != -INFINITY) {
#pragma unroll
                for (int n = NE - 1; n >= 0; --n) {
                    const unsigned long long has = __ballot(v[n] == m);
                    if (has) li = n * 64 + __ffsll(has) - 1;
                }
#pragma unroll
                for (int n = 0; n < NE; ++n)
                    if (n * 64 + lane == li) v[n] = -INFINITY;
            }
        } else {
            for (int e = lane; e < E; e += 64) {
                bool taken = false;
#pragma unroll
                for (int j = 0; j < KMAX; ++j)
                    if (j < round) taken = taken || (e == ci[j]);
                const float x = lr[e];
                if (!taken && x >= -1e30f && (x > m || li == E)) {
                    m = x;
                    li = e;
                }
            }
            const float w = rt_wave_max(m);
            int lowest = m == w && li < E ? li : E;
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1)
                lowest = min(lowest, __shfl_xor(lowest, off, 64));
            m = w;
            li = lowest;
        }
        cv[round] = m == -INFINITY ? -1e30f : m;
        ci[round] = li;
    }

    if (pre_softmax) {
        // full-E softmax: cv[0] IS the max — snapshot before the
        // in-place exp overwrites it
        const float fm = cv[0];
        float ls = 0.f;
        for (int e = lane; e < E; e += 64) ls += __expf(lr[e] - fm);
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1)
            ls += __shfl_down(ls, off, 64);
        ls = __shfl(ls, 0, 64);
#pragma unroll
        for (int j = 0; j < KMAX; ++j)
            if (j < k) cv[j] = __expf(cv[j] - fm) / ls;
    } else if (act_sigmoid) {
#pragma unroll
        for (int j = 0; j < KMAX; ++j)
            if (j < k) cv[j] = 1.f / (1.f + __expf(-cv[j]));
    } else {
        const float m0 = cv[0];
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < KMAX; ++j)
            if (j < k) {
                cv[j] = __expf(cv[j] - m0);
                s += cv[j];
            }
#pragma unroll
        for (int j = 0; j < KMAX; ++j)
            if (j < k) cv[j] /= s;
    }
    if (normalize) {
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < KMAX; ++j)
            if (j < k) s += cv[j];
#pragma unroll
        for (int j = 0; j < KMAX; ++j)
            if (j < k) cv[j] /= fmaxf(s, 1e-20f);
    }
    if (lane == 0) {
#pragma unroll
        for (int j = 0; j < KMAX; ++j)
            if (j < k) {
                vals[(long)row * k + j] = cv[j];
                idx[(long)row * k + j] = ci[j];
            }
    }
}

template <int NE>
__global__ __launch_bounds__(256) void router_topk_kernel(
    float* __restrict__ vals,        // (T, k)
    long* __restrict__ idx,          // (T, k)
    const float* __restrict__ logits,  // (T, E)
    const int T, const int E, const int k,
    const int act_sigmoid, const int pre_softmax, const int normalize) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= T) return;
    rt_row<NE>(vals, idx, logits + (long)row * E, row, E, k, act_sigmoid, pre_softmax, normalize);
}

// Logits of up to 16 experts in 32 bits, of rows in 16 or 32, and the choice among them. A
// workgroup has R rows and all experts: 8 channels a thread and turn, the sums over the waves
// through LDS, then a wave a row chooses. Few rows are bound by latency, which is why this is one
// launch for three (conversion to 32 bits, the library's product, the choice): 8 experts of 4096, 2
// chosen, 1 row 12.8 -> 5.1 us, 128 rows 15.0 -> 5.9, 511 18.4 -> 8.9; 16 of 5120, 100 rows 16.9 ->
// 11.8, 511 21.5 -> 18.2. From 1024 rows on four share what they read of w: 8 experts 24.6 -> 12.2,
// 4096 rows 35.3 -> 31.9; of more experts such rows are the library's (16, 4000 rows 40.7 against 54.9).
template <typename T, int EP, int R>
__global__ __launch_bounds__(512) void router_few_kernel(
    float* __restrict__ vals, long* __restrict__ idx, const T* __restrict__ x,
    const float* __restrict__ w, const int rows, const int E, const int K, const int k,
    const int act_sigmoid, const int pre_softmax, const int normalize) {
    __shared__ float part[8][R * EP], logits[R * EP];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int row0 = blockIdx.x * R;
    float acc[R][EP];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int e = 0; e < EP; ++e) acc[r][e] = 0.f;
    for (int c = threadIdx.x * 8; c < K; c += 4096) {
        Vec8<T> xs[R];
#pragma unroll
        for (int r = 0; r < R; ++r) xs[r] = load_vec8(x + (long)min(row0 + r, rows - 1) * K + c);
#pragma unroll
        for (int e = 0; e < EP; ++e) {
            const Vec8<float> we = load_vec8(w + (long)min(e, E - 1) * K + c);
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int i = 0; i < 8; ++i) acc[r][e] += VecTraits<T>::to_float(xs[r].v[i]) * we.v[i];
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int e = 0; e < EP; ++e) {
            const float v = wave_reduce_sum(acc[r][e]);
            if (lane == 0) part[wid][r * EP + e] = v;
        }
    __syncthreads();
    if (threadIdx.x < R * EP) {
        float v = part[0][threadIdx.x];
#pragma unroll
        for (int i = 1; i < 8; ++i) v += part[i][threadIdx.x];
        logits[threadIdx.x] = v;
    }
    __syncthreads();
    if (wid < R && row0 + wid < rows)
        rt_row<1>(vals, idx, logits + wid * EP, row0 + wid, E, k, act_sigmoid, pre_softmax, normalize);
}

}  // namespace

// The choice of rows x (T, K) among E <= 16 experts with weights w (E, K) in fp32.
void router_few(torch::Tensor vals, torch::Tensor idx, torch::Tensor x, torch::Tensor w, long top_k,
                long act_sigmoid, long pre_softmax, long normalize) {
    TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && x.size(1) == w.size(1) && x.size(1) % 8 == 0 &&
                x.size(1) > 0, "router_few: shapes");
    const int rows = x.size(0), E = w.size(0), K = x.size(1);
    TORCH_CHECK(E >= top_k && E <= 16 && top_k >= 1 && top_k <= KMAX, "router_few: up to 16 experts");
    TORCH_CHECK(x.is_cuda() && w.is_cuda() && x.device() == w.device() && vals.device() == x.device() &&
                idx.device() == x.device(), "router_few: tensors of one GPU");
    TORCH_CHECK(x.is_contiguous() && w.is_contiguous() && w.scalar_type() == at::ScalarType::Float &&
                ((size_t)x.data_ptr() | (size_t)w.data_ptr()) % 16 == 0, "router_few: layout");
    TORCH_CHECK(vals.numel() == rows * top_k && idx.numel() == rows * top_k && vals.is_contiguous() &&
                idx.is_contiguous() && vals.scalar_type() == at::ScalarType::Float &&
                idx.scalar_type() == at::ScalarType::Long, "router_few: out shapes");
    if (rows == 0) return;
    auto stream = at::hip::getCurrentHIPStream();
    const bool four = rows >= 1024;
#define RF_GO(T, EP, R)                                                                            \
    hipLaunchKernelGGL((router_few_kernel<T, EP, R>), dim3((rows + R - 1) / R), dim3(512), 0,      \
                       stream, vals.data_ptr<float>(), idx.data_ptr<long>(),                       \
                       (const T*)x.data_ptr(), w.data_ptr<float>(), rows, E, K, (int)top_k,        \
                       (int)act_sigmoid, (int)pre_softmax, (int)normalize)
#define RF_T(T)                                                                                    \
    do {                                                                                           \
        if (E <= 8 && four) RF_GO(T, 8, 4);                                                        \
        else if (E <= 8) RF_GO(T, 8, 1);                                                           \
        else RF_GO(T, 16, 1);                                                                      \
    } while (0)
    if (x.scalar_type() == at::ScalarType::BFloat16) RF_T(__hip_bfloat16);
    else if (x.scalar_type() == at::ScalarType::Half) RF_T(__half);
    else if (x.scalar_type() == at::ScalarType::Float) RF_T(float);
    else TORCH_CHECK(false, "router_few: x in fp32, bf16 or f16");
#undef RF_T
#undef RF_GO
    HIP_CHECK_KERNEL();
}

void router_topk(torch::Tensor vals, torch::Tensor idx, torch::Tensor logits,
                 long top_k, long act_sigmoid, long pre_softmax,
                 long normalize) {
    TORCH_CHECK(logits.dim() == 2 && logits.is_contiguous() &&
                logits.scalar_type() == at::ScalarType::Float, "logits f32");
    const int T = logits.size(0), E = logits.size(1);
    TORCH_CHECK(top_k >= 1 && top_k <= KMAX, "top_k <= 8");
    TORCH_CHECK(vals.numel() == T * top_k && idx.numel() == T * top_k &&
                vals.scalar_type() == at::ScalarType::Float &&
                idx.scalar_type() == at::ScalarType::Long, "out shapes");
    auto stream = at::hip::getCurrentHIPStream();
    const int threads = 256;          // 4 waves; one wave per row
    const int blocks = (T + 3) / 4;
    if (T == 0) return;
#define RT_GO(NE)                                                                      \
    hipLaunchKernelGGL((router_topk_kernel<NE>), dim3(blocks), dim3(threads), 0,       \
                       stream, vals.data_ptr<float>(), idx.data_ptr<long>(),           \
                       logits.data_ptr<float>(), T, E, (int)top_k,                     \
                       (int)act_sigmoid, (int)pre_softmax, (int)normalize)
    if (E <= 64) RT_GO(1);
    else if (E <= 128) RT_GO(2);
    else if (E <= 256) RT_GO(4);
    else if (E <= 512) RT_GO(8);
    else RT_GO(0);
#undef RT_GO
    HIP_CHECK_KERNEL();
}
