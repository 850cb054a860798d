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
__global__ __launch_bounds__(256) void router_topk_kernel(
    float* __restrict__ vals,        // (T, k)
    long* __restrict__ idx,          // (T, k)
    const float* __restrict__ logits,  // (T, E)
    const int T, const int E, const int k,
    const int act_sigmoid, const int pre_softmax, const int normalize) {
    const int wid = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * 4 + wid;
    if (row >= T) return;
    const float* lr = logits + (long)row * E;

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

}  // namespace

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
