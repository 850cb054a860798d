// Fused post-QKV-GEMM decode plumbing (a big slice of the reference's K2
// fused TKG block, attention_block_tkg): one kernel takes the fused
// qkv GEMM output (B, S, (Hq+2Hkv)*D), applies RoPE to q and k, scatters
// k and v into the linear KV cache at (seq_id, position), and emits q in
// the (B, Hq, S, D) layout the decode-attention kernel wants. Replaces
// 3 transpose-copies + rope + kv_update (5 kernel launches + 4 extra HBM
// round trips per layer per step).
//
// Also: silu/gelu on a fused gate|up GEMM output without the chunk copies.

#include "common.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

template <typename T, typename CT>
__global__ void qkv_rope_update_kernel(
    T* __restrict__ q_out,           // (B, Hq, S, D)
    const T* __restrict__ qkv,       // (B, S, (Hq+2Hkv)*D)
    const float* __restrict__ cosb,  // (B, S, D)
    const float* __restrict__ sinb,
    CT* __restrict__ k_cache,        // (Bc, Hkv, Smax, D)
    CT* __restrict__ v_cache,
    const int* __restrict__ positions,  // (B, S)
    const int* __restrict__ seq_ids,    // (B,)
    const int B, const int S, const int Hq, const int Hkv,
    const int D, const int Bc, const int Smax) {
    using VT = VecTraits<T>;
    const int half = D / 2;
    const int Ht = Hq + 2 * Hkv;
    // direct 2D grid: blockIdx.x = (b, s) row, blockIdx.y covers Ht*half —
    // the grid-stride formulation spent its cycles on per-iteration 64-bit
    // div/mod (measured 45 GB/s at prefill scale)
    {
        const int bs = blockIdx.x;
        const int b = bs / S;
        const int s = bs % S;
        const int idx = blockIdx.y * blockDim.x + threadIdx.x;
        if (idx >= Ht * half) return;
        const int h = idx / half;
        const int i = idx % half;

        const T* src = qkv + (((long)b * S + s) * Ht + h) * D;
        const float x1f = VT::to_float(src[i]);
        const float x2f = VT::to_float(src[i + half]);

        float o1f, o2f;
        if (h < Hq + Hkv) {  // rope for q and k
            const float c = cosb[((long)b * S + s) * D + i];
            const float sn = sinb[((long)b * S + s) * D + i];
            o1f = x1f * c - x2f * sn;
            o2f = x2f * c + x1f * sn;
        } else {             // v: plain copy
            o1f = x1f;
            o2f = x2f;
        }

        if (h < Hq) {
            T* dst = q_out + (((long)b * Hq + h) * S + s) * D;
            dst[i] = VT::from_float(o1f);
            dst[i + half] = VT::from_float(o2f);
        } else {
            const int row = seq_ids[b];
            const int pos = positions[(long)b * S + s];
            if (row < 0 || row >= Bc || pos < 0 || pos >= Smax) return;
            const bool is_k = h < Hq + Hkv;
            const int hk = is_k ? h - Hq : h - Hq - Hkv;
            CT* cache = is_k ? k_cache : v_cache;
            CT* dst = cache + (((long)row * Hkv + hk) * Smax + pos) * D;
            dst[i] = VecTraits<CT>::from_float(o1f);
            dst[i + half] = VecTraits<CT>::from_float(o2f);
        }
    }
}

// The same for head sizes of 16 L, with optional per-head RMS norms of q and k before the rope and
// with pages (a flat slot per token, caches (slots, Hkv, D)) as well as rows. A lane takes 8
// channels of each half of a head, L lanes a head: 16 B loads and stores, the norm a sum over L
// lanes. Bound by memory: 8192 tokens of (32 + 2 x 8) heads of 128 (200 MB in and out) took 91 us
// a channel pair at a time; a model step over them 12.94 -> 12.72 ms.
// With norms or pages it stands for norms, rope, copies and cache write of their own: a prompt of
// 2048 tokens, (32 + 2 x 4) heads, 2 layers 1550 -> 1285 us; 512 tokens onto 3500 in pages,
// (32 + 2 x 8) heads, 4 layers 1780 -> 1660 us.
template <typename T, typename CT, int L>
__global__ void __launch_bounds__(256)
qkv_rope_vec_kernel(T* __restrict__ q_out, const T* __restrict__ qkv,
                    const float* __restrict__ qkv_parts, const int nparts,
                    const float* __restrict__ cosb, const float* __restrict__ sinb,
                    CT* __restrict__ k_cache, CT* __restrict__ v_cache,
                    const int* __restrict__ positions, const int* __restrict__ seq_ids,
                    const int* __restrict__ slots, const T* __restrict__ qw,
                    const T* __restrict__ kw, const float eps, const int rows, const int S,
                    const int Hq, const int Hkv, const int Bc, const long Smax) {
    using VT = VecTraits<T>;
    constexpr int D = 16 * L, half = D / 2;
    const int Ht = Hq + 2 * Hkv, per = Ht * L;
    const long item = (long)blockIdx.x * 256 + threadIdx.x;
    const int bs = (int)(item / per);
    if (bs >= rows) return;                      // whole heads: `per` is a multiple of L
    const int in = (int)(item - (long)bs * per), h = in / L, i = (in % L) * 8;
    const int b = bs / S, s = bs - b * S;
    const long at0 = ((long)bs * Ht + h) * D + i;
    float x1[8], x2[8];
    if (nparts == 0) {
        const Vec8<T> a = load_vec8(qkv + at0), c = load_vec8(qkv + at0 + half);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            x1[j] = VT::to_float(a.v[j]);
            x2[j] = VT::to_float(c.v[j]);
        }
    } else {                                     // the parts of a split product
        const long plane = (long)rows * Ht * D;
        const float* p = qkv_parts + at0;
        Vec8<float> a = load_vec8(p), c = load_vec8(p + half);
        int k = 1;
        for (; k + 2 <= nparts; k += 2) {
            const Vec8<float> a1 = load_vec8(p + k * plane), c1 = load_vec8(p + k * plane + half);
            const Vec8<float> a2 = load_vec8(p + (k + 1) * plane),
                              c2 = load_vec8(p + (k + 1) * plane + half);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                a.v[j] += a1.v[j] + a2.v[j];
                c.v[j] += c1.v[j] + c2.v[j];
            }
        }
        if (k < nparts) {
            const Vec8<float> a1 = load_vec8(p + k * plane), c1 = load_vec8(p + k * plane + half);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                a.v[j] += a1.v[j];
                c.v[j] += c1.v[j];
            }
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            x1[j] = a.v[j];
            x2[j] = c.v[j];
        }
    }
    if (h < Hq + Hkv) {
        const T* w = h < Hq ? qw : kw;
        if (w) {
            float ssq = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j) ssq += x1[j] * x1[j] + x2[j] * x2[j];
            ssq = group_reduce_sum<L>(ssq);
            const float inv = rsqrtf(ssq / D + eps);
            const Vec8<T> w1 = load_vec8(w + i), w2 = load_vec8(w + half + i);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                x1[j] = x1[j] * inv * VT::to_float(w1.v[j]);
                x2[j] = x2[j] * inv * VT::to_float(w2.v[j]);
            }
        }
        const Vec8<float> cv = load_vec8(cosb + (long)bs * D + i);
        const Vec8<float> sv = load_vec8(sinb + (long)bs * D + i);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float o1 = x1[j] * cv.v[j] - x2[j] * sv.v[j];
            x2[j] = x2[j] * cv.v[j] + x1[j] * sv.v[j];
            x1[j] = o1;
        }
    }
    if (h < Hq) {
        Vec8<T> o1, o2;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            o1.v[j] = VT::from_float(x1[j]);
            o2.v[j] = VT::from_float(x2[j]);
        }
        T* dst = q_out + (((long)b * Hq + h) * S + s) * D + i;
        store_vec8(dst, o1);
        store_vec8(dst + half, o2);
        return;
    }
    const bool is_k = h < Hq + Hkv;
    const int hk = is_k ? h - Hq : h - Hq - Hkv;
    long at;
    if (slots) {
        const long slot = slots[bs];
        if (slot < 0 || slot >= Smax) return;    // Smax: slots of the whole cache
        at = slot * Hkv + hk;
    } else {
        const int row = seq_ids[b], pos = positions[bs];
        if (row < 0 || row >= Bc || pos < 0 || pos >= Smax) return;
        at = ((long)row * Hkv + hk) * Smax + pos;
    }
    Vec8<CT> o1, o2;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        o1.v[j] = VecTraits<CT>::from_float(x1[j]);
        o2.v[j] = VecTraits<CT>::from_float(x2[j]);
    }
    CT* dst = (is_k ? k_cache : v_cache) + at * D + i;
    store_vec8(dst, o1);
    store_vec8(dst + half, o2);
}

template <typename T, bool GELU>
__global__ void act_mul_fused_kernel(
    T* __restrict__ out,             // (rows, I)
    const T* __restrict__ gate_up,   // (rows, 2I): [gate | up]
    const long rows, const int I) {
    using VT = VecTraits<T>;
    // blockIdx.x = row, blockIdx.y covers I/8 (see qkv kernel note on the
    // div/mod cost of the grid-stride form)
    {
        const long r = blockIdx.x;
        const int c8 = blockIdx.y * blockDim.x + threadIdx.x;
        if (c8 >= I / 8) return;
        Vec8<T> g = load_vec8(gate_up + r * 2 * I + c8 * 8);
        Vec8<T> u = load_vec8(gate_up + r * 2 * I + I + c8 * 8);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            float gf = VT::to_float(g.v[j]);
            float uf = VT::to_float(u.v[j]);
            float a;
            if constexpr (GELU) {
                const float cc = 0.7978845608028654f;
                a = 0.5f * gf * (1.f + tanhf(cc * (gf + 0.044715f * gf * gf * gf)));
            } else {
                a = gf / (1.f + __expf(-gf));
            }
            g.v[j] = VT::from_float(a * uf);
        }
        store_vec8(out + r * I + c8 * 8, g);
    }
}

#define DISPATCH_FT(TYPE, NAME, ...)                                           \
    [&] {                                                                      \
        if (TYPE == at::ScalarType::BFloat16) {                                \
            using scalar_t = __hip_bfloat16;                                   \
            return __VA_ARGS__();                                              \
        } else if (TYPE == at::ScalarType::Half) {                             \
            using scalar_t = __half;                                           \
            return __VA_ARGS__();                                              \
        } else if (TYPE == at::ScalarType::Float) {                            \
            using scalar_t = float;                                            \
            return __VA_ARGS__();                                              \
        } else {                                                               \
            TORCH_CHECK(false, NAME ": unsupported dtype");                    \
        }                                                                      \
    }()

void qkv_rope_update(torch::Tensor q_out, torch::Tensor qkv,
                     torch::Tensor cosb, torch::Tensor sinb,
                     torch::Tensor k_cache, torch::Tensor v_cache,
                     torch::Tensor positions, torch::Tensor seq_ids,
                     long Hq, long Hkv, c10::optional<torch::Tensor> q_norm,
                     c10::optional<torch::Tensor> k_norm, double eps,
                     c10::optional<torch::Tensor> slots) {
    // qkv: (B, S, width), or its parts in fp32, (parts, B, S, width) beside a q_out of 16 bits
    const int nparts = qkv.dim() == 4 ? (int)qkv.size(0) : 0;
    const int B = q_out.size(0), S = q_out.size(2);
    const int D = k_cache.size(3);
    const int Bc = k_cache.size(0), Smax = k_cache.size(2);
    TORCH_CHECK(qkv.size(-1) == (Hq + 2 * Hkv) * D &&
                qkv.numel() == (long)std::max(nparts, 1) * B * S * qkv.size(-1),
                "qkv width mismatch");
    TORCH_CHECK(qkv.is_contiguous(), "qkv must be contiguous");
    TORCH_CHECK(qkv.scalar_type() == (nparts ? at::ScalarType::Float : q_out.scalar_type()),
                "qkv: type");
    const int ht_half = (int)(Hq + 2 * Hkv) * (D / 2);
    dim3 blocks((unsigned)(B * S), (unsigned)((ht_half + 255) / 256));
    auto stream = at::hip::getCurrentHIPStream();
    const bool fp8 = k_cache.scalar_type() == at::ScalarType::Float8_e4m3fn;
    const size_t bits = (size_t)qkv.data_ptr() | (size_t)q_out.data_ptr() |
                        (size_t)k_cache.data_ptr() | (size_t)v_cache.data_ptr() |
                        (size_t)cosb.data_ptr() | (size_t)sinb.data_ptr() |
                        (q_norm ? (size_t)q_norm->data_ptr() : 0) |
                        (k_norm ? (size_t)k_norm->data_ptr() : 0);
    const bool vec = (D == 32 || D == 64 || D == 128 || D == 256) && bits % 16 == 0 && D <= cosb.size(-1);
    TORCH_CHECK(vec || (!q_norm && !k_norm && !slots && !nparts),
                "qkv_rope_update: norms, pages and parts need head sizes 32, 64, 128 or 256");
    TORCH_CHECK(fp8 || k_cache.scalar_type() == q_out.scalar_type(), "cache/new dtype mismatch");
    if (vec) {
        for (const auto* w : {&q_norm, &k_norm})
            if (w->has_value())
                TORCH_CHECK((*w)->numel() == D && (*w)->is_contiguous() &&
                            (*w)->scalar_type() == q_out.scalar_type(), "qkv_rope_update: norm");
        if (slots)
            TORCH_CHECK(slots->scalar_type() == at::ScalarType::Int && slots->is_contiguous() &&
                        slots->numel() == (long)B * S && k_cache.size(2) == Hkv, "slots");
        const long items = (long)B * S * (Hq + 2 * Hkv) * (D / 16), nb = (items + 255) / 256;
        TORCH_CHECK(nb < (1L << 31), "qkv_rope_update: too many tokens");
        if (nb == 0) return;
        const long smax = slots ? k_cache.size(0) * k_cache.size(1) : Smax;
#define QKV_VEC(CT, LL)                                                                            \
    hipLaunchKernelGGL((qkv_rope_vec_kernel<scalar_t, CT, LL>), dim3((unsigned)nb), dim3(256), 0,  \
        stream, (scalar_t*)q_out.data_ptr(), (const scalar_t*)(nparts ? nullptr : qkv.data_ptr()), \
        nparts ? qkv.data_ptr<float>() : nullptr, nparts,                                          \
        cosb.data_ptr<float>(), sinb.data_ptr<float>(), (CT*)k_cache.data_ptr(),                   \
        (CT*)v_cache.data_ptr(), slots ? nullptr : positions.data_ptr<int>(),                      \
        slots ? nullptr : seq_ids.data_ptr<int>(), slots ? slots->data_ptr<int>() : nullptr,       \
        q_norm ? (const scalar_t*)q_norm->data_ptr() : nullptr,                                    \
        k_norm ? (const scalar_t*)k_norm->data_ptr() : nullptr, (float)eps, B * S, S, (int)Hq,     \
        (int)Hkv, Bc, smax)
#define QKV_VEC_D(CT)                                                                              \
    do {                                                                                           \
        if (D == 32) { QKV_VEC(CT, 2); } else if (D == 64) { QKV_VEC(CT, 4); }                     \
        else if (D == 128) { QKV_VEC(CT, 8); } else { QKV_VEC(CT, 16); }                           \
    } while (0)
        DISPATCH_FT(q_out.scalar_type(), "qkv_rope_update", [&] {
            if (fp8) {
                QKV_VEC_D(__hip_fp8_e4m3);
            } else {
                QKV_VEC_D(scalar_t);
            }
        });
#undef QKV_VEC_D
#undef QKV_VEC
        HIP_CHECK_KERNEL();
        return;
    }
    DISPATCH_FT(qkv.scalar_type(), "qkv_rope_update", [&] {
        if (fp8) {
            hipLaunchKernelGGL((qkv_rope_update_kernel<scalar_t, __hip_fp8_e4m3>),
                               blocks, dim3(256), 0, stream,
                               (scalar_t*)q_out.data_ptr(), (const scalar_t*)qkv.data_ptr(),
                               cosb.data_ptr<float>(), sinb.data_ptr<float>(),
                               (__hip_fp8_e4m3*)k_cache.data_ptr(),
                               (__hip_fp8_e4m3*)v_cache.data_ptr(),
                               positions.data_ptr<int>(), seq_ids.data_ptr<int>(),
                               B, S, (int)Hq, (int)Hkv, D, Bc, Smax);
        } else {
            hipLaunchKernelGGL((qkv_rope_update_kernel<scalar_t, scalar_t>),
                               blocks, dim3(256), 0, stream,
                               (scalar_t*)q_out.data_ptr(), (const scalar_t*)qkv.data_ptr(),
                               cosb.data_ptr<float>(), sinb.data_ptr<float>(),
                               (scalar_t*)k_cache.data_ptr(), (scalar_t*)v_cache.data_ptr(),
                               positions.data_ptr<int>(), seq_ids.data_ptr<int>(),
                               B, S, (int)Hq, (int)Hkv, D, Bc, Smax);
        }
    });
    HIP_CHECK_KERNEL();
}

void silu_mul_fused(torch::Tensor out, torch::Tensor gate_up) {
    const int I2 = gate_up.size(-1);
    const long rows = gate_up.numel() / I2;
    const int I = I2 / 2;
    TORCH_CHECK(I % 8 == 0, "intermediate size must be a multiple of 8");
    dim3 blocks((unsigned)rows, (unsigned)((I / 8 + 255) / 256));
    auto stream = at::hip::getCurrentHIPStream();
    DISPATCH_FT(gate_up.scalar_type(), "silu_mul_fused", [&] {
        hipLaunchKernelGGL((act_mul_fused_kernel<scalar_t, false>), blocks,
                           dim3(256), 0, stream,
                           (scalar_t*)out.data_ptr(), (const scalar_t*)gate_up.data_ptr(),
                           rows, I);
    });
    HIP_CHECK_KERNEL();
}

void gelu_tanh_mul_fused(torch::Tensor out, torch::Tensor gate_up) {
    const int I2 = gate_up.size(-1);
    const long rows = gate_up.numel() / I2;
    const int I = I2 / 2;
    TORCH_CHECK(I % 8 == 0, "intermediate size must be a multiple of 8");
    dim3 blocks((unsigned)rows, (unsigned)((I / 8 + 255) / 256));
    auto stream = at::hip::getCurrentHIPStream();
    DISPATCH_FT(gate_up.scalar_type(), "gelu_tanh_mul_fused", [&] {
        hipLaunchKernelGGL((act_mul_fused_kernel<scalar_t, true>), blocks,
                           dim3(256), 0, stream,
                           (scalar_t*)out.data_ptr(), (const scalar_t*)gate_up.data_ptr(),
                           rows, I);
    });
    HIP_CHECK_KERNEL();
}
