// Memory-bound elementwise/normalization kernels for gfx950.
//
// RMSNorm (K7-analog), fused residual-add RMSNorm, SiLU*up / GELU*up
// (the K5 MLP activation seam) and RoPE apply (rotate-half convention).
// All bf16/f16 paths use 16-byte vectorized loads (guide G13: scalar bf16
// loads cost ~2x); RMSNorm is two-pass with the second pass served from L1/L2.

#include "common.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

// ---------------------------------------------------------------------------
// RMSNorm: one 256-thread workgroup per row, grid-stride over rows.
// ---------------------------------------------------------------------------
template <typename T, bool FUSED_ADD>
__global__ void rmsnorm_kernel(
    T* __restrict__ out, const T* __restrict__ x, T* __restrict__ residual,
    const T* __restrict__ weight, const float eps, const int rows, const int H) {
    __shared__ float red[16];
    using VT = VecTraits<T>;
    for (int row = blockIdx.x; row < rows; row += gridDim.x) {
        const T* xr = x + (long)row * H;
        T* rr = FUSED_ADD ? residual + (long)row * H : nullptr;
        float ssq = 0.f;
        for (int i = threadIdx.x * 8; i < H; i += blockDim.x * 8) {
            Vec8<T> v = load_vec8(xr + i);
            if constexpr (FUSED_ADD) {
                Vec8<T> r = load_vec8(rr + i);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    float f = VT::to_float(v.v[j]) + VT::to_float(r.v[j]);
                    v.v[j] = VT::from_float(f);
                    ssq += f * f;
                }
                store_vec8(rr + i, v);  // residual stream updated in place
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    float f = VT::to_float(v.v[j]);
                    ssq += f * f;
                }
            }
        }
        ssq = block_reduce_sum(ssq, red);
        const float inv = rsqrtf(ssq / H + eps);
        const T* src = FUSED_ADD ? rr : xr;
        T* orow = out + (long)row * H;
        for (int i = threadIdx.x * 8; i < H; i += blockDim.x * 8) {
            Vec8<T> v = load_vec8(src + i);
            Vec8<T> w = load_vec8(weight + i);
#pragma unroll
            for (int j = 0; j < 8; ++j)
                v.v[j] = VT::from_float(VT::to_float(v.v[j]) * inv * VT::to_float(w.v[j]));
            store_vec8(orow + i, v);
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// residual += y; out = RMSNorm(residual), with y in 16 bits or as `parts` planes in fp32 (the
// parts of K of a product, tile_gemm.hip), which are added up on the way. A row's values stay in
// registers between the sum and the norm: V times 8 a thread. A decode step waits for it twice a
// layer, so a row of few rows takes as many threads as it has 16-byte pieces and the planes' loads
// go out together.
// ---------------------------------------------------------------------------
template <typename T, bool PARTS, int V>
__global__ __launch_bounds__(1024) void add_norm_kernel(
    T* __restrict__ out, T* __restrict__ residual, const void* __restrict__ y,
    const T* __restrict__ weight, const float eps, const int H, const int parts,
    const long plane) {
    __shared__ float red[16];
    using VT = VecTraits<T>;
    const long row = blockIdx.x;
    float f[V][8];
    float ssq = 0.f;
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const int i = (v * blockDim.x + threadIdx.x) * 8;
        if (i >= H) continue;
        const Vec8<T> r = load_vec8(residual + row * H + i);
        if constexpr (PARTS) {
            const float* p = (const float*)y + row * H + i;
            Vec8<float> a = load_vec8(p);
            int k = 1;
            for (; k + 3 <= parts; k += 3) {
                const Vec8<float> b = load_vec8(p + k * plane), c = load_vec8(p + (k + 1) * plane),
                                  d = load_vec8(p + (k + 2) * plane);
#pragma unroll
                for (int j = 0; j < 8; ++j) a.v[j] += b.v[j] + c.v[j] + d.v[j];
            }
            for (; k < parts; ++k) {
                const Vec8<float> b = load_vec8(p + k * plane);
#pragma unroll
                for (int j = 0; j < 8; ++j) a.v[j] += b.v[j];
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) f[v][j] = a.v[j];
        } else {
            const Vec8<T> a = load_vec8((const T*)y + row * H + i);
#pragma unroll
            for (int j = 0; j < 8; ++j) f[v][j] = VT::to_float(a.v[j]);
        }
        Vec8<T> o;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            f[v][j] += VT::to_float(r.v[j]);
            ssq += f[v][j] * f[v][j];
            o.v[j] = VT::from_float(f[v][j]);
            f[v][j] = VT::to_float(o.v[j]);      // what is normed is the residual as it is kept
        }
        store_vec8(residual + row * H + i, o);
    }
    ssq = block_reduce_sum(ssq, red);
    const float inv = rsqrtf(ssq / H + eps);
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const int i = (v * blockDim.x + threadIdx.x) * 8;
        if (i >= H) continue;
        const Vec8<T> w = load_vec8(weight + i);
        Vec8<T> o;
#pragma unroll
        for (int j = 0; j < 8; ++j) o.v[j] = VT::from_float(f[v][j] * inv * VT::to_float(w.v[j]));
        store_vec8(out + row * H + i, o);
    }
}

// ---------------------------------------------------------------------------
// SiLU(gate) * up and GELU-tanh(gate) * up
// ---------------------------------------------------------------------------
template <typename T, bool GELU>
__global__ void act_mul_kernel(
    T* __restrict__ out, const T* __restrict__ gate, const T* __restrict__ up,
    const long n) {
    using VT = VecTraits<T>;
    const long i0 = ((long)blockIdx.x * blockDim.x + threadIdx.x) * 8;
    const long stride = (long)gridDim.x * blockDim.x * 8;
    for (long i = i0; i < n; i += stride) {
        Vec8<T> g = load_vec8(gate + i);
        Vec8<T> u = load_vec8(up + i);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            float gf = VT::to_float(g.v[j]);
            float uf = VT::to_float(u.v[j]);
            float a;
            if constexpr (GELU) {
                // tanh approximation of GELU
                const float c = 0.7978845608028654f;  // sqrt(2/pi)
                a = 0.5f * gf * (1.f + tanhf(c * (gf + 0.044715f * gf * gf * gf)));
            } else {
                a = gf / (1.f + __expf(-gf));
            }
            g.v[j] = VT::from_float(a * uf);
        }
        store_vec8(out + i, g);
    }
}

// ---------------------------------------------------------------------------
// RoPE apply (rotate-half): q (B,Hq,S,D), k (B,Hkv,S,D) in place.
// cos/sin: (B,S,D) fp32. Each thread handles the pair (i, i+D/2), i < D/2;
// lanes cover consecutive i so both halves load coalesced.
// ---------------------------------------------------------------------------
template <typename T>
__global__ void rope_kernel(
    T* __restrict__ q, T* __restrict__ k,
    const float* __restrict__ cosb, const float* __restrict__ sinb,
    const int B, const int Hq, const int Hkv, const int S, const int D) {
    using VT = VecTraits<T>;
    const int half = D / 2;
    const long total = (long)B * (Hq + Hkv) * S * half;
    const long stride = (long)gridDim.x * blockDim.x;
    for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += stride) {
        const int i = idx % half;
        long rest = idx / half;
        const int s = rest % S;
        rest /= S;
        const int h = rest % (Hq + Hkv);
        const int b = rest / (Hq + Hkv);
        T* base = (h < Hq)
            ? q + (((long)b * Hq + h) * S + s) * D
            : k + (((long)b * Hkv + (h - Hq)) * S + s) * D;
        const float c = cosb[((long)b * S + s) * D + i];
        const float sn = sinb[((long)b * S + s) * D + i];
        const float x1 = VT::to_float(base[i]);
        const float x2 = VT::to_float(base[i + half]);
        base[i] = VT::from_float(x1 * c - x2 * sn);
        base[i + half] = VT::from_float(x2 * c + x1 * sn);
    }
}

// ---------------------------------------------------------------------------
// Host wrappers
// ---------------------------------------------------------------------------
#define DISPATCH_FLOAT_TYPES(TYPE, NAME, ...)                                  \
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

static int ew_grid(long work_items, int block) {
    long blocks = (work_items + block - 1) / block;
    if (blocks > 2048) blocks = 2048;  // grid-stride the rest (guide G11)
    if (blocks < 1) blocks = 1;
    return (int)blocks;
}

void rms_norm(torch::Tensor out, torch::Tensor x, torch::Tensor weight, double eps) {
    const int H = x.size(-1);
    const long rows = x.numel() / H;
    TORCH_CHECK(H % 8 == 0, "hidden size must be a multiple of 8");
    auto stream = at::hip::getCurrentHIPStream();
    DISPATCH_FLOAT_TYPES(x.scalar_type(), "rms_norm", [&] {
        hipLaunchKernelGGL(
            (rmsnorm_kernel<scalar_t, false>), dim3(ew_grid(rows, 1)), dim3(256), 0, stream,
            (scalar_t*)out.data_ptr(), (const scalar_t*)x.data_ptr(), nullptr,
            (const scalar_t*)weight.data_ptr(), (float)eps, (int)rows, H);
    });
    HIP_CHECK_KERNEL();
}

void rms_norm_fused_add(torch::Tensor out, torch::Tensor x, torch::Tensor residual,
                        torch::Tensor weight, double eps) {
    const int H = x.size(-1);
    const long rows = x.numel() / H;
    TORCH_CHECK(H % 8 == 0, "hidden size must be a multiple of 8");
    auto stream = at::hip::getCurrentHIPStream();
    DISPATCH_FLOAT_TYPES(x.scalar_type(), "rms_norm_fused_add", [&] {
        hipLaunchKernelGGL(
            (rmsnorm_kernel<scalar_t, true>), dim3(ew_grid(rows, 1)), dim3(256), 0, stream,
            (scalar_t*)out.data_ptr(), (const scalar_t*)x.data_ptr(),
            (scalar_t*)residual.data_ptr(), (const scalar_t*)weight.data_ptr(),
            (float)eps, (int)rows, H);
    });
    HIP_CHECK_KERNEL();
}

// out = RMSNorm(residual += y): y of residual's shape and type, or (parts, rows, H) in fp32
void add_norm(torch::Tensor out, torch::Tensor residual, torch::Tensor y, torch::Tensor weight,
              double eps) {
    const int H = residual.size(-1);
    const long rows = H ? residual.numel() / H : 0;
    const bool planes = y.scalar_type() == at::ScalarType::Float &&
                        residual.scalar_type() != at::ScalarType::Float;
    TORCH_CHECK(H % 8 == 0 && H <= 32768, "add_norm: rows of up to 32768, a multiple of 8");
    TORCH_CHECK(out.is_contiguous() && residual.is_contiguous() && y.is_contiguous() &&
                weight.is_contiguous() && out.numel() == residual.numel() &&
                weight.numel() == H && out.scalar_type() == residual.scalar_type() &&
                weight.scalar_type() == residual.scalar_type(), "add_norm: operands");
    TORCH_CHECK(planes ? y.dim() == 3 && y.numel() == y.size(0) * rows * H && y.size(0) > 0
                       : y.scalar_type() == residual.scalar_type() && y.numel() == rows * H,
                "add_norm: y");
    TORCH_CHECK((((size_t)out.data_ptr() | (size_t)residual.data_ptr() | (size_t)y.data_ptr() |
                  (size_t)weight.data_ptr()) & 15) == 0, "add_norm: alignment");
    if (rows == 0) return;
    const int parts = planes ? (int)y.size(0) : 1;
    // many rows: 256 threads each, several rows a CU; few: one value of 16 bytes a thread
    const int wide = (H / 8 + 63) / 64 * 64;
    int threads = std::min(wide, rows >= 512 && H <= 8192 ? 256 : 1024);
    const int V = (H / 8 + threads - 1) / threads;
    auto stream = at::hip::getCurrentHIPStream();
#define ADD_NORM(P, VV)                                                                          \
    hipLaunchKernelGGL((add_norm_kernel<scalar_t, P, VV>), dim3((unsigned)rows), dim3(threads),  \
                       0, stream, (scalar_t*)out.data_ptr(), (scalar_t*)residual.data_ptr(),     \
                       y.data_ptr(), (const scalar_t*)weight.data_ptr(), (float)eps, H, parts,   \
                       rows * H)
#define ADD_NORM_V(P)                                                                            \
    do {                                                                                         \
        if (V == 1) ADD_NORM(P, 1);                                                              \
        else if (V == 2) ADD_NORM(P, 2);                                                         \
        else ADD_NORM(P, 4);                                                                     \
    } while (0)
    DISPATCH_FLOAT_TYPES(residual.scalar_type(), "add_norm", [&] {
        if (planes) ADD_NORM_V(true);
        else ADD_NORM_V(false);
    });
#undef ADD_NORM_V
#undef ADD_NORM
    HIP_CHECK_KERNEL();
}

void silu_mul(torch::Tensor out, torch::Tensor gate, torch::Tensor up) {
    const long n = gate.numel();
    TORCH_CHECK(n % 8 == 0, "numel must be a multiple of 8");
    auto stream = at::hip::getCurrentHIPStream();
    DISPATCH_FLOAT_TYPES(gate.scalar_type(), "silu_mul", [&] {
        hipLaunchKernelGGL((act_mul_kernel<scalar_t, false>),
                           dim3(ew_grid(n / 8, 256)), dim3(256), 0, stream,
                           (scalar_t*)out.data_ptr(), (const scalar_t*)gate.data_ptr(),
                           (const scalar_t*)up.data_ptr(), n);
    });
    HIP_CHECK_KERNEL();
}

void gelu_tanh_mul(torch::Tensor out, torch::Tensor gate, torch::Tensor up) {
    const long n = gate.numel();
    TORCH_CHECK(n % 8 == 0, "numel must be a multiple of 8");
    auto stream = at::hip::getCurrentHIPStream();
    DISPATCH_FLOAT_TYPES(gate.scalar_type(), "gelu_tanh_mul", [&] {
        hipLaunchKernelGGL((act_mul_kernel<scalar_t, true>),
                           dim3(ew_grid(n / 8, 256)), dim3(256), 0, stream,
                           (scalar_t*)out.data_ptr(), (const scalar_t*)gate.data_ptr(),
                           (const scalar_t*)up.data_ptr(), n);
    });
    HIP_CHECK_KERNEL();
}

void rope_apply(torch::Tensor q, torch::Tensor k, torch::Tensor cosb, torch::Tensor sinb) {
    TORCH_CHECK(q.dim() == 4 && k.dim() == 4, "q/k must be (B,H,S,D)");
    const int B = q.size(0), Hq = q.size(1), S = q.size(2), D = q.size(3);
    const int Hkv = k.size(1);
    TORCH_CHECK(cosb.scalar_type() == at::ScalarType::Float, "cos/sin must be fp32");
    TORCH_CHECK(cosb.dim() == 3 && cosb.size(2) == D, "cos must be (B,S,D)");
    const long total = (long)B * (Hq + Hkv) * S * (D / 2);
    auto stream = at::hip::getCurrentHIPStream();
    DISPATCH_FLOAT_TYPES(q.scalar_type(), "rope_apply", [&] {
        hipLaunchKernelGGL((rope_kernel<scalar_t>),
                           dim3(ew_grid(total, 256)), dim3(256), 0, stream,
                           (scalar_t*)q.data_ptr(), (scalar_t*)k.data_ptr(),
                           cosb.data_ptr<float>(), sinb.data_ptr<float>(),
                           B, Hq, Hkv, S, D);
    });
    HIP_CHECK_KERNEL();
}
