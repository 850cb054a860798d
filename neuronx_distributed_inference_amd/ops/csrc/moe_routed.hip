// Routed experts of a MoE layer, from the router's choice to the layer's output, in four
// launches: a table of row tiles, gate and up projection with the gated activation, down
// projection, weighted sum of each token's experts.
//
// Bounds: with few rows an expert the weight stream (every chosen expert's weights once from
// HBM); with many the matrix cores, and before those the LDS (128 B/clk a CU).
//
//   * Workgroup = 8 waves, MT rows of one expert x 256 columns. K goes in steps of 128 B of a
//     weight row (128 deep with 8-bit weights, and then 64 rows at most) through a ring of three
//     LDS buffers, global_load_lds throughout, one raw barrier a step and a counted vmcnt: two
//     steps are in flight while one is computed.
//   * The row tiles of an expert want the same weights: the list of workgroups (8 row tiles x
//     all column tiles, rows fastest) is cut into 8 contiguous parts, one for each XCD, so that
//     they meet in one L2. The list covers real tiles only; the grid is sized for the worst
//     case and the rest leaves at once.
//   * Gate and up columns of the same number are in the same lane: the activation needs no
//     exchange and the two projections no round trip through memory. A lane holds 4 adjacent
//     columns of a row (weights are the first operand).
//   * The down projection writes 32-bit rows, and a second kernel adds each token's rows in
//     the order of its choice: the same sum in every run. fp32 atomics into the output instead
//     took longer than the product itself (2048 tokens x 8 experts x 2048 columns: 201 of
//     341 us; 284 of 1831 us for 4096 tokens x 2 x 4096).
//
// The three products of a layer in us, before = moe_grouped_kernel (64 rows x 256 columns, a
// launch each for gate, up and activation, atomics):
//   128 experts of 2048 x 768, 8 a token:  2048 tokens 776 -> 364 (weights at the 4.9 TB/s of
//     a large copy: 247);
//     512 tokens 379 -> 266;  8 experts of 4096 x 14336, 2 a token: 4096 tokens 6379 -> 3290
//     (bf16 products alone 1850), 256 tokens 688 -> 604 (577 at that rate), 128 tokens in 8 bits
//     376 -> 309 (288).
// Row tiles (32, 64, 128), gate + up and down with its sum: 32 rows an expert 164+102, 144+92,
// 144+100 (64 rows 224+138, 172+118, 150+118); 128 rows 358+234, 237+185, 202+164;
// 8 experts in 8 bits, 32 rows: 198+117, 185+143 (32 fills more of the chip); 128 rows 474+280,
//   380+267 (128 rows x 128 columns: 440+258).

#include "common.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

namespace {

typedef __bf16 mr_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 mr_f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 mr_bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 mr_f16x2 __attribute__((ext_vector_type(2)));
typedef float mr_f32x4 __attribute__((ext_vector_type(4)));

template <typename T> struct MrMfma;
template <> struct MrMfma<__hip_bfloat16> {
    using vec8 = mr_bf16x8;
    using vec2 = mr_bf16x2;
    static DEV_INLINE mr_f32x4 mfma(vec8 a, vec8 b, mr_f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
    template <bool HI> static DEV_INLINE vec2 from_fp8(unsigned p) {
        return __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(p, 1.f, HI);
    }
};
template <> struct MrMfma<__half> {
    using vec8 = mr_f16x8;
    using vec2 = mr_f16x2;
    static DEV_INLINE mr_f32x4 mfma(vec8 a, vec8 b, mr_f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
    template <bool HI> static DEV_INLINE vec2 from_fp8(unsigned p) {
        return __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(p, 1.f, HI);
    }
};

// 16 bytes a lane to the 1 KB of LDS at the wave-uniform `dst`. Written out: the compiler would
// wait for every such load in flight before each LDS read. No register result; the kernel
// waits (vmcnt) before the barrier that hands the buffer over.
DEV_INLINE void mr_load_lds(const char* src, unsigned dst) {
    const unsigned at = __builtin_amdgcn_readfirstlane(dst);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                 :: "s"(at), "v"(src) : "memory", "m0");
}

template <int N>
DEV_INLINE void mr_vm_wait() {
    asm volatile("s_waitcnt vmcnt(%c0)" ::"i"(N) : "memory");
}

DEV_INLINE float mr_act(float g, int gelu) {
    if (gelu) {
        const float u = 0.7978845608028654f * (g + 0.044715f * g * g * g);
        return 0.5f * g * (1.f + tanhf(u));
    }
    return g / (1.f + __expf(-g));
}

template <bool F8, int MT>
struct MrTile {
    static_assert(!F8 || MT < 128, "the ring would not fit");
    static constexpr int BN = 256;
    static constexpr int BK = F8 ? 128 : 64;          // 128 B of a weight row
    static constexpr int XH = BK / 64;                // 128 B images of x a step
    static constexpr int WM = MT == 128 ? 2 : 1;      // waves along the rows
    static constexpr int WN = 8 / WM;
    static constexpr int MI = MT / WM / 16;
    static constexpr int NI = BN / WN / 16;
    static constexpr int XB = XH * MT * 128;
    static constexpr int STEP = XB + BN * 128;        // bytes of a ring buffer
};

template <typename T, bool F8, bool GLU, int MT>
__global__ void __launch_bounds__(512, 2)
moe_routed_kernel(void* __restrict__ y, const T* __restrict__ x, const char* __restrict__ w0,
                  const char* __restrict__ w1, const float* __restrict__ s0,
                  const float* __restrict__ s1, const int* __restrict__ tiles,
                  const int* __restrict__ gather, const int N, const int K, const int col0,
                  const int ncols, const int ntn, const int gelu) {
    using MF = MrMfma<T>;
    using vec8 = typename MF::vec8;
    using C = MrTile<F8, MT>;
    constexpr int MI = C::MI, NI = C::NI, XH = C::XH;
    constexpr int BNO = GLU ? C::BN / 2 : C::BN;      // output columns of a workgroup
    constexpr int WP = C::BN / 64;                    // 1 KB pieces of W a wave stages
    constexpr int XP = XH * MT / 8;                   // pieces of x in all
    constexpr int XW = (XP + 7) / 8;                  // and of a wave that has any
    constexpr int ES = F8 ? 1 : 2;
    constexpr int GRP = 8;                            // row tiles of a group
    extern __shared__ __attribute__((aligned(16))) char smem[];

    // workgroup -> tile of the list, contiguous parts for the XCDs
    const int nreal = tiles[0], total = nreal * ntn, per = (total + 7) >> 3;
    const int slot_wg = blockIdx.x >> 3, li = (blockIdx.x & 7) * per + slot_wg;
    if (slot_wg >= per || li >= total) return;        // uniform over the workgroup
    const int grp = li / (GRP * ntn), rows_grp = min(GRP, nreal - grp * GRP);
    const int in = li - grp * GRP * ntn, rt = grp * GRP + in % rows_grp;
    const int n0 = (in / rows_grp) * BNO;             // first column, of the slab
    const int e = tiles[1 + 2 * rt], rows = tiles[2 + 2 * rt];
    const long m0 = (long)rt * MT;

    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm0 = (wid / C::WN) * (MI * 16), wn = wid % C::WN;
    const int lrow = lane & 15, ls = lane >> 4, prow = lane >> 3;
    const int pslot = (lane & 7) ^ prow;              // source side of the XOR swizzle
    const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) char*)smem;

    const bool x_wave = XP >= 8 || wid < XP;
    const char* xsrc[XW];
    unsigned xdst[XW];
#pragma unroll
    for (int i = 0; i < XW; ++i) {
        const int piece = (x_wave ? wid * XW : 0) + i, img = piece / (MT / 8);
        const int r = (piece % (MT / 8)) * 8 + prow;
        const long src = gather ? (r < rows ? gather[m0 + r] : 0) : m0 + r;
        xsrc[i] = reinterpret_cast<const char*>(x + src * K) + img * 128 + pslot * 16;
        xdst[i] = lds0 + piece * 1024;
    }
    const char* wsrc[WP];
    unsigned wdst[WP];
#pragma unroll
    for (int i = 0; i < WP; ++i) {
        const int piece = wid * WP + i, r = piece * 8 + prow;
        const bool up = GLU && r >= C::BN / 2;
        const int n = min(col0 + n0 + (up ? r - C::BN / 2 : r), N - 1);
        wsrc[i] = (up ? w1 : w0) + ((long)e * N + n) * K * ES + pslot * 16;
        wdst[i] = lds0 + C::XB + piece * 1024;
    }
    auto stage = [&](int t, unsigned buf) {
        if (x_wave) {
#pragma unroll
            for (int i = 0; i < XW; ++i) mr_load_lds(xsrc[i] + t * (C::BK * 2), xdst[i] + buf);
        }
#pragma unroll
        for (int i = 0; i < WP; ++i) mr_load_lds(wsrc[i] + t * 128, wdst[i] + buf);
    };

    mr_f32x4 acc[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = {0.f, 0.f, 0.f, 0.f};
    // row of W's image that fragment j of this wave starts at: with GLU the first half of the
    // fragments are gate columns, the second the same up columns
    auto wrow = [&](int j) {
        constexpr int NH = NI / 2;
        return GLU ? (j / NH) * (C::BN / 2) + (wn * NH + j % NH) * 16 : (wn * NI + j) * 16;
    };
    auto compute = [&](unsigned buf) {
        const char* xb = smem + buf + (wm0 + lrow) * 128;
        const char* wb = smem + buf + C::XB + lrow * 128;
#pragma unroll
        for (int kq = 0; kq < C::BK / 32; ++kq) {
            vec8 a[MI], b[NI];
            const int sx = ((kq & 1) * 4 + ls) ^ (lrow & 7);
#pragma unroll
            for (int i = 0; i < MI; ++i)
                a[i] = *reinterpret_cast<const vec8*>(xb + (kq >> 1) * (MT * 128) + i * 2048 +
                                                      sx * 16);
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                if constexpr (F8) {
                    const int sw = (kq * 2 + (ls >> 1)) ^ (lrow & 7);
                    const uint2 p = *reinterpret_cast<const uint2*>(
                        wb + wrow(j) * 128 + sw * 16 + (ls & 1) * 8);
                    typename MF::vec2 q[4] = {
                        MF::template from_fp8<false>(p.x), MF::template from_fp8<true>(p.x),
                        MF::template from_fp8<false>(p.y), MF::template from_fp8<true>(p.y)};
                    b[j] = *reinterpret_cast<const vec8*>(q);
                } else {
                    b[j] = *reinterpret_cast<const vec8*>(wb + wrow(j) * 128 + sx * 16);
                }
            }
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NI; ++j) acc[i][j] = MF::mfma(b[j], a[i], acc[i][j]);
        }
    };

    const int nk = K / C::BK;
    const bool active = wm0 < rows;                   // a wave without rows only stages
    stage(0, 0);
    if (nk > 1) stage(1, C::STEP);
    unsigned cur = 0, nxt = 2 * C::STEP;
    for (int t = 0; t < nk; ++t) {
        if (t + 1 < nk) {
            if (XP >= 8 || !x_wave) mr_vm_wait<WP + (XP >= 8 ? XW : 0)>();
            else mr_vm_wait<WP + XW>();
        } else {
            mr_vm_wait<0>();
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        // the buffer computed in the turn before is free
        if (t + 2 < nk) stage(t + 2, nxt);
        if (active) compute(cur);
        cur = cur == 2 * C::STEP ? 0 : cur + C::STEP;
        nxt = nxt == 2 * C::STEP ? 0 : nxt + C::STEP;
    }
    if (!active) return;

    constexpr int NO = GLU ? NI / 2 : NI;
#pragma unroll
    for (int j = 0; j < NO; ++j) {
        const int c = n0 + (wn * NO + j) * 16 + ls * 4;      // column of the slab
        if (c >= ncols) continue;
        mr_f32x4 sg = {1.f, 1.f, 1.f, 1.f}, su = sg;
        if constexpr (F8) {
            sg = *reinterpret_cast<const mr_f32x4*>(s0 + (long)e * N + col0 + c);
            if (GLU) su = *reinterpret_cast<const mr_f32x4*>(s1 + (long)e * N + col0 + c);
        }
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const int m = wm0 + i * 16 + lrow;
            if (m >= rows) continue;
            mr_f32x4 v = acc[i][j] * sg;
            if constexpr (GLU) {
                const mr_f32x4 u = acc[i][j + NO] * su;
                T o[4];
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    o[r] = VecTraits<T>::from_float(mr_act(v[r], gelu) * u[r]);
                *reinterpret_cast<uint2*>(reinterpret_cast<T*>(y) + (m0 + m) * ncols + c) =
                    *reinterpret_cast<const uint2*>(o);
            } else {
                *reinterpret_cast<mr_f32x4*>(reinterpret_cast<float*>(y) + (m0 + m) * ncols + c) = v;
            }
        }
    }
}

// out[t, col0 + c] = sum over the token's choices of weight * y[row of the choice, c]
template <typename T, int TOPK>
__global__ void __launch_bounds__(256)
moe_routed_sum_kernel(T* __restrict__ out, const float* __restrict__ y,
                      const int* __restrict__ inv, const float* __restrict__ weights,
                      const int ntok, const int topk, const int N, const int col0,
                      const int ncols) {
    const int per = ncols / 8;
    const long id = (long)blockIdx.x * 256 + threadIdx.x;
    if (id >= (long)ntok * per) return;
    const int t = (int)(id / per), c = (int)(id % per) * 8;
    const int k = TOPK ? TOPK : topk;
    float v[8] = {};
#pragma unroll
    for (int j = 0; j < k; ++j) {
        const int row = inv[(long)t * k + j];
        const float wt = weights ? weights[(long)t * k + j] : 1.f;
        const float* p = y + (long)max(row, 0) * ncols + c;
        float4 a = *reinterpret_cast<const float4*>(p);
        float4 b = *reinterpret_cast<const float4*>(p + 4);
        if (row < 0) a = b = float4{0.f, 0.f, 0.f, 0.f};     // another rank's expert
        v[0] += a.x * wt; v[1] += a.y * wt; v[2] += a.z * wt; v[3] += a.w * wt;
        v[4] += b.x * wt; v[5] += b.y * wt; v[6] += b.z * wt; v[7] += b.w * wt;
    }
    Vec8<T> o;
#pragma unroll
    for (int i = 0; i < 8; ++i) o.v[i] = VecTraits<T>::from_float(v[i]);
    store_vec8(out + (long)t * N + col0 + c, o);
}

// The table: tiles[0] = number of row tiles, then (expert, rows) of each; gather = token of a
// tile row (padding rows stay unwritten: readers go by `rows`); inv = tile row of a choice, or
// -1 where the expert is not one of the El from `first`. One workgroup: counts and ranks by LDS
// atomics, the scan over experts a wave's. (Rows within an expert may come in any order: each
// is multiplied by itself, and the sum goes by `inv`.) 16384 choices of 128 experts: 63 us with
// a scan by one thread and a search per tile, before the 10 launches it also replaces.
template <typename I>
__global__ void __launch_bounds__(1024)
moe_route_kernel(int* __restrict__ tiles, int* __restrict__ gather, int* __restrict__ inv,
                 const I* __restrict__ idx, const int n, const int El, const long first,
                 const int topk, const int mt) {
    extern __shared__ int rsm[];
    int *count = rsm, *next = rsm + El;
    for (int e = threadIdx.x; e < El; e += 1024) count[e] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += 1024) {
        const long e = (long)idx[i] - first;
        if (e >= 0 && e < El) atomicAdd(&count[e], 1);
    }
    __syncthreads();
    if (threadIdx.x < 64) {
        const int lane = threadIdx.x;
        int carry = 0;
        for (int base = 0; base < El; base += 64) {
            const int e = base + lane, c = e < El ? count[e] : 0, nt = (c + mt - 1) / mt;
            int s = nt;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const int up = __shfl_up(s, off, 64);
                if (lane >= off) s += up;
            }
            const int start = carry + s - nt;
            if (e < El) next[e] = start * mt;
            for (int j = 0; j < nt; ++j) {
                tiles[1 + 2 * (start + j)] = e;
                tiles[2 + 2 * (start + j)] = min(mt, c - j * mt);
            }
            carry += __shfl(s, 63, 64);
        }
        if (lane == 0) tiles[0] = carry;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += 1024) {
        const long e = (long)idx[i] - first;
        int row = -1;
        if (e >= 0 && e < El) {
            row = atomicAdd(&next[e], 1);
            gather[row] = i / topk;
        }
        inv[i] = row;
    }
}

template <typename T, bool F8, bool GLU, int MT>
void mr_launch(void* y, const torch::Tensor& x, const torch::Tensor& w0, const torch::Tensor& w1,
               const float* s0, const float* s1, const torch::Tensor& tiles, const int* gather,
               int max_tiles, int col0, int ncols, int gelu, hipStream_t st) {
    using C = MrTile<F8, MT>;
    constexpr int LDS = 3 * C::STEP, BNO = GLU ? C::BN / 2 : C::BN;
    // a limit of the function, the same in every call
    (void)hipFuncSetAttribute((const void*)moe_routed_kernel<T, F8, GLU, MT>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    const int ntn = (ncols + BNO - 1) / BNO;
    const long grid = ((long)max_tiles * ntn + 7) / 8 * 8;
    TORCH_CHECK(grid < (1L << 31), "moe_routed: too many tiles");
    hipLaunchKernelGGL((moe_routed_kernel<T, F8, GLU, MT>), dim3((unsigned)grid), dim3(512), LDS, st, y,
                       (const T*)x.data_ptr(), (const char*)w0.data_ptr(),
                       (const char*)w1.data_ptr(), s0, s1, tiles.data_ptr<int>(), gather,
                       (int)w0.size(1), (int)w0.size(2), col0, ncols, ntn, gelu);
    HIP_CHECK_KERNEL();
}

template <bool GLU>
void mr_dispatch(void* y, const torch::Tensor& x, const torch::Tensor& w0,
                 const torch::Tensor& w1, const float* s0, const float* s1,
                 const torch::Tensor& tiles, const int* gather, int mt, int col0, int ncols,
                 int gelu) {
    const int max_tiles = (int)((tiles.numel() - 1) / 2);
    auto st = at::hip::getCurrentHIPStream();
    const bool f8 = s0 != nullptr, bf = x.scalar_type() == at::ScalarType::BFloat16;
#define MR(TT, FF, MM) mr_launch<TT, FF, GLU, MM>(y, x, w0, w1, s0, s1, tiles, gather, max_tiles, \
                                                  col0, ncols, gelu, st)
#define MR_M(TT)                                                                                  \
    do {                                                                                          \
        if (f8 && mt == 64) MR(TT, true, 64);                                                     \
        else if (f8) MR(TT, true, 32);                                                            \
        else if (mt == 128) MR(TT, false, 128);                                                   \
        else if (mt == 64) MR(TT, false, 64);                                                     \
        else MR(TT, false, 32);                                                                   \
    } while (0)
    if (bf) MR_M(__hip_bfloat16);
    else MR_M(__half);
#undef MR_M
#undef MR
}

void mr_check(const torch::Tensor& x, const torch::Tensor& w, const c10::optional<torch::Tensor>& s,
              const torch::Tensor& tiles, long mt) {
    TORCH_CHECK(mt == 32 || mt == 64 || (mt == 128 && !s.has_value()),
                "moe_routed: mt must be 32, 64 or, with 16-bit weights, 128");
    TORCH_CHECK(x.dim() == 2 && w.dim() == 3 && x.size(1) == w.size(2), "moe_routed: shapes");
    TORCH_CHECK(x.is_contiguous() && w.is_contiguous() && tiles.is_contiguous(),
                "moe_routed: contiguous tensors required");
    TORCH_CHECK(x.scalar_type() == at::ScalarType::BFloat16 ||
                x.scalar_type() == at::ScalarType::Half, "moe_routed: bf16/f16 only");
    TORCH_CHECK((size_t)x.data_ptr() % 16 == 0 && (size_t)w.data_ptr() % 16 == 0,
                "moe_routed: 16-byte alignment");
    TORCH_CHECK(tiles.scalar_type() == at::ScalarType::Int && tiles.numel() % 2 == 1, "tiles");
    TORCH_CHECK(w.size(2) % (s.has_value() ? 128 : 64) == 0 && w.size(1) % 16 == 0,
                "moe_routed: K must be a multiple of 64 (8-bit weights: 128), N of 16");
    if (s.has_value()) {
        TORCH_CHECK(w.scalar_type() == at::ScalarType::Byte &&
                    s->scalar_type() == at::ScalarType::Float && s->is_contiguous() &&
                    s->numel() == w.size(0) * w.size(1), "moe_routed: 8-bit weights and scales");
    } else {
        TORCH_CHECK(w.scalar_type() == x.scalar_type(), "moe_routed: weight type");
    }
}

}  // namespace

void moe_route(torch::Tensor tiles, torch::Tensor gather, torch::Tensor inv, torch::Tensor idx,
               long num_local, long first, long mt) {
    TORCH_CHECK(idx.dim() == 2 && idx.is_contiguous(), "moe_route: idx (T, k) contiguous");
    TORCH_CHECK(num_local >= 1 && num_local <= 8192, "moe_route: experts");
    const long n = idx.numel();
    TORCH_CHECK(n < (1L << 30) && inv.numel() == n, "moe_route: sizes");
    const long most = (n + std::min(n, num_local) * (mt - 1)) / mt;    // tiles at worst
    TORCH_CHECK(tiles.numel() >= 1 + 2 * most && gather.numel() >= most * mt, "moe_route: tables");
    TORCH_CHECK(tiles.scalar_type() == at::ScalarType::Int &&
                gather.scalar_type() == at::ScalarType::Int &&
                inv.scalar_type() == at::ScalarType::Int, "moe_route: int32 tables");
    auto st = at::hip::getCurrentHIPStream();
    const int lds = 2 * (int)num_local * 4;
#define MR_ROUTE(I) hipLaunchKernelGGL(moe_route_kernel<I>, dim3(1), dim3(1024), lds, st,         \
        tiles.data_ptr<int>(), gather.data_ptr<int>(), inv.data_ptr<int>(), idx.data_ptr<I>(),    \
        (int)n, (int)num_local, first, (int)idx.size(1), (int)mt)
    TORCH_CHECK(idx.scalar_type() == at::ScalarType::Long ||
                idx.scalar_type() == at::ScalarType::Int, "moe_route: idx int32 or int64");
    if (idx.scalar_type() == at::ScalarType::Long) {
        MR_ROUTE(long);
    } else {
        MR_ROUTE(int);
    }
#undef MR_ROUTE
    HIP_CHECK_KERNEL();
}

void moe_routed_glu(torch::Tensor h, torch::Tensor x, torch::Tensor w_gate, torch::Tensor w_up,
                    c10::optional<torch::Tensor> s_gate, c10::optional<torch::Tensor> s_up,
                    torch::Tensor tiles, c10::optional<torch::Tensor> gather, long mt, long gelu) {
    mr_check(x, w_gate, s_gate, tiles, mt);
    mr_check(x, w_up, s_up, tiles, mt);
    const long rows = (tiles.numel() - 1) / 2 * mt;
    TORCH_CHECK(w_gate.sizes() == w_up.sizes() && s_gate.has_value() == s_up.has_value(),
                "moe_routed_glu: gate and up");
    TORCH_CHECK(h.dim() == 2 && h.is_contiguous() && h.scalar_type() == x.scalar_type() &&
                h.size(0) >= rows && h.size(1) == w_gate.size(1), "moe_routed_glu: h");
    TORCH_CHECK(gather.has_value() ? gather->scalar_type() == at::ScalarType::Int &&
                                         gather->numel() >= rows
                                   : x.size(0) >= rows, "moe_routed_glu: rows");
    mr_dispatch<true>(h.data_ptr(), x, w_gate, w_up, s_gate ? s_gate->data_ptr<float>() : nullptr,
                      s_up ? s_up->data_ptr<float>() : nullptr, tiles,
                      gather ? gather->data_ptr<int>() : nullptr, (int)mt, 0,
                      (int)w_gate.size(1), (int)gelu);
}

// `ws` holds the products of as many columns at a time as it has room for
void moe_routed_down(torch::Tensor out, torch::Tensor ws, torch::Tensor h, torch::Tensor w_down,
                     c10::optional<torch::Tensor> s_down, torch::Tensor tiles, torch::Tensor inv,
                     c10::optional<torch::Tensor> weights, long mt) {
    mr_check(h, w_down, s_down, tiles, mt);
    const long rows = (tiles.numel() - 1) / 2 * mt, N = w_down.size(1), T = out.size(0);
    TORCH_CHECK(h.size(0) >= rows && out.dim() == 2 && out.is_contiguous() && out.size(1) == N &&
                out.scalar_type() == h.scalar_type(), "moe_routed_down: shapes");
    TORCH_CHECK(T > 0 && inv.numel() % T == 0 && inv.scalar_type() == at::ScalarType::Int &&
                inv.is_contiguous(), "moe_routed_down: inv");
    if (weights.has_value())
        TORCH_CHECK(weights->scalar_type() == at::ScalarType::Float &&
                    weights->numel() == inv.numel() && weights->is_contiguous(),
                    "moe_routed_down: weights");
    const long room = ws.numel() / rows / 256 * 256;
    TORCH_CHECK(ws.scalar_type() == at::ScalarType::Float && ws.is_contiguous() &&
                (room > 0 || ws.numel() >= rows * N), "moe_routed_down: workspace");
    const long slab = ws.numel() >= rows * N ? N : room;
    const int topk = (int)(inv.numel() / T);
    auto st = at::hip::getCurrentHIPStream();
    for (long c = 0; c < N; c += slab) {
        const int nc = (int)std::min(slab, N - c);
        mr_dispatch<false>(ws.data_ptr(), h, w_down, w_down,
                           s_down ? s_down->data_ptr<float>() : nullptr, nullptr, tiles, nullptr,
                           (int)mt, (int)c, nc, 0);
        const long blocks = (T * (nc / 8) + 255) / 256;
#define MR_SUM(TT, KK) hipLaunchKernelGGL((moe_routed_sum_kernel<TT, KK>), dim3((unsigned)blocks),  \
        dim3(256), 0, st, (TT*)out.data_ptr(), ws.data_ptr<float>(), inv.data_ptr<int>(),          \
        weights ? weights->data_ptr<float>() : nullptr, (int)T, topk, (int)N, (int)c, nc)
#define MR_SUMK(TT)                                                                                \
    do {                                                                                           \
        if (topk == 8) {                                                                           \
            MR_SUM(TT, 8);                                                                         \
        } else if (topk == 2) {                                                                    \
            MR_SUM(TT, 2);                                                                         \
        } else {                                                                                   \
            MR_SUM(TT, 0);                                                                         \
        }                                                                                          \
    } while (0)
        if (h.scalar_type() == at::ScalarType::BFloat16) {
            MR_SUMK(__hip_bfloat16);
        } else {
            MR_SUMK(__half);
        }
#undef MR_SUMK
#undef MR_SUM
        HIP_CHECK_KERNEL();
    }
}
