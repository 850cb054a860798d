// Token-generation (decode) attention for gfx950 — the K2-analog
// (ref attention_block_tkg, modules/attention/attention_base.py:1186-1381).
//
// Memory-bound split-KV design. 16-bit models with head sizes 64 and 128 take the matrix-core
// kernel further down; fp32 and the other head sizes take this one:
//  * pass 1: grid (nsplit, Hkv*Sq, B), 256-thread workgroups (4 waves).
//    Lane groups of D/8 lanes stream K/V rows with 16-B loads (8 bf16 per
//    lane = one ds-free register path; guide G13). Each group computes the
//    q.k dots for all GQ query heads of its KV head at once, so the KV
//    bytes are read ONCE per (b, hkv) regardless of GQA ratio, online
//    softmax in registers, cross-group combine via __shfl_xor butterflies,
//    cross-wave combine via LDS, per-split partials (m, l, o) to workspace.
//  * pass 2: combines the nsplit partials per (b, hq, sq) row.
//
// The split over the sequence gives the chip >> 256 workgroups at decode
// batch sizes (256 CUs in 8 XCDs need large grids) and is the same
// structure flash-decoding (seq-sharded KV, ref C5) extends across GPUs.

#include "common.h"
#include "attention_row.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

constexpr float M_INIT = -1e30f;

// PAGED=false: linear cache (Bc, Hkv, Smax, D), row l at seq row seq_ids[b].
// PAGED=true: paged cache (num_blocks, block_size, Hkv, D) walked through
// block_table (B, max_blocks); Smax is the per-sequence capacity
// max_blocks*block_size.
// CT = cache storage type (T itself, or fp8-e4m3 when the KV cache is
// quantized; the k-scale is folded into the softmax scale by the host and
// the v-scale applied in pass 2).
// 2-way packed dot (v_dot2): halves the QK VALU work and the q-register
// footprint.
typedef __bf16 dot2_bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 dot2_f16x2 __attribute__((ext_vector_type(2)));
template <typename T> struct Dot2 {
    static constexpr bool ok = false;
    using v2 = float;
    static __device__ __forceinline__ float dot(v2, v2, float c) { return c; }
    static __device__ __forceinline__ v2 pack(float, float) { return 0.f; }
};
template <> struct Dot2<__hip_bfloat16> {
    static constexpr bool ok = true;
    using v2 = dot2_bf16x2;
    static __device__ __forceinline__ float dot(v2 a, v2 b, float c) {
        return __builtin_amdgcn_fdot2_f32_bf16(a, b, c, false);
    }
    static __device__ __forceinline__ v2 pack(float a, float b) {
        v2 r; r[0] = (__bf16)a; r[1] = (__bf16)b; return r;
    }
};
template <> struct Dot2<__half> {
    static constexpr bool ok = true;
    using v2 = dot2_f16x2;
    static __device__ __forceinline__ float dot(v2 a, v2 b, float c) {
        return __builtin_amdgcn_fdot2(a, b, c, false);
    }
    static __device__ __forceinline__ v2 pack(float a, float b) {
        v2 r; r[0] = (_Float16)a; r[1] = (_Float16)b; return r;
    }
};

template <typename T, typename CT, int D, int GQ, bool PAGED>
__global__ __launch_bounds__(256) void decode_attn_pass1(
    float* __restrict__ o_part,        // (B, Hq, Sq, nsplit, D)
    float* __restrict__ ml_part,       // (B, Hq, Sq, nsplit, 2)
    const T* __restrict__ q,           // (B, Hq, Sq, D) — Hq = Hkv*gq
    const CT* __restrict__ k_cache,    // (Bc, Hkv, Smax, D)
    const CT* __restrict__ v_cache,
    const int* __restrict__ positions, // (B, Sq) per-query absolute position
    const int* __restrict__ seq_ids,   // (B,) (linear) / unused (paged)
    const int* __restrict__ block_table,  // (B, max_blocks) when PAGED
    const float scale, const int window, const int ring,
    const int Hkv, const int Sq, const int gq,
    const int Smax, const int chunk, const int nsplit,
    const int block_size, const int max_blocks) {
    using VT = VecTraits<T>;
    constexpr int GS = D / 8;          // lanes per group
    constexpr int NG = 256 / GS;       // groups per workgroup

    const int split = blockIdx.x;
    const int hkv = blockIdx.y / Sq;
    const int sq = blockIdx.y % Sq;
    const int b = blockIdx.z;
    const int Hq = Hkv * gq;

    const int lane = threadIdx.x & (WAVE_SIZE - 1);
    const int wid = threadIdx.x / WAVE_SIZE;
    const int grp = threadIdx.x / GS;         // 0..NG-1
    const int c = threadIdx.x % GS;           // lane-in-group

    const int row = seq_ids[b];
    // query at absolute position p attends cache rows [0, p]
    const int eff_len = positions[(long)b * Sq + sq] + 1;
    int lo = 0;
    int span_hi = eff_len;
    int pmax = 0;
    if (ring) {
        // RING cache (compact sliding-window layers): slot s holds the
        // newest position == s (mod Smax); all written slots are scanned
        // and masked by true position below. pmax = max over VALID (>=0)
        // positions of the row — ragged chunked-prefill batches carry
        // trailing -1 pads (CPU ref ops/__init__.py uses positions.amax).
        pmax = -1;
        for (int s = 0; s < Sq; ++s)
            pmax = max(pmax, positions[(long)b * Sq + s]);
        span_hi = min(pmax + 1, Smax);
    } else if (window > 0 && eff_len > window) {
        lo = eff_len - window;
    }
    // window < 0: Llama4 CHUNKED attention with chunk size -window — the
    // query attends only rows in its own chunk [(p/C)*C, p]
    else if (window < 0) lo = ((eff_len - 1) / (-window)) * (-window);
    const int split_lo = max(lo, split * chunk);
    const int split_hi = min(span_hi, (split + 1) * chunk);

    // ---- q into registers, pre-scaled ----
    constexpr bool PK = Dot2<T>::ok && std::is_same<T, CT>::value;
    using D2 = Dot2<T>;
    typename D2::v2 q_pk[PK ? GQ : 1][4];
    float q_reg[PK ? 1 : GQ][8];
#pragma unroll
    for (int g = 0; g < GQ; ++g) {
        if (g < gq) {
            const long qoff = ((((long)b * Hq) + hkv * gq + g) * Sq + sq) * D + c * 8;
            Vec8<T> qv = load_vec8(q + qoff);
            if constexpr (PK) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    q_pk[g][j] = D2::pack(VT::to_float(qv.v[2 * j]) * scale,
                                          VT::to_float(qv.v[2 * j + 1]) * scale);
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    q_reg[g][j] = VT::to_float(qv.v[j]) * scale;
            }
        }
    }

    float m[GQ], lsum[GQ], o_acc[GQ][8];
#pragma unroll
    for (int g = 0; g < GQ; ++g) {
        m[g] = M_INIT;
        lsum[g] = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) o_acc[g][j] = 0.f;
    }

    // ---- stream K/V rows (next row's loads issued before computing the
    // current one so the HBM latency hides under the dot/softmax VALU) ----
    if ((PAGED || row >= 0) && split_lo < split_hi) {
        const CT* kbase = PAGED ? k_cache : k_cache + (((long)row * Hkv + hkv) * Smax) * D;
        const CT* vbase = PAGED ? v_cache : v_cache + (((long)row * Hkv + hkv) * Smax) * D;
        // unconditional prefetch with clamped addresses — a conditional
        // ("load or keep") makes hipcc branch around the loads and wait
        // vmcnt(0) per iteration (guide §5 trap 4(c))
        auto row_addr = [&](int l, bool& valid) -> long {
            if constexpr (PAGED) {
                const int blk = block_table[(long)b * max_blocks + l / block_size];
                valid = blk >= 0;
                return (((long)max(blk, 0) * block_size + l % block_size) * Hkv + hkv) * D + c * 8;
            }
            valid = true;
            return (long)l * D + c * 8;
        };
        // per-group CONTIGUOUS row runs: a group streams rows
        // [g_lo, g_hi) back to back, so each group is one sequential HBM
        // stream (the strided l += NG layout read 256B chunks at 4 KB
        // stride — DRAM-page/channel hostile, same pathology measured on
        // the skinny GEMM). Online softmax is order-free, so the group->row
        // assignment is irrelevant to the math.
        const int span = split_hi - split_lo;
        const int rpg = (span + NG - 1) / NG;
        const int g_lo = split_lo + grp * rpg;
        const int g_hi = min(g_lo + rpg, split_hi);
        // row-compute body (shared by the 2-deep software pipeline legs)
        auto attn_row = [&](int l, bool valid_cur, const Vec8<CT>& kv_cur,
                            const Vec8<CT>& vv_cur) {
            if (PAGED && !valid_cur) return;
            if (ring) {
                const int p_s = pmax - ((pmax - l) % Smax);  // slot's true pos
                if (p_s >= eff_len ||
                    (window > 0 && p_s <= eff_len - 1 - window))
                    return;
            }
            const Vec8<CT>& vv_use = vv_cur;

            float s[GQ];
            if constexpr (PK) {
                const typename D2::v2* kp =
                    reinterpret_cast<const typename D2::v2*>(kv_cur.v);
#pragma unroll
                for (int g = 0; g < GQ; ++g) {
                    if (g >= gq) continue;
                    float d = 0.f;
#pragma unroll
                    for (int j = 0; j < 4; ++j) d = D2::dot(q_pk[g][j], kp[j], d);
                    s[g] = group_reduce_sum<GS>(d);
                }
            } else {
                float kf[8];
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    kf[j] = VecTraits<CT>::to_float(kv_cur.v[j]);
#pragma unroll
                for (int g = 0; g < GQ; ++g) {
                    if (g >= gq) continue;
                    float d = 0.f;
#pragma unroll
                    for (int j = 0; j < 8; ++j) d += q_reg[g][j] * kf[j];
                    s[g] = group_reduce_sum<GS>(d);  // all GS lanes get the dot
                }
            }
#pragma unroll
            for (int g = 0; g < GQ; ++g) {
                if (g >= gq) continue;
                const float mn = fmaxf(m[g], s[g]);
                const float corr = __expf(m[g] - mn);
                const float p = __expf(s[g] - mn);
                lsum[g] = lsum[g] * corr + p;
                m[g] = mn;
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    o_acc[g][j] = o_acc[g][j] * corr + p * VecTraits<CT>::to_float(vv_use.v[j]);
            }
        };

        // 2-deep pipeline: two row buffers alternate, so at each wait
        // point the OTHER buffer's load is still in flight and the
        // waited-on load has had ~2 iterations to land (depth-1 exposed
        // most of the HBM latency per row: the register copy forces the
        // vmcnt wait before the next load can issue).
        // Clamps: empty ranges and tails re-load a safe row.
        bool v0, v1;
        long off0 = row_addr(min(g_lo, split_hi - 1), v0);
        Vec8<CT> k0 = load_vec8(kbase + off0);
        Vec8<CT> w0 = load_vec8(vbase + off0);
        long off1 = row_addr((g_lo + 1 < g_hi) ? g_lo + 1
                                               : min(g_lo, split_hi - 1), v1);
        Vec8<CT> k1 = load_vec8(kbase + off1);
        Vec8<CT> w1 = load_vec8(vbase + off1);
        for (int l = g_lo; l < g_hi; l += 2) {
            {
                const bool vc = v0;
                const Vec8<CT> kc = k0, wc = w0;
                const int ln = (l + 2 < g_hi) ? l + 2 : l;
                off0 = row_addr(ln, v0);
                k0 = load_vec8(kbase + off0);
                w0 = load_vec8(vbase + off0);
                attn_row(l, vc, kc, wc);
            }
            if (l + 1 < g_hi) {
                const bool vc = v1;
                const Vec8<CT> kc = k1, wc = w1;
                const int ln = (l + 3 < g_hi) ? l + 3 : l + 1;
                off1 = row_addr(ln, v1);
                k1 = load_vec8(kbase + off1);
                w1 = load_vec8(vbase + off1);
                attn_row(l + 1, vc, kc, wc);
            }
        }
    }

    // ---- combine groups within the wave (xor butterfly over group bits) ----
#pragma unroll
    for (int off = GS; off < WAVE_SIZE; off <<= 1) {
#pragma unroll
        for (int g = 0; g < GQ; ++g) {
            if (g >= gq) continue;
            const float m_o = __shfl_xor(m[g], off, WAVE_SIZE);
            const float l_o = __shfl_xor(lsum[g], off, WAVE_SIZE);
            const float mn = fmaxf(m[g], m_o);
            const float f_s = __expf(m[g] - mn);
            const float f_o = __expf(m_o - mn);
            lsum[g] = lsum[g] * f_s + l_o * f_o;
            m[g] = mn;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float oo = __shfl_xor(o_acc[g][j], off, WAVE_SIZE);
                o_acc[g][j] = o_acc[g][j] * f_s + oo * f_o;
            }
        }
    }

    // ---- combine the 4 waves through LDS ----
    __shared__ float o_lds[4][GQ > 4 ? GQ : 4][D];
    __shared__ float ml_lds[4][GQ > 4 ? GQ : 4][2];
    if (lane < GS) {
#pragma unroll
        for (int g = 0; g < GQ; ++g) {
            if (g >= gq) continue;
#pragma unroll
            for (int j = 0; j < 8; ++j) o_lds[wid][g][c * 8 + j] = o_acc[g][j];
            if (c == 0) {
                ml_lds[wid][g][0] = m[g];
                ml_lds[wid][g][1] = lsum[g];
            }
        }
    }
    __syncthreads();
    if (wid == 0 && lane < GS) {
        for (int g = 0; g < gq; ++g) {
            float mm = M_INIT, ll = 0.f, oo[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) oo[j] = 0.f;
            for (int w = 0; w < 4; ++w) {
                const float mw = ml_lds[w][g][0];
                const float lw = ml_lds[w][g][1];
                const float mn = fmaxf(mm, mw);
                const float f_s = __expf(mm - mn);
                const float f_w = __expf(mw - mn);
                ll = ll * f_s + lw * f_w;
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    oo[j] = oo[j] * f_s + o_lds[w][g][c * 8 + j] * f_w;
                mm = mn;
            }
            const long base =
                ((((long)b * Hq + hkv * gq + g) * Sq + sq) * nsplit + split);
#pragma unroll
            for (int j = 0; j < 8; ++j) o_part[base * D + c * 8 + j] = oo[j];
            if (c == 0) {
                ml_part[base * 2 + 0] = mm;
                ml_part[base * 2 + 1] = ll;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Matrix-core pass 1: 16-bit models, head sizes 64 and 128, cache in the model's type or e4m3.
//
// Bound by the stream of K and V. The lane-group kernel above spends about 40 vector
// instructions a row and query head on products, exponentials and lane sums (129 us where the
// stream takes 83, 274 us of an 8-bit cache where it takes 33); here a wave takes 32 keys at a
// time through the matrix pipe and the vector units are left with one exponential a score:
//   * S^T = K Q^T on 16x16x32 tiles: the rows are keys, the columns up to 16 (query token,
//     head of the group) pairs, so every K row is used by all of them. The A operand is 16
//     contiguous bytes of a key row.
//   * O = P V: the C layout of S^T gives a lane 4 consecutive keys of its column in each of
//     the two 16-key tiles, which is the A operand of P for the same 32 keys in another
//     order. V rows are read in that order, 16 bytes of channels a lane (a whole row for
//     16 lanes), and turned in registers: one byte permutation makes a B operand word. Which
//     channels a column of the product stands for is free, so nothing else moves.
//   * P enters as three 16-bit parts that add up to its 24 bits. (Two parts: 64 rows of 2048 73.1
//     us for 73.9, of an 8-bit cache 38.6 for 40.7. 32-bit matrix instructions, which need no
//     parts: 81 and 55.) fp16 has no exponents for small parts: there P is lifted by 2^7, and its
//     reference follows a 32-key step down that stays more than 2^8 below it, so that P at each
//     step's largest lies in [2^-1, 2^15]. The accumulator is scaled up meanwhile, by 2^64 at
//     most: far from overflow, and what lies deeper is less than a 32-bit sum keeps. One key
//     whose values are 10^-4 of the others' ahead of 60000 at e^-19, fp16, error 2-norm: 1.9e-4
//     (two parts and one reference 4.2e-3, 32-bit multiply-adds of scaled queries 5.1e-4).
//   * The next 32 keys are on their way while these are computed: straight to LDS (STAGED), into
//     a place of the wave's own, so that no wave waits for another, and from there to the
//     registers just before they are computed. What a CU holds in flight is some 140 lines of
//     128 bytes, and a load that asks for 64 bytes of each of 16 rows (K as the matrix operand
//     wants it; 32 bytes in 8 bits) takes a line for half of one: staged, every load is of whole
//     lines, and past the caches. (Streaming alone, 64 rows of 1024 to 2048 keys: 71.6 us as
//     operands, 61.5 as whole lines, not cached.) Caches that start off 16 bytes go straight to
//     two register buffers, as all did. Waves of a workgroup take 32-key tiles in turn and meet in
//     LDS once at the end.
//   * The accumulator is rescaled only when a maximum grew by more than 2^8.
// Measured in a captured graph (MI355X, bf16, 32/8 heads of 128, lengths half to full, before ->
// now, stream rate): 64 rows of 2048 131 -> 76 us (5.3 TB/s); 16 of 8192 136 -> 73; 128 of 512
// 68 -> 40; 256 of 168 57 -> 28; 1 of 300 18.2 -> 7.8; 1 of 8192 55 -> 12; 13 rows of 8000, 64/8
// heads 271 -> 72 us, e4m3 279 -> 48 us. Straight to registers -> staged: 64 rows of 2048 75.5 ->
// 66.5 us (6.1 TB/s), in pages 88 -> 78.5; 256 of 168 36.0 -> 31.8; 13 of 8000, e4m3, 44.7 -> 35.1;
// 100 of 1200, heads of 64, 41.0 -> 36.6; 1 row the same. Error against 64 bits, bf16: 1.66e-3 (the rounding of
// the result), before 1.66e-3 to 3.5e-3 (the scaled query was rounded too).
typedef __bf16 dm_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 dm_f16x8 __attribute__((ext_vector_type(8)));
typedef float dm_f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned dm_u32x4 __attribute__((ext_vector_type(4)));

template <typename T> struct DmTraits;
template <> struct DmTraits<__hip_bfloat16> {
    using vec8 = dm_bf16x8;
    using elem = __bf16;
    static DEV_INLINE dm_f32x4 mfma(vec8 a, vec8 b, dm_f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
    // a 16-bit part of each value, taken off it
    static DEV_INLINE vec8 part(float (&e)[8]) {
        vec8 p;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            p[j] = (__bf16)e[j];
            e[j] -= (float)p[j];
        }
        return p;
    }
    static DEV_INLINE unsigned cvt2(unsigned w, bool hi) {   // two e4m3 -> two bf16, exact
        return __builtin_bit_cast(unsigned, hi
            ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, true)
            : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, false));
    }
};
template <> struct DmTraits<__half> {
    using vec8 = dm_f16x8;
    using elem = _Float16;
    static DEV_INLINE dm_f32x4 mfma(vec8 a, vec8 b, dm_f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
    static DEV_INLINE vec8 part(float (&e)[8]) {
        dm_u32x4 p;
#pragma unroll
        for (int j = 0; j < 4; ++j) {          // towards zero: in pairs, what is left is exact
            const auto h = __builtin_amdgcn_cvt_pkrtz(e[2 * j], e[2 * j + 1]);
            p[j] = __builtin_bit_cast(unsigned, h);
            e[2 * j] -= (float)h[0];
            e[2 * j + 1] -= (float)h[1];
        }
        return __builtin_bit_cast(vec8, p);
    }
    static DEV_INLINE unsigned cvt2(unsigned w, bool hi) {
        return __builtin_bit_cast(unsigned, hi
            ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, true)
            : __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, false));
    }
};

// NE elements of the cache's type in whole words, and as 16-bit pairs
template <int NE, bool F8> struct DmRaw {
    static constexpr int W = NE * (F8 ? 1 : 2) / 4;
    unsigned w[W];
    DEV_INLINE void load(const char* p) {
        if constexpr (W == 4) *reinterpret_cast<int4*>(w) = *reinterpret_cast<const int4*>(p);
        else if constexpr (W == 2) *reinterpret_cast<int2*>(w) = *reinterpret_cast<const int2*>(p);
        else w[0] = *reinterpret_cast<const unsigned*>(p);
    }
    template <typename T> DEV_INLINE void pairs(unsigned (&o)[NE / 2]) const {
#pragma unroll
        for (int i = 0; i < NE / 2; ++i) {
            if constexpr (F8) o[i] = DmTraits<T>::cvt2(w[i >> 1], i & 1);
            else o[i] = w[i];
        }
    }
};

// 16 bytes a lane to the 1 KB of LDS at dst; past the caches, which a step's keys would only sweep
DEV_INLINE void dm_load_lds(const char* src, char* dst) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) unsigned int*)src,
                                     (__attribute__((address_space(3))) unsigned int*)dst, 16, 0, 2);
}

constexpr float DM_GROWTH = 8.f;   // log2 growth of a maximum that is put off
constexpr float DM_DEPTH = 64.f;   // and how far below the largest score P may count from (fp16)
constexpr int DM_TILE = 32;        // keys of a wave's step
constexpr int DM_LEAST = 128;      // keys of a split: one step of each wave

template <typename T, typename CT, int D, bool PAGED, int WPR, bool STAGED>
__global__ __launch_bounds__(256, 2) void decode_mfma_kernel(
    T* __restrict__ out,               // (B, Hq, Sq, D), written when nsplit == 1
    float* __restrict__ o_part,        // (B, Hq, Sq, nsplit, D)
    float* __restrict__ ml_part,       // (B, Hq, Sq, nsplit, 2)
    const T* __restrict__ q, const CT* __restrict__ k_cache, const CT* __restrict__ v_cache,
    const int* __restrict__ positions, const int* __restrict__ seq_ids,
    const int* __restrict__ block_table, const float* __restrict__ sinks,
    float* __restrict__ lse_out, const float scale, const float v_scale, const int window,
    const int ring, const int Hkv, const int Sq, const int gq, const int Smax, const int nsplit,
    const int block_size, const int max_blocks, const int B) {
    using DT = DmTraits<T>;
    using vec8 = typename DT::vec8;
    constexpr bool F8 = sizeof(CT) == 1;
    constexpr bool F16 = std::is_same<T, __half>::value;
    constexpr float LIFT = F16 ? 7.f : 0.f;
    constexpr int NKS = D / 32;            // k-steps of K Q^T
    constexpr int DV = D / 16;             // channels a lane holds of a V row
    constexpr int ES = sizeof(CT);

    const int ncol = gq * Sq;
    const int nct = (ncol + 15) >> 4;
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // uniform: so are the loops
    const int n = lane & 15, g = lane >> 4;
    // a set of columns is WPR waves' work (see launch_decode); the last ones may have none
    const int sub = wid % WPR, slot0 = wid - sub;
    int split, y, b;
    bool idle = false;
    if constexpr (WPR == 4) {
        split = blockIdx.x;
        y = blockIdx.y;
        b = blockIdx.z;
    } else {                                   // (no splits)
        const long set = (long)blockIdx.x * (4 / WPR) + wid / WPR;
        idle = set >= (long)B * Hkv * nct;
        split = 0;
        b = idle ? B - 1 : (int)(set / (Hkv * nct));
        y = idle ? 0 : (int)(set % (Hkv * nct));
    }
    const int hkv = y / nct;
    const int c0 = (y % nct) * 16;
    const int nc = min(16, ncol - c0), ncw = min(16, ncol);    // ncw: columns of a wave's LDS
    const int Hq = Hkv * gq;

    const int row = idle ? -1 : PAGED ? 0 : seq_ids[b];
    const int col = min(c0 + n, ncol - 1);
    const int sq = col / gq;
    const int head = hkv * gq + col % gq;
    const int qpos = (c0 + n < ncol && row >= 0) ? positions[(long)b * Sq + sq] : -1;

    // keys [k_lo, k_hi) that any column sees; a column's own first key
    int key_lo = 0, pmax = -1, span = qpos + 1, first = qpos < 0 ? 0x7fffffff : 0;
    if (ring) {
        for (int s = 0; s < Sq; ++s) pmax = max(pmax, positions[(long)b * Sq + s]);
        span = row >= 0 ? min(pmax + 1, Smax) : 0;
    } else {
        if (window > 0) key_lo = max(0, qpos - window + 1);
        else if (window < 0) key_lo = qpos >= 0 ? qpos / -window * -window : 0;
        if (qpos >= 0) first = key_lo;
    }
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) {
        span = max(span, __shfl_xor(span, off, WAVE_SIZE));
        first = min(first, __shfl_xor(first, off, WAVE_SIZE));
    }
    // the splits share the keys that are seen (see launch_decode)
    const int all_hi = __builtin_amdgcn_readfirstlane(min(span, Smax));
    const int all_lo = min(__builtin_amdgcn_readfirstlane(ring ? 0 : first), all_hi);
    const int seen = all_lo / DM_TILE * DM_TILE;
    const int chunk = max(DM_LEAST, ((all_hi - seen + nsplit - 1) / nsplit + DM_TILE - 1) / DM_TILE * DM_TILE);
    const int k_hi = min(all_hi, seen + (split + 1) * chunk);
    const int k_lo = max(all_lo, seen + split * chunk);
    const int t_lo = k_lo / DM_TILE, t_hi = k_lo < k_hi ? (k_hi + DM_TILE - 1) / DM_TILE : 0;
    // position of the key in cache row l: l itself; in a ring the newest one that is l modulo
    // Smax, which is base + l up to the newest row and base + l - Smax behind it
    const int ring_base = ring && pmax >= 0 ? pmax - pmax % Smax : 0;
    const int ring_at = ring && pmax >= 0 ? pmax % Smax : 0x7fffffff;
    if (ring && window > 0) key_lo = max(0, qpos - window + 1);

    vec8 qf[NKS];
    {
        const T* qp = q + (((long)b * Hq + head) * Sq + sq) * D + g * 8;
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) qf[ks] = *reinterpret_cast<const vec8*>(qp + ks * 32);
    }

    const long lin = PAGED ? 0 : ((long)max(row, 0) * Hkv + hkv) * (long)Smax * D * ES;
    const char* kbase = reinterpret_cast<const char*>(k_cache) + lin;
    const char* vbase = reinterpret_cast<const char*>(v_cache) + lin;
    const int last = k_hi - 1;

    // pages: lanes 0..31 each look up a key of the tile, a step ahead of its use
    auto page_key = [&](int t) -> int { return max(min(t * DM_TILE + (lane & 31), last), 0); };
    auto page_load = [&](int t) -> int {
        if constexpr (!PAGED) return 0;
        return block_table[(long)b * max_blocks + page_key(t) / block_size];
    };
    struct Buf {
        DmRaw<8, F8> k[2][NKS];
        DmRaw<DV, F8> v[8];
        unsigned bad;              // bit j: key j of the lane has no page
    };
    // STAGED: the wave's tile in LDS, K then V, 16-byte pieces of a row in the order piece ^ turn(row)
    extern __shared__ __attribute__((aligned(16))) float dm_lds[];
    constexpr int ROWB = D * ES, PPR = ROWB / 16, RPI = 64 / PPR, TILE_B = DM_TILE * ROWB;
    char* const tile = reinterpret_cast<char*>(dm_lds) + wid * 2 * TILE_B;
    auto turn = [](int r) { return PPR == 4 ? (r >> 1) & 3 : r & (PPR - 1); };
    auto stage = [&](int t, int blk) -> unsigned {
        unsigned bad = 0;
        int prow = 0;                  // cache row of the lane's key, -1: no page
        if constexpr (PAGED) prow = blk < 0 ? -1 : blk * block_size + page_key(t) % block_size;
#pragma unroll
        for (int i = 0; i < DM_TILE / RPI; ++i) {
            const int r = i * RPI + lane / PPR;
            const int at = ((lane % PPR) ^ turn(r)) * 16;
            const char *kp, *vp;
            if constexpr (PAGED) {
                const long off = ((long)max(__shfl(prow, r, WAVE_SIZE), 0) * Hkv + hkv) * ROWB + at;
                kp = kbase + off;
                vp = vbase + off;
            } else {
                const unsigned off = (unsigned)(min(t * DM_TILE + r, last) * ROWB) + at;
                kp = kbase + off;
                vp = vbase + off;
            }
            dm_load_lds(kp, tile + i * 1024);
            dm_load_lds(vp, tile + TILE_B + i * 1024);
        }
        if constexpr (PAGED) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                bad |= ((unsigned)__shfl(prow, (j >> 2) * 16 + g * 4 + (j & 3), WAVE_SIZE) >> 31) << j;
        }
        return bad;
    };
    auto fetch = [&](Buf& u) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                const int r = kb * 16 + n, at = (ks * 32 + g * 8) * ES;
                u.k[kb][ks].load(tile + r * ROWB + (((at >> 4) ^ turn(r)) << 4) + (at & 15));
            }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int r = (j >> 2) * 16 + g * 4 + (j & 3), at = n * DV * ES;
            u.v[j].load(tile + TILE_B + r * ROWB + (((at >> 4) ^ turn(r)) << 4) + (at & 15));
        }
    };
    auto load = [&](Buf& u, int t, int blk) {
        u.bad = 0;
        int prow = 0;                  // cache row of the lane's key, -1: no page
        if constexpr (PAGED) prow = blk < 0 ? -1 : blk * block_size + page_key(t) % block_size;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            const char* p;
            if constexpr (PAGED) {
                const int r = __shfl(prow, kb * 16 + n, WAVE_SIZE);
                p = kbase + ((long)max(r, 0) * Hkv + hkv) * (D * ES);
            } else {
                p = kbase + (unsigned)(min(t * DM_TILE + kb * 16 + n, last) * (D * ES));
            }
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) u.k[kb][ks].load(p + (ks * 32 + g * 8) * ES);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int kk = (j >> 2) * 16 + g * 4 + (j & 3);
            const char* p;
            if constexpr (PAGED) {
                const int r = __shfl(prow, kk, WAVE_SIZE);
                u.bad |= ((unsigned)r >> 31) << j;
                p = vbase + ((long)max(r, 0) * Hkv + hkv) * (D * ES);
            } else {
                p = vbase + (unsigned)(min(t * DM_TILE + kk, last) * (D * ES));
            }
            u.v[j].load(p + n * DV * ES);
        }
    };

    dm_f32x4 o[DV];
#pragma unroll
    for (int i = 0; i < DV; ++i) o[i] = {0.f, 0.f, 0.f, 0.f};
    // of column n; what P counts from, l: of this lane's keys, largest score so far (fp16)
    float m = -INFINITY, l = 0.f, top = -INFINITY;
    const float sc = scale * 1.4426950408889634f;

    auto step = [&](Buf& u, int t) {
        dm_f32x4 s[2];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            s[kb] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                unsigned w[4];
                u.k[kb][ks].template pairs<T>(w);
                s[kb] = DT::mfma(__builtin_bit_cast(vec8, dm_u32x4{w[0], w[1], w[2], w[3]}),
                                 qf[ks], s[kb]);
            }
        }
        float x[8], mx = -INFINITY;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int key = t * DM_TILE + (j >> 2) * 16 + g * 4 + (j & 3);
            const int at = key + ring_base - (key > ring_at ? Smax : 0);
            bool ok = (key < k_hi) & (key >= k_lo) & (at <= qpos) & (at >= key_lo);
            if constexpr (PAGED) ok = ok & !((u.bad >> j) & 1);
            x[j] = ok ? s[j >> 2][j & 3] * sc : -INFINITY;
            mx = fmaxf(mx, x[j]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16, WAVE_SIZE));
        mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE_SIZE));
        bool move = mx > m + DM_GROWTH || (m == -INFINITY && mx > m);
        float mn = fmaxf(m, mx);
        if constexpr (F16) {               // and down to a step that stays far below
            top = fmaxf(top, mx);
            if (mx < m - DM_GROWTH && mx != -INFINITY) {
                mn = fmaxf(mx, top - DM_DEPTH);
                move = mn < m;
            }
        }
        if (__any(move)) {
            const float f = m == -INFINITY ? 0.f : exp2f(m - mn);
            m = mn;
            l *= f;
            // the accumulator's rows are columns g*4 + r
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float fr = __shfl(f, g * 4 + r, WAVE_SIZE);
#pragma unroll
                for (int i = 0; i < DV; ++i) o[i][r] *= fr;
            }
        }
        const float mu = m == -INFINITY ? 0.f : m - LIFT;
        float e[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            e[j] = __builtin_amdgcn_exp2f(x[j] - mu);
            l += e[j];
        }
        vec8 p[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) p[c] = DT::part(e);
        // V: pairs of channels of 8 keys -> for each channel, pairs of keys
        unsigned vp[8][DV / 2];
#pragma unroll
        for (int j = 0; j < 8; ++j) u.v[j].template pairs<T>(vp[j]);
        if constexpr (PAGED) {             // whatever stands in for a missing page: not 0 * NaN
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const unsigned keep = ((u.bad >> j) & 1) - 1u;
#pragma unroll
                for (int i = 0; i < DV / 2; ++i) vp[j][i] &= keep;
            }
        }
#pragma unroll
        for (int i = 0; i < DV; ++i) {
            dm_u32x4 w;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                w[e] = __builtin_amdgcn_perm(vp[2 * e + 1][i >> 1], vp[2 * e][i >> 1],
                                             (i & 1) ? 0x07060302u : 0x05040100u);
            const vec8 vb = __builtin_bit_cast(vec8, w);
#pragma unroll
            for (int c = 0; c < 3; ++c) o[i] = DT::mfma(p[c], vb, o[i]);
        }
    };

    if constexpr (STAGED) {
        if (t_lo + sub < t_hi) {
            int t = t_lo + sub;
            unsigned bad = stage(t, page_load(t));
            int blk = page_load(t + WPR);
            for (;; t += WPR) {
                Buf u;
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                fetch(u);
                u.bad = bad;
                if (t + WPR >= t_hi) {
                    step(u, t);
                    break;
                }
                // into registers before the next tile lands in their place
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                bad = stage(t + WPR, blk);
                blk = page_load(t + 2 * WPR);
                step(u, t);
            }
        }
        __syncthreads();                       // the tiles' place is the waves' meeting place
    } else if (t_lo + sub < t_hi) {
        Buf u0, u1;
        int t = t_lo + sub;
        int blk = page_load(t), next = page_load(t + WPR);
        load(u0, t, blk);
        for (;;) {
            // past the end the loads repeat the last key: no branch between them and their use
            blk = page_load(t + 2 * WPR);
            load(u1, t + WPR, next);
            step(u0, t);
            t += WPR;
            if (t >= t_hi) break;
            next = page_load(t + 2 * WPR);
            load(u0, t + WPR, blk);
            step(u1, t);
            t += WPR;
            if (t >= t_hi) break;
        }
    }
    l += __shfl_xor(l, 16, WAVE_SIZE);
    l += __shfl_xor(l, 32, WAVE_SIZE);
    m -= LIFT;

    // ---- the waves of a set meet ----
    float* o_lds = dm_lds;                     // [4][ncw][D]
    float* ml_lds = dm_lds + 4 * ncw * D;      // [4][16][2]
    if (g == 0) {
        ml_lds[(wid * 16 + n) * 2] = m;
        ml_lds[(wid * 16 + n) * 2 + 1] = l;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (g * 4 + r >= nc) continue;
        float* p = o_lds + (wid * ncw + g * 4 + r) * D + n * DV;
#pragma unroll
        for (int i = 0; i < DV; i += 4)
            *reinterpret_cast<float4*>(p + i) =
                float4{o[i][r], o[i + 1][r], o[i + 2][r], o[i + 3][r]};
    }
    __syncthreads();
    // (whole waves, for the rows that are done again: a column is 32 or 16 lanes of one)
    if (idle) return;
    for (int base = sub * 64; base < nc * (D / 4); base += WPR * 64) {
        const bool in = base + lane < nc * (D / 4);
        const int idx = in ? base + lane : base;
        const int cl = idx / (D / 4), d = idx % (D / 4) * 4;
        const int cc = c0 + cl;
        const int hh = hkv * gq + cc % gq;
        float ms = -INFINITY, ls = 0.f;
#pragma unroll
        for (int w = slot0; w < slot0 + WPR; ++w) ms = fmaxf(ms, ml_lds[(w * 16 + cl) * 2]);
        float4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = slot0; w < slot0 + WPR; ++w) {
            const float lw = ml_lds[(w * 16 + cl) * 2 + 1];
            if (lw == 0.f) continue;       // no key seen
            // (no maximum, but a sum: it is NaN, as of a query that is, and stays)
            const float f = ms == -INFINITY ? 1.f : exp2f(ml_lds[(w * 16 + cl) * 2] - ms);
            ls += f * lw;
            const float4 y = *reinterpret_cast<const float4*>(o_lds + (w * ncw + cl) * D + d);
            acc.x += f * y.x;
            acc.y += f * y.y;
            acc.z += f * y.z;
            acc.w += f * y.w;
        }
        // columns whose sums are finite and whose values are not: see attention_row.h
        const bool lost = !((acc.x + acc.y) * 0.f + (acc.z + acc.w) * 0.f == 0.f) && ls == ls;
        unsigned long long bad = __ballot(lost);
        while (bad) {
            const int first_lane = __ffsll(bad) - 1, cb = (base + first_lane) / (D / 4);
            const int cq = (c0 + cb) / gq, pos = row >= 0 ? positions[(long)b * Sq + cq] : -1;
            int from = 0;
            if (window > 0) from = max(0, pos - window + 1);
            else if (window < 0 && !ring) from = pos >= 0 ? pos / -window * -window : 0;
            float mr, lr, y[D / 64];
            attend_row<D>(q + (((long)b * Hq + hkv * gq + (c0 + cb) % gq) * Sq + cq) * D,
                          k_cache, v_cache, k_lo, k_hi, sc, [&](int key) -> long {
                const int at = key + ring_base - (key > ring_at ? Smax : 0);
                if (at > pos || at < from) return -1;
                if constexpr (PAGED) {
                    const int p = block_table[(long)b * max_blocks + key / block_size];
                    return p < 0 ? -1 : (((long)p * block_size + key % block_size) * Hkv + hkv) * D;
                }
                return (((long)max(row, 0) * Hkv + hkv) * (long)Smax + key) * D;
            }, mr, lr, y);
            float z[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) z[e] = __shfl(y[e % (D / 64)], (d + e) / (D / 64), WAVE_SIZE);
            if (cl == cb) {
                ms = mr;
                ls = lr;
                acc = float4{z[0], z[1], z[2], z[3]};
            }
            bad &= ~__ballot(cl == cb);
        }
        if (!in) continue;
        const long rowid = ((long)b * Hq + hh) * Sq + cc / gq;
        const float mn = ms * 0.6931471805599453f;     // natural units from here on
        if (nsplit > 1) {
            *reinterpret_cast<float4*>(o_part + (rowid * nsplit + split) * D + d) = acc;
            if (d == 0) {
                ml_part[(rowid * nsplit + split) * 2] = mn;
                ml_part[(rowid * nsplit + split) * 2 + 1] = ls;
            }
            continue;
        }
        float f = 1.f;
        if (sinks != nullptr) {        // a sink joins the denominator only
            const float mt = fmaxf(mn, sinks[hh]);
            f = __expf(mn - mt);
            ls = ls * f + __expf(sinks[hh] - mt);
            if (lse_out != nullptr && d == 0) lse_out[rowid] = mt + __logf(ls);
        } else if (lse_out != nullptr && d == 0) {
            lse_out[rowid] = ls > 0.f ? mn + __logf(ls) : -INFINITY;
        }
        const float inv = ls > 0.f ? v_scale * f / ls : 0.f;
        T* po = out + rowid * D + d;
        po[0] = VecTraits<T>::from_float(acc.x * inv);
        po[1] = VecTraits<T>::from_float(acc.y * inv);
        po[2] = VecTraits<T>::from_float(acc.z * inv);
        po[3] = VecTraits<T>::from_float(acc.w * inv);
    }
}

// Pass 2: out row = sum over splits of exp(m_i - m) o_i / L. A group of D/4 lanes takes every
// G-th split of a row (G: the splits' number rounded up to a power of two, at most all groups of
// the workgroup) and the groups of a row meet in LDS, so that a row of 64 splits is 8 dependent
// loads and not 64 (D = 128), and rows of few splits share a workgroup.
template <typename T, int D>
__global__ __launch_bounds__(256) void decode_attn_pass2(
    T* __restrict__ out,               // (B, Hq, Sq, D)
    const float* __restrict__ o_part,  // (B, Hq, Sq, nsplit, D)
    const float* __restrict__ ml_part, // (B, Hq, Sq, nsplit, 2)
    const int nsplit, const int G, const long rows, const float v_scale,
    const float* __restrict__ sinks,   // (Hq,) learned sink logits or null
    const int Hq, const int Sq,
    float* __restrict__ lse_out) {     // (B,Hq,Sq) log-sum-exp, or null —
                                       // the cross-rank flash-decoding handle
    using VT = VecTraits<T>;
    constexpr int LPG = D / 4, NG = 256 / LPG;
    __shared__ float4 s_o[256];
    __shared__ float s_ml[NG][2];
    const int grp = threadIdx.x / LPG, c = threadIdx.x % LPG;
    const long rowid = (long)blockIdx.x * (NG / G) + grp / G;
    float m = M_INIT, l = 0.f;
    float4 acc = {0.f, 0.f, 0.f, 0.f};
    if (rowid < rows) {
        for (int i = grp % G; i < nsplit; i += G) {
            const float mi = ml_part[(rowid * nsplit + i) * 2];
            const float li = ml_part[(rowid * nsplit + i) * 2 + 1];
            const float4 oi = *reinterpret_cast<const float4*>(o_part + (rowid * nsplit + i) * D + c * 4);
            const float mn = fmaxf(m, mi);
            const float f = __expf(m - mn), fi = __expf(mi - mn);
            m = mn;
            l = l * f + li * fi;
            acc.x = acc.x * f + oi.x * fi;
            acc.y = acc.y * f + oi.y * fi;
            acc.z = acc.z * f + oi.z * fi;
            acc.w = acc.w * f + oi.w * fi;
        }
    }
    s_o[threadIdx.x] = acc;
    if (c == 0) {
        s_ml[grp][0] = m;
        s_ml[grp][1] = l;
    }
    __syncthreads();
    if (grp % G != 0 || rowid >= rows) return;
    float ms = M_INIT, L = 0.f;
    for (int w = 0; w < G; ++w) ms = fmaxf(ms, s_ml[grp + w][0]);
    if (sinks != nullptr) {  // sink joins the softmax denominator only
        const int h = (int)((rowid / Sq) % Hq);
        ms = fmaxf(ms, sinks[h]);
        L += __expf(sinks[h] - ms);
    }
    acc = {0.f, 0.f, 0.f, 0.f};
    for (int w = 0; w < G; ++w) {
        const float f = __expf(s_ml[grp + w][0] - ms);
        L += s_ml[grp + w][1] * f;
        const float4 y = s_o[(grp + w) * LPG + c];
        acc.x += y.x * f;
        acc.y += y.y * f;
        acc.z += y.z * f;
        acc.w += y.w * f;
    }
    const float inv = (L > 0.f) ? v_scale / L : 0.f;
    if (lse_out != nullptr && c == 0)
        lse_out[rowid] = (L > 0.f) ? ms + __logf(L) : -INFINITY;
    T* po = out + rowid * D + c * 4;
    po[0] = VT::from_float(acc.x * inv);
    po[1] = VT::from_float(acc.y * inv);
    po[2] = VT::from_float(acc.z * inv);
    po[3] = VT::from_float(acc.w * inv);
}

// ---------------------------------------------------------------------------
// the shares of a decode row's keys, where the caller adds them up
struct DecodeShares {
    torch::Tensor o, ml;         // (B, Hq, Sq, n, D) and (B, Hq, Sq, n, 2) in fp32
    int n = 1;                   // 1: none, the result is there
    long most = 0;               // that the caller takes
};

template <typename T, typename CT, int D, int GQ>
static void launch_decode(torch::Tensor& out, const torch::Tensor& q,
                          const torch::Tensor& k_cache, const torch::Tensor& v_cache,
                          const torch::Tensor& seq_lens, const torch::Tensor& seq_ids,
                          float scale, int window, int gq,
                          const torch::Tensor* block_table = nullptr,
                          int block_size = 0, float v_scale = 1.0f,
                          const torch::Tensor* sinks = nullptr,
                          torch::Tensor* lse_out = nullptr,
                          int ring = 0, DecodeShares* shares = nullptr) {
    const int B = q.size(0), Hq = q.size(1), Sq = q.size(2);
    const bool paged = block_table != nullptr;
    const int Hkv = paged ? k_cache.size(2) : k_cache.size(1);
    const int max_blocks = paged ? (int)block_table->size(1) : 0;
    const int Smax = paged ? max_blocks * block_size : (int)k_cache.size(2);
    if (Smax == 0) ring = 0;               // the kernels divide by a ring's size
    constexpr bool MFMA = !std::is_same<T, float>::value && (D == 64 || D == 128);
    const int nct = (gq * Sq + 15) / 16;
    // Splits over the keys. Matrix-core kernel: two workgroups fit a CU, so 512 fill the chip;
    // more only add partial sums to write and combine (64 rows of 2048: 68 us at 512, 72 at
    // 1024, 73 at 2048; 13 rows of 8000 of 8 heads in 8 bits 36 / 38 / 44), as rows of unequal length even out over
    // the CUs by themselves. A split keeps 128 rows, one step of each wave (1 row of 300: 7.8 us;
    // 256: 8.4), 256 in long caches where the combining pass weighs more (1 row of 8192: 11.8 us
    // with 256, 13.5 with 128). Their number goes by the capacity, which the host knows; what
    // they share by the keys that a row sees, so that short rows keep them busy too. 32/8 heads
    // of 128, shares of the capacity -> of the row: 1 row of 700 in a cache of 8192 10.1 -> 9.2 us,
    // of 1000 (or a window of 1024) in 32768 18.9 -> 12.5, 16 rows of 700 in 8192 25.7 -> 15.0 (in
    // pages 27.8 -> 15.9), full rows the same (16 of half to full 8192 73.3, 73.7; 64 of 2048
    // 73.5, 73.9).
    // Lane-group kernel: >= 1024 workgroups when possible, chunks of >= 128 rows.
    int nsplit, chunk = 0;
    if constexpr (MFMA) {
        const int least = Smax <= 2048 ? DM_LEAST : 2 * DM_LEAST;
        nsplit = 512 / std::max(1, B * Hkv * nct);
        nsplit = std::max(1, std::min({nsplit, (Smax + least - 1) / least, 64}));
    } else {
        nsplit = 1024 / std::max(1, B * Hkv * Sq);
        nsplit = std::max(1, std::min({nsplit, (Smax + 127) / 128, 64}));
        chunk = (Smax + nsplit - 1) / nsplit;
    }

    auto opts = torch::TensorOptions().dtype(torch::kFloat32).device(q.device());
    const bool parts = !MFMA || nsplit > 1;
    auto o_part = torch::empty({parts ? (long)B * Hq * Sq * nsplit * D : 0}, opts);
    auto ml_part = torch::empty({parts ? (long)B * Hq * Sq * nsplit * 2 : 0}, opts);
    auto stream = at::hip::getCurrentHIPStream();

    dim3 grid1(nsplit, Hkv * Sq, B);
    if constexpr (MFMA) {
        if (B == 0 || Sq == 0) return;
        const int nc = std::min(16, gq * Sq);
        const bool staged = ((size_t)k_cache.data_ptr() | (size_t)v_cache.data_ptr()) % 16 == 0;
        const size_t lds = std::max((4 * nc * D + 4 * 16 * 2) * sizeof(float),
                                    staged ? 4 * 2 * DM_TILE * D * sizeof(CT) : 0);
        const long sets = (long)B * Hkv * nct;
        // Waves of a set of columns (of one row's KV head). Where rows are short a workgroup is
        // gone after a step or two of its waves, and what it waits for on the way (positions,
        // pages, the first keys, the other waves) is most of its time: a wave a set takes more
        // steps, and all sets are there at once. Longer rows are bound by their bytes, for which 4
        // waves have more on the way; in 8 bits a row of many has half as many bytes, and a row of
        // few wants all the waves there are. 4 waves' time over one's, half to full caches of
        // 64, 128, 200, 256, 384 keys (8 KV heads of 4 query heads; 1 and 8 are like it):
        //   sets           768                      1536                     4096
        //   128, 16 bits   1.21 1.17 1.15 1.08 1.04  1.31 1.09 1.00 0.94 0.88  1.67 1.26 1.24 0.97 0.92
        //   128, e4m3      1.23 1.09 1.12 0.96 0.98  1.42 1.22 1.10 1.02 0.97  1.89 1.59 1.43 1.28 1.20
        //   64, 16 bits    0.94 0.93 0.90 0.92 0.91  1.15 1.10 0.99 0.95 0.87  1.58 1.33 1.18 1.02 1.00
        //   64, e4m3       0.89 0.85 0.80 0.75 0.71  1.17 1.06 0.96 0.96 0.88  1.66 1.37 1.27 1.13 1.11
        // (1024 sets: 64 in 16 bits 1.26 1.22 1.15, e4m3 0.94 0.92 0.86; 2048: e4m3 1.16 and 1.01
        // at 384.) In 16 bits the line is at 7 tiles: 224 keys 1.15 0.97 1.05, heads of 64 0.94
        // 1.01 1.11; 248 1.06 0.95 1.03 and 0.91 0.95 1.02. 256 rows of 168, heads of 128: 37.4 ->
        // 30.7 us.
        const int span = window ? std::min(Smax, std::abs(window) + Sq + DM_TILE) : Smax;
        const bool f8 = sizeof(CT) == 1;
        const bool alone = nsplit == 1 && sets >= (D == 128 ? 768 : f8 ? 2048 : 1024) &&
                           span <= DM_TILE * (f8 && sets >= 2048 ? 12 : 7);
        TORCH_CHECK(sets < (1L << 31), "attention_decode: too many rows");
        const dim3 grid = alone ? dim3((unsigned)((sets + 3) / 4)) : dim3(nsplit, Hkv * nct, B);
#define DM_GO(PG, W)                                                                        \
        do {                                                                                \
            if (staged) DM_RUN(PG, W, true);                                                \
            else DM_RUN(PG, W, false);                                                      \
        } while (0)
#define DM_RUN(PG, W, ST)                                                                   \
        hipLaunchKernelGGL((decode_mfma_kernel<T, CT, D, PG, W, ST>), grid, dim3(256), lds, stream, \
                           (T*)out.data_ptr(), o_part.data_ptr<float>(),                    \
                           ml_part.data_ptr<float>(), (const T*)q.data_ptr(),               \
                           (const CT*)k_cache.data_ptr(), (const CT*)v_cache.data_ptr(),    \
                           seq_lens.data_ptr<int>(), seq_ids.data_ptr<int>(),               \
                           PG ? block_table->data_ptr<int>() : nullptr,                     \
                           sinks ? sinks->data_ptr<float>() : nullptr,                      \
                           lse_out ? lse_out->data_ptr<float>() : nullptr, scale, v_scale,  \
                           window, ring, Hkv, Sq, gq, Smax, nsplit, block_size, max_blocks, B)
        if (paged) {
            if (alone) DM_GO(true, 1);
            else DM_GO(true, 4);
        } else {
            if (alone) DM_GO(false, 1);
            else DM_GO(false, 4);
        }
#undef DM_GO
#undef DM_RUN
        HIP_CHECK_KERNEL();
        if (nsplit == 1) return;
        if (shares && nsplit <= shares->most) {
            shares->o = o_part;
            shares->ml = ml_part;
            shares->n = nsplit;
            return;
        }
    } else if (paged) {
        hipLaunchKernelGGL((decode_attn_pass1<T, CT, D, GQ, true>), grid1, dim3(256), 0, stream,
                           o_part.data_ptr<float>(), ml_part.data_ptr<float>(),
                           (const T*)q.data_ptr(), (const CT*)k_cache.data_ptr(),
                           (const CT*)v_cache.data_ptr(), seq_lens.data_ptr<int>(),
                           seq_ids.data_ptr<int>(), block_table->data_ptr<int>(),
                           scale, window, 0, Hkv, Sq, gq, Smax, chunk, nsplit,
                           block_size, max_blocks);
    } else {
        hipLaunchKernelGGL((decode_attn_pass1<T, CT, D, GQ, false>), grid1, dim3(256), 0, stream,
                           o_part.data_ptr<float>(), ml_part.data_ptr<float>(),
                           (const T*)q.data_ptr(), (const CT*)k_cache.data_ptr(),
                           (const CT*)v_cache.data_ptr(), seq_lens.data_ptr<int>(),
                           seq_ids.data_ptr<int>(), nullptr,
                           scale, window, ring, Hkv, Sq, gq, Smax, chunk, nsplit, 0, 0);
    }
    HIP_CHECK_KERNEL();
    constexpr int NG = 256 / (D / 4);
    const long rows = (long)B * Hq * Sq;
    int G = 1;
    while (G < nsplit && G < NG) G *= 2;
    dim3 grid2((unsigned)((rows + NG / G - 1) / (NG / G)));
    hipLaunchKernelGGL((decode_attn_pass2<T, D>), grid2, dim3(256), 0, stream,
                       (T*)out.data_ptr(), o_part.data_ptr<float>(),
                       ml_part.data_ptr<float>(), nsplit, G, rows, v_scale,
                       sinks ? sinks->data_ptr<float>() : nullptr, Hq, Sq,
                       lse_out ? lse_out->data_ptr<float>() : nullptr);
    HIP_CHECK_KERNEL();
}

template <typename T, int D>
static void dispatch_gq(torch::Tensor& out, const torch::Tensor& q,
                        const torch::Tensor& k_cache, const torch::Tensor& v_cache,
                        const torch::Tensor& seq_lens, const torch::Tensor& seq_ids,
                        float scale, int window, int gq,
                        const torch::Tensor* bt = nullptr, int bs = 0,
                        float v_scale = 1.0f, const torch::Tensor* sinks = nullptr,
                        torch::Tensor* lse_out = nullptr, int ring = 0,
                        DecodeShares* shares = nullptr) {
    const bool fp8 = k_cache.scalar_type() == at::ScalarType::Float8_e4m3fn;
    if constexpr (!std::is_same<T, float>::value && (D == 64 || D == 128)) {
        // the matrix-core kernel takes heads in columns: any ratio
        TORCH_CHECK(gq <= 8 || (bt == nullptr && lse_out == nullptr),
                    "GQA ratio > 8 not supported yet (got ", gq, ")");
        if (fp8)
            launch_decode<T, __hip_fp8_e4m3, D, 1>(out, q, k_cache, v_cache, seq_lens, seq_ids, scale,
                                                   window, gq, bt, bs, v_scale, sinks, lse_out, ring,
                                                   shares);
        else
            launch_decode<T, T, D, 1>(out, q, k_cache, v_cache, seq_lens, seq_ids, scale, window, gq,
                                      bt, bs, v_scale, sinks, lse_out, ring, shares);
        return;
    }
#define GQ_CASE(CT)                                                                     \
    do {                                                                                \
        if (gq <= 1)                                                                    \
            launch_decode<T, CT, D, 1>(out, q, k_cache, v_cache, seq_lens, seq_ids,     \
                                       scale, window, gq, bt, bs, v_scale, sinks,       \
                                       lse_out, ring);                                  \
        else if (gq <= 2)                                                               \
            launch_decode<T, CT, D, 2>(out, q, k_cache, v_cache, seq_lens, seq_ids,     \
                                       scale, window, gq, bt, bs, v_scale, sinks,       \
                                       lse_out, ring);                                  \
        else if (gq <= 4)                                                               \
            launch_decode<T, CT, D, 4>(out, q, k_cache, v_cache, seq_lens, seq_ids,     \
                                       scale, window, gq, bt, bs, v_scale, sinks,       \
                                       lse_out, ring);                                  \
        else if (gq <= 8)                                                               \
            launch_decode<T, CT, D, 8>(out, q, k_cache, v_cache, seq_lens, seq_ids,     \
                                       scale, window, gq, bt, bs, v_scale, sinks,       \
                                       lse_out, ring);                                  \
        else                                                                            \
            TORCH_CHECK(false, "GQA ratio > 8 not supported yet (got ", gq, ")");       \
    } while (0)
    if (fp8) {
        GQ_CASE(__hip_fp8_e4m3);
    } else {
        GQ_CASE(T);
    }
#undef GQ_CASE
}

void attention_decode_paged(torch::Tensor out, torch::Tensor q,
                            torch::Tensor k_cache, torch::Tensor v_cache,
                            torch::Tensor seq_lens, torch::Tensor block_table,
                            double scale, long window) {
    // paged cache (num_blocks, block_size, Hkv, D); `seq_lens` carries
    // per-query POSITIONS, shape (B, Sq)
    TORCH_CHECK(q.dim() == 4 && k_cache.dim() == 4, "bad shapes");
    TORCH_CHECK(seq_lens.numel() == q.size(0) * q.size(2),
                "positions must be (B, Sq)");
    const int D = q.size(3);
    const int Hq = q.size(1), Hkv = k_cache.size(2);
    const int bs = k_cache.size(1);
    TORCH_CHECK(Hq % Hkv == 0, "Hq must be a multiple of Hkv");
    const int gq = Hq / Hkv;
    auto seq_ids = seq_lens;  // unused in the paged path

#define CASE_P(T)                                                               \
    do {                                                                        \
        if (D == 128)                                                           \
            dispatch_gq<T, 128>(out, q, k_cache, v_cache, seq_lens, seq_ids,    \
                                (float)scale, (int)window, gq, &block_table, bs); \
        else if (D == 64)                                                       \
            dispatch_gq<T, 64>(out, q, k_cache, v_cache, seq_lens, seq_ids,     \
                               (float)scale, (int)window, gq, &block_table, bs); \
        else                                                                    \
            TORCH_CHECK(false, "paged decode: head_dim 64/128 only");           \
    } while (0)

    if (q.scalar_type() == at::ScalarType::BFloat16) {
        CASE_P(__hip_bfloat16);
    } else if (q.scalar_type() == at::ScalarType::Half) {
        CASE_P(__half);
    } else if (q.scalar_type() == at::ScalarType::Float) {
        CASE_P(float);
    } else {
        TORCH_CHECK(false, "attention_decode_paged: unsupported dtype");
    }
#undef CASE_P
}

void attention_decode(torch::Tensor out, torch::Tensor q,
                      torch::Tensor k_cache, torch::Tensor v_cache,
                      torch::Tensor seq_lens, torch::Tensor seq_ids,
                      double scale, long window,
                      c10::optional<torch::Tensor> sinks_opt,
                      c10::optional<torch::Tensor> lse_opt,
                      long ring) {
    // lse_opt: fp32 (B, Hq, Sq), filled with per-query log-sum-exp — the
    // cross-rank flash-decoding combine handle
    // `seq_lens` carries per-query POSITIONS, shape (B, Sq)
    TORCH_CHECK(q.dim() == 4 && k_cache.dim() == 4, "bad shapes");
    TORCH_CHECK(seq_lens.numel() == q.size(0) * q.size(2),
                "positions must be (B, Sq)");
    const int D = q.size(3);
    const int Hq = q.size(1), Hkv = k_cache.size(1);
    TORCH_CHECK(Hq % Hkv == 0, "Hq must be a multiple of Hkv");
    const int gq = Hq / Hkv;
    TORCH_CHECK(q.is_contiguous() && k_cache.is_contiguous() && v_cache.is_contiguous(),
                "contiguous tensors required");
    torch::Tensor sinks_t;
    const torch::Tensor* sinks = nullptr;
    if (sinks_opt.has_value()) {
        sinks_t = sinks_opt->to(torch::kFloat32).contiguous();
        sinks = &sinks_t;
    }
    torch::Tensor* lse_ptr = nullptr;
    torch::Tensor lse_t;
    if (lse_opt.has_value()) {
        lse_t = *lse_opt;
        TORCH_CHECK(lse_t.scalar_type() == torch::kFloat32 &&
                    lse_t.numel() == (long)q.size(0) * Hq * q.size(2),
                    "lse must be fp32 (B,Hq,Sq)");
        lse_ptr = &lse_t;
    }

#define CASE_T(T)                                                               \
    do {                                                                        \
        if (D == 128)                                                           \
            dispatch_gq<T, 128>(out, q, k_cache, v_cache, seq_lens, seq_ids,    \
                                (float)scale, (int)window, gq, nullptr, 0,      \
                                1.0f, sinks, lse_ptr, (int)ring);               \
        else if (D == 64)                                                       \
            dispatch_gq<T, 64>(out, q, k_cache, v_cache, seq_lens, seq_ids,     \
                               (float)scale, (int)window, gq, nullptr, 0,       \
                               1.0f, sinks, lse_ptr, (int)ring);                \
        else if (D == 32)                                                       \
            dispatch_gq<T, 32>(out, q, k_cache, v_cache, seq_lens, seq_ids,     \
                               (float)scale, (int)window, gq, nullptr, 0,       \
                               1.0f, sinks, lse_ptr, (int)ring);                \
        else if (D == 256)                                                      \
            dispatch_gq<T, 256>(out, q, k_cache, v_cache, seq_lens, seq_ids,    \
                                (float)scale, (int)window, gq, nullptr, 0,      \
                                1.0f, sinks, lse_ptr, (int)ring);               \
        else                                                                    \
            TORCH_CHECK(false, "head_dim must be 32/64/128/256, got ", D);      \
    } while (0)

    if (q.scalar_type() == at::ScalarType::BFloat16) {
        CASE_T(__hip_bfloat16);
    } else if (q.scalar_type() == at::ScalarType::Half) {
        CASE_T(__half);
    } else if (q.scalar_type() == at::ScalarType::Float) {
        CASE_T(float);
    } else {
        TORCH_CHECK(false, "attention_decode: unsupported dtype");
    }
#undef CASE_T
}

torch::Tensor tile_gemm(torch::Tensor x, torch::Tensor w, c10::optional<torch::Tensor> bias,
                        long splits, bool parts, long glu);
long tile_gemm_splits(long M, long N, long K, long glu, bool whole);
torch::Tensor shares_gemm(const torch::Tensor& o, const torch::Tensor& ml, long n, const torch::Tensor& w);

// Values of all shares that a workgroup of the product adds up, at most: 256 workgroups read theirs from
// the L2 where the kernel before would read each once. Both kernels / one, us: 6 shares of 256 (32 heads
// of 64, context 700) 11.8 / 10.0, 6 of 1024 (32 heads of 128) 16.6 / 15.6, 16 of 256 14.1 / 13.6, but 32
// of 1024 (context 8000) 22.1 / 23.5 and 36.4 / 42.1 (64 heads).
constexpr long DECODE_SHARES = 8192;

// attention_decode of one token of one row (16 bits, heads of 64 or 128) and the product with w
// (N, Hq * D): as tile_gemm leaves it, its parts of K or the result.
torch::Tensor attention_decode_product(torch::Tensor q, torch::Tensor k_cache, torch::Tensor v_cache,
                                       torch::Tensor positions, torch::Tensor seq_ids, double scale,
                                       long window, torch::Tensor w) {
    TORCH_CHECK(q.dim() == 4 && k_cache.dim() == 4 && q.size(0) == 1 && q.size(2) == 1 &&
                positions.numel() == 1, "attention_decode_product: one token of one row");
    const int D = q.size(3), Hq = q.size(1), Hkv = k_cache.size(1);
    TORCH_CHECK((D == 64 || D == 128) && Hq % Hkv == 0 && w.dim() == 2 && w.size(1) == (long)Hq * D &&
                w.scalar_type() == q.scalar_type(), "attention_decode_product: shapes and types");
    TORCH_CHECK(q.is_contiguous() && k_cache.is_contiguous() && v_cache.is_contiguous(),
                "contiguous tensors required");
    torch::Tensor out = torch::empty_like(q);
    const long splits = tile_gemm_splits(1, w.size(0), w.size(1), 0, false);
    TORCH_CHECK(splits > 0, "attention_decode_product: product not taken");
    DecodeShares shares;
    shares.most = DECODE_SHARES / ((w.size(1) / 64 + splits - 1) / splits * 64);
#define ADP(T, DD)                                                                                 \
    dispatch_gq<T, DD>(out, q, k_cache, v_cache, positions, seq_ids, (float)scale, (int)window,    \
                       Hq / Hkv, nullptr, 0, 1.0f, nullptr, nullptr, 0, &shares)
    if (q.scalar_type() == at::ScalarType::BFloat16) {
        if (D == 128) ADP(__hip_bfloat16, 128);
        else ADP(__hip_bfloat16, 64);
    } else {
        TORCH_CHECK(q.scalar_type() == at::ScalarType::Half, "attention_decode_product: 16 bits");
        if (D == 128) ADP(__half, 128);
        else ADP(__half, 64);
    }
#undef ADP
    if (shares.n > 1) return shares_gemm(shares.o, shares.ml, shares.n, w);
    return tile_gemm(out.view({1, (long)Hq * D}), w, c10::nullopt, 0, true, 0);
}
