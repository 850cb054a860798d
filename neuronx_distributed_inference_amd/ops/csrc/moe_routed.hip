// Routed experts of a MoE layer, from the router's choice to the layer's output, in four
// launches: a table of row tiles, gate and up projection with the gated activation, down
// projection, weighted sum of each token's experts.
//
// Bounds: with few rows an expert the weight stream (every chosen expert's weights once from
// HBM); with many the matrix cores, and before those the LDS (128 B/clk a CU).
//
//   * Workgroup = 8 waves, MT rows of one expert x 256 columns. K goes in steps of 128 B of a
//     weight row (128 deep with 8-bit weights, and then 64 rows at most) through a ring of three
//     or four LDS buffers (as many as 160 KB hold), global_load_lds throughout, one raw barrier a
//     step and a counted vmcnt: all but one of the buffers are in flight.
//   * A second row tile of an expert reads its weights again (from the L2 at best) and adds a
//     round of workgroups, so the height goes by the rows an expert has by chance and not only on
//     average: 2048 tokens x 8 of 128 experts (128 rows +- 11) take 128 tiles of 160 rows, and
//     would take 190 of 128.
//   * The last round of workgroups, where it would fill half of the chip or less, takes its tiles in
//     halves of 128 columns, in rings of their own: a token of 8 of 128 experts (48 tiles)
//     42 -> 31 us with its table and sum, 128 tokens of 8 experts in 16 bits (3 1/2 rounds) 467 ->
//     453, 512 in 8 bits 630 -> 592. More than half of the chip's tiles stay whole: their halves would be
//     a round more.
//   * An expert's weights that no other row tile wants come past the caches: at 2048 tokens of 128
//     experts 347 -> 317 us, 64 tokens 221 -> 198; 128 tokens of 8 experts in 16 bits 515 -> 467, in
//     8 bits 281 -> 264. Where another wants them they are shared in the L2 (1024 tokens of 8 experts
//     with all past it 935 -> 980). The tallest tiles of more choices than one holds for each expert are
//     bound by the matrix cores, and there the question itself costs 1 to 2 %: a kernel without it.
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
//   * Down projections of few tiles (8 experts x 16 column tiles leave half of the CUs without
//     one) are shared out by steps: 256 workgroups take equal runs of the list's steps, across
//     tiles, their loads running on into the next tile, and leave a part for each tile they
//     touch; the kernel that adds up the choices adds the parts as well. 8 experts of 14336 x
//     4096 in 8 bits, 32 rows each: 122 -> 89 us (5.3 TB/s). Runs of whole tiles for all
//     products (a workgroup a CU) gained nothing where there are many: 360 and 353 us at 2048
//     tokens of 128 experts, 3206 and 3307 for 4096 tokens of 8.
//
// The layer's products with their table and sum in us, tiles of 32, 64 and 128 rows in a ring of
// three, all in step and through the caches -> now:
//   128 experts of 2048 x 768, 8 a token:  64 tokens 228 -> 199, 1024 300 -> 255, 2048 410 -> 313,
//     3000 487 -> 459, 4096 610 -> 521
//   8 experts of 4096 x 14336, 2 a token:  16 tokens 558 -> 434, 128 586 -> 453, 256 630 -> 475,
//     1024 1115 -> 917, 2048 1700;  in 8 bits 16 tokens 305 -> 226, 128 320 -> 262, 200 349 -> 279,
//     256 400 -> 378
// Row tiles there (rows an expert on average: times of tiles of 32, 64, 96, 128, 160 rows):
//   128 experts  32: 261 228 232 238 245;  64: 359 297 252 263 264;  128: 565 425 400 380 322;
//     188: 741 544 485 476 509;  256: 990 693 587 575 532
//   8 experts in 8 bits (32, 48, 64 rows)  4: 241 242 240;  32: 295 261 268;  40: 339 288 285;
//     50: 362 369 284;  64: 462 398 388

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

// The same, past the caches where `once` (the same for the wave). The branch is hidden from the
// compiler, which would double the tallest tiles' registers for it: 317 -> 362 us at 2048 tokens of 128
// experts.
DEV_INLINE void mr_load_lds_once(const char* src, unsigned dst, int once) {
    const unsigned at = __builtin_amdgcn_readfirstlane(dst);
    once = __builtin_amdgcn_readfirstlane(once);
    asm volatile("s_mov_b32 m0, %0\n\t"
                 "s_cmp_lg_u32 %2, 0\n\t"
                 "s_cbranch_scc1 1f\n\t"
                 "global_load_lds_dwordx4 %1, off\n\t"
                 "s_branch 2f\n"
                 "1:\n\t"
                 "global_load_lds_dwordx4 %1, off nt\n"
                 "2:"
                 :: "s"(at), "v"(src), "s"(once) : "memory", "m0", "scc");
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

// HALF: a tile of half the columns
template <bool F8, int MT, bool HALF>
struct MrTile {
    static constexpr int BN = HALF ? 128 : 256;
    static constexpr int BK = F8 ? 128 : 64;          // 128 B of a weight row
    static constexpr int XH = BK / 64;                // 128 B images of x a step
    static constexpr int WM = HALF || MT >= 96 ? 2 : 1;       // waves along the rows
    static constexpr int WN = 8 / WM;
    static constexpr int MI = (MT / 16 + WM - 1) / WM;
    static constexpr int NI = BN / WN / 16;
    static constexpr int XB = XH * MT * 128;
    static constexpr int STEP = XB + BN * 128;        // bytes of a ring buffer
    static constexpr int D = STEP * 4 <= 163840 ? 4 : 3;
    static_assert(STEP * D <= 163840, "the ring does not fit");
};

typedef const __attribute__((address_space(4))) int* mr_table;     // read by scalar loads
constexpr int MR_WGS = 256;          // workgroups of a launch at most: one a CU
constexpr int MR_GRP = 8;            // row tiles of a group

// Where a launch's workgroups stop inside tiles, and not only at their ends (see the top): tiles
// that fill the last round of the chip badly, with 8 steps or more for every workgroup.
// Shares of one expert's row tiles read its weights at different times, whole tiles together, so
// that up to half of a round gains however its rows lie (8 experts of 8192 x 2048 in 8 bits, 400
// tokens, 16 tiles 170 -> 147 us), and more than that only where few experts have a second tile
// (`crowded`) and the shares are long: 8 of 14336 x 4096 in 16 bits, 128 rows each 639 -> 561, 10
// tiles 606 -> 594, but 13 tiles 666 -> 709, 11 of 96 rows 637 -> 649; 4 of 8192 x 4096, 12 tiles
// 294 -> 368; 64 of 1408 x 2048, 4 tokens (16 steps a workgroup) 82.5 -> 86.7.
constexpr int MR_CROWDED = 1 << 30;  // in tiles[0]: an eighth more row tiles than experts with rows
DEV_INLINE bool mr_shares(const int total, const int nk, const bool crowded) {
    const int rounds = (total + MR_WGS - 1) / MR_WGS;
    if (rounds > 2 || total * 100 >= rounds * MR_WGS * 85 || total * nk < MR_WGS * 8) return false;
    return total <= MR_WGS / 2 || (!crowded && total * nk >= MR_WGS * 16);
}

struct MrArgs {
    void* y;
    const void* x;
    const char *w0, *w1;
    const float *s0, *s1;
    const int *tiles, *gather;
    int N, K, col0, ncols, ntn, gelu;
};

// A tile of the list (of its columns, the half `side`), or with `share` workgroup wg's `left` steps
// from step k0 of tile li0 on.
template <typename T, bool F8, bool GLU, int MT, bool ONCE, bool HALF>
DEV_INLINE void mr_work(const MrArgs& a_, const int nreal, const bool share, const int wg, const int li0,
                        const int k0, int left, const int side) {
    using MF = MrMfma<T>;
    using vec8 = typename MF::vec8;
    using C = MrTile<F8, MT, HALF>;
    constexpr int MI = C::MI, NI = C::NI, XH = C::XH, D = C::D;
    constexpr int BNO = (GLU ? 128 : 256);            // output columns of a tile
    constexpr int WP = C::BN / 64;                    // 1 KB pieces of W a wave stages
    constexpr int XP = XH * MT / 8;                   // pieces of x in all: a wave takes every 8th
    constexpr int XW = (XP + 7) / 8;
    constexpr int ES = F8 ? 1 : 2;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    void* __restrict__ const y = a_.y;
    const T* __restrict__ const x = (const T*)a_.x;
    const char* __restrict__ const w0 = a_.w0;
    const char* __restrict__ const w1 = a_.w1;
    const float* __restrict__ const s0 = a_.s0;
    const float* __restrict__ const s1 = a_.s1;
    const int N = a_.N, K = a_.K, col0 = a_.col0, ncols = a_.ncols, ntn = a_.ntn, gelu = a_.gelu;
    mr_table tiles = (mr_table)(size_t)a_.tiles, gather = (mr_table)(size_t)a_.gather;
    const int nk = K / C::BK;

    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wid / C::WN, wn = wid % C::WN;     // fragments wm, wm + WM, ... of the rows
    const int lrow = lane & 15, ls = lane >> 4, prow = lane >> 3;
    const int pslot = (lane & 7) ^ prow;              // source side of the XOR swizzle
    const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) char*)smem;

    // tile of the list -> row tile, first column (of the slab)
    auto place = [&](int li, int& rt, int& n0) {
        const int grp = li / (MR_GRP * ntn), rows_grp = min(MR_GRP, nreal - grp * MR_GRP);
        const int in = li - grp * MR_GRP * ntn;
        rt = grp * MR_GRP + in % rows_grp;
        n0 = (in / rows_grp) * BNO + (HALF ? side * (BNO / 2) : 0);
    };

    // ---- loads: a cursor that runs ahead of the products, into the next tile too ----
    int s_li = li0, s_k = k0, s_left = left;
    const char* xsrc[XW];
    const char* wsrc[WP];
    int once = 0;                                     // no other row tile has these weights
    auto sources = [&]() {
        int rt, n0;
        place(s_li, rt, n0);
        const int e = tiles[1 + 2 * rt], rows = tiles[2 + 2 * rt];
        const int m0 = rt * MT;
        if constexpr (ONCE) {                         // (without branches, as in mr_load_lds_once)
            const int before = max(rt - 1, 0), after = min(rt + 1, nreal - 1);
            once = !((int)(before != rt) & (int)(tiles[1 + 2 * before] == e) |
                     (int)(after != rt) & (int)(tiles[1 + 2 * after] == e));
        }
        // Whole tiles start at different steps and wrap round: in step they would all ask for the
        // same 128 bytes of rows a power of two apart, which few of the memory channels hold
        // (8 experts in 16 bits, 32 rows each: 516 -> 501 us; 2048 tokens of 128: 0.87 -> 0.85 of
        // the time before; in 8 bits the same). Row tiles of the same weights keep together.
        if (!share) s_k = (e * ntn + n0 / BNO) % nk;
#pragma unroll
        for (int i = 0; i < XW; ++i) {
            const int piece = min(wid + 8 * i, XP - 1), img = piece / (MT / 8);
            const int r0 = (piece % (MT / 8)) * 8;
            long src = m0 + r0 + prow;
            if (GLU && gather) {                      // rows past the end repeat the first token
                int id = 0;
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const int g = gather[m0 + r0 + q];
                    id = prow == q ? g : id;
                }
                src = r0 + prow < rows ? id : 0;
            }
            xsrc[i] = reinterpret_cast<const char*>(x + src * K) + img * 128 + pslot * 16;
        }
#pragma unroll
        for (int i = 0; i < WP; ++i) {
            const int r = (wid * WP + i) * 8 + prow;
            const bool up = GLU && r >= C::BN / 2;
            const int n = min(col0 + n0 + (up ? r - C::BN / 2 : r), N - 1);
            wsrc[i] = (up ? w1 : w0) + ((long)e * N + n) * K * ES + pslot * 16;
        }
    };
    const bool more = wid < XP % 8;                   // this wave loads a piece of x more
    auto stage = [&](unsigned buf) {
        const unsigned xd = lds0 + buf + wid * 1024, wd = lds0 + buf + C::XB + wid * (WP * 1024);
#pragma unroll
        for (int i = 0; i < XP / 8; ++i) mr_load_lds(xsrc[i] + s_k * (C::BK * 2), xd + i * 8192);
        if (XP % 8 && more) mr_load_lds(xsrc[XW - 1] + s_k * (C::BK * 2), xd + (XW - 1) * 8192);
#pragma unroll
        for (int i = 0; i < WP; ++i) {
            if constexpr (ONCE) mr_load_lds_once(wsrc[i] + s_k * 128, wd + i * 1024, once);
            else mr_load_lds(wsrc[i] + s_k * 128, wd + i * 1024);
        }
        --s_left;
        if (++s_k == nk) {
            s_k = 0;
            if (share) {
                ++s_li;
                if (s_left > 0) sources();
            }
        }
    };
    // wait until at most n steps of this wave's loads are in flight
    auto wait_steps = [&](int n) {
        constexpr int L0 = WP + XP / 8, L1 = L0 + 1;
        if (D > 3 && n >= 2) {
            if (XP % 8 && more) mr_vm_wait<2 * L1>();
            else mr_vm_wait<2 * L0>();
        } else if (n >= 1) {
            if (XP % 8 && more) mr_vm_wait<L1>();
            else mr_vm_wait<L0>();
        } else {
            mr_vm_wait<0>();
        }
    };

    mr_f32x4 acc[MI][NI];
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NI; ++j) acc[i][j] = {0.f, 0.f, 0.f, 0.f};
    };
    // row of W's image that fragment j of this wave starts at: with GLU the first half of the
    // fragments are gate columns, the second the same up columns
    auto wrow = [&](int j) {
        constexpr int NH = NI / 2;
        return GLU ? (j / NH) * (C::BN / 2) + (wn * NH + j % NH) * 16 : (wn * NI + j) * 16;
    };
    auto compute = [&](unsigned buf, auto frags) {
        constexpr int MF_ = decltype(frags)::value;
        const char* xb = smem + buf + (wm * 16 + lrow) * 128;
        const char* wb = smem + buf + C::XB + lrow * 128;
#pragma unroll
        for (int kq = 0; kq < C::BK / 32; ++kq) {
            vec8 a[MF_], b[NI];
            const int sx = ((kq & 1) * 4 + ls) ^ (lrow & 7);
#pragma unroll
            for (int i = 0; i < MF_; ++i)
                a[i] = *reinterpret_cast<const vec8*>(xb + (kq >> 1) * (MT * 128) +
                                                      i * (C::WM * 2048) + sx * 16);
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
            for (int i = 0; i < MF_; ++i)
#pragma unroll
                for (int j = 0; j < NI; ++j) acc[i][j] = MF::mfma(b[j], a[i], acc[i][j]);
            // (all halves' fragments at once would not fit the registers)
            if constexpr (MI * NI > 16) __builtin_amdgcn_sched_barrier(0);
        }
    };

    // ---- products: the cursor of the tile at hand ----
    int li = li0, k = k0, rt, n0, rows;
    auto enter = [&]() {
        place(li, rt, n0);
        rows = tiles[2 + 2 * rt];
        clear();
    };
    enter();
    sources();
    int staged = 0;
    unsigned cur = 0, nxt = 0;
    for (; staged < D - 1 && s_left > 0; ++staged) {
        stage(nxt);
        nxt += C::STEP;
    }
    for (;;) {
        const int steps = min(nk - k, left);
        // a loop of its own for the tiles where a wave has rows in half of its fragments at most:
        // with both in one loop the accumulators are copied at every step
        auto run = [&](auto frags) {
            for (int i = 0; i < steps; ++i) {
                // `staged` steps are on the way or there, the oldest is the one at hand
                wait_steps(staged - 1);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                // the buffer computed in the turn before is free
                if (s_left > 0) {
                    stage(nxt);
                    nxt = nxt == (D - 1) * C::STEP ? 0 : nxt + C::STEP;
                } else {
                    --staged;
                }
                compute(cur, frags);
                cur = cur == (D - 1) * C::STEP ? 0 : cur + C::STEP;
            }
        };
        constexpr int FEW = (MI + 1) / 2;
        if (rows > (FEW * C::WM + wm) * 16) run(std::integral_constant<int, MI>{});
        else run(std::integral_constant<int, FEW>{});
        left -= steps;

        // ---- the tile, or this workgroup's share of it, is done ----
        constexpr int NO = GLU ? NI / 2 : NI;
        const long m0 = share ? (long)(wg + li) * MT : (long)rt * MT;
        const int pitch = share ? C::BN : ncols;
        const int e = tiles[1 + 2 * rt];
        int row = wm * 16 + lrow;
        asm volatile("" : "+v"(row));     // not hoisted: addresses would not fit the registers
#pragma unroll
        for (int j = 0; j < NO; ++j) {
            const int ct = (wn * NO + j) * 16 + ls * 4, c = n0 + ct;     // column of the slab
            if (c >= ncols) continue;
            mr_f32x4 sg = {1.f, 1.f, 1.f, 1.f}, su = sg;
            if constexpr (F8) {
                sg = *reinterpret_cast<const mr_f32x4*>(s0 + (long)e * N + col0 + c);
                if (GLU) su = *reinterpret_cast<const mr_f32x4*>(s1 + (long)e * N + col0 + c);
            }
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                const int m = i * (C::WM * 16) + row;
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
                    *reinterpret_cast<mr_f32x4*>(reinterpret_cast<float*>(y) + (m0 + m) * pitch +
                                                 (share ? ct : c)) = v;
                }
            }
        }
        if (GLU || left == 0) break;
        // the scales' loads end here, for the compiler too: it would wait for them, and with them
        // for all loads in flight, at every step
        if constexpr (F8) __builtin_amdgcn_s_waitcnt(0x0f70);     // vmcnt(0)
        k = 0;
        ++li;
        enter();
    }
}

template <typename T, bool F8, bool GLU, int MT, bool ONCE>
__global__ void __launch_bounds__(512, 2)
moe_routed_kernel(const MrArgs a, const int can_share) {
    const int head = ((mr_table)(size_t)a.tiles)[0], nreal = head & (MR_CROWDED - 1);
    const int total = nreal * a.ntn, nk = a.K / MrTile<F8, MT, false>::BK;
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    // the workgroup's part of the list; every exit is uniform over the workgroup
    if (!GLU && can_share && mr_shares(total, nk, head & MR_CROWDED)) {
        if (slot >= MR_WGS / 8) return;
        const int wg = xcd * (MR_WGS / 8) + slot;
        const long all = (long)total * nk;
        const int from = (int)(wg * all / MR_WGS), left = (int)((wg + 1) * all / MR_WGS) - from;
        if (left)
            mr_work<T, F8, GLU, MT, ONCE, false>(a, nreal, true, wg, from / nk, from % nk, left, 0);
        return;
    }
    const int rest = total % MR_WGS, halved = rest <= MR_WGS / 2 ? rest : 0, whole = total - halved;
    const int per = (whole + 7) >> 3, per_half = (2 * halved + 7) >> 3;
    if (slot < per) {
        const int li = xcd * per + slot;
        if (li < whole) mr_work<T, F8, GLU, MT, ONCE, false>(a, nreal, false, 0, li, 0, nk, 0);
    } else if (slot < per + per_half) {
        const int h = xcd * per_half + slot - per;
        if (h < 2 * halved)
            mr_work<T, F8, GLU, MT, ONCE, true>(a, nreal, false, 0, whole + (h >> 1), 0, nk, h & 1);
    }
}

// out[t, col0 + c] = sum over the token's choices of weight * y[row of the choice, c]. Where the
// products' workgroups stop inside tiles (share_tile: rows of one), workgroup w's share of tile li
// is a tile of 256 columns at w + li, and a row is the sum of its tile's shares in their order.
template <typename T, int TOPK>
__global__ void __launch_bounds__(256)
moe_routed_sum_kernel(T* __restrict__ out, const float* __restrict__ y,
                      const int* __restrict__ inv, const float* __restrict__ weights,
                      const int* __restrict__ tiles, const int ntok, const int topk, const int N,
                      const int col0, const int ncols, const int ntn, const int nk,
                      const int share_tile) {
    const int per = ncols / 8;
    const long id = (long)blockIdx.x * 256 + threadIdx.x;
    if (id >= (long)ntok * per) return;
    const int t = (int)(id / per), c = (int)(id % per) * 8;
    const int k = TOPK ? TOPK : topk;
    const int head = tiles[0], nreal = head & (MR_CROWDED - 1), total = nreal * ntn;
    const bool share = share_tile && mr_shares(total, nk, head & MR_CROWDED);
    float v[8] = {};
    auto add = [&](int row, float wt, float4 a, float4 b) {
        if (row < 0) a = b = float4{0.f, 0.f, 0.f, 0.f};     // another rank's expert
        v[0] += a.x * wt; v[1] += a.y * wt; v[2] += a.z * wt; v[3] += a.w * wt;
        v[4] += b.x * wt; v[5] += b.y * wt; v[6] += b.z * wt; v[7] += b.w * wt;
    };
    if (!share) {                      // (a loop of its own: all choices' loads go out together)
#pragma unroll
        for (int j = 0; j < k; ++j) {
            const int row = inv[(long)t * k + j];
            const float wt = weights ? weights[(long)t * k + j] : 1.f;
            const float* p = y + (long)max(row, 0) * ncols + c;
            add(row, wt, *reinterpret_cast<const float4*>(p), *reinterpret_cast<const float4*>(p + 4));
        }
    } else {
#pragma unroll
        for (int j = 0; j < k; ++j) {
            const int row = inv[(long)t * k + j];
            const float wt = weights ? weights[(long)t * k + j] : 1.f;
            const int rt = max(row, 0) / share_tile, grp = rt / MR_GRP;
            const int rows_grp = min(MR_GRP, nreal - grp * MR_GRP);
            const int li = grp * MR_GRP * ntn + (c >> 8) * rows_grp + rt % MR_GRP;
            const long all = (long)total * nk, s0 = (long)li * nk;
            const int w0 = (int)(((s0 + 1) * MR_WGS - 1) / all);
            const int n = (int)(((s0 + nk) * MR_WGS - 1) / all) - w0 + 1;
            const long step = (long)share_tile * 256;
            const float* p = y + (w0 + li) * step + (max(row, 0) % share_tile) * 256 + (c & 255);
            float4 a = *reinterpret_cast<const float4*>(p);
            float4 b = *reinterpret_cast<const float4*>(p + 4);
            for (int i = 1; i < n; ++i) {
                p += step;
                const float4 a1 = *reinterpret_cast<const float4*>(p);
                const float4 b1 = *reinterpret_cast<const float4*>(p + 4);
                a.x += a1.x; a.y += a1.y; a.z += a1.z; a.w += a1.w;
                b.x += b1.x; b.y += b1.y; b.z += b1.z; b.w += b1.w;
            }
            add(row, wt, a, b);
        }
    }
    Vec8<T> o;
#pragma unroll
    for (int i = 0; i < 8; ++i) o.v[i] = VecTraits<T>::from_float(v[i]);
    store_vec8(out + (long)t * N + col0 + c, o);
}

DEV_INLINE int mr_wave_sum(int x) {    // of a wave's values, in every lane, by DPP
#define MR_STEP(CTRL, ROWS) x += __builtin_amdgcn_update_dpp(0, x, CTRL, ROWS, 0xf, false)
    MR_STEP(0x111, 0xf);               // row_shr 1, 2, 4, 8
    MR_STEP(0x112, 0xf);
    MR_STEP(0x114, 0xf);
    MR_STEP(0x118, 0xf);
    MR_STEP(0x142, 0xa);               // row_bcast 15, 31
    MR_STEP(0x143, 0xc);
#undef MR_STEP
    return __builtin_amdgcn_readlane(x, 63);
}

// The table: tiles[0] = number of row tiles (and MR_CROWDED), then (expert, rows) of each; gather =
// token of a tile row (padding rows stay unwritten: readers go by `rows`); inv = tile row of a
// choice, or -1 where the expert is not one of the El from `first`. Rows of an expert stand in the
// order of their choices, so that a row's tile, and the shares that its sum is made of, are the
// same in every run. A workgroup an expert: all of them count all choices (LDS atomics), which spares a
// launch and a wait between counts and rows, and each ranks its own by ballots, its 16 waves a
// run of the choices each. 16384 choices of 128 experts: 20 us by one workgroup (rows in any
// order), 11 now. Few choices wait for one load after the other: 4 waves, and what the first pass
// read stays in registers (2 and 128 choices of 8 experts 4.3 and 4.6 -> 3.4 and 3.7 us).
template <typename I>
__global__ void __launch_bounds__(1024)
moe_route_kernel(int* __restrict__ tiles, int* __restrict__ gather, int* __restrict__ inv,
                 const I* __restrict__ idx, const int n, const int El, const long first,
                 const int topk, const int mt) {
    extern __shared__ int count[];                    // [El]
    __shared__ int s_mine[16];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, own = blockIdx.x;
    const int nw = blockDim.x >> 6;
    for (int e = threadIdx.x; e < El; e += blockDim.x) count[e] = 0;
    const int run = ((n + nw - 1) / nw + 63) / 64 * 64, lo = wid * run, hi = min(n, lo + run);
    int mine = 0, e[8];                               // -1: not one of the El, -2: past the end
    // eight loads at a time: what the kernel waits for
    auto load = [&](int i0) {
        long v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = (long)idx[min(i0 + u * 64 + lane, n - 1)] - first;
#pragma unroll
        for (int u = 0; u < 8; ++u)
            e[u] = i0 + u * 64 + lane >= hi ? -2 : v[u] >= 0 && v[u] < El ? (int)v[u] : -1;
    };
    if (lo < hi) load(lo);
    __syncthreads();
    for (int i0 = lo; i0 < hi; i0 += 512) {
        if (i0 != lo) load(i0);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            if (e[u] >= 0) atomicAdd(&count[e[u]], 1);
            mine += __popcll(__ballot(e[u] == own));
        }
    }
    if (lane == 0) s_mine[wid] = mine;
    __syncthreads();
    int before = 0, all = 0, used = 0;                // tiles of the experts before, of all; experts
    for (int x = lane; x < El; x += 64) {             // (each wave by itself)
        const int nt = (count[x] + mt - 1) / mt;
        all += nt;
        before += x < own ? nt : 0;
        used += nt > 0;
    }
    const int start = mr_wave_sum(before);
    int row = 0;
    for (int w = 0; w < wid; ++w) row += s_mine[w];
    const int c = count[own];
    for (int j = threadIdx.x; j * mt < c; j += blockDim.x) {
        tiles[1 + 2 * (start + j)] = own;
        tiles[2 + 2 * (start + j)] = min(mt, c - j * mt);
    }
    if (own == 0 && wid == 0) {
        all = mr_wave_sum(all);
        used = mr_wave_sum(used);
        if (lane == 0) tiles[0] = all | ((long)all * 8 >= (long)used * 9 ? MR_CROWDED : 0);
    }
    row += start * mt;
    for (int i0 = lo; i0 < hi; i0 += 512) {
        if (run > 512) load(i0);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = i0 + u * 64 + lane;
            const bool is = e[u] == own;
            const unsigned long long m = __ballot(is);
            if (is) {
                const int at = row + __popcll(m & ((1ull << lane) - 1));
                gather[at] = i / topk;
                inv[i] = at;
            } else if (own == 0 && e[u] == -1) {
                inv[i] = -1;
            }
            row += __popcll(m);
        }
    }
}

template <typename T, bool F8, bool GLU, int MT, bool ONCE = true>
void mr_launch(void* y, const torch::Tensor& x, const torch::Tensor& w0, const torch::Tensor& w1,
               const float* s0, const float* s1, const torch::Tensor& tiles, const int* gather,
               int max_tiles, int col0, int ncols, int gelu, int share, hipStream_t st) {
    using C = MrTile<F8, MT, false>;
    using H = MrTile<F8, MT, true>;
    constexpr int LDS = std::max(C::D * C::STEP, H::D * H::STEP), BNO = GLU ? C::BN / 2 : C::BN;
    // a limit of the function, the same in every call
    (void)hipFuncSetAttribute((const void*)moe_routed_kernel<T, F8, GLU, MT, ONCE>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    const int ntn = (ncols + BNO - 1) / BNO;
    TORCH_CHECK((long)max_tiles * ntn < (1L << 30), "moe_routed: too many tiles");
    // a workgroup a tile, up to half of MR_WGS more for those in halves, and what rounding eighths up
    // takes; shares need all MR_WGS, whatever the table turns out to hold
    const long units = (long)max_tiles * ntn + std::min((long)max_tiles * ntn, MR_WGS / 2L) + 14;
    const long grid = std::max(share ? (long)MR_WGS : 0, (units + 7) / 8 * 8);
    const MrArgs a{y, x.data_ptr(), (const char*)w0.data_ptr(), (const char*)w1.data_ptr(), s0, s1,
                   tiles.data_ptr<int>(), gather, (int)w0.size(1), (int)w0.size(2), col0, ncols, ntn,
                   gelu};
    hipLaunchKernelGGL((moe_routed_kernel<T, F8, GLU, MT, ONCE>), dim3((unsigned)grid), dim3(512),
                       LDS, st, a, share);
    HIP_CHECK_KERNEL();
}

template <bool GLU>
void mr_dispatch(void* y, const torch::Tensor& x, const torch::Tensor& w0,
                 const torch::Tensor& w1, const float* s0, const float* s1,
                 const torch::Tensor& tiles, const int* gather, int mt, int col0, int ncols,
                 int gelu, int share) {
    const int max_tiles = (int)((tiles.numel() - 1) / 2);
    auto st = at::hip::getCurrentHIPStream();
    const bool f8 = s0 != nullptr, bf = x.scalar_type() == at::ScalarType::BFloat16;
    // more choices than a tile holds for each expert: hardly one has its weights to itself
    const bool many = max_tiles > 2 * w0.size(0);
#define MR(TT, FF, ...) mr_launch<TT, FF, GLU, __VA_ARGS__>(y, x, w0, w1, s0, s1, tiles, gather,  \
                                                            max_tiles, col0, ncols, gelu, share, st)
#define MR_M(TT)                                                                                  \
    do {                                                                                          \
        if (f8 && mt == 64) MR(TT, true, 64);                                                     \
        else if (f8 && mt == 48) MR(TT, true, 48);                                                \
        else if (f8) MR(TT, true, 32);                                                            \
        else if (mt == 160 && many) MR(TT, false, 160, false);                                    \
        else if (mt == 160) MR(TT, false, 160);                                                   \
        else if (mt == 128) MR(TT, false, 128);                                                   \
        else if (mt == 96) MR(TT, false, 96);                                                     \
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
    TORCH_CHECK(mt == 32 || mt == 64 || (s.has_value() ? mt == 48
                                                       : mt == 96 || mt == 128 || mt == 160),
                "moe_routed: mt must be 32, 64, with 8-bit weights 48, with 16-bit 96, 128, 160");
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
    const int lds = (int)num_local * 4;
    // runs of 512 choices are read once (see the kernel): 4 waves for up to four of them
    const int threads = n <= 2048 ? 256 : 1024;
#define MR_ROUTE(I) hipLaunchKernelGGL(moe_route_kernel<I>, dim3((unsigned)num_local), dim3(threads), lds, st,      \
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
                      (int)w_gate.size(1), (int)gelu, 0);
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
    const int nk = (int)(w_down.size(2) / (s_down.has_value() ? 128 : 64));
    // shares: of at most 2 * MR_WGS tiles (mr_shares); workgroup w's of tile li stands at w + li,
    // so that there are fewer than tiles and workgroups together
    const long most = std::min(2L * MR_WGS, (tiles.numel() - 1) / 2 * ((N + 255) / 256));
    const bool share = slab == N && ws.numel() >= (MR_WGS + most) * mt * 256;
    auto st = at::hip::getCurrentHIPStream();
    for (long c = 0; c < N; c += slab) {
        const int nc = (int)std::min(slab, N - c);
        mr_dispatch<false>(ws.data_ptr(), h, w_down, w_down,
                           s_down ? s_down->data_ptr<float>() : nullptr, nullptr, tiles, nullptr,
                           (int)mt, (int)c, nc, 0, share);
        const long blocks = (T * (nc / 8) + 255) / 256;
#define MR_SUM(TT, KK) hipLaunchKernelGGL((moe_routed_sum_kernel<TT, KK>), dim3((unsigned)blocks),  \
        dim3(256), 0, st, (TT*)out.data_ptr(), ws.data_ptr<float>(), inv.data_ptr<int>(),          \
        weights ? weights->data_ptr<float>() : nullptr, tiles.data_ptr<int>(), (int)T, topk,       \
        (int)N, (int)c, nc, (nc + 255) / 256, nk, share ? (int)mt : 0)
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
