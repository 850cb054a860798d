// Flash attention over many query tokens for gfx950: whole prompts (K1/K11-analog; ref
// nkilib attention_cte called at attention_base.py:722-744 and the in-repo sliding-window
// NKI kernel modules/sliding_window/attention.py:38-477) and portions of prompts whose
// earlier tokens are already in the linear or paged cache.
//
// What bounds it: the matrix cores and, next to them, one exponential per score. Everything
// else is kept off the vector units:
//   * A workgroup takes 128 query rows of ONE kv head, 32 a wave. Rows are (token, head of
//     the group) pairs, so the heads that share K and V share its tiles in LDS, a chunk of
//     a few tokens still fills the rows, and the causal border is 128/gq tokens wide.
//   * Scores are made transposed, S^T = K Q^T (mfma 32x32x16): a lane owns ONE query row, so
//     the running maximum, the sum and the rescaling are plain registers (one exchange with
//     the other half wave for the maximum of 64 keys, none for the sum until the end).
//   * P never leaves the registers: the C layout of S^T holds, for a lane, runs of 4
//     consecutive keys; read as the B operand of O^T = V^T P^T they are the same 16 keys in
//     another order, and V^T is read in that order. V stays row-major in LDS: ds_read_b64_tr
//     transposes 4 keys x 16 channels on the way to the registers.
//   * Over a cache P enters the second product as three 16-bit parts (HILO), which add up to its
//     24 bits: single tokens are attended with 32-bit probabilities, and several do not get less.
//     (One part more than the two that random inputs need for the same measured error: 512 tokens
//     over 4000, linear 69 -> 81 us, paged 83 -> 98.) In fp16, which has no exponents for small
//     parts, P is lifted by 2^7 and its reference follows a tile that stays more than 2^8 below
//     it, so that P at each tile's largest lies in [2^-1, 2^15]; the accumulator is scaled up
//     meanwhile, by 2^64 at most. Prompts from an empty cache: one 16-bit part, as ever.
//   * The accumulator is rescaled only when a row's maximum grew by more than 2^8 since the
//     last time; probabilities and sums share the stale maximum, so nothing is lost.
//   * K and V tiles of 64 keys go straight to LDS (global_load_lds, 16 B a lane), two
//     buffers, one barrier a tile: the next tile flies while this one is computed. Slots of
//     16 B are XOR-swizzled on the source side so that neither the row reads of K nor the
//     transposing reads of V meet in a bank.
//
//   * Over pages that hold whole tiles (a multiple of 64 rows) a tile is one page number and one
//     address, kept in scalar registers; a tile without a page is left out. Page numbers, divisions
//     and marks for each key row took as many vector instructions as the exponentials: 512 tokens
//     over 3500 in pages of 64 90 -> 74 us, 64 tokens 24 -> 18. Other page sizes keep the row form.
//   * Over a cache a wave has priority while it multiplies with V: its SIMD's other wave then
//     computes exponentials beside it (74.6 -> 72.4 us; 200 tokens over 2000, heads of 64, 29.6 ->
//     27.7). Prompts from an empty cache have it where flash_run says so.
//
// Rows with few tiles to share (short chunks over a long cache) are split over the keys as
// well: fp32 partial sums per split and a small combining kernel.
//
// Measured (MI355X, bf16, 32 query / 8 kv heads; before: 16x16x32 tiles, P through LDS, V
// transposed by the staging stores; several tokens over a cache: one workgroup a token):
//   prompt of 8192, head size 128     2168 -> 608 us (904 TFLOP/s; two thirds of it is the
//                                     matrix pipe, the rest exponentials it does not hide)
//   prompt of 2048, head size 128/64  179 -> 54 us / 145 -> 39 us
//   prompt of 512 / 128               40 -> 16 us / 16 -> 9 us
//   512 tokens over 4000, linear/paged 1574 -> 72 us / 1749 -> 72 us (pages of 16 or 32: 87)
//   64 tokens over 4000, linear       237 -> 34 us, in pages 24 -> 18
//   32 rows of 6 tokens over 2000     351 -> 50 us (a verification step)
//   1 row of 2 tokens over 2000       28 -> 18 us
// No size was found at which several tokens are better off one by one. Error against 64 bits
// over a cache, bf16, 2-norm: 1.7e-3 (the rounding of the result; one by one 2.4e-3, fp16 2.1e-4
// and 3.0e-4); with one key far ahead of 60000 at e^-19 whose values are 10^-4 of the others',
// fp16: 2.0e-4 (one by one 4.0e-4; with two parts and one reference 6.2e-2).

#include "common.h"
#include "attention_row.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

namespace {

typedef __bf16 fa_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 fa_f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 fa_bf16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 fa_f16x4 __attribute__((ext_vector_type(4)));
typedef short fa_s16x4 __attribute__((ext_vector_type(4)));
typedef unsigned fa_u32x4 __attribute__((ext_vector_type(4)));
typedef float fa_f32x16 __attribute__((ext_vector_type(16)));

template <typename T> struct FaTraits;
template <> struct FaTraits<__hip_bfloat16> {
    using vec8 = fa_bf16x8;
    using vec4 = fa_bf16x4;
    using elem = __bf16;
    static DEV_INLINE fa_f32x16 mfma(vec8 a, vec8 b, fa_f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
    // a 16-bit part of each value, taken off it
    static DEV_INLINE vec8 part(float (&e)[8]) {
        vec8 p;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            p[j] = (elem)e[j];
            e[j] -= (float)p[j];
        }
        return p;
    }
};
template <> struct FaTraits<__half> {
    using vec8 = fa_f16x8;
    using vec4 = fa_f16x4;
    using elem = _Float16;
    static DEV_INLINE fa_f32x16 mfma(vec8 a, vec8 b, fa_f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
    static DEV_INLINE vec8 part(float (&e)[8]) {
        fa_u32x4 p;
#pragma unroll
        for (int j = 0; j < 4; ++j) {          // towards zero: in pairs, what is left is exact
            const auto h = __builtin_amdgcn_cvt_pkrtz(e[2 * j], e[2 * j + 1]);
            p[j] = __builtin_bit_cast(unsigned, h);
            e[2 * j] -= (float)h[0];
            e[2 * j + 1] -= (float)h[1];
        }
        return __builtin_bit_cast(vec8, p);
    }
};

constexpr int QROWS = 128;      // query rows of a workgroup
constexpr int KT = 64;          // keys of a tile
constexpr float FA_GROWTH = 8.f;  // log2 growth of a maximum that is put off
constexpr float FA_DEPTH = 64.f;  // and how far below the largest score P may count from (fp16)

// the other half wave's value
DEV_INLINE float half_swap(float x) {
    const unsigned u = __builtin_bit_cast(unsigned, x);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return __builtin_bit_cast(float, (threadIdx.x & 32) ? r[0] : r[1]);
}

// 16 bytes a lane from `src` to the 1 KB of LDS at the wave-uniform `dst`. Written out, because
// the compiler puts a wait for every such load in flight before each transposing LDS read, of
// any buffer. It has no register result; the kernel waits (vmcnt) before the barrier that
// hands the tile over.
DEV_INLINE void fa_load_lds(const void* src, unsigned dst) {
    const unsigned at = __builtin_amdgcn_readfirstlane(dst);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                 :: "s"(at), "v"(src) : "memory", "m0");
}

struct FaArgs {
    const int* positions;    // (B, S) position of each query (-1: padding), or null: token index
    const int* seq_ids;      // (B,) cache row, or null: batch row
    const int* block_table;  // (B, max_blocks), paged caches
    const int* starts;       // (B + 1,) packed prompts: first row of each in q and out (rows, Hq, D), or null
    const float* sinks;      // (Hq,) or null
    float* o_part;           // (nsplit, B, Hq, S, D), nsplit > 1
    float* ml_part;          // (nsplit, B, Hq, S, 2)
    long ob, oh, os;         // element strides of out over (b, head, token)
    float scale;
    int window, B, Hq, Hkv, S, cap;   // cap: key rows of a sequence
    int Smax, block_size, max_blocks; // linear row capacity / paged geometry
    int turned;                       // rows' tiles from which on their order is reversed, or 0 (flash_launch)
    int nsplit, nqt, clamp_rows;      // clamp_rows: a negative seq_id reads row 0 (else: no keys)
};

// where the keys are: a row of a linear cache, pages, or pages that hold whole tiles
enum FaKeys { ROWS, PAGES, TILE_PAGES };

// FIRST: a wave has priority while it multiplies with V
template <typename T, int D, int KEYS, bool HILO, bool FIRST>
__global__ __launch_bounds__(256, 2) void flash_kernel(
    T* __restrict__ out, const T* __restrict__ q, const T* __restrict__ k,
    const T* __restrict__ v, const FaArgs a) {
    using FT = FaTraits<T>;
    using vec8 = typename FT::vec8;
    using vec4 = typename FT::vec4;
    constexpr bool PAGED = KEYS == PAGES;  // a page number for each key row
    constexpr int ROWB = D * 2;            // bytes of a key row
    constexpr int SLOTS = ROWB / 16;       // 16-byte slots of a row: 16 or 8
    constexpr int RPI = 64 / SLOTS;        // rows that one wave-wide load stages: 4 or 8
    constexpr int NLD = KT / 4 / RPI;      // loads a wave issues per tile and operand
    constexpr int TILE_B = KT * ROWB;
    constexpr int NKS = D / 16;            // k-steps of Q K^T
    constexpr int NDB = D / 32;            // 32-channel blocks of the output
    constexpr int NP = HILO ? 3 : 1;       // 16-bit parts of P
    constexpr bool FOLLOW = HILO && std::is_same<T, __half>::value;
    constexpr float LIFT = FOLLOW ? 7.f : 0.f;

    extern __shared__ __attribute__((aligned(16))) char smem[];
    // [2 buffers][K tile | V tile], then block bounds and the paged tiles' bad-row marks
    int* s_bounds = reinterpret_cast<int*>(smem + 4 * TILE_B);
    int* s_bad = s_bounds + 8;             // [2][1 + KT], paged only

    const int NH = a.B * a.Hkv;
    int hg, rest;
    {
        // kv heads go round the 8 XCDs, so that one L2 serves a head's K and V; the longest
        // (last) rows of all heads start first
        const int id = blockIdx.x;
        if ((NH & 7) == 0) {
            const int per = NH >> 3, t = id >> 3;
            hg = (id & 7) + 8 * (t % per);
            rest = t / per;
        } else {
            hg = id % NH;
            rest = id / NH;
        }
    }
    if (a.turned && rest >= a.turned) rest = a.nqt - 1 - (rest - a.turned);
    const int qt = a.nqt - 1 - rest / a.nsplit;
    const int split = rest % a.nsplit;
    const int b = hg / a.Hkv, hkv = hg % a.Hkv;
    const int gq = a.Hq / a.Hkv;
    // packed: S is the longest prompt's; the workgroups past a shorter one have nothing to do
    const int row0 = a.starts ? a.starts[b] : 0;
    const int R = gq * (a.starts ? a.starts[b + 1] - row0 : a.S);
    if (qt * QROWS >= R) return;

    const int lane = threadIdx.x & 63;
    const int wid = threadIdx.x >> 6;
    const int half = lane >> 5;
    const int r_own = qt * QROWS + wid * 32 + (lane & 31);
    const int rr = min(r_own, R - 1);
    const int token = rr / gq;
    const int head = hkv * gq + rr % gq;
    const int row = a.seq_ids ? a.seq_ids[b] : b;

    int qpos = a.positions ? a.positions[(long)b * a.S + token] : token;
    if (r_own >= R || (row < 0 && !a.clamp_rows)) qpos = -1;
    // the lane's own first visible key; positions past the capacity see what is left of theirs
    const int key_lo = a.window > 0 ? qpos - a.window + 1
                                    : a.window < 0 ? qpos / -a.window * -a.window : 0;
    const bool past = __any(qpos >= a.cap);
    qpos = min(qpos, a.cap - 1);

    // bounds of the wave's and the workgroup's valid rows
    int wmin = qpos < 0 ? 0x7fffffff : qpos, wmax = qpos;
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) {
        wmin = min(wmin, __shfl_xor(wmin, off, WAVE_SIZE));
        wmax = max(wmax, __shfl_xor(wmax, off, WAVE_SIZE));
    }
    if (lane == 0) {
        s_bounds[wid * 2] = wmin;
        s_bounds[wid * 2 + 1] = wmax;
    }
    // Q as the B operand: column = the lane's row, 8 channels at half*8 of each k-step
    vec8 qf[NKS];
    {
        const T* qp = q + (a.starts ? ((long)(row0 + token) * a.Hq + head)
                                    : ((long)b * a.Hq + head) * a.S + token) * D + half * 8;
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) qf[ks] = *reinterpret_cast<const vec8*>(qp + ks * 16);
    }
    // landed before the first tile is on its way: no wait for them inside the loop
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) asm volatile("" : "+v"(qf[ks]));
    __syncthreads();
    int bmin = s_bounds[0], bmax = s_bounds[1];
#pragma unroll
    for (int w = 1; w < 4; ++w) {
        bmin = min(bmin, s_bounds[w * 2]);
        bmax = max(bmax, s_bounds[w * 2 + 1]);
    }
    bmin = __builtin_amdgcn_readfirstlane(bmin);
    bmax = __builtin_amdgcn_readfirstlane(bmax);
    wmin = __builtin_amdgcn_readfirstlane(wmin);
    wmax = __builtin_amdgcn_readfirstlane(wmax);
    const int C = a.window < 0 ? -a.window : 0;
    int lo = 0;
    if (a.window > 0) lo = max(0, bmin - a.window + 1);
    else if (C) lo = (bmin / C) * C;
    if (bmax < 0) lo = 0;
    // the wave's own first visible key, and from where on every key is inside all its windows
    const int w_lo = a.window > 0 ? max(0, wmin - a.window + 1) : (C && wmax >= 0 ? (wmin / C) * C : 0);
    const int w_in = past && a.window ? 0x7fffffff
                     : a.window > 0   ? wmax - a.window + 1
                                      : (C && wmax >= 0 ? (wmax / C) * C : 0);

    int t_lo = lo / KT, t_hi = (bmax + KT) / KT;      // tiles [t_lo, t_hi); none when bmax < 0
    if (a.nsplit > 1) {
        const int per = (t_hi - t_lo + a.nsplit - 1) / a.nsplit;
        t_lo += split * per;
        t_hi = min(t_hi, t_lo + per);
    }

    const float c0 = a.scale * 1.4426950408889634f;   // scores in log2 units
    // c multiplies masked scores too, which are -inf: positive, so that they stay it
    const float sign = c0 == 0.f ? 0.f : c0 < 0.f ? -1.f : 1.f, c = c0 == 0.f ? 1.f : fabsf(c0);

    // ---- staging: this lane's rows and source slots ----
    const int st_row = wid * (KT / 4) + lane / SLOTS;  // + i * RPI
    const int st_p = lane % SLOTS;
    const long lin = KEYS != ROWS ? 0 : ((long)max(row, 0) * a.Hkv + hkv) * (long)a.Smax * D;
    auto swz_k = [](int r) { return D == 128 ? (r & 15) : ((r >> 1) & 7); };
    auto swz_v = [](int r) { return D == 128 ? ((r & 3) << 2) : (((r >> 1) & 1) << 2); };
    const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) char*)smem;
    int blk[NLD];                                      // paged: the next tile's page numbers
    // of whole tiles: the pages of the tile at hand, of the one on its way and of the one after
    const int* pages = KEYS == TILE_PAGES ? a.block_table + (long)b * a.max_blocks : nullptr;
    int page = 0, page_now = 0, page_next = 0;
    auto load_blocks = [&](int t) {
        if constexpr (KEYS == TILE_PAGES) page_next = pages[t * KT / a.block_size];
        if constexpr (PAGED) {
#pragma unroll
            for (int i = 0; i < NLD; ++i) {
                const int key = min(t * KT + st_row + i * RPI, bmax);
                blk[i] = a.block_table[(long)b * a.max_blocks + key / a.block_size];
            }
        }
    };
    auto stage = [&](int t, int buf) {
        const unsigned kd = lds0 + buf * 2 * TILE_B + wid * (TILE_B / 4);
        const unsigned vd = kd + TILE_B;
        long first = 0;                                // of the tile's keys in its page
        if constexpr (KEYS == TILE_PAGES)
            first = ((long)max(page_next, 0) * a.block_size + t * KT % a.block_size) * a.Hkv + hkv;
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            const int r = st_row + i * RPI;
            const int key = min(t * KT + r, bmax);
            long off;
            if constexpr (KEYS == TILE_PAGES)
                off = (first + (long)(key - t * KT) * a.Hkv) * D;
            else if constexpr (PAGED)
                off = (((long)max(blk[i], 0) * a.block_size + key % a.block_size) * a.Hkv + hkv) * D;
            else
                off = lin + (long)key * D;
            const T* ks = k + off + (st_p ^ swz_k(r)) * 8;
            const T* vs = v + off + (st_p ^ swz_v(r)) * 8;
            fa_load_lds(ks, kd + i * 1024);
            fa_load_lds(vs, vd + i * 1024);
        }
        if constexpr (PAGED) {
            // rows without a page are marked; their values are cleared once they have landed
            if (st_p == 0) {
#pragma unroll
                for (int i = 0; i < NLD; ++i) {
                    const bool bad = blk[i] < 0;
                    s_bad[buf * (KT + 1) + 1 + st_row + i * RPI] = bad;
                    if (bad) s_bad[buf * (KT + 1)] = t;
                }
            }
        }
    };

    fa_f32x16 o[NDB];
#pragma unroll
    for (int i = 0; i < NDB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[i][r] = 0.f;
    // m: what P counts from (log2 units); l: this half's sum; top: the largest score (FOLLOW)
    float m = -INFINITY, l = 0.f, top = -INFINITY;

    // fragment addresses within a tile
    const int ka_row = lane & 31;
    const int vi = lane & 15;
    const int va_row = half * 4 + (vi >> 2);
    const int va_d = ((lane >> 4) & 1) * 16 + (vi & 3) * 4;

    if constexpr (PAGED) {
        if (threadIdx.x < 2) s_bad[threadIdx.x * (KT + 1)] = -1;
        __syncthreads();
    }
    if (t_lo < t_hi) {
        load_blocks(t_lo);
        page_now = page_next;
        stage(t_lo, 0);
        if (t_lo + 1 < t_hi) load_blocks(t_lo + 1);
    }
    for (int t = t_lo; t < t_hi; ++t) {
        const int buf = (t - t_lo) & 1;
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        if constexpr (PAGED) {
            // a row without a page: its V row (whatever page 0 holds) must not reach 0 * V
#pragma unroll
            for (int i = 0; i < NLD; ++i) {
                const int r = st_row + i * RPI;
                if (s_bad[buf * (KT + 1) + 1 + r])
                    *reinterpret_cast<int4*>(smem + buf * 2 * TILE_B + TILE_B + r * ROWB + st_p * 16)
                        = int4{0, 0, 0, 0};
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        page = page_now;
        if (t + 1 < t_hi) {
            page_now = page_next;
            stage(t + 1, buf ^ 1);
            if (t + 2 < t_hi) load_blocks(t + 2);
        }
        const int k0 = t * KT;
        if (k0 > wmax || k0 + KT <= w_lo) continue;     // nothing here for this wave
        if (KEYS == TILE_PAGES && page < 0) continue;   // nor keys that anyone sees
        const char* kb = smem + buf * 2 * TILE_B;
        const char* vb = kb + TILE_B;

        fa_f32x16 s[2];
#pragma unroll
        for (int n = 0; n < 2; ++n) {
#pragma unroll
            for (int r = 0; r < 16; ++r) s[n][r] = 0.f;
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                const int r = n * 32 + ka_row;
                const vec8 ka = *reinterpret_cast<const vec8*>(
                    kb + r * ROWB + (((ks * 2 + half) ^ swz_k(r)) << 4));
                s[n] = FT::mfma(ka, qf[ks], s[n]);
            }
        }
        // four reads ahead of the products, not one (what the compiler does by itself)
        __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
        for (int i = 0; i < 2 * NKS - 4; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
        if (sign != 1.f) {
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int r = 0; r < 16; ++r) s[n][r] *= sign;
        }
        bool masked = (k0 + KT - 1 > wmin) || (k0 < w_in);
        if constexpr (PAGED) masked = masked || s_bad[buf * (KT + 1)] == t;
        if (masked) {
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int kk = n * 32 + 8 * (r >> 2) + 4 * half + (r & 3);
                    bool ok = k0 + kk <= qpos && k0 + kk >= key_lo;
                    if constexpr (PAGED) ok = ok && !s_bad[buf * (KT + 1) + 1 + kk];
                    s[n][r] = ok ? s[n][r] : -INFINITY;
                }
        }
        float mx = s[0][0];
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[n][r]);
        mx = fmaxf(mx, half_swap(mx)) * c;
        bool move = mx > m + FA_GROWTH || (m == -INFINITY && mx > m);
        float mn = fmaxf(m, mx);
        if constexpr (FOLLOW) {                         // and down to a tile that stays far below
            top = fmaxf(top, mx);
            if (mx < m - FA_GROWTH && mx != -INFINITY) {
                mn = fmaxf(mx, top - FA_DEPTH);
                move = mn < m;
            }
        }
        if (__any(move)) {
            const float f = m == -INFINITY ? 0.f : exp2f(m - mn);
            m = mn;
            l *= f;
#pragma unroll
            for (int i = 0; i < NDB; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[i][r] *= f;
        }
        const float mu = m == -INFINITY ? 0.f : m - LIFT;   // (0: a row that has seen no key yet)
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float e = __builtin_amdgcn_exp2f(fmaf(s[n][r], c, -mu));
                l += e;
                s[n][r] = e;
            }
        // (this wave before the other of its SIMD: that one's exponentials are to run beside these
        // products, and not both waves' products in turns)
        if constexpr (FIRST) __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            vec8 p[NP];
            {
                float e[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) e[j] = s[kt >> 1][(kt & 1) * 8 + j];
                if constexpr (HILO) {
#pragma unroll
                    for (int c = 0; c < NP; ++c) p[c] = FT::part(e);
                } else {
#pragma unroll
                    for (int j = 0; j < 8; ++j) p[0][j] = (typename FT::elem)e[j];
                }
            }
#pragma unroll
            for (int db = 0; db < NDB; ++db) {
                vec8 va;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int r = kt * 16 + j * 8 + va_row;
                    const int d = db * 32 + va_d;
                    const char* at = vb + r * ROWB + (((d >> 3) ^ swz_v(r)) << 4) + (d & 7) * 2;
                    const fa_s16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (__attribute__((address_space(3))) fa_s16x4*)at);
                    const vec4 y = __builtin_bit_cast(vec4, x);
#pragma unroll
                    for (int e = 0; e < 4; ++e) va[j * 4 + e] = y[e];
                }
#pragma unroll
                for (int c = 0; c < NP; ++c) o[db] = FT::mfma(va, p[c], o[db]);
            }
        }
        __builtin_amdgcn_sched_group_barrier(0x100, 8, 1);
#pragma unroll
        for (int i = 0; i < 4 * NDB - 4; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, NP, 1);
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 4 * NP, 1);
        if constexpr (FIRST) __builtin_amdgcn_s_setprio(0);
    }

    // ---- epilogue: rows of 4 channels from 8*(r>>2) + 4*half ----
    l += half_swap(l);
    m -= LIFT;
    if constexpr (HILO) {
        // rows whose sums are finite and whose values are not: see attention_row.h
        float z[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < NDB; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) z[r & 3] += o[i][r] * 0.f;
        const bool lost = !((z[0] + z[1]) + (z[2] + z[3]) == 0.f);
        const unsigned long long bad =
            __ballot(lost && l == l && l != 0.f && qpos >= 0 && r_own < R);
        for (unsigned rest = (unsigned)bad | (unsigned)(bad >> 32); rest; rest &= rest - 1) {
            const int own = __ffs(rest) - 1;
            const long at = ((long)b * a.Hq + __shfl(head, own, WAVE_SIZE)) * a.S +
                            __shfl(token, own, WAVE_SIZE);
            float mr, lr, acc[D / 64];
            attend_row<D>(q + at * D, k, v, max(__shfl(key_lo, own, WAVE_SIZE), t_lo * KT),
                          min(__shfl(qpos, own, WAVE_SIZE) + 1, t_hi * KT), c0,
                          [&](int key) -> long {
                if constexpr (KEYS != ROWS) {
                    const int p = a.block_table[(long)b * a.max_blocks + key / a.block_size];
                    return p < 0 ? -1 : (((long)p * a.block_size + key % a.block_size) * a.Hkv + hkv) * D;
                }
                return lin + (long)key * D;
            }, mr, lr, acc);
            // through the tile buffer that the last tile did not use, a part for each wave
            float* row_lds = reinterpret_cast<float*>(smem + ((t_hi - t_lo) & 1) * 2 * TILE_B +
                                                      wid * (TILE_B / 2));
#pragma unroll
            for (int e = 0; e < D / 64; ++e) row_lds[lane * (D / 64) + e] = acc[e];
            __builtin_amdgcn_wave_barrier();
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if ((lane & 31) == own) {
                m = mr;
                l = lr;
#pragma unroll
                for (int i = 0; i < NDB; ++i)
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        o[i][r] = row_lds[i * 32 + 8 * (r >> 2) + 4 * half + (r & 3)];
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_wave_barrier();
        }
    }
    if (r_own >= R) return;
    // padding (tiles that are whole for the others ran unmasked), or no key seen. A sum that is
    // NaN, as of a query that is, has no maximum either and stays
    if (qpos < 0 || l == 0.f) {
        m = -INFINITY;
        l = 0.f;
#pragma unroll
        for (int i = 0; i < NDB; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[i][r] = 0.f;
    }
    if (a.nsplit > 1) {
        const long at = (((long)split * a.B + b) * a.Hq + head) * a.S + token;
        if (half == 0) {
            a.ml_part[at * 2] = m;
            a.ml_part[at * 2 + 1] = l;
        }
        if (l == 0.f) return;                           // nothing seen: the weight is 0
        float* po = a.o_part + at * D;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *reinterpret_cast<float4*>(po + db * 32 + 8 * g + 4 * half) =
                    float4{o[db][g * 4], o[db][g * 4 + 1], o[db][g * 4 + 2], o[db][g * 4 + 3]};
        return;
    }
    float f = 1.f;
    if (a.sinks != nullptr && m != -INFINITY) {         // a sink joins the denominator only
        const float sk = a.sinks[head] * 1.4426950408889634f, mt = fmaxf(m, sk);
        f = exp2f(m - mt);
        l = l * f + exp2f(sk - mt);
    }
    const float inv = l > 0.f ? f / l : 0.f;
    T* po = out + (a.starts ? row0 * a.os : b * a.ob) + head * a.oh + token * a.os;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            vec4 y;
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = (typename FT::elem)(o[db][g * 4 + e] * inv);
            *reinterpret_cast<vec4*>(po + db * 32 + 8 * g + 4 * half) = y;
        }
}

// out row = sum over splits of 2^(m_i - m) o_i / l; a wave a row
template <typename T, int D>
__global__ __launch_bounds__(256) void flash_combine_kernel(T* __restrict__ out, const FaArgs a) {
    const long rows = (long)a.B * a.Hq * a.S;
    const long rowid = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (rowid >= rows) return;
    const int lane = threadIdx.x & 63;
    const int token = (int)(rowid % a.S);
    const int head = (int)(rowid / a.S % a.Hq);
    const int b = (int)(rowid / a.S / a.Hq);
    float m = -INFINITY;
    for (int i = 0; i < a.nsplit; ++i) m = fmaxf(m, a.ml_part[(i * rows + rowid) * 2]);
    if (a.sinks != nullptr && m != -INFINITY) m = fmaxf(m, a.sinks[head] * 1.4426950408889634f);
    constexpr int PER = D / 64;
    float acc[PER], L = 0.f;
#pragma unroll
    for (int j = 0; j < PER; ++j) acc[j] = 0.f;
    for (int i = 0; i < a.nsplit; ++i) {
        const float mi = a.ml_part[(i * rows + rowid) * 2];
        const float li = a.ml_part[(i * rows + rowid) * 2 + 1];
        if (li == 0.f) continue;
        const float f = mi == -INFINITY ? 1.f : exp2f(mi - m);      // (1: a sum of NaN)
        L += f * li;
#pragma unroll
        for (int j = 0; j < PER; ++j) acc[j] += f * a.o_part[(i * rows + rowid) * D + lane * PER + j];
    }
    if (a.sinks != nullptr && m != -INFINITY) L += exp2f(a.sinks[head] * 1.4426950408889634f - m);
    const float inv = L > 0.f ? 1.f / L : 0.f;
    T* po = out + b * a.ob + head * a.oh + token * a.os + lane * PER;
#pragma unroll
    for (int j = 0; j < PER; ++j) po[j] = VecTraits<T>::from_float(acc[j] * inv);
}

template <typename T, int D, int KEYS, bool HILO, bool FIRST = HILO>
void flash_launch(torch::Tensor& out, const torch::Tensor& q, const torch::Tensor& k,
                  const torch::Tensor& v, FaArgs& a, bool even, hipStream_t stream) {
    const int gq = a.Hq / a.Hkv;
    a.nqt = (int)(((long)gq * a.S + QROWS - 1) / QROWS);
    const size_t lds = 4 * KT * D * 2 + 8 * sizeof(int) + (KEYS == PAGES ? 2 * (KT + 1) * sizeof(int) : 0);
    // a limit of the function on the device at hand, the same in every call
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&flash_kernel<T, D, KEYS, HILO, FIRST>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    const long blocks = (long)a.B * a.Hkv * a.nqt * a.nsplit;
    // Workgroups that are all there at once, two to a CU: the second ones in the other order, so that a
    // CU with one of the longest rows gets one of the shortest (1500 tokens 37.9 -> 35.6 us, 2048 50.5
    // -> 47.2, 4 prompts of 512 20.3 -> 19.3, heads of 64 2 to 4 %). One a CU has no second; more than
    // 512 take the places that come free, longest first. Windows make rows alike (20.3 -> 20.6).
    constexpr int CUS = 256;
    const long heads = (long)a.B * a.Hkv;
    a.turned = !HILO && even && a.window == 0 && blocks > CUS && blocks <= 2 * CUS ? (int)(CUS / heads) : 0;
    TORCH_CHECK(blocks < (1l << 31), "flash attention: too many query rows");
    hipLaunchKernelGGL((flash_kernel<T, D, KEYS, HILO, FIRST>), dim3((unsigned)blocks), dim3(256), lds, stream,
                       (T*)out.data_ptr(), (const T*)q.data_ptr(), (const T*)k.data_ptr(),
                       (const T*)v.data_ptr(), a);
    HIP_CHECK_KERNEL();
    if (a.nsplit > 1) {
        const long rows = (long)a.B * a.Hq * a.S;
        hipLaunchKernelGGL((flash_combine_kernel<T, D>), dim3((unsigned)((rows + 3) / 4)), dim3(256),
                           0, stream, (T*)out.data_ptr(), a);
        HIP_CHECK_KERNEL();
    }
}

void flash_run(torch::Tensor& out, const torch::Tensor& q, const torch::Tensor& k,
               const torch::Tensor& v, FaArgs& a, c10::optional<torch::Tensor>& sinks_opt) {
    const int D = q.size(3);
    TORCH_CHECK(q.dim() == 4 && k.dim() == 4 && v.dim() == 4 && out.dim() == 4, "bad shapes");
    TORCH_CHECK(q.is_contiguous() && k.is_contiguous() && v.is_contiguous(),
                "contiguous tensors required");
    TORCH_CHECK(((size_t)k.data_ptr() | (size_t)v.data_ptr()) % 16 == 0,
                "flash attention: K/V are staged 16 bytes at a time");
    TORCH_CHECK(out.sizes() == q.sizes() && out.stride(3) == 1 && out.stride(2) % 4 == 0 &&
                out.stride(1) % 4 == 0 && out.stride(0) % 4 == 0, "flash attention: bad output layout");
    TORCH_CHECK(k.sizes() == v.sizes() && k.size(3) == D, "flash attention: K/V shapes differ");
    TORCH_CHECK(k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type() &&
                out.scalar_type() == q.scalar_type(), "flash attention: one dtype for q, k, v and out");
    TORCH_CHECK(a.Hkv > 0 && a.Hq % a.Hkv == 0, "Hq must divide by Hkv");
    TORCH_CHECK(D == 64 || D == 128, "flash attention: head_dim 64/128 only");
    if (q.numel() == 0) return;
    if (k.numel() == 0) {
        out.zero_();
        return;
    }
    torch::Tensor sinks_t;
    if (sinks_opt.has_value()) {
        sinks_t = sinks_opt->to(torch::kFloat32).contiguous();
        TORCH_CHECK(sinks_t.numel() == a.Hq, "sinks must be (Hq,)");
        a.sinks = sinks_t.data_ptr<float>();
    }
    a.ob = out.stride(0);
    a.oh = out.stride(1);
    a.os = out.stride(a.starts ? 0 : 2);
    torch::Tensor o_part, ml_part;
    if (a.nsplit > 1) {
        auto opts = torch::TensorOptions().dtype(torch::kFloat32).device(q.device());
        const long rows = (long)a.nsplit * a.B * a.Hq * a.S;
        o_part = torch::empty({rows * D}, opts);
        ml_part = torch::empty({rows * 2}, opts);
        a.o_part = o_part.data_ptr<float>();
        a.ml_part = ml_part.data_ptr<float>();
    }
    auto stream = at::hip::getCurrentHIPStream();
    const bool paged = a.block_table != nullptr, tiles = paged && a.block_size % KT == 0;
    const bool extend = a.positions != nullptr;
    // Packed prompts of several lengths: the grid counts the longest's tiles for each, and says neither
    // how many workgroups have work nor which of them are long.
    const bool even = !a.starts || q.size(0) == (long)a.B * a.S;
    // Priority for prompts: between 1.4 and two rounds of workgroups a CU's second place is filled all the
    // way, and it pays as it does over a cache, where rows are long. Heads of 128, one prompt of 2816, 2880,
    // 2944, 3072, 3584, 4096 tokens (704 to 1024 workgroups) 81.1 / 82.0, 83.4 / 83.3, 86.5 / 85.3, 94.6 / 90.5,
    // 126 / 115, 156 / 146 us; 3 of 940 and of 1300 40.3 / 37.8 and 61.0 / 58.1, 4 of 900 46.2 / 44.5, but 5 of
    // 700 39.8 / 39.5, 6 of 600 37.8 / 38.3, 8 of 370 26.9 / 28.9, 12 of 250 25.7 / 26.2. Chunks of 512 and 2048
    // keys 41.1 / 39.8 and 87.9 / 82.8 (4096 tokens); a window has short rows: of 512 38.1 / 39.2 (3 of 1024), of
    // 1024 59.8 / 63.1 (2848 tokens). 576 and 640 workgroups lose 2 and 4 %, 1256 to 1504 between +1 and -3;
    // heads of 64 up to 6. (A kernel of its own: a branch around it in one kernel costs the others 1 to 3 %.)
    const long groups = ((long)a.Hq / a.Hkv * a.S + QROWS - 1) / QROWS * a.B * a.Hkv;
    const bool first = even && groups >= 720 && groups <= 1024 && a.S >= 900 &&
                       (a.window <= 0 || a.window >= a.S);
#define FA_D(T, D)                                                                        \
    do {                                                                                  \
        if (tiles) flash_launch<T, D, TILE_PAGES, true>(out, q, k, v, a, even, stream);   \
        else if (paged) flash_launch<T, D, PAGES, true>(out, q, k, v, a, even, stream);   \
        else if (extend) flash_launch<T, D, ROWS, true>(out, q, k, v, a, even, stream);   \
        else if (D == 128 && first) flash_launch<T, 128, ROWS, false, true>(out, q, k, v, a, even, stream); \
        else flash_launch<T, D, ROWS, false>(out, q, k, v, a, even, stream);              \
    } while (0)
#define FA_GO(T)                                                                          \
    do {                                                                                  \
        if (D == 128) FA_D(T, 128);                                                       \
        else FA_D(T, 64);                                                                 \
    } while (0)
    if (q.scalar_type() == at::ScalarType::BFloat16) FA_GO(__hip_bfloat16);
    else if (q.scalar_type() == at::ScalarType::Half) FA_GO(__half);
    else TORCH_CHECK(false, "flash_prefill: bf16/f16 only");
#undef FA_GO
#undef FA_D
}

FaArgs flash_args(const torch::Tensor& q, double scale, long window) {
    FaArgs a{};
    a.scale = (float)scale;
    a.window = (int)window;
    a.B = q.size(0);
    a.Hq = q.size(1);
    a.S = q.size(2);
    a.nsplit = 1;
    return a;
}

// Splits over the keys: two workgroups fit a CU, so fill 512 places, but leave a split at least 4
// tiles (256 keys) of a row that fills the capacity, below which combining costs more. (Rows' own
// lengths are on the device: a short row's tiles are shared by as many splits. 6 tokens over 300
// of 32768 15 us, one workgroup a token 46; over 1000 of 32768, 8 rows, 20 and 109.)
int flash_splits(const FaArgs& a) {
    const long tiles = ((long)a.Hq / a.Hkv * a.S + QROWS - 1) / QROWS * a.B * a.Hkv;
    const long most = std::max(1, a.cap / (4 * KT));
    return (int)std::max(1l, std::min({512 / std::max(1l, tiles), most, 16l}));
}

}  // namespace

void flash_prefill(torch::Tensor out, torch::Tensor q, torch::Tensor k,
                   torch::Tensor v, double scale, long window,
                   c10::optional<torch::Tensor> sinks_opt) {
    FaArgs a = flash_args(q, scale, window);
    a.Hkv = k.size(1);
    a.cap = a.Smax = k.size(2);
    TORCH_CHECK(k.size(0) == a.B && k.size(2) == a.S, "flash_prefill: K/V must match q");
    flash_run(out, q, k, v, a, sinks_opt);
}

void flash_prefill_cached(torch::Tensor out, torch::Tensor q,
                          torch::Tensor k_cache, torch::Tensor v_cache,
                          torch::Tensor seq_ids, double scale, long window,
                          c10::optional<torch::Tensor> sinks_opt) {
    // K/V read from the (Bc, Hkv, Smax, D) cache rows just written —
    // prefill straight off the cache, no fresh K/V tensors
    auto sid = seq_ids.to(torch::kInt32).contiguous();
    FaArgs a = flash_args(q, scale, window);
    a.Hkv = k_cache.size(1);
    a.Smax = k_cache.size(2);
    a.cap = std::min(a.S, a.Smax);
    a.seq_ids = sid.data_ptr<int>();
    a.clamp_rows = 1;   // rows of -1 are batch padding: read row 0, the host drops the result
    TORCH_CHECK(sid.numel() == a.B, "seq_ids must be (B,)");
    flash_run(out, q, k_cache, v_cache, a, sinks_opt);
}

// The same for prompts one after the other without padding: q and out (rows, Hq, 1, D), prompt b
// from row starts[b] to starts[b + 1], the longest of `longest` tokens.
void flash_prefill_packed(torch::Tensor out, torch::Tensor q, torch::Tensor k_cache,
                          torch::Tensor v_cache, torch::Tensor seq_ids, torch::Tensor starts,
                          long longest, double scale, long window) {
    FaArgs a = flash_args(q, scale, window);
    TORCH_CHECK(a.S == 1 && longest > 0 && starts.scalar_type() == at::kInt &&
                starts.is_contiguous() && seq_ids.scalar_type() == at::kInt &&
                seq_ids.is_contiguous() && starts.numel() == seq_ids.numel() + 1 &&
                starts.is_cuda() && seq_ids.is_cuda(), "flash_prefill_packed: prompts");
    a.B = seq_ids.numel();
    a.S = (int)longest;
    a.Hkv = k_cache.size(1);
    a.Smax = k_cache.size(2);
    a.cap = std::min(a.S, a.Smax);
    a.seq_ids = seq_ids.data_ptr<int>();
    a.starts = starts.data_ptr<int>();
    a.clamp_rows = 1;
    c10::optional<torch::Tensor> none;
    flash_run(out, q, k_cache, v_cache, a, none);
}

// Several query tokens a sequence against the cache, each attending the rows up to its own
// position (chunked prefill, prefix prefill, verification). Linear cache: block_table absent.
void flash_extend(torch::Tensor out, torch::Tensor q, torch::Tensor k_cache,
                  torch::Tensor v_cache, torch::Tensor positions,
                  c10::optional<torch::Tensor> seq_ids_opt,
                  c10::optional<torch::Tensor> block_table_opt, double scale, long window,
                  c10::optional<torch::Tensor> sinks_opt) {
    FaArgs a = flash_args(q, scale, window);
    const bool paged = block_table_opt.has_value();
    a.Hkv = k_cache.size(paged ? 2 : 1);
    auto pos = positions.to(torch::kInt32).contiguous();
    TORCH_CHECK(pos.numel() == (long)a.B * a.S, "positions must be (B, Sq)");
    a.positions = pos.data_ptr<int>();
    torch::Tensor sid, bt;
    if (paged) {
        bt = block_table_opt->to(torch::kInt32).contiguous();
        TORCH_CHECK(bt.dim() == 2 && bt.size(0) == a.B, "block_table must be (B, blocks)");
        TORCH_CHECK(a.Hkv > 0 && a.Hq / a.Hkv <= 8, "GQA ratio > 8 not supported yet (got ",
                    a.Hkv > 0 ? a.Hq / a.Hkv : 0, ")");
        a.block_table = bt.data_ptr<int>();
        a.block_size = k_cache.size(1);
        a.max_blocks = bt.size(1);
        a.cap = a.max_blocks * a.block_size;
        if (bt.numel() == 0) {
            out.zero_();
            return;
        }
    } else {
        TORCH_CHECK(seq_ids_opt.has_value() && seq_ids_opt->numel() == a.B, "seq_ids must be (B,)");
        sid = seq_ids_opt->to(torch::kInt32).contiguous();
        a.seq_ids = sid.data_ptr<int>();
        a.cap = a.Smax = k_cache.size(2);
    }
    a.nsplit = flash_splits(a);
    flash_run(out, q, k_cache, v_cache, a, sinks_opt);
}
