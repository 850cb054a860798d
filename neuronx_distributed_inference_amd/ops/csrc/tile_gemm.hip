// y (M, N) = x (M, K) @ w (N, K)^T in 16 bits, up to 512 rows: the products of decoding and of short
// prompts, bound by the weights' bytes, which come once, straight to LDS.
//
// A workgroup holds a ring of D chunks (64 of K, 128 bytes a row) of its tiles of x and w, filled
// by global_load_lds and waited for by count, with one barrier a chunk. What fills the memory
// pipes is the bytes on the way: 64 to 128 KB a CU. K is split so that all 256 CUs have a tile;
// the parts stay in fp32 and the kernel that follows (residual sum and norm, rope) adds them up,
// so that a split costs no launch. With GLU a wave has the gate and the up rows of its columns and
// writes silu(gate) (or gelu) * up, which saves a launch and both in 16 bits. Two products whose
// sum the next kernel wants (a mixer's two output projections) go in one launch.

#include "common.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

namespace {

typedef __bf16 tg_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 tg_f16x8 __attribute__((ext_vector_type(8)));
typedef float tg_f32x4 __attribute__((ext_vector_type(4)));

template <typename T> struct TgMfma;
template <> struct TgMfma<__hip_bfloat16> {
    using vec8 = tg_bf16x8;
    static DEV_INLINE tg_f32x4 mfma(vec8 a, vec8 b, tg_f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
};
template <> struct TgMfma<__half> {
    using vec8 = tg_f16x8;
    static DEV_INLINE tg_f32x4 mfma(vec8 a, vec8 b, tg_f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
};

template <int N> DEV_INLINE void tg_wait() {
    asm volatile("s_waitcnt vmcnt(%c0)" ::"i"(N) : "memory");
}

// wait until at most `left` chunks of G loads are in flight
template <int G, int MAX> DEV_INLINE void tg_wait_chunks(int left) {
    if constexpr (MAX == 0) {
        tg_wait<0>();
    } else {
        if (left >= MAX) tg_wait<G * MAX>();
        else tg_wait_chunks<G, MAX - 1>(left);
    }
}

template <int AUX> DEV_INLINE void tg_load(const char* src, char* dst) {
    __builtin_amdgcn_global_load_lds(
        (const __attribute__((address_space(1))) unsigned int*)src,
        (__attribute__((address_space(3))) unsigned int*)dst, 16, 0, AUX);
}

constexpr int TG_BK = 64;    // K of a chunk: 128 bytes a row

struct TgArgs {
    void* y;             // (M, N), or (M, N / 2) with GLU
    float* part;         // (splits, M, N) fp32 when splits > 1
    const void* x;       // (M, K)
    const void* w;       // (N, K)
    const void* x2;      // a second product of the same sizes, parts after the first's, or null
    const void* w2;
    const void* bias;    // (N,) or null
    int M, N, K, splits, mblocks, ntiles, per_xcd, work;
    unsigned xbytes, xbytes2;    // from a row of x to the next
};

// none; silu and the tanh form of gelu of the gate
enum TgGlu { PLAIN, SILU, GELU };

template <int GLU> DEV_INLINE float tg_act(float z) {
    if constexpr (GLU == GELU)
        return 0.5f * z * (1.f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
    return z / (1.f + __expf(-z));
}


// A workgroup of WM x WN waves makes BM x BN outputs (of one of `splits` parts of K), a wave
// BM/WM x BN/WN of them. D chunks of w and DX of x are in LDS or on the way there. Where they
// differ, half of the waves load w and half x: a wave's loads are waited for in their order, and
// one that has both would wait for w as early as for x, which is near (L2).
template <typename T, int BM, int BN, int WM, int WN, int D, int DX, int GLU, bool ONCE>
__global__ __launch_bounds__(64 * WM * WN) void tile_gemm_kernel(const TgArgs a) {
    using MF = TgMfma<T>;
    using vec8 = typename MF::vec8;
    constexpr int NW = WM * WN;
    constexpr int FM = BM / WM / 16, FN = BN / WN / 16;
    constexpr int XPT = BM / 8, WPT = BN / 8;          // pieces of 8 rows, 1 KB, a wave's load
    constexpr bool APART = DX != D;
    constexpr int LW = APART ? NW / 2 : NW;            // waves that load w (and x)
    constexpr int XP = XPT >= LW ? XPT / LW : 1, WP = WPT / LW;
    static_assert(WPT % LW == 0 && (XPT % LW == 0 || XPT < LW), "pieces");
    static_assert(!GLU || FN % 2 == 0, "gate and up of a column in one wave");
    constexpr int XB = BM * 128, WB = BN * 128, W0 = DX * XB;    // bytes of a chunk; w's ring
    extern __shared__ __attribute__((aligned(16))) char smem[];

    // workgroups go round the XCDs: each gets one run of the work, row blocks of a tile of w
    // next to each other
    const int item = (blockIdx.x & 7) * a.per_xcd + (blockIdx.x >> 3);
    if (item >= a.work) return;
    const int mb = item % a.mblocks;
    const int rest = item / a.mblocks;
    const int nt = rest % a.ntiles, slice = rest / a.ntiles;
    const int m0 = mb * BM;
    const int chunks = a.K / TG_BK;
    const bool second = slice >= a.splits;
    const int part = second ? slice - a.splits : slice;
    const int c_lo = (int)((long)part * chunks / a.splits);
    const int n = (int)((long)(part + 1) * chunks / a.splits) - c_lo;     // >= 1: splits <= chunks

    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lw = wid % LW;
    const bool has_w = !APART || wid < LW, has_x = !APART || wid >= LW;
    const int depth = has_w ? D : DX;
    const int wm = wid / WN, wn = wid % WN;
    const int lrow = lane & 15, lslot = lane >> 4;

    // where the lane's 16 bytes of each piece come from; LDS rows hold 16-byte slots in the order
    // slot ^ (row & 7), so that 8 rows of one slot lie in different banks. Rows past the end
    // repeat the last one.
    const int prow = lane >> 3;
    const unsigned kbytes = (unsigned)a.K * sizeof(T), xbytes = second ? a.xbytes2 : a.xbytes;
    unsigned xo[XP], wo[WP];
#pragma unroll
    for (int i = 0; i < XP; ++i) {
        const int r = (lw * XP + i) % XPT * 8 + prow;
        xo[i] = (unsigned)min(r, a.M - 1 - m0) * xbytes + ((lane & 7) ^ (r & 7)) * 16;
    }
#pragma unroll
    for (int i = 0; i < WP; ++i) {
        const int r = (lw * WP + i) * 8 + prow;
        unsigned row;
        if constexpr (GLU) {
            // of a wave's rows half are gate and half are up, of the same columns
            constexpr int PW = BN / WN;
            const int in = r % PW;
            row = min(r / PW * (PW / 2) + in % (PW / 2), a.N / 2 - 1 - nt * (BN / 2)) +
                  (in >= PW / 2 ? a.N / 2 : 0);
        } else {
            row = min(r, a.N - 1 - nt * BN);
        }
        wo[i] = row * kbytes + ((lane & 7) ^ (r & 7)) * 16;
    }
    const char* x0 = (const char*)(second ? a.x2 : a.x) + (long)m0 * xbytes + (long)c_lo * 128;
    const char* w0 = (const char*)(second ? a.w2 : a.w) + (long)nt * (GLU ? BN / 2 : BN) * kbytes + (long)c_lo * 128;
    // tiles start at different chunks and wrap round: in step they would all ask for the same
    // 128 bytes of rows a power of two apart, which few of the memory channels hold
    int at = ((blockIdx.x >> 3) / a.mblocks) % n;
    int to = 0;                                        // buffer of the next chunk loaded
    auto stage = [&]() {
        if (has_w) {
            char* base = smem + W0 + to * WB;
            const char* wp = w0 + (long)at * 128;
#pragma unroll
            for (int i = 0; i < WP; ++i)
                tg_load<ONCE ? 2 : 0>(wp + wo[i], base + (lw * WP + i) * 1024);
        }
        if (has_x) {
            char* base = smem + to * XB;
            const char* xp = x0 + (long)at * 128;
#pragma unroll
            for (int i = 0; i < XP; ++i) tg_load<0>(xp + xo[i], base + ((lw * XP + i) % XPT) * 1024);
        }
        at = at + 1 == n ? 0 : at + 1;
        to = to + 1 == depth ? 0 : to + 1;
    };
    // until at most `left` chunks of the wave's loads are in flight; ALL: as many as a full ring has
    auto wait = [&](int left) {
        if (!APART) tg_wait_chunks<XP + WP, D - 1>(left);
        else if (has_w) tg_wait_chunks<WP, D - 1>(left);
        else tg_wait_chunks<XP, DX - 1>(left);
    };
    auto wait_full = [&]() {
        if (!APART) tg_wait<(XP + WP) * (D - 2)>();
        else if (has_w) tg_wait<WP * (D - 2)>();
        else tg_wait<XP * (DX - 2)>();
    };

    tg_f32x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = {0.f, 0.f, 0.f, 0.f};

    int off[2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
        off[h] = lrow * 128 + (((h * 4 + lslot) ^ (lrow & 7)) << 4);
    const int xoff = wm * (BM / WM) * 128, woff = W0 + wn * (BN / WN) * 128;
    vec8 xa[2][FM], wb[2][FN];
    auto read = [&](int bx, int bw, int h) {
        const char* xs = smem + bx * XB + xoff + off[h];
        const char* ws = smem + bw * WB + woff + off[h];
#pragma unroll
        for (int j = 0; j < FN; ++j) wb[h][j] = *reinterpret_cast<const vec8*>(ws + j * 2048);
#pragma unroll
        for (int i = 0; i < FM; ++i) xa[h][i] = *reinterpret_cast<const vec8*>(xs + i * 2048);
    };
    auto mma = [&](int h) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = MF::mfma(wb[h][j], xa[h][i], acc[i][j]);
    };

#pragma unroll
    for (int i = 0; i < D; ++i)
        if (i < n && (i < DX || has_w)) stage();
    wait(min(depth, n) - 1);
    __builtin_amdgcn_s_barrier();
    read(0, 0, 0);
    int bx = 0, bw = 0, t = 0;
    // The second half of a chunk is read before the products of the first, and the first half of
    // the next chunk before those of the second. Between them every wave has read the chunk, which
    // its successor a ring on then overwrites, and has its loads of the next one.
    for (; t < n - D; ++t) {
        const int nx = bx == DX - 1 ? 0 : bx + 1, nw = bw == D - 1 ? 0 : bw + 1;
        read(bx, bw, 1);
        mma(0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        wait_full();
        __builtin_amdgcn_s_barrier();
        read(nx, nw, 0);
        stage();
        mma(1);
        bx = nx;
        bw = nw;
    }
    for (; t < n; ++t) {
        const int nx = bx == DX - 1 ? 0 : bx + 1, nw = bw == D - 1 ? 0 : bw + 1;
        read(bx, bw, 1);
        mma(0);
        if (t + 1 < n) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            wait(min(depth - 2, n - t - 2));
            __builtin_amdgcn_s_barrier();
            read(nx, nw, 0);
            if (APART && !has_w && t + DX < n) stage();
        }
        mma(1);
        bx = nx;
        bw = nw;
    }

    // w's rows stand in the products' rows: register r of acc[i][j] is column j * 16 +
    // lane / 16 * 4 + r of row i * 16 + lane % 16
    constexpr int FC = GLU ? FN / 2 : FN, CW = GLU ? BN / 2 : BN;
    const int cols = GLU ? a.N / 2 : a.N;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int m = m0 + wm * (BM / WM) + i * 16 + lrow;
        if (m >= a.M) continue;
#pragma unroll
        for (int j = 0; j < FC; ++j) {
            const int c = nt * CW + wn * (CW / WN) + j * 16 + lslot * 4;
            if (c >= cols) continue;
            tg_f32x4 v = acc[i][j];
            if constexpr (GLU) {
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = tg_act<GLU>(v[r]) * acc[i][j + FC][r];
            } else if (a.part) {
                *reinterpret_cast<tg_f32x4*>(a.part + ((long)slice * a.M + m) * a.N + c) = v;
                continue;
            } else if (a.bias) {
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] += VecTraits<T>::to_float(((const T*)a.bias)[c + r]);
            }
            __align__(8) T o[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] = VecTraits<T>::from_float(v[r]);
            *reinterpret_cast<int2*>((T*)a.y + (long)m * cols + c) = *reinterpret_cast<int2*>(o);
        }
    }
}

// tile_gemm_kernel for one row of attention's output that is still in shares of its keys (n of each
// head's D values, with their maxima and sums): 4 waves add up the chunk of K that the workgroup
// has, which is little, while the others have their first D chunks of w on the way. A wave reads
// back from LDS what it loaded itself, so these wait for the sum, once, and never for each other.
// Bound by latency, hence one launch for two: 2048 x 2048 behind 6 shares of 32 heads of 64, attention
// included, 11.8 -> 10.0 us (see DECODE_SHARES for where the line lies).
template <typename T, int BN, int WN, int D>
__global__ __launch_bounds__(64 * (WN + 4)) void shares_gemm_kernel(const TgArgs a,
                                                                    const float* __restrict__ o,
                                                                    const float* __restrict__ ml,
                                                                    const int shares, const int HD) {
    using MF = TgMfma<T>;
    using VT = VecTraits<T>;
    using vec8 = typename MF::vec8;
    constexpr int FN = BN / WN / 16, WP = BN / 8 / WN, WB = BN * 128;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    T* const xs = reinterpret_cast<T*>(smem + D * WB);       // of the workgroup's part of K

    const int item = (blockIdx.x & 7) * a.per_xcd + (blockIdx.x >> 3);
    if (item >= a.work) return;
    const int nt = item % a.ntiles, slice = item / a.ntiles;
    const int chunks = a.K / TG_BK;
    const int c_lo = (int)((long)slice * chunks / a.splits);
    const int n = (int)((long)(slice + 1) * chunks / a.splits) - c_lo;
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    if (wid >= WN) {
        constexpr int U = 8;                                 // shares whose loads go out together
        for (int i = (threadIdx.x - WN * 64) * 4; i < n * TG_BK; i += 1024) {
            const int k = c_lo * TG_BK + i, head = k / HD;
            const float* op = o + (long)head * shares * HD + k % HD;
            const float* mp = ml + (long)head * shares * 2;
            float m = -1e30f, l = 0.f;
            tg_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
            for (int s0 = 0; s0 < shares; s0 += U) {
                tg_f32x4 v[U];
                float2 p[U];
                float mn = m;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int s = min(s0 + u, shares - 1);
                    p[u] = *reinterpret_cast<const float2*>(mp + s * 2);
                    v[u] = *reinterpret_cast<const tg_f32x4*>(op + (long)s * HD);
                }
#pragma unroll
                for (int u = 0; u < U; ++u) mn = fmaxf(mn, p[u].x);
                const float f = __expf(m - mn);
                m = mn;
                l *= f;
                acc *= f;
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (s0 + u < shares) {
                        const float e = __expf(p[u].x - m);
                        l += p[u].y * e;
                        acc += v[u] * e;
                    }
            }
            const float inv = l > 0.f ? 1.f / l : 0.f;
            __align__(8) T r[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) r[j] = VT::from_float(acc[j] * inv);
            *reinterpret_cast<int2*>(xs + i) = *reinterpret_cast<int2*>(r);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        return;
    }

    const int lrow = lane & 15, lslot = lane >> 4, prow = lane >> 3;
    const unsigned kbytes = (unsigned)a.K * sizeof(T);
    unsigned wo[WP];
#pragma unroll
    for (int i = 0; i < WP; ++i) {
        const int q = (wid * WP + i) * 8 + prow;
        wo[i] = min(q, a.N - 1 - nt * BN) * kbytes + ((lane & 7) ^ (q & 7)) * 16;
    }
    const char* w0 = (const char*)a.w + (long)nt * BN * kbytes + (long)c_lo * 128;
    const int first = (blockIdx.x >> 3) % n;                 // as in tile_gemm_kernel
    int at = first, to = 0;
    auto stage = [&]() {
        char* base = smem + to * WB + wid * (WP * 1024);
        const char* wp = w0 + (long)at * 128;
#pragma unroll
        for (int i = 0; i < WP; ++i) tg_load<2>(wp + wo[i], base + i * 1024);
        at = at + 1 == n ? 0 : at + 1;
        to = to + 1 == D ? 0 : to + 1;
    };
    tg_f32x4 acc[FN];
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[j] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < D; ++i)
        if (i < n) stage();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    int bw = 0, c = first;
    for (int t = 0; t < n; ++t) {
        tg_wait_chunks<WP, D - 1>(n - 1 - t);
        vec8 xa[2], wb[2][FN];
        const char* wp = smem + bw * WB + wid * (WP * 1024) + lrow * 128;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            xa[h] = *reinterpret_cast<const vec8*>(xs + c * TG_BK + h * 32 + lslot * 8);
#pragma unroll
            for (int j = 0; j < FN; ++j)
                wb[h][j] = *reinterpret_cast<const vec8*>(
                    wp + j * 2048 + (((h * 4 + lslot) ^ (lrow & 7)) << 4));
        }
        if (t + D < n) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            stage();
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[j] = MF::mfma(wb[h][j], xa[h], acc[j]);
        c = c + 1 == n ? 0 : c + 1;
        bw = bw + 1 == D ? 0 : bw + 1;
    }
    if (lrow) return;                                        // (16 times the same row)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const int col = nt * BN + wid * (BN / WN) + j * 16 + lslot * 4;
        if (col >= a.N) continue;
        if (a.part) {
            *reinterpret_cast<tg_f32x4*>(a.part + (long)slice * a.N + col) = acc[j];
            continue;
        }
        __align__(8) T r[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) r[q] = VT::from_float(acc[j][q]);
        *reinterpret_cast<int2*>((T*)a.y + col) = *reinterpret_cast<int2*>(r);
    }
}

// y = sum of the parts (+ bias)
template <typename T>
__global__ __launch_bounds__(256) void tile_sum_kernel(T* __restrict__ y,
                                                       const float* __restrict__ part,
                                                       const T* __restrict__ bias, const long MN,
                                                       const int N, const int splits) {
    const long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= MN) return;
    tg_f32x4 s = *reinterpret_cast<const tg_f32x4*>(part + i);
    for (int k = 1; k < splits; ++k) s += *reinterpret_cast<const tg_f32x4*>(part + k * MN + i);
    __align__(8) T o[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (bias) s[r] += VecTraits<T>::to_float(bias[i % N + r]);
        o[r] = VecTraits<T>::from_float(s[r]);
    }
    *reinterpret_cast<int2*>(y + i) = *reinterpret_cast<int2*>(o);
}

// The tile of a shape. A chunk of w (BN rows of 128 bytes) is what a workgroup streams, x comes
// again and again from the L2: few rows take small tiles with a deep ring, so that a CU has 64 KB
// and more on the way; many rows take tall ones, for fewer reads of x and w from LDS a product.
enum TgTile { T16, T16N, T32, T32N, T64, T64N, T64W, T128, T128N, T128W, T128B, T192, T256, T256W };

struct TgPlan {
    TgTile tile;
    int bm, bn, splits, tiles;
};

// parts of K that are worth their sum, see below
long tg_parts(long M, long K, long tiles, bool whole) {
    const bool small = whole ? M > 64 && M <= 128 && K >= 512 : true;
    if (small && K <= 768 && tiles * (K / 128) <= (M <= 16 ? 128 : 64)) return K / 128;
    return std::min(16L, std::max(std::min(8L, K / 256), K / 384));
}

// What is not taken (splits == 0) goes to the library. Times of 16-bit products on weights that
// are not in a cache, 32-bit parts left to the next kernel, here / library (or the kernels with a
// ring of 3 chunks that were here before):
//   rows   (6144, 4096)  (4096, 4096)  (28672, 4096)  (4096, 14336)  (57344, 8192)
//   1       10.7 / 13.6    7.7 / 10.3    40.7 /  49.9   20.9 / 27.4   150 / 160
//   16      11.0 / 16.2    8.1 / 13.2    39.9 /  51.7   20.7 / 26.8   151 / 164
//   64      12.9 / 19.7   10.0 / 15.5    43.6 /  54.3   23.4 / 32.4   166 / 184
//   128     17.0 / 21.4   14.0 / 18.9    50.5 /  60.4   29.8 / 43.2   154 / 221
//   192     21.7 / 26.2   17.1 / 20.3    62.1 /  79     35.3 / 66.9   224 / 232
//   256     22.5 / 27.2   17.8 / 25.2    64.7 /  84.1   37.9 / 53.4   268 / 239
//   512     34.9 / 38.2   25.5 / 29.7     123 /   105   62.1 / 89.2   442 / 375
// so up to 256 rows, unless the tiles of more than 128 rows need a second round of the chip, and
// up to 512 rows where the tiles of the outputs alone leave CUs idle. Parts of K fill the 256 CUs
// once, each with 4 chunks or more, and 6 where there are more than 8 of them: a part is as many
// bytes to write and to read as it has of weights at 128 rows and 4 chunks. Product and the norm
// that adds up, with 2 chunks or more / so: 93 rows (2048, 2048) 15.2 / 12.9 us, 128 rows
// (1024, 2048) 14.2 / 12.2, 64 rows (1024, 3072) 9.9 / 9.4, 256 rows (1024, 1024) 13.1 / 10.9,
// 1 row (2048, 1024) 6.5 / 6.0; 128 rows (1024, 4096) in 16 / 10 / 8 parts 15.5 / 14.4 / 14.6,
// 256 rows 15.0 / 14.5 / 16.0. A K of up to 768 in parts of 2 chunks, where these are at most 64
// workgroups (128 for up to 16 rows): parts of 2 / of 4, 1 row (2048, 512) 5.4 / 5.7 us, (1024, 256)
// 5.1 / 5.5, 93 rows (512, 256) 7.7 / 8.7, (1024, 512) 8.6 / 9.3, (768, 768) 9.2 / 9.7, 64 rows (1024, 512)
// 6.7 / 6.9; with more of them 93 rows (4096, 512) 11.4 / 10.9, 400 (1024, 512) 11.6 / 11.1, (2048, 256)
// 12.0 / 10.4, 48 (768, 768) even, and of a longer K 64 (512, 1024) 7.5 / 6.9. Where the sum is a launch of its
// own, see below, only of a K from 512 on and for 65 to 128 rows: 93 (512, 512) 7.8 / 8.2, (2048, 512)
// 8.4 / 9.0; else 48 (512, 512) 5.8 / 5.6, 1 (768, 768) 5.4 / 5.0, and 2 parts / one 93 (512, 256) 7.1 / 6.2,
// 1 (1024, 256) 4.4 / 3.2.
// From 128 rows on what bounds them is what a CU takes in, x and w together: 40 to 43 GB/s in every
// tile tried (chunks of x laid out in a row changed nothing, deeper rings of either no more), so a
// tile of 192 rows, which reads w once for them, and x apart from w in time: 129 to 192 rows
// 71.8 -> 62.9, 39.7 -> 35.0, 23.1 -> 20.8 (160 rows of the third, fourth and first shape). 193 to 256
// rows in one tile as well, its w apart from the cache as nothing else reads it (tiles of 128 x 256 read
// w twice): 256 rows of the third shape 69.5 -> 64.7, (32000, 4096) 76 -> 70, (8192, 28672) 139 -> 134,
// (10240, 8192) 51.3 -> 50.0; more than 256 rows would fill a second tile in part only: 300 rows of
// the first shape 33.9 with it, 28.4 without. Gate|up of few columns takes tiles of
// 128 also where 256 would leave half of the CUs idle: 128 rows of the third shape 72.0 -> 50.5.
// 33 to 64 rows of x are a third of what a tile of 128 columns takes in: tiles of 256 where these fill
// the chip's rounds. 64 rows, 128 / 256 columns: (128256, 4096) 177 / 170 us, (57344, 8192) 148 / 138,
// (65536, 2048) 46.1 / 43.5; in 2.3 rounds (151936, 2048) 116 / 120, in half of one (28672, 4096) 42 / 64.
// `whole`: no kernel follows that would add up parts. Then up to 64 rows take tiles of half the width
// where these fill most of the chip undivided, also where those of the full width in two parts are
// a little faster by themselves: the sum is a launch of its own, some 3 us. 48 rows, undivided /
// two parts without their sum / library: (11408, 2048) 14.3 / 13.4 / 17.6 us, (16384, 2048)
// 15.5 / 16.6 / 19.1, (12288, 4096) 23.6 / 22.5 / 25.2; 100 rows of the last 33.0 / 27.2 / 32.4.
// From there to 128 rows tiles of 128 columns, for 256 in twice as many parts, where K is short and
// they or their parts take 180 CUs: 128 rows (32000, 4096) 59.0 -> 52.3 us, (32000, 2048) 38.9 -> 29.1,
// (24576, 4096) 51.0 -> 46.8, (16384, 4096) 39.8 -> 36.9; on 157 CUs (20000, 4096) 42.9 -> 44.5, and
// (32000, 8192) 94.1 -> 95.2.
TgPlan tg_plan(long M, long N, long K, bool glu, bool whole) {
    TgPlan p{T16, 16, 128, 0};
    if (M < 1 || M > 512 || N < 64 || N % (glu ? 8 : 4) || K < (whole && !glu ? 128 : 256) || K % TG_BK ||
        K * N * 2 >= (1L << 32))
        return p;
    // half the width where that many more tiles spare parts of K, or with GLU fill the chip
    const bool narrow = glu ? N < 25600 : N <= 4096 || (whole && M <= 64 && N > 8192 && N <= 16384);
    const long wides = (N + 255) / 256, rounds = (wides + 255) / 256;
    const long tiles128 = (N + 127) / 128;
    const bool filled = whole && K <= 4096 && tiles128 <= 256 && tiles128 * (256 / tiles128) >= 180;
    const bool wide = wides * 100 >= rounds * 256 * 85;
    if (M <= 16) p = narrow ? TgPlan{T16N, 16, 64, 0} : TgPlan{T16, 16, 128, 0};
    else if (M <= 32) p = narrow ? TgPlan{T32N, 32, 64, 0} : TgPlan{T32, 32, 128, 0};
    else if (M <= 64 && wide) p = {T64W, 64, 256, 0};
    else if (M <= 64) p = narrow ? TgPlan{T64N, 64, 64, 0} : TgPlan{T64, 64, 128, 0};
    else if (M <= 128 && narrow && glu) p = {T128N, 128, 64, 0};
    else if (M <= 128 && (glu ? N < 49152 : N * K < (60 << 20) || filled)) p = {T128, 128, 128, 0};
    else if (M <= 128) p = {T128W, 128, 256, 0};
    else if (N * K <= (20 << 20)) p = {T128B, 128, 128, 0};
    else if (M <= 192) p = {T192, 192, 128, 0};
    else if (M <= 256) p = {T256, 256, 128, 0};
    else p = {T256W, 128, 256, 0};
    const long tiles = (M + p.bm - 1) / p.bm * ((N + p.bn - 1) / p.bn);
    if (M > 128 && tiles > 256) return p;
    if (M > 256 && (tiles > 128 || glu)) return p;
    p.tiles = (int)tiles;
    p.splits = glu ? 1 : (int)std::max(1L, std::min(256 / tiles, tg_parts(M, K, tiles, whole)));
    return p;
}

template <typename T, int BM, int BN, int WM, int WN, int D, int GLU, bool ONCE, int DX = D>
void tg_go(TgArgs& a, hipStream_t stream) {
    a.mblocks = (a.M + BM - 1) / BM;
    a.ntiles = (a.N + BN - 1) / BN;
    a.work = a.mblocks * a.ntiles * a.splits * (a.w2 ? 2 : 1);
    a.per_xcd = (a.work + 7) / 8;
    constexpr int LDS = (DX * BM + D * BN) * 128;
    static_assert(LDS <= 163840, "the rings do not fit");
    auto* k = tile_gemm_kernel<T, BM, BN, WM, WN, D, DX, GLU, ONCE>;
    TORCH_CHECK(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    LDS) == hipSuccess, "tile_gemm: LDS");
    hipLaunchKernelGGL(k, dim3(a.per_xcd * 8), dim3(64 * WM * WN), LDS, stream, a);
    HIP_CHECK_KERNEL();
}

template <typename T, int GLU>
void tg_tile(TgArgs& a, TgTile tile, hipStream_t s) {
    switch (tile) {
        case T16: tg_go<T, 16, 128, 1, 4, 4, GLU, true>(a, s); break;
        case T16N: tg_go<T, 16, 64, 1, 2, 8, GLU, true>(a, s); break;
        case T32: tg_go<T, 32, 128, 1, 4, 4, GLU, true>(a, s); break;
        case T32N: tg_go<T, 32, 64, 1, 2, 6, GLU, true>(a, s); break;
        case T64: tg_go<T, 64, 128, 1, 4, 3, GLU, true>(a, s); break;
        case T64N: tg_go<T, 64, 64, 2, 2, 5, GLU, true>(a, s); break;
        case T64W: tg_go<T, 64, 256, 1, 8, 3, GLU, true>(a, s); break;
        case T128: tg_go<T, 128, 128, 2, 4, 5, GLU, true>(a, s); break;
        case T128N: tg_go<T, 128, 64, 4, 2, 6, GLU, true>(a, s); break;
        case T128W: tg_go<T, 128, 256, 2, 4, 3, GLU, true>(a, s); break;
        case T128B: tg_go<T, 128, 128, 2, 4, 5, GLU, false>(a, s); break;
        case T192: tg_go<T, 192, 128, 4, 2, 5, GLU, true, 3>(a, s); break;
        case T256: tg_go<T, 256, 128, 4, 2, 3, GLU, true>(a, s); break;
        case T256W: tg_go<T, 128, 256, 2, 4, 3, GLU, false>(a, s); break;
    }
}

}  // namespace

// Parts of K that tile_gemm takes for this shape, 0: none, it is the library's.
long tile_gemm_splits(long M, long N, long K, long glu, bool whole) {
    return tg_plan(M, N, K, glu != PLAIN, whole).splits;
}

namespace {

// rows of x may lie further apart than they are long (columns of a wider tensor)
void tg_operands(const torch::Tensor& x, const torch::Tensor& w) {
    TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && x.size(1) == w.size(1), "tile_gemm: shapes");
    TORCH_CHECK(x.is_cuda() && w.device() == x.device(), "tile_gemm: operands of one GPU");
    TORCH_CHECK(x.stride(1) == 1 && (x.size(0) < 2 || (x.stride(0) >= x.size(1) &&
                x.stride(0) % 8 == 0 && x.stride(0) < (1L << 20))) && w.is_contiguous() &&
                x.scalar_type() == w.scalar_type(), "tile_gemm: rows of one type");
    TORCH_CHECK(((size_t)x.data_ptr() | (size_t)w.data_ptr()) % 16 == 0, "tile_gemm: alignment");
    TORCH_CHECK(x.scalar_type() == at::kBFloat16 || x.scalar_type() == at::kHalf,
                "tile_gemm: bf16/f16 only");
}

unsigned tg_row_bytes(const torch::Tensor& x) {
    return (unsigned)(x.size(0) < 2 ? x.size(1) : x.stride(0)) * 2;
}

void tg_launch(TgArgs& a, TgTile tile, bool bf, long glu) {
    auto stream = at::hip::getCurrentHIPStream();
    if (bf) {
        if (glu == SILU) tg_tile<__hip_bfloat16, SILU>(a, tile, stream);
        else if (glu == GELU) tg_tile<__hip_bfloat16, GELU>(a, tile, stream);
        else tg_tile<__hip_bfloat16, PLAIN>(a, tile, stream);
    } else {
        TORCH_CHECK(glu != GELU, "tile_gemm: gelu in bf16 only");
        if (glu == SILU) tg_tile<__half, SILU>(a, tile, stream);
        else tg_tile<__half, PLAIN>(a, tile, stream);
    }
}

}  // namespace

// x (M, K) @ w (N, K)^T. `splits` 0: as planned, which leaves (splits, M, N) parts in fp32 where
// there are several (`parts`) or sums them up. `glu`: silu (1) or gelu (2) of the first half of the
// columns times the second.
torch::Tensor tile_gemm(torch::Tensor x, torch::Tensor w, c10::optional<torch::Tensor> bias,
                        long splits, bool parts, long glu) {
    tg_operands(x, w);
    TORCH_CHECK(glu >= PLAIN && glu <= GELU, "tile_gemm: glu");
    const bool bf = x.scalar_type() == at::ScalarType::BFloat16;
    TgArgs a{};
    a.M = x.size(0);
    a.K = x.size(1);
    a.N = w.size(0);
    a.xbytes = tg_row_bytes(x);
    const TgPlan plan = tg_plan(a.M, a.N, a.K, glu, !parts);
    TORCH_CHECK(plan.splits > 0, "tile_gemm: shape not taken");
    TORCH_CHECK(splits >= 0 && splits <= a.K / TG_BK && !(glu && splits > 1), "tile_gemm: splits");
    a.splits = splits ? splits : plan.splits;
    TORCH_CHECK(!bias || (!parts && !glu && bias->is_contiguous() && bias->numel() == a.N &&
                          bias->scalar_type() == x.scalar_type()), "tile_gemm: bias");
    torch::Tensor y, part;
    if (a.splits > 1) {
        part = torch::empty({a.splits, a.M, a.N}, x.options().dtype(torch::kFloat32));
        a.part = part.data_ptr<float>();
    }
    if (a.splits == 1 || !parts) {
        y = torch::empty({a.M, glu ? a.N / 2 : a.N}, x.options());
        a.y = y.data_ptr();
    }
    a.x = x.data_ptr();
    a.w = w.data_ptr();
    a.bias = bias ? bias->data_ptr() : nullptr;
    auto stream = at::hip::getCurrentHIPStream();
    tg_launch(a, plan.tile, bf, glu);
    if (a.splits == 1) return y;
    if (parts) return part;
    const long MN = (long)a.M * a.N;
    const dim3 grid((unsigned)((MN / 4 + 255) / 256));
    if (bf)
        hipLaunchKernelGGL((tile_sum_kernel<__hip_bfloat16>), grid, dim3(256), 0, stream,
                           (__hip_bfloat16*)a.y, a.part, (const __hip_bfloat16*)a.bias, MN, a.N,
                           a.splits);
    else
        hipLaunchKernelGGL((tile_sum_kernel<__half>), grid, dim3(256), 0, stream, (__half*)a.y,
                           a.part, (const __half*)a.bias, MN, a.N, a.splits);
    HIP_CHECK_KERNEL();
    return y;
}

// Parts of K of x @ w^T and then of x2 @ w2^T, products of one shape: (2 n, M, N) in fp32.
torch::Tensor tile_gemm_pair(torch::Tensor x, torch::Tensor w, torch::Tensor x2, torch::Tensor w2) {
    tg_operands(x, w);
    tg_operands(x2, w2);
    TORCH_CHECK(x.sizes() == x2.sizes() && w.sizes() == w2.sizes() &&
                x.scalar_type() == x2.scalar_type(), "tile_gemm_pair: shapes");
    TgArgs a{};
    a.M = x.size(0);
    a.K = x.size(1);
    a.N = w.size(0);
    const TgPlan plan = tg_plan(a.M, a.N, a.K, false, false);
    TORCH_CHECK(plan.splits > 0, "tile_gemm_pair: shape not taken");
    // the two fill the CUs together; 4 parts each where K has 4 chunks for each, and from there on half as
    // many as one product takes (product and the norm that adds up, 2 / 4 parts each of K 1024: 16 rows
    // (512, 1024) 8.0 / 6.9 us, 100 rows (1024, 1024) 12.9 / 11.5; 4 / 8 of K 2048: 100 rows (2048, 2048)
    // 16.3 / 19.0, 48 rows (1024, 2048) 9.6 / 10.3)
    const long worth = std::max(std::min(4L, (long)a.K / 256), tg_parts(a.M, a.K, 256, false) / 2);
    a.splits = (int)std::max(1L, std::min(128L / plan.tiles, worth));
    torch::Tensor part = torch::empty({2 * a.splits, a.M, a.N}, x.options().dtype(torch::kFloat32));
    a.part = part.data_ptr<float>();
    a.x = x.data_ptr();
    a.w = w.data_ptr();
    a.x2 = x2.data_ptr();
    a.w2 = w2.data_ptr();
    a.xbytes = tg_row_bytes(x);
    a.xbytes2 = tg_row_bytes(x2);
    tg_launch(a, plan.tile, x.scalar_type() == at::kBFloat16, PLAIN);
    return part;
}

namespace {

template <typename T, int BN, int WN, int D>
void tg_shares_go(TgArgs& a, const float* o, const float* ml, int shares, int HD, hipStream_t stream) {
    a.mblocks = 1;
    a.ntiles = (a.N + BN - 1) / BN;
    a.work = a.ntiles * a.splits;
    a.per_xcd = (a.work + 7) / 8;
    const int longest = (a.K / TG_BK + a.splits - 1) / a.splits, lds = D * BN * 128 + longest * 128;
    TORCH_CHECK(lds <= 163840, "shares_gemm: K");
    auto* k = shares_gemm_kernel<T, BN, WN, D>;
    // (a limit of the function, the same in every call)
    TORCH_CHECK(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    163840) == hipSuccess, "shares_gemm: LDS");
    hipLaunchKernelGGL(k, dim3(a.per_xcd * 8), dim3(64 * (WN + 4)), lds, stream, a, o, ml, shares, HD);
    HIP_CHECK_KERNEL();
}

}  // namespace

// o (heads, n, D) and ml (heads, n, 2): attention's shares of one row. Their sum @ w^T, with its
// parts of K as tile_gemm leaves them.
torch::Tensor shares_gemm(const torch::Tensor& o, const torch::Tensor& ml, long n, const torch::Tensor& w) {
    TgArgs a{};
    a.M = 1;
    a.K = w.size(1);
    a.N = w.size(0);
    const long heads = ml.numel() / (2 * n);
    const int HD = (int)(a.K / heads);
    TORCH_CHECK(o.numel() == n * a.K && heads * HD == a.K && HD % 4 == 0, "shares_gemm: shares");
    TORCH_CHECK(w.is_contiguous() && (size_t)w.data_ptr() % 16 == 0 && w.device() == o.device(),
                "shares_gemm: weight");
    const TgPlan plan = tg_plan(1, a.N, a.K, false, false);
    TORCH_CHECK(plan.splits > 0, "shares_gemm: shape not taken");
    a.splits = plan.splits;
    torch::Tensor y;
    if (a.splits > 1) {
        y = torch::empty({a.splits, 1, a.N}, o.options());
        a.part = y.data_ptr<float>();
    } else {
        y = torch::empty({1, a.N}, w.options());
        a.y = y.data_ptr();
    }
    a.w = w.data_ptr();
    auto s = at::hip::getCurrentHIPStream();
    const float *op = o.data_ptr<float>(), *mp = ml.data_ptr<float>();
    const bool narrow = plan.tile == T16N;
    if (w.scalar_type() == at::kBFloat16) {
        if (narrow) tg_shares_go<__hip_bfloat16, 64, 2, 8>(a, op, mp, (int)n, HD, s);
        else tg_shares_go<__hip_bfloat16, 128, 4, 4>(a, op, mp, (int)n, HD, s);
    } else {
        if (narrow) tg_shares_go<__half, 64, 2, 8>(a, op, mp, (int)n, HD, s);
        else tg_shares_go<__half, 128, 4, 4>(a, op, mp, (int)n, HD, s);
    }
    return y;
}
