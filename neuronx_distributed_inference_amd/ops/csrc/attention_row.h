// One query row against its visible keys in 32-bit multiply-adds, by one wave.
//
// The matrix-core kernels multiply whole tiles of V by probabilities that are 0 where a row does
// not see a key, and by the small parts of those that are not. With finite values nothing is
// wrong with that. A value that is not (an overflow in a later token of the same portion, in a
// row before a window) gives 0 * Inf = NaN to rows that do not see it, and Inf - Inf to those that
// do. The kernels notice at the end: sums that are finite under an accumulator that is not. Such
// rows, and no others, are done again here, where a key that is not seen is not read.
#pragma once

#include "common.h"

// slot(key): element offset of the key's row in k and v, or -1 where it is not seen. m (log2
// units), l: maximum and sum; acc: channels lane * D/64 and on.
template <int D, typename T, typename CT, typename Slot>
DEV_INLINE void attend_row(const T* q, const CT* k, const CT* v, const int lo, const int hi,
                           const float scale_log2, Slot slot, float& m, float& l,
                           float (&acc)[D / 64]) {
    constexpr int PER = D / 64;
    const int lane = threadIdx.x & 63;
    m = -INFINITY;
    l = 0.f;
#pragma unroll
    for (int e = 0; e < PER; ++e) acc[e] = 0.f;
#pragma unroll 1                             // rarely run: few registers
    for (int base = lo; base < hi; base += 64) {
        const long off = base + lane < hi ? slot(base + lane) : -1;
        float s = -INFINITY;
        if (off >= 0) {
            float d = 0.f;
#pragma unroll 2
            for (int c = 0; c < D; c += 8) {
                const Vec8<T> a = load_vec8(q + c);
                const Vec8<CT> x = load_vec8(k + off + c);
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    d += VecTraits<T>::to_float(a.v[i]) * VecTraits<CT>::to_float(x.v[i]);
            }
            s = d * scale_log2;
        }
        const float mn = fmaxf(m, wave_reduce_max(s));
        const float f = m == -INFINITY ? 0.f : exp2f(m - mn);
        const float p = off < 0 ? 0.f : exp2f(s - (mn == -INFINITY ? 0.f : mn));
        m = mn;
        l = l * f + wave_reduce_sum(p);
#pragma unroll
        for (int e = 0; e < PER; ++e) acc[e] *= f;
        const int n = min(64, hi - base);
#pragma unroll 4
        for (int j = 0; j < n; ++j) {
            const long at = __shfl(off, j, WAVE_SIZE);
            const float pj = __shfl(p, j, WAVE_SIZE);
            if (at < 0) continue;
#pragma unroll
            for (int e = 0; e < PER; ++e)
                acc[e] += pj * VecTraits<CT>::to_float(v[at + lane * PER + e]);
        }
    }
}
