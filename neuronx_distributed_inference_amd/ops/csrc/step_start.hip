// What a model step does before its first product, in a launch each. A decode step of a small
// model is a chain of some 50 launches of 2 to 10 us, of which these were 12 (embedding rows, two
// clamps and two gathers for rope, casts of positions and rows, the first norm; 4 copies into the
// captured graph's inputs), and 30 for paged caches: nothing in them takes time but the launch,
// about 2.3 us behind one another. Steps, before -> now: 1 row of a 1B model (4 layers) 251 ->
// 231 us, 13 rows of 70B (2 layers) 807 -> 749, 48 rows of a hybrid decoder (4 layers, paged)
// 891 -> 823; prompts (launched one by one): 93 tokens 547 -> 484, 512 tokens onto 3500 in pages
// 1589 -> 1526.

#include "common.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include <c10/macros/Macros.h>

namespace {

// Prompts of a batch one after the other without padding, by value: a row finds its own in here.
constexpr int PROMPTS = 256;
struct Packed {
    int n, S;                  // prompts; tokens between their first ones in ids and positions
    int starts[PROMPTS + 1];   // first row of each
};

// One workgroup per token: h = embedding row, x = its RMS norm, cos and sin = rope's table rows at
// the position (clamped into the table), position and cache row as int32. V values of 16 bytes of
// a row a thread. PACKED: rows are the tokens of prompts alone (before: every product, norm and
// activation of the model ran over the padding as well; 5 prompts of up to 777 tokens of an 8B model,
// 4 layers, 4040 rows of which 2700 to 3200 are tokens, 5.68 -> 5.08 ms, 93 tokens of a 1B model
// in a bucket of 124 382 -> 333 us, most of it the launches that padded); sid32 is then a row's
// cache row, and the first workgroup writes out where prompts start and their cache rows.
template <typename T, int V, typename S, bool PACKED>
__global__ __launch_bounds__(1024) void step_start_kernel(
    T* __restrict__ h, T* __restrict__ x, float* __restrict__ cos, float* __restrict__ sin,
    int* __restrict__ pos32, int* __restrict__ sid32, const long* __restrict__ ids,
    const long* __restrict__ positions, const S* __restrict__ seq_ids,
    const T* __restrict__ table, const float* __restrict__ cos_table,
    const float* __restrict__ sin_table, const T* __restrict__ weight, const float eps,
    const int H, const int D, const int B, const long vocab, const long table_rows,
    const std::conditional_t<PACKED, Packed, int> packed, int* __restrict__ starts,
    int* __restrict__ prompt_sid) {
    __shared__ float red[16];
    using VT = VecTraits<T>;
    const long row = blockIdx.x;
    long from = row;
    if constexpr (PACKED) {
        int lo = 0, hi = packed.n;                 // starts[lo] <= row < starts[hi]
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (packed.starts[mid] <= row) lo = mid;
            else hi = mid;
        }
        from = (long)lo * packed.S + row - packed.starts[lo];
        if (threadIdx.x == 0) sid32[row] = (int)seq_ids[lo];
        if (row == 0)
            for (int i = threadIdx.x; i <= packed.n; i += blockDim.x) {
                starts[i] = packed.starts[i];
                if (i < packed.n) prompt_sid[i] = (int)seq_ids[i];
            }
    }
    const long id = ids[from], pos = positions[from];
    CUDA_KERNEL_ASSERT(id >= 0 && id < vocab);
    const long at = min(max(pos, 0l), table_rows - 1);
    for (int i = threadIdx.x * 4; i < D; i += blockDim.x * 4) {
        *reinterpret_cast<float4*>(cos + row * D + i) =
            *reinterpret_cast<const float4*>(cos_table + at * D + i);
        *reinterpret_cast<float4*>(sin + row * D + i) =
            *reinterpret_cast<const float4*>(sin_table + at * D + i);
    }
    if (threadIdx.x == 0) {
        pos32[row] = (int)pos;
        if constexpr (!PACKED)
            if (seq_ids && row < B) sid32[row] = (int)seq_ids[row];
    }
    Vec8<T> v[V];
    float ssq = 0.f;
#pragma unroll
    for (int k = 0; k < V; ++k) {
        const int i = (k * blockDim.x + threadIdx.x) * 8;
        if (i >= H) continue;
        v[k] = load_vec8(table + id * H + i);
        store_vec8(h + row * H + i, v[k]);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float f = VT::to_float(v[k].v[j]);
            ssq += f * f;
        }
    }
    ssq = block_reduce_sum(ssq, red);
    const float inv = rsqrtf(ssq / H + eps);
#pragma unroll
    for (int k = 0; k < V; ++k) {
        const int i = (k * blockDim.x + threadIdx.x) * 8;
        if (i >= H) continue;
        const Vec8<T> w = load_vec8(weight + i);
        Vec8<T> o;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            o.v[j] = VT::from_float(VT::to_float(v[k].v[j]) * inv * VT::to_float(w.v[j]));
        store_vec8(x + row * H + i, o);
    }
}

// Flat cache slots of positions: page of the sequence's table * block size + offset, -1 for
// padding (negative positions) and missing pages; positions past the table count into its last
// page, as offsets do.
template <typename O, typename TT, typename P>
__global__ __launch_bounds__(256) void slot_mapping_kernel(
    O* __restrict__ slots, const TT* __restrict__ table, const P* __restrict__ positions,
    const long n, const int S, const long cols, const long block_size) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const long p = positions[i], pos = max(p, 0l);
    const long page = table[i / S * cols + min(pos / block_size, cols - 1)];
    slots[i] = (O)(p >= 0 && page >= 0 ? page * block_size + pos % block_size : -1);
}

// Tokens of each prompt of a batch, (count, 1), or (count, 0) where they do not stand at the front
// or a position behind them is not negative. One workgroup a prompt.
template <typename M, typename P>
__global__ __launch_bounds__(256) void prompt_lengths_kernel(int2* __restrict__ out,
                                                             const M* __restrict__ mask,
                                                             const P* __restrict__ positions,
                                                             const int S) {
    __shared__ int s_n[4], s_far[4], s_near[4];
    const long b = blockIdx.x;
    int n = 0, far = -1, near = 0;             // last token; -1: no padded prompt
    for (int i = threadIdx.x; i < S; i += 256) {
        const M m = mask[b * S + i];
        if (m != 0) {
            ++n;
            far = i;
            if (m != 1) near = -1;             // not a mask of tokens
        } else if (positions[b * S + i] >= 0) {
            near = -1;                         // its cache row would be written
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        n += __shfl_xor(n, off, WAVE_SIZE);
        far = max(far, __shfl_xor(far, off, WAVE_SIZE));
        near = min(near, __shfl_xor(near, off, WAVE_SIZE));
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        s_n[w] = n;
        s_far[w] = far;
        s_near[w] = near;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < 4; ++i) {
            n += s_n[i];
            far = max(far, s_far[i]);
            near = min(near, s_near[i]);
        }
        out[b] = int2{n, far == n - 1 && near >= 0};
    }
}

// int32 positions and cache rows, and the number of valid positions of a row. One workgroup a row.
template <typename P, typename S>
__global__ __launch_bounds__(256) void step_layout_kernel(
    int* __restrict__ pos32, int* __restrict__ sid32, int* __restrict__ nvalid,
    const P* __restrict__ positions, const S* __restrict__ seq_ids, const int L) {
    __shared__ int s_n[4];
    const long b = blockIdx.x;
    int n = 0;
    for (int i = threadIdx.x; i < L; i += 256) {
        const int p = (int)positions[b * L + i];
        pos32[b * L + i] = p;
        n += p >= 0;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off, WAVE_SIZE);
    if ((threadIdx.x & 63) == 0) s_n[threadIdx.x >> 6] = n;
    __syncthreads();
    if (threadIdx.x == 0) {
        nvalid[b] = s_n[0] + s_n[1] + s_n[2] + s_n[3];
        sid32[b] = (int)seq_ids[b];
    }
}

// Page table of rows that own their pages one after another: row s has s * M .. s * M + M - 1,
// negative rows none.
template <typename S>
__global__ __launch_bounds__(256) void linear_table_kernel(int* __restrict__ table,
                                                           const S* __restrict__ seq_ids,
                                                           const int M) {
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j >= M) return;
    const long s = seq_ids[blockIdx.y];
    table[(long)blockIdx.y * M + j] = s >= 0 ? (int)(s * M + j) : -1;
}

constexpr int COPIES = 8;
struct CopyArgs {
    char* dst[COPIES];
    const char* src[COPIES];
    long bytes[COPIES];
};

// Several copies in one launch: workgroups of row y share copy y, 16 bytes a thread where both
// ends are aligned.
__global__ __launch_bounds__(256) void copy_many_kernel(const CopyArgs a) {
    char* d = a.dst[blockIdx.y];
    const char* s = a.src[blockIdx.y];
    const long n = a.bytes[blockIdx.y], step = (long)gridDim.x * 256;
    const long id = (long)blockIdx.x * 256 + threadIdx.x;
    long done = 0;
    if ((((size_t)d | (size_t)s) & 15) == 0) {
        for (long i = id; i < n / 16; i += step) ((int4*)d)[i] = ((const int4*)s)[i];
        done = n / 16 * 16;
    }
    for (long i = done + id; i < n; i += step) d[i] = s[i];
}

bool on(const torch::Tensor& t, at::ScalarType type) {
    return t.is_cuda() && t.is_contiguous() && t.scalar_type() == type;
}

bool whole(const torch::Tensor& t) {
    return t.is_cuda() && t.is_contiguous() &&
           (t.scalar_type() == at::ScalarType::Long || t.scalar_type() == at::ScalarType::Int);
}

}  // namespace

namespace {

void start_run(torch::Tensor h, torch::Tensor x, torch::Tensor cos, torch::Tensor sin,
               torch::Tensor pos32, c10::optional<torch::Tensor> sid32, torch::Tensor ids,
               torch::Tensor positions, c10::optional<torch::Tensor> seq_ids, torch::Tensor table,
               torch::Tensor cos_table, torch::Tensor sin_table, torch::Tensor weight, double eps,
               const Packed* packed, int* starts, int* prompt_sid) {
    const long rows = pos32.numel();
    const int H = table.size(1), D = cos_table.size(1);
    const auto type = table.scalar_type();
    const bool bf = type == at::ScalarType::BFloat16;
    TORCH_CHECK(bf || type == at::ScalarType::Half, "step_start: bf16/f16 only");
    TORCH_CHECK(on(ids, at::kLong) && on(positions, at::kLong) &&
                positions.numel() == ids.numel() && (packed || ids.numel() == rows) &&
                on(pos32, at::kInt), "step_start: ids and positions");
    TORCH_CHECK(on(table, type) && on(weight, type) && on(h, type) && on(x, type) && H % 8 == 0 &&
                H <= 32768 && weight.numel() == H && h.numel() == rows * H && x.numel() == rows * H,
                "step_start: rows");
    TORCH_CHECK(on(cos_table, at::kFloat) && on(sin_table, at::kFloat) && on(cos, at::kFloat) &&
                on(sin, at::kFloat) && D % 4 == 0 && cos_table.size(0) > 0 &&
                sin_table.sizes() == cos_table.sizes() && cos.numel() == rows * D &&
                sin.numel() == rows * D, "step_start: rope tables");
    TORCH_CHECK((((size_t)h.data_ptr() | (size_t)x.data_ptr() | (size_t)table.data_ptr() |
                  (size_t)weight.data_ptr() | (size_t)cos.data_ptr() | (size_t)sin.data_ptr() |
                  (size_t)cos_table.data_ptr() | (size_t)sin_table.data_ptr()) & 15) == 0,
                "step_start: alignment");
    const int B = seq_ids ? (int)seq_ids->numel() : 0;
    TORCH_CHECK(!seq_ids || (sid32 && whole(*seq_ids) && on(*sid32, at::kInt) &&
                             sid32->numel() == (packed ? rows : B) && B <= rows),
                "step_start: rows of the cache");
    if (rows == 0) return;
    const bool s64 = !seq_ids || seq_ids->scalar_type() == at::kLong;
    const int wide = (H / 8 + 63) / 64 * 64;
    const int threads = std::min(wide, rows >= 512 && H <= 8192 ? 256 : 1024);
    const int V = (H / 8 + threads - 1) / threads;
    auto stream = at::hip::getCurrentHIPStream();
#define START(T, VV, S, PK, ARG)                                                                   \
    hipLaunchKernelGGL((step_start_kernel<T, VV, S, PK>), dim3((unsigned)rows), dim3(threads), 0,  \
                       stream, (T*)h.data_ptr(), (T*)x.data_ptr(), cos.data_ptr<float>(),          \
                       sin.data_ptr<float>(), pos32.data_ptr<int>(),                               \
                       sid32 ? sid32->data_ptr<int>() : nullptr, ids.data_ptr<long>(),             \
                       positions.data_ptr<long>(),                                                 \
                       seq_ids ? (const S*)seq_ids->data_ptr() : nullptr,                          \
                       (const T*)table.data_ptr(), cos_table.data_ptr<float>(),                    \
                       sin_table.data_ptr<float>(), (const T*)weight.data_ptr(), (float)eps, H, D, \
                       B, table.size(0), cos_table.size(0), ARG, starts, prompt_sid)
#define START_P(T, VV, S)                                                                          \
    do {                                                                                           \
        if (packed) START(T, VV, S, true, *packed);                                                \
        else START(T, VV, S, false, 0);                                                            \
    } while (0)
#define START_V(T, S)                                                                              \
    do {                                                                                           \
        if (V == 1) START_P(T, 1, S);                                                              \
        else if (V == 2) START_P(T, 2, S);                                                         \
        else START_P(T, 4, S);                                                                     \
    } while (0)
    if (bf) {
        if (s64) START_V(__hip_bfloat16, long);
        else START_V(__hip_bfloat16, int);
    } else {
        if (s64) START_V(__half, long);
        else START_V(__half, int);
    }
#undef START_V
#undef START_P
#undef START
    HIP_CHECK_KERNEL();
}

}  // namespace

void step_start(torch::Tensor h, torch::Tensor x, torch::Tensor cos, torch::Tensor sin,
                torch::Tensor pos32, c10::optional<torch::Tensor> sid32, torch::Tensor ids,
                torch::Tensor positions, c10::optional<torch::Tensor> seq_ids, torch::Tensor table,
                torch::Tensor cos_table, torch::Tensor sin_table, torch::Tensor weight,
                double eps) {
    start_run(h, x, cos, sin, pos32, sid32, ids, positions, seq_ids, table, cos_table, sin_table,
              weight, eps, nullptr, nullptr, nullptr);
}

// Of (B, S) ids and positions the first lengths[b] of each row, one after the other (rows of h, x,
// cos, sin, pos32 and sid32). starts: (prompts + 1,), prompt_sid: (prompts,).
void step_start_packed(torch::Tensor h, torch::Tensor x, torch::Tensor cos, torch::Tensor sin,
                       torch::Tensor pos32, torch::Tensor sid32, torch::Tensor starts,
                       torch::Tensor prompt_sid, torch::Tensor ids, torch::Tensor positions,
                       torch::Tensor seq_ids, torch::Tensor table, torch::Tensor cos_table,
                       torch::Tensor sin_table, torch::Tensor weight, double eps,
                       const std::vector<long>& lengths) {
    const long n = lengths.size();
    TORCH_CHECK(n > 0 && n <= PROMPTS && ids.dim() == 2 && ids.size(0) == n &&
                seq_ids.numel() == n && on(starts, at::kInt) && starts.numel() == n + 1 &&
                on(prompt_sid, at::kInt) && prompt_sid.numel() == n, "step_start_packed: prompts");
    Packed p{};
    p.n = (int)n;
    p.S = (int)ids.size(1);
    long at = 0;
    for (long i = 0; i < n; ++i) {
        TORCH_CHECK(lengths[i] > 0 && lengths[i] <= p.S, "step_start_packed: lengths");
        p.starts[i] = (int)at;
        at += lengths[i];
        TORCH_CHECK(at < (1L << 31), "step_start_packed: too many tokens");
    }
    p.starts[n] = (int)at;
    TORCH_CHECK(pos32.numel() == at, "step_start_packed: rows");
    start_run(h, x, cos, sin, pos32, sid32, ids, positions, seq_ids, table, cos_table, sin_table,
              weight, eps, &p, starts.data_ptr<int>(), prompt_sid.data_ptr<int>());
}

// (prompts, 2): tokens of each, and whether they alone have positions and stand at the front
void prompt_lengths(torch::Tensor out, torch::Tensor mask, torch::Tensor positions) {
    const auto type = mask.scalar_type();
    TORCH_CHECK(mask.dim() == 2 && mask.is_cuda() && mask.is_contiguous() &&
                (type == at::kLong || type == at::kInt || type == at::kBool) && whole(positions) &&
                positions.sizes() == mask.sizes() && on(out, at::kInt) &&
                out.numel() == 2 * mask.size(0), "prompt_lengths");
    const long B = mask.size(0);
    if (B == 0) return;
    auto stream = at::hip::getCurrentHIPStream();
#define LENGTHS(M, P)                                                                              \
    hipLaunchKernelGGL((prompt_lengths_kernel<M, P>), dim3((unsigned)B), dim3(256), 0, stream,     \
                       (int2*)out.data_ptr<int>(), (const M*)mask.data_ptr(),                      \
                       positions.data_ptr<P>(), (int)mask.size(1))
#define LENGTHS_P(M)                                                                               \
    do {                                                                                           \
        if (positions.scalar_type() == at::kLong) LENGTHS(M, long);                                \
        else LENGTHS(M, int);                                                                      \
    } while (0)
    if (type == at::kLong) LENGTHS_P(long);
    else if (type == at::kInt) LENGTHS_P(int);
    else LENGTHS_P(bool);
#undef LENGTHS_P
#undef LENGTHS
    HIP_CHECK_KERNEL();
}

void slot_mapping(torch::Tensor slots, torch::Tensor table, torch::Tensor positions,
                  long block_size) {
    TORCH_CHECK(whole(table) && whole(positions) && table.dim() == 2 && positions.dim() == 2 &&
                table.size(0) >= positions.size(0) && table.size(1) > 0 && block_size > 0 &&
                whole(slots) && slots.numel() == positions.numel(), "slot_mapping");
    const long n = positions.numel();
    if (n == 0) return;
    auto stream = at::hip::getCurrentHIPStream();
    const bool t64 = table.scalar_type() == at::kLong, p64 = positions.scalar_type() == at::kLong;
    const bool o64 = slots.scalar_type() == at::kLong;
#define SLOTS(O, TT, P)                                                                            \
    hipLaunchKernelGGL((slot_mapping_kernel<O, TT, P>), dim3((unsigned)((n + 255) / 256)),         \
                       dim3(256), 0, stream, slots.data_ptr<O>(), table.data_ptr<TT>(),            \
                       positions.data_ptr<P>(), n, (int)positions.size(1), table.size(1),          \
                       block_size)
#define SLOTS_O(TT, P)                                                                             \
    do {                                                                                           \
        if (o64) SLOTS(long, TT, P);                                                               \
        else SLOTS(int, TT, P);                                                                    \
    } while (0)
    if (t64 && p64) SLOTS_O(long, long);
    else if (t64) SLOTS_O(long, int);
    else if (p64) SLOTS_O(int, long);
    else SLOTS_O(int, int);
#undef SLOTS_O
#undef SLOTS
    HIP_CHECK_KERNEL();
}

void step_layout(torch::Tensor pos32, torch::Tensor sid32, torch::Tensor nvalid,
                 torch::Tensor positions, torch::Tensor seq_ids) {
    TORCH_CHECK(whole(positions) && positions.dim() == 2 && whole(seq_ids) &&
                on(pos32, at::kInt) && pos32.numel() == positions.numel() && on(sid32, at::kInt) &&
                on(nvalid, at::kInt) && nvalid.numel() == positions.size(0) &&
                seq_ids.numel() == positions.size(0) && sid32.numel() == positions.size(0),
                "step_layout");
    const long B = positions.size(0);
    if (B == 0) return;
    auto stream = at::hip::getCurrentHIPStream();
    const bool p64 = positions.scalar_type() == at::kLong, s64 = seq_ids.scalar_type() == at::kLong;
#define LAYOUT(P, S)                                                                               \
    hipLaunchKernelGGL((step_layout_kernel<P, S>), dim3((unsigned)B), dim3(256), 0, stream,        \
                       pos32.data_ptr<int>(), sid32.data_ptr<int>(), nvalid.data_ptr<int>(),       \
                       positions.data_ptr<P>(), seq_ids.data_ptr<S>(), (int)positions.size(1))
    if (p64 && s64) LAYOUT(long, long);
    else if (p64) LAYOUT(long, int);
    else if (s64) LAYOUT(int, long);
    else LAYOUT(int, int);
#undef LAYOUT
    HIP_CHECK_KERNEL();
}

void linear_table(torch::Tensor table, torch::Tensor seq_ids) {
    TORCH_CHECK(on(table, at::kInt) && table.dim() == 2 && whole(seq_ids) &&
                seq_ids.numel() == table.size(0) && table.size(0) <= 65535, "linear_table");
    if (table.numel() == 0) return;
    const int M = table.size(1);
    auto stream = at::hip::getCurrentHIPStream();
    const dim3 grid((M + 255) / 256, (unsigned)table.size(0));
    if (seq_ids.scalar_type() == at::kLong)
        hipLaunchKernelGGL((linear_table_kernel<long>), grid, dim3(256), 0, stream,
                           table.data_ptr<int>(), seq_ids.data_ptr<long>(), M);
    else
        hipLaunchKernelGGL((linear_table_kernel<int>), grid, dim3(256), 0, stream,
                           table.data_ptr<int>(), seq_ids.data_ptr<int>(), M);
    HIP_CHECK_KERNEL();
}

// dst[i] = src[i], all of the current device, contiguous, of one type and size
void copy_many(std::vector<torch::Tensor> dst, std::vector<torch::Tensor> src) {
    TORCH_CHECK(dst.size() == src.size(), "copy_many: as many sources as destinations");
    auto stream = at::hip::getCurrentHIPStream();
    for (size_t base = 0; base < dst.size(); base += COPIES) {
        CopyArgs a{};
        const int n = (int)std::min<size_t>(COPIES, dst.size() - base);
        long most = 0;
        for (int i = 0; i < n; ++i) {
            const auto &d = dst[base + i], &s = src[base + i];
            TORCH_CHECK(on(d, s.scalar_type()) && on(s, s.scalar_type()) &&
                        d.sizes() == s.sizes(), "copy_many: like tensors on the GPU");
            a.dst[i] = (char*)d.data_ptr();
            a.src[i] = (const char*)s.data_ptr();
            a.bytes[i] = (long)(s.numel() * s.element_size());
            most = std::max(most, a.bytes[i]);
        }
        if (most == 0) continue;
        const dim3 grid((unsigned)std::min(1024l, (most + 4095) / 4096), n);
        hipLaunchKernelGGL(copy_many_kernel, grid, dim3(256), 0, stream, a);
        HIP_CHECK_KERNEL();
    }
}
