// The launches of plain decoder layers over prompts, one after the other. A prompt of up to 512 rows
// is 8 launches of 5 to 25 us a layer, which Python makes in some 90 us a layer: the GPU waits for
// the host. 93 tokens of a 1B model, 4 layers: 484 -> 380 us.

#include <torch/extension.h>
#include <vector>

long tile_gemm_splits(long M, long N, long K, long glu, bool whole);
torch::Tensor tile_gemm(torch::Tensor x, torch::Tensor w, c10::optional<torch::Tensor> bias,
                        long splits, bool parts, long glu);
void add_norm(torch::Tensor out, torch::Tensor residual, torch::Tensor y, torch::Tensor weight,
              double eps);
void qkv_rope_update(torch::Tensor q_out, torch::Tensor qkv, torch::Tensor cosb, torch::Tensor sinb,
                     torch::Tensor k_cache, torch::Tensor v_cache, torch::Tensor positions,
                     torch::Tensor seq_ids, long Hq, long Hkv, c10::optional<torch::Tensor> q_norm,
                     c10::optional<torch::Tensor> k_norm, double eps,
                     c10::optional<torch::Tensor> slots);
bool lt_linear(torch::Tensor y, torch::Tensor x, torch::Tensor w, c10::optional<torch::Tensor> bias,
               bool timed);
void silu_mul_fused(torch::Tensor out, torch::Tensor gate_up);
void flash_prefill_packed(torch::Tensor out, torch::Tensor q, torch::Tensor k_cache,
                          torch::Tensor v_cache, torch::Tensor seq_ids, torch::Tensor starts,
                          long longest, double scale, long window);
void flash_prefill_cached(torch::Tensor out, torch::Tensor q, torch::Tensor k_cache,
                          torch::Tensor v_cache, torch::Tensor seq_ids, double scale, long window,
                          c10::optional<torch::Tensor> sinks);

namespace {

// x @ w^T, as parts of K where the tiled kernel has it so; the library's where that kernel does not
// take it
torch::Tensor product(const torch::Tensor& x, const torch::Tensor& w, bool glu) {
    const long rows = x.size(0), N = w.size(0);
    if (tile_gemm_splits(rows, N, x.size(1), glu, glu))
        return tile_gemm(x, w, c10::nullopt, 0, !glu, glu);
    torch::Tensor y = torch::empty({rows, N}, x.options());
    if (!lt_linear(y, x, w, c10::nullopt, false)) y = at::linear(x, w);   // no algorithm for the shape
    if (!glu) return y;
    torch::Tensor o = torch::empty({rows, N / 2}, x.options());
    silu_mul_fused(o, y);
    return o;
}

}  // namespace

// weights: 8 a layer, those of q|k|v, output, the norm after it, gate|up, down and the norm after
// that, key and value cache rows; sizes: 3 a layer, query heads, KV heads, window; numbers: 3 a
// layer, the norms' eps and the scale. h (B, S, H), the residual stream, is updated; x is its
// norm. The normed output, or nothing, with nothing done, where an operand is not as the kernels
// take it, or a product of whole prompts not the tiled kernel's. Packed prompts: h (rows, 1, H),
// with a cache row for each row in seq_ids and each prompt's in prompt_sid, starts and `longest`
// as flash_prefill_packed has them.
c10::optional<torch::Tensor> prompt_layers(torch::Tensor h, torch::Tensor x, torch::Tensor cos,
                                           torch::Tensor sin, torch::Tensor positions,
                                           torch::Tensor seq_ids,
                                           const std::vector<torch::Tensor>& weights,
                                           const std::vector<long>& sizes,
                                           const std::vector<double>& numbers,
                                           c10::optional<torch::Tensor> starts,
                                           c10::optional<torch::Tensor> prompt_sid, long longest) {
    const size_t layers = weights.size() / 8;
    TORCH_CHECK(weights.size() == layers * 8 && sizes.size() == layers * 3 &&
                numbers.size() == layers * 3 && h.dim() == 3 && x.sizes() == h.sizes() &&
                x.is_contiguous() && starts.has_value() == prompt_sid.has_value() &&
                (!starts || h.size(1) == 1), "prompt_layers: operands");
    const long B = h.size(0), S = h.size(1), H = h.size(2), rows = B * S;
    const auto type = h.scalar_type();
    for (size_t i = 0; i < layers; ++i) {
        const torch::Tensor* w = &weights[i * 8];
        const long D = w[6].size(3), Hq = sizes[i * 3], Hkv = sizes[i * 3 + 1];
        for (int j : {0, 1, 3, 4})
            if (w[j].scalar_type() != type || !w[j].is_contiguous() ||
                (size_t)w[j].data_ptr() % 16 || !w[j].is_cuda())
                return c10::nullopt;
        for (int j : {6, 7})
            if (w[j].scalar_type() != type || !w[j].is_contiguous() ||
                (size_t)w[j].data_ptr() % 16)
                return c10::nullopt;
        if (w[0].size(0) != (Hq + 2 * Hkv) * D || w[0].size(1) != H || w[1].size(0) != H ||
            w[1].size(1) != Hq * D || cos.size(-1) < D ||
            ((size_t)cos.data_ptr() | (size_t)sin.data_ptr()) % 16 || w[3].size(1) != H ||
            w[4].size(0) != H || 2 * w[4].size(1) != w[3].size(0) || w[4].size(1) % 8 ||
            (size_t)x.data_ptr() % 16)
            return c10::nullopt;
        if (!starts && (!tile_gemm_splits(rows, w[0].size(0), H, false, false) ||
                        !tile_gemm_splits(rows, H, Hq * D, false, false) ||
                        !tile_gemm_splits(rows, w[3].size(0), H, true, true) ||
                        !tile_gemm_splits(rows, H, w[4].size(1), false, false)))
            return c10::nullopt;
    }
    torch::Tensor xs = x.view({rows, H});
    for (size_t i = 0; i < layers; ++i) {
        const torch::Tensor* w = &weights[i * 8];
        const long D = w[6].size(3), Hq = sizes[i * 3], Hkv = sizes[i * 3 + 1];
        torch::Tensor y = product(xs, w[0], false);
        const long N = w[0].size(0);
        torch::Tensor q = torch::empty({B, Hq, S, D}, x.options());
        qkv_rope_update(q, y.dim() == 3 ? y.view({y.size(0), B, S, N}) : y.view({B, S, N}), cos, sin,
                        w[6], w[7], positions, seq_ids, Hq, Hkv, c10::nullopt, c10::nullopt, 0.0,
                        c10::nullopt);
        torch::Tensor o = torch::empty({B, S, Hq, D}, x.options());
        const double scale = numbers[i * 3 + 2];
        const long window = sizes[i * 3 + 2];
        if (starts)
            flash_prefill_packed(o.transpose(1, 2), q, w[6], w[7], *prompt_sid, *starts, longest,
                                 scale, window);
        else
            flash_prefill_cached(o.transpose(1, 2), q, w[6], w[7], seq_ids, scale, window,
                                 c10::nullopt);
        y = product(o.view({rows, Hq * D}), w[1], false);
        torch::Tensor n = torch::empty_like(xs);
        add_norm(n, h, y, w[2], numbers[i * 3]);
        y = product(product(n, w[3], true), w[4], false);
        xs = torch::empty_like(xs);
        add_norm(xs, h, y, w[5], numbers[i * 3 + 1]);
    }
    return xs.view({B, S, H});
}
