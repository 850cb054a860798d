// The launches of plain decoder layers over a short prompt, one after the other. A prompt of up to
// 512 rows is 8 launches of 5 to 25 us a layer, which Python makes in some 90 us a layer: the GPU
// waits for the host. 93 tokens of a 1B model, 4 layers: 484 -> 380 us.

#include <torch/extension.h>
#include <vector>

long tile_gemm_splits(long M, long N, long K, bool glu);
torch::Tensor tile_gemm(torch::Tensor x, torch::Tensor w, c10::optional<torch::Tensor> bias,
                        long splits, bool parts, bool glu);
void add_norm(torch::Tensor out, torch::Tensor residual, torch::Tensor y, torch::Tensor weight,
              double eps);
void qkv_rope_update(torch::Tensor q_out, torch::Tensor qkv, torch::Tensor cosb, torch::Tensor sinb,
                     torch::Tensor k_cache, torch::Tensor v_cache, torch::Tensor positions,
                     torch::Tensor seq_ids, long Hq, long Hkv, c10::optional<torch::Tensor> q_norm,
                     c10::optional<torch::Tensor> k_norm, double eps,
                     c10::optional<torch::Tensor> slots);
void flash_prefill_cached(torch::Tensor out, torch::Tensor q, torch::Tensor k_cache,
                          torch::Tensor v_cache, torch::Tensor seq_ids, double scale, long window,
                          c10::optional<torch::Tensor> sinks);

// weights: 8 a layer, those of q|k|v, output, the norm after it, gate|up, down and the norm after
// that, key and value cache rows; sizes: 3 a layer, query heads, KV heads, window; numbers: 3 a
// layer, the norms' eps and the scale. h (B, S, H), the residual stream, is updated; x is its
// norm. The normed output, or nothing, with nothing done, where a product is not the tiled
// kernel's or rope does not take its parts.
c10::optional<torch::Tensor> prompt_layers(torch::Tensor h, torch::Tensor x, torch::Tensor cos,
                                           torch::Tensor sin, torch::Tensor positions,
                                           torch::Tensor seq_ids,
                                           const std::vector<torch::Tensor>& weights,
                                           const std::vector<long>& sizes,
                                           const std::vector<double>& numbers) {
    const size_t layers = weights.size() / 8;
    TORCH_CHECK(weights.size() == layers * 8 && sizes.size() == layers * 3 &&
                numbers.size() == layers * 3 && h.dim() == 3 && x.sizes() == h.sizes() &&
                x.is_contiguous(), "prompt_layers: operands");
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
            w[4].size(0) != H || 2 * w[4].size(1) != w[3].size(0) || (size_t)x.data_ptr() % 16 ||
            !tile_gemm_splits(rows, w[0].size(0), H, false) ||
            !tile_gemm_splits(rows, H, Hq * D, false) ||
            !tile_gemm_splits(rows, w[3].size(0), H, true) ||
            !tile_gemm_splits(rows, H, w[4].size(1), false))
            return c10::nullopt;
    }
    torch::Tensor xs = x.view({rows, H});
    for (size_t i = 0; i < layers; ++i) {
        const torch::Tensor* w = &weights[i * 8];
        const long D = w[6].size(3), Hq = sizes[i * 3], Hkv = sizes[i * 3 + 1];
        torch::Tensor y = tile_gemm(xs, w[0], c10::nullopt, 0, true, false);
        const long N = w[0].size(0);
        torch::Tensor q = torch::empty({B, Hq, S, D}, x.options());
        qkv_rope_update(q, y.dim() == 3 ? y.view({y.size(0), B, S, N}) : y.view({B, S, N}), cos, sin,
                        w[6], w[7], positions, seq_ids, Hq, Hkv, c10::nullopt, c10::nullopt, 0.0,
                        c10::nullopt);
        torch::Tensor o = torch::empty({B, S, Hq, D}, x.options());
        flash_prefill_cached(o.transpose(1, 2), q, w[6], w[7], seq_ids, numbers[i * 3 + 2],
                             sizes[i * 3 + 2], c10::nullopt);
        y = tile_gemm(o.view({rows, Hq * D}), w[1], c10::nullopt, 0, true, false);
        torch::Tensor n = torch::empty_like(xs);
        add_norm(n, h, y, w[2], numbers[i * 3]);
        y = tile_gemm(tile_gemm(n, w[3], c10::nullopt, 0, false, true), w[4], c10::nullopt, 0, true,
                      false);
        xs = torch::empty_like(xs);
        add_norm(xs, h, y, w[5], numbers[i * 3 + 1]);
    }
    return xs.view({B, S, H});
}
