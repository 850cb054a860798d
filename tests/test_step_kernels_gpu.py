"""GPU tests of the kernels that a model step is made of beside attention: tiled products whose
parts of K the next kernel adds up, residual sum and norm, and the layers that run on them."""

import pytest
import torch

pytestmark = pytest.mark.gpu

from neuronx_distributed_inference_amd import ops

F64 = torch.float64
EPS16 = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _product(M, N, K, dtype, seed=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    x = torch.randn(M, K, device="cuda", generator=g).to(dtype)
    w = (torch.randn(N, K, device="cuda", generator=g) * 0.05).to(dtype)
    exact = x.to(F64) @ w.to(F64).t()
    # K sums in 32 bits: at most K roundings of 2^-24 of the largest partial sum
    sums = K * 2.0 ** -24 * (x.to(F64).abs() @ w.to(F64).abs().t())
    return x, w, exact, sums


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [
    (1, 64, 256), (1, 4100, 320), (2, 2048, 2048), (16, 6144, 512), (17, 4352, 256),
    (32, 100, 1088), (33, 11408, 256), (48, 4092, 4096), (64, 4100, 576), (65, 132, 2048),
    (93, 3072, 2048), (128, 4096, 256), (127, 16384, 4096), (129, 68, 320), (200, 4096, 4096),
    (256, 6144, 4096), (257, 2048, 2048), (300, 4096, 512), (512, 4096, 256)])
def test_tile_gemm(M, N, K, dtype):
    x, w, exact, sums = _product(M, N, K, dtype)
    plan = ops._tile_takes(x, w)
    assert plan >= 1
    for splits in {1, 2, plan, K // 64}:
        parts = ops._C.tile_gemm(x, w, None, splits, True)
        assert parts.dim() == (3 if splits > 1 else 2)
        if splits > 1:
            got, limit = parts.to(F64).sum(0), sums
        else:
            got, limit = parts.to(F64), sums + EPS16[dtype] * exact.abs()
        assert ((got - exact).abs() <= limit + 1e-30).all()
        bias = torch.linspace(-1, 1, N, device="cuda").to(dtype)
        y = ops._C.tile_gemm(x, w, bias, splits)
        want = exact + bias.to(F64)
        assert y.dtype == dtype
        assert ((y.to(F64) - want).abs() <= 2 * sums + EPS16[dtype] * want.abs() + 1e-7).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [(1, 64, 256), (7, 28672, 512), (16, 1000, 320), (32, 16384, 256),
                                   (40, 72, 256), (64, 25608, 256), (65, 16384, 256),
                                   (128, 28672, 256), (200, 2056, 2048), (256, 28672, 1024)])
def test_tile_gemm_glu(M, N, K, dtype):
    x, w, exact, sums = _product(M, N, K, dtype)
    y = ops._C.tile_gemm(x, w, glu=True)
    g, u = exact[:, : N // 2], exact[:, N // 2:]
    want = torch.nn.functional.silu(g) * u
    # the slope of silu stays below 1.1; its exp and division are good to 2^-20
    limit = 1.1 * sums[:, : N // 2] * u.abs() + g.abs() * sums[:, N // 2:] \
        + (EPS16[dtype] + 2.0 ** -20) * want.abs() + 1e-7
    assert ((y.to(F64) - want).abs() <= limit).all()


@pytest.mark.parametrize("M,N,K", [(33, 48904, 320), (64, 49160, 256), (47, 65528, 576)])
def test_tile_gemm_wide(M, N, K):
    """Tiles of 64 rows and 256 columns: rows and columns short of them, fewer chunks than the ring."""
    test_tile_gemm(M, N, K, torch.bfloat16)
    test_tile_gemm_glu(M, N, K, torch.float16)


@pytest.mark.parametrize("M,N,K", [(193, 20616, 1088), (224, 6152, 4096), (255, 31000, 768)])
def test_tile_gemm_256_rows(M, N, K):
    """The tile of 256 rows: rows and columns short of it, a ring that ends in each of its slots."""
    assert N * K > 20 << 20
    test_tile_gemm(M, N, K, torch.bfloat16)
    test_tile_gemm_glu(M, N, K, torch.float16)


@pytest.mark.parametrize("M,N,K", [(1, 4096, 192), (1, 60, 256), (8, 66, 256), (8, 64, 260),
                                   (513, 4096, 4096), (512, 28672, 4096), (129, 57344, 8192)])
def test_tile_gemm_leaves_to_the_library(M, N, K):
    assert ops._C.tile_gemm_splits(M, N, K, False) == 0


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,H,parts", [(1, 8, 0), (1, 2048, 1), (3, 4096, 8), (64, 8192, 5),
                                          (5, 520, 4), (2, 32768, 2), (600, 4096, 0),
                                          (513, 16384, 3), (700, 8192, 2)])
def test_add_norm(rows, H, parts, dtype):
    g = torch.Generator(device="cuda")
    g.manual_seed(rows + H)
    shape = (parts, rows, H) if parts else (rows, H)
    y = torch.randn(shape, device="cuda", generator=g)
    y = y if parts else y.to(dtype)
    res = torch.randn(rows, H, device="cuda", generator=g).to(dtype)
    w = torch.randn(H, device="cuda", generator=g).to(dtype)
    total = res.to(F64) + (y.to(F64).sum(0) if parts else y.to(F64))
    out = ops.add_norm(y, res, w, 1e-5)
    # the residual as it is kept, under the root mean square of the sum
    want = res.to(F64) * torch.rsqrt(total.square().mean(-1, keepdim=True) + 1e-5) * w.to(F64)
    # one rounding of each result, some of 2^-24 before it
    assert ((res.to(F64) - total).abs() <= EPS16[dtype] * total.abs() + 1e-5).all()
    assert ((out.to(F64) - want).abs() <= (EPS16[dtype] + 2.0 ** -16) * want.abs() + 1e-4).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("parts", [1, 2, 3, 8])
@pytest.mark.parametrize("normed", [False, True])
def test_qkv_rope_update_adds_parts(parts, normed, dtype):
    B, S, Hq, Hkv, D = 3, 2, 8, 2, 64
    g = torch.Generator(device="cuda")
    g.manual_seed(parts)
    y = torch.randn(parts, B, S, (Hq + 2 * Hkv) * D, device="cuda", generator=g)
    ang = torch.randn(B, S, D // 2, device="cuda", generator=g).repeat(1, 1, 2)
    pos = torch.randint(0, 16, (B, S), device="cuda", generator=g, dtype=torch.int32)
    pos[:, 1] = pos[:, 0] + 1
    ids = torch.arange(B, device="cuda", dtype=torch.int32)
    norms = None
    if normed:
        norms = tuple(torch.randn(D, device="cuda", generator=g).to(dtype) for _ in range(2)) + (1e-6,)
    caches = [torch.zeros(B, Hkv, 20, D, device="cuda", dtype=dtype) for _ in range(2)]
    q = ops.qkv_rope_update(y, ang.cos(), ang.sin(), *caches, pos, ids, Hq, Hkv, norms=norms,
                            dtype=dtype)
    wide = [torch.zeros(B, Hkv, 20, D, dtype=F64) for _ in range(2)]
    want = ops.qkv_rope_update(y.to(F64).sum(0).cpu(), ang.to(F64).cos().cpu(),
                               ang.to(F64).sin().cpu(), *wide, pos.cpu(), ids.cpu(), Hq, Hkv,
                               norms=norms and tuple(t.cpu().to(F64) for t in norms[:2]) + (1e-6,))
    for a, b in zip([q] + caches, [want] + wide):
        # rope adds two products: a rounding each of the parts' sums and the angles in 32 bits
        assert ((a.cpu().to(F64) - b).abs() <= EPS16[dtype] * b.abs() + 1e-4).all()


def _small_llama(dtype, layers=2, moe=False, **kw):
    from neuronx_distributed_inference_amd.config import EngineConfig
    from neuronx_distributed_inference_amd.models.llama.modeling_llama import (
        LlamaForCausalLM, LlamaInferenceConfig)
    from neuronx_distributed_inference_amd.models.mixtral.modeling_mixtral import (
        MixtralForCausalLM, MixtralInferenceConfig)

    ec = EngineConfig(batch_size=2, max_batch_size=2, seq_len=160, max_length=160,
                      torch_dtype=dtype, tp_degree=1, output_logits=True, fused_qkv=True,
                      fused_gate_up=True, enable_batch_bucketing=False, **kw)
    sizes = dict(neuron_config=ec, hidden_size=512, intermediate_size=1024,
                 num_hidden_layers=layers, num_attention_heads=8, num_key_value_heads=2,
                 head_dim=64, vocab_size=512, max_position_embeddings=320, rms_norm_eps=1e-5,
                 rope_theta=10000.0, hidden_act="silu", tie_word_embeddings=False)
    if moe:
        sizes.update(num_local_experts=4, num_experts_per_tok=4)   # no choice that rounding flips
    with torch.device("cuda"):
        lm = (MixtralForCausalLM(MixtralInferenceConfig(**sizes)) if moe else
              LlamaForCausalLM(LlamaInferenceConfig(**sizes))).eval()
    g = torch.Generator(device="cuda")
    g.manual_seed(0)
    for name, p in lm.model.named_parameters():
        if "norm" in name:
            p.data.uniform_(0.5, 1.5, generator=g)
        elif p.element_size() > 1:                           # (8 bits: a cache)
            p.data.normal_(0, 0.05, generator=g)
    return lm


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("moe", [False, True])
@pytest.mark.parametrize("hook", ["layer", "norm", "o_proj", "down", "final", "global"])
def test_fused_layers_and_layers_with_hooks(hook, moe, dtype):
    """A hook sees its module's tensors, from the chain of modules; without one the fused layers
    give the same logits and cache."""
    if moe and hook == "down":
        pytest.skip("no down projection")
    lm = _small_llama(dtype, moe=moe)
    ids = torch.randint(0, 512, (2, 70), device="cuda")
    step = torch.randint(0, 512, (2, 1), device="cuda")

    def run():
        lm.reset()
        with torch.inference_mode():
            a = lm(input_ids=ids).logits
            b = lm(input_ids=step, position_ids=torch.full((2, 1), 70, device="cuda")).logits
        return a.float(), b.float(), lm.model.kv_mgr.get_cache(1)[0].data.float().clone()

    fused = run()
    layer = lm.model.layers[1]
    seen = []
    note = lambda *a: seen.append(1)  # noqa: E731
    if hook == "global":
        h = torch.nn.modules.module.register_module_forward_hook(note)
    else:
        mod = {"layer": layer, "norm": layer.post_attention_layernorm,
               "o_proj": layer.self_attn.o_proj, "final": lm.model.norm,
               "down": getattr(layer.mlp, "down_proj", None)}[hook]
        h = mod.register_forward_hook(note)
    try:
        plain = run()
    finally:
        h.remove()
    assert len(seen) >= 2
    # 16-bit activations of two layers, rounded at other places
    tol = 0.03 if dtype == "bfloat16" else 0.004
    for a, b in zip(fused, plain):
        assert (a - b).norm() <= tol * b.norm()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("mt,f8,T,E,k,H,I", [
    # tiles filled to the last row, by half and by one; experts without rows
    (96, False, 200, 4, 2, 320, 192), (160, False, 330, 4, 2, 256, 128), (128, False, 70, 4, 2, 64, 64),
    (160, False, 81, 4, 4, 1088, 64), (48, True, 99, 4, 2, 384, 256), (64, True, 33, 8, 1, 256, 128),
    # shares of tiles: fewer tiles than workgroups, between one and two rounds of them
    (32, False, 40, 8, 2, 4096, 2048), (96, False, 300, 8, 2, 4096, 1088), (48, True, 128, 8, 2, 4096, 3584),
    (64, False, 130, 16, 2, 4608, 512), (160, False, 7, 3, 3, 8192, 1344)])
def test_moe_routed_tile_heights_and_shares(mt, f8, T, E, k, H, I, dtype, monkeypatch):
    """As test_moe_routed_experts, for tiles of one height and with the down projection shared out
    or not (a workspace too small for shares): rounded activations and results, 32-bit sums."""
    monkeypatch.setattr(ops, "_moe_tile_rows", lambda *a: mt)
    g = torch.Generator(device="cuda")
    g.manual_seed(mt + T)
    x = torch.randn(T, H, device="cuda", generator=g).to(dtype)
    logits = torch.randn(T, E, device="cuda", generator=g)
    logits[:, 0] += 3.0                                      # one expert of many rows
    wt, idx = torch.softmax(logits, -1).topk(k, dim=-1)
    w = [(torch.randn(E, *s, device="cuda", generator=g) * 0.05).to(dtype)
         for s in ((I, H), (I, H), (H, I))]
    scales, ref = None, [v.to(F64) for v in w]
    if f8:
        w, scales = zip(*[ops.fp8_moe_quantize(v) for v in w])
        ref = [ops.fp8_moe_dequant(v, s).to(F64) for v, s in zip(w, scales)]
    want = torch.zeros(T, H, dtype=F64, device="cuda")
    for e in range(E):
        t, j = (idx == e).nonzero(as_tuple=True)
        xe = x[t].to(F64)
        h = torch.nn.functional.silu(xe @ ref[0][e].t()) * (xe @ ref[1][e].t())
        want.index_add_(0, t, (h @ ref[2][e].t()) * wt[t, j].to(F64).unsqueeze(1))
    for room in (1 << 30, 4 * H * mt):
        monkeypatch.setattr(ops, "MOE_WORKSPACE", room)
        got = ops.moe_routed_experts(x, wt, idx, *w, scales=scales, num_experts=E)
        assert (got.to(F64) - want).norm() < EPS16[dtype] * want.norm()
        assert torch.equal(got, ops.moe_routed_experts(x, wt, idx, *w, scales=scales, num_experts=E))


@pytest.mark.parametrize("mt,f8,T,H,I", [
    # 8 row tiles, two an expert, times 32 (whole tiles only), 33, 48 and 49 (too many for halves) tiles
    # of columns, the last one's second half without any where I is 64 past a tile
    (32, False, 33, 128, 4096), (32, False, 63, 128, 4160), (64, False, 65, 64, 6144),
    (64, False, 127, 64, 6208), (48, True, 49, 128, 4224), (32, True, 64, 256, 6272),
    # 4 row tiles: weights that one tile has to itself; 12 of the tallest
    (128, False, 100, 64, 8256), (96, False, 81, 64, 12288), (160, False, 330, 64, 2816),
    # the down projection's tiles in halves too
    (32, False, 20, 16448, 64), (48, True, 33, 16640, 128), (160, False, 150, 16512, 64)])
def test_moe_routed_last_round(mt, f8, T, H, I, monkeypatch):
    """All of 4 experts for each token: lists of tiles that end in whole tiles and in halves."""
    test_moe_routed_tile_heights_and_shares(mt, f8, T, 4, 4, H, I, torch.bfloat16, monkeypatch)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,S,H,D,seq", [(1, 1, 8, 4, None), (3, 5, 2048, 64, torch.int64), (64, 1, 4096, 128, torch.int32),
                                         (1, 600, 8192, 128, torch.int64), (2, 2, 32768, 256, None)])
def test_step_start(B, S, H, D, seq, dtype):
    """Rows and rope tables to the bit, the norm within the rounding of its result."""
    V, L = 50, 40
    table = torch.randn(V, H, device="cuda").to(dtype)
    cos, sin = torch.randn(2, L, D, device="cuda")
    w = torch.randn(H, device="cuda").to(dtype)
    ids = torch.randint(0, V, (B, S), device="cuda")
    pos = torch.randint(-3, L + 9, (B, S), device="cuda")
    sid = None if seq is None else torch.randint(-1, 9, (B,), device="cuda").to(seq)
    assert ops.step_start_takes(ids, pos, sid, table, cos)
    h, x, c, s, p32, s32 = ops.step_start(ids, pos, sid, table, cos, sin, w, 1e-5)
    assert torch.equal(h, table[ids]) and torch.equal(p32, pos.int())
    at = pos.clamp(0, L - 1)
    assert torch.equal(c, cos[at]) and torch.equal(s, sin[at])
    assert (s32 is None) if sid is None else torch.equal(s32, sid.int())
    r = h.to(F64)
    want = r * torch.rsqrt(r.square().mean(-1, keepdim=True) + 1e-5) * w.to(F64)
    assert ((x.to(F64) - want).abs() <= (EPS16[dtype] + 1e-5) * want.abs() + 1e-7).all()
    for bad in (ids.int(), ids.t() if B > 1 and S > 1 else ids.cpu(), ids[:, :0]):
        assert not ops.step_start_takes(bad, pos, sid, table, cos)


@pytest.mark.parametrize("tdt", [torch.int64, torch.int32])
@pytest.mark.parametrize("pdt", [torch.int64, torch.int32])
def test_slots_layouts_and_tables(tdt, pdt):
    """The index kernels against the same index arithmetic on the CPU, to the bit."""
    from neuronx_distributed_inference_amd.models.hybrid_base import HybridDecoderModel
    from neuronx_distributed_inference_amd.modules.kvcache.block_kv_cache_manager import (
        generate_slot_mapping)
    from neuronx_distributed_inference_amd.ops.seqmix import StepLayout

    for B, S, M, bs in ((1, 1, 1, 1), (3, 300, 5, 7), (65, 2, 9, 64)):
        table = torch.randint(-1, 1000, (B + 1, M)).to(tdt)
        pos = torch.randint(-4, M * bs + 9, (B, S)).to(pdt)
        for out in (torch.int64, torch.int32):
            got = generate_slot_mapping(table.cuda(), pos.cuda(), bs, out)
            assert got.dtype == out
            assert torch.equal(got.cpu(), generate_slot_mapping(table, pos, bs, out))
        seq = torch.randint(-1, 7, (B,)).to(tdt)
        a, b = StepLayout(pos.cuda(), seq.cuda()), StepLayout(pos, seq)
        for n in ("positions", "seq_ids", "nvalid"):
            assert getattr(a, n).dtype == torch.int32
            assert torch.equal(getattr(a, n).cpu(), getattr(b, n)), n
        model = type("M", (), {"max_blocks_per_seq": M * 300})()
        model.kv_mgr = type("K", (), {"num_blocks": 10 ** 6, "state": type("S", (), {"num_slots": 8})})()
        tables = [HybridDecoderModel.begin_step(model, pos.to(d), seq.to(d), None) for d in ("cuda", "cpu")]
        assert torch.equal(tables[0].cpu().long(), tables[1])


def test_copy_many():
    g = torch.Generator(device="cuda").manual_seed(0)
    src = [torch.randint(0, 255, (n,), device="cuda", generator=g, dtype=torch.uint8)
           for n in (0, 1, 15, 16, 4097, 70001, 3, 5, 31, 64)]
    src += [src[4][1:], src[5][::2], torch.randn(3, 5), torch.randn(2, 3, device="cuda").t(),
            torch.arange(9, device="cuda")]
    dst = [torch.zeros(t.shape, dtype=t.dtype, device="cuda") for t in src[:-1]]
    dst.append(torch.zeros(9, device="cuda"))            # another type
    ops.copy_many(dst, src)
    for d, s in zip(dst, src):
        assert torch.equal(d, s.to(d.device, d.dtype))


WINDOWED = [
    # S, H, G, D, page, start, options
    (2, 4, 4, 64, 16, 0, {}),
    (33, 12, 4, 128, 24, 200, dict(window=70, keep_first=3, r=True, gate="full")),
    (127, 4, 1, 64, 64, 5, dict(window=64, keep_first=80, r=True)),
    (128, 8, 8, 128, 16, 0, dict(chunk=48, sink=True, gate="head")),
    (300, 16, 4, 128, 64, 0, dict(window=100, keep_first=4, r=True, gate="full")),
    (77, 6, 2, 64, 16, 40, dict(window=50, gate="full")),
    (65, 16, 1, 64, 24, 611, dict(window=1, slopes=True, q_temp=(0.3, 64))),
    (130, 6, 2, 128, 16, 70, dict(window=130, keep_first=64, chunk=90, softcap=20.0, r=True)),
    (64, 2, 2, 64, 64, 1000, dict(softcap=5.0, sink=True, slopes=True)),
    (3, 64, 1, 128, 16, 333, dict(keep_first=9, window=32, sink=True, gate="head"))]


def _windowed(S, H, G, D, page, start, opts, seed=0):
    """Arguments of seqmix.paged_attention for rows of unequal length, the last tokens padding."""
    g = torch.Generator().manual_seed(seed + S + D)
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    B, opts = 3, dict(opts)
    pos = torch.stack([start + 17 * b + torch.arange(S) for b in range(B)])
    for b in range(1, B):
        if S > b:
            pos[b, S - b:] = -1
    nb = (start + 17 * B + S) // page + 1
    table = torch.randperm(B * nb, generator=g).view(B, nb).int()
    kc, vc = (rnd(B * nb, page, G, D).bfloat16() for _ in range(2))
    q = rnd(B, S, H * D + 8).bfloat16()[..., : H * D]
    if opts.pop("r", False):
        opts.update(r1=torch.rand(H, generator=g), r2=torch.rand(H, generator=g) * 0.3)
    if opts.pop("slopes", False):
        opts["slopes"] = torch.rand(H, generator=g) * 0.05
    if opts.pop("sink", False):
        opts["sink"] = rnd(H)
    gate = opts.pop("gate", None)
    if gate:
        opts.update(gate=rnd(B, S, H * D if gate == "full" else H).bfloat16(),
                    gate_per_head=gate == "head")
    return q, kc, vc, pos, table, D ** -0.5, H, opts


def _windowed_error(args):
    from neuronx_distributed_inference_amd.ops import ref, seqmix

    q, kc, vc, pos, table, scale, H, opts = args
    want = ref.paged_attention(q.reshape(*q.shape[:2], H, -1), kc, vc, pos, table, scale, **opts)
    cu = lambda t: t.cuda() if torch.is_tensor(t) else t  # noqa: E731
    rows = torch.empty(*q.shape[:2], q.shape[2] + 8, dtype=q.dtype, device="cuda")
    rows[..., : q.shape[2]] = q.cuda()
    step = seqmix.StepLayout(pos.cuda(), torch.arange(q.shape[0], device="cuda"))
    got = seqmix.paged_attention(rows[..., : q.shape[2]], kc.cuda(), vc.cuda(), step, table.cuda(), scale, H,
                                 **{k: cu(v) for k, v in opts.items()})
    ok = pos >= 0
    got, want = got.cpu().to(F64)[ok], want.to(F64)[ok]
    return ((got - want).norm() / want.norm()).item()


@pytest.mark.parametrize("S,H,G,D,page,start,opts", WINDOWED)
def test_windowed_attention_of_portions(S, H, G, D, page, start, opts):
    """Rows that end inside tiles, windows, kept keys and blocks that begin and end inside them,
    every option, against the plain reference: the result's rounding (2^-9) and as much for P's
    16 bits and the hardware logarithm."""
    assert _windowed_error(_windowed(S, H, G, D, page, start, opts)) < 2.0 ** -8


@pytest.mark.parametrize("H,G,D,page,start,opts", [
    (4, 4, 64, 16, 0, {}), (12, 4, 128, 24, 200, dict(window=70, keep_first=3, r=True, gate="full")),
    (16, 4, 128, 64, 700, dict(window=1024, keep_first=4, r=True, gate="full")),
    (17, 1, 64, 64, 255, dict(window=256, keep_first=300, sink=True, gate="head")),
    (40, 2, 128, 16, 95, dict(chunk=48, keep_first=60, softcap=20.0)),
    (16, 1, 64, 24, 2211, dict(slopes=True, q_temp=(0.3, 64))), (3, 1, 128, 16, 31, dict(window=1, r=True))])
def test_windowed_attention_of_single_tokens(H, G, D, page, start, opts):
    """One key to several rounds of the waves, more heads than a tile has columns, every option:
    the result's rounding (2^-9) and as much for the hardware logarithm and exponential."""
    q, kc, vc, pos, table, scale, H, o = _windowed(3, H, G, D, page, start, opts)
    for s in range(3):
        one = lambda t: t[:, s:s + 1] if torch.is_tensor(t) and t.dim() == 3 and t.shape[1] == 3 else t  # noqa: E731
        args = (q[:, s:s + 1], kc, vc, pos[:, s:s + 1], table, scale, H, {k: one(v) for k, v in o.items()})
        assert _windowed_error(args) < 2.0 ** -8


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
def test_windowed_attention_of_single_tokens_values_not_finite(D, bad):
    """A value that is not finite reaches the rows that see its key, as such, and no others."""
    from neuronx_distributed_inference_amd.ops import seqmix

    H, G, page, n = 6, 2, 16, 300
    q, kc, vc, _, table, scale, H, o = _windowed(2, H, G, D, page, n, dict(window=100, keep_first=2))
    pos = torch.tensor([[n], [n + 3], [n + 9]])
    clean = vc.clone()
    for b, key in ((0, n - 50), (1, n - 96), (2, 1), (2, 50)):     # seen; seen; kept; not seen
        vc[table[b, key // page], key % page, 0, 5] = bad
    step = seqmix.StepLayout(pos.cuda(), torch.arange(3, device="cuda"))
    run = lambda v: seqmix.paged_attention(q[:, :1].contiguous().cuda(), kc.cuda(), v.cuda(), step,  # noqa: E731
                                           table.cuda(), scale, H, **o).cpu().float().view(3, H, D)
    got, want = run(vc), run(clean)
    hit = torch.zeros(3, H, D, dtype=torch.bool)
    hit[:, :H // G, 5] = True
    assert torch.equal(torch.isfinite(got), ~hit)
    assert (torch.isnan(got[hit]) if bad != bad else got[hit] == bad).all()
    assert (got[~hit] - want[~hit]).abs().max() < 2.0 ** -7 * want.abs().max()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K,glu", [
    (129, 5124, 4160, False), (160, 21000, 1024, False), (191, 32764, 704, False), (192, 6144, 4096, False),
    (193, 32768, 704, False), (129, 28680, 768, True), (192, 21000, 1024, True), (65, 28672, 256, True),
    (128, 49152, 256, True), (128, 49144, 320, True)])
def test_tile_gemm_rings_of_their_own(M, N, K, glu, dtype):
    """Tiles of 192 rows, whose halves of the waves load x and w through rings of unequal length:
    fewer chunks than either ring, as many, more; and the other tiles at the border."""
    x, w, exact, sums = _product(M, N, K, dtype)
    if glu:
        g, u = exact.chunk(2, dim=1)
        want = torch.nn.functional.silu(g) * u
        gs, us = sums.chunk(2, dim=1)
        limit = 1.1 * gs * u.abs() + us * g.abs() + (EPS16[dtype] + 2.0 ** -18) * want.abs() + 1e-6
        got = ops._C.tile_gemm(x, w, glu=True).to(F64)
        assert ((got - want).abs() <= limit).all()
        return
    for splits in {1, 2, ops._tile_takes(x, w), K // 64}:
        parts = ops._C.tile_gemm(x, w, None, splits, True).to(F64)
        got, limit = (parts.sum(0), sums) if splits > 1 else (parts, sums + EPS16[dtype] * exact.abs())
        assert ((got - exact).abs() <= limit + 1e-30).all()


@pytest.mark.parametrize("kind", ["linear", "ring", "paged", "fp8", "window"])
@pytest.mark.parametrize("B,Hkv,gq,Sq,D", [(257, 3, 4, 1, 128), (257, 8, 1, 3, 64), (193, 8, 8, 1, 64),
                                           (343, 3, 1, 1, 64), (257, 7, 5, 4, 128), (683, 3, 1, 3, 64),
                                           (64, 8, 4, 1, 128)])
def test_decode_attention_of_many_short_rows(kind, B, Hkv, gq, Sq, D):
    """A wave a row (the last workgroup's may have none) against the same rows in small
    batches, which four waves or splits of the keys serve: both round the result once (2^-9). A
    wave a row from 768 sets of columns on (heads of 64: 1024, in 8 bits 2048); the last shape has
    fewer, and heads of 64 in 8 bits take some of the others with four waves."""
    sets = B * Hkv * -(-gq * Sq // 16)
    assert (sets >= (768 if D == 128 else 1024)) == (B != 64) and 20 * Hkv * -(-gq * Sq // 16) < 768
    g = torch.Generator(device="cuda").manual_seed(B)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).bfloat16()  # noqa: E731
    cap, Hq = 96 if kind != "window" else 700, Hkv * gq
    q = rnd(B, Hq, Sq, D)
    pos = torch.randint(0, 2 * cap if kind == "ring" else cap - Sq, (B, 1), device="cuda", generator=g) \
        + torch.arange(Sq, device="cuda")
    if kind == "paged":
        k, v = rnd(B * 6, 16, Hkv, D), rnd(B * 6, 16, Hkv, D)
        table = torch.randperm(B * 6, device="cuda", generator=g).view(B, 6).int()
        table[3, 2:] = -1
        run = lambda a, b: ops.attention_decode_paged(q[a:b], k, v, pos[a:b], table[a:b])  # noqa: E731
    else:
        k, v = rnd(B, Hkv, cap, D), rnd(B, Hkv, cap, D)
        if kind == "fp8":
            k, v = k.to(torch.float8_e4m3fn), v.to(torch.float8_e4m3fn)
        rows = torch.randperm(B, device="cuda", generator=g).int()
        kw = {"ring": dict(sliding_window=cap, ring=True), "window": dict(sliding_window=40)}.get(kind, {})
        run = lambda a, b: ops.attention_decode(q[a:b], k, v, pos[a:b], rows[a:b], **kw)  # noqa: E731
    got = run(0, B)
    want = torch.cat([run(a, min(a + 20, B)) for a in range(0, B, 20)])
    err = (got.to(F64) - want.to(F64)).norm(dim=-1) / want.to(F64).norm(dim=-1).clamp(min=1e-3)
    assert torch.isfinite(got).all() and err.max() < 2.0 ** -7 and err.mean() < 2.0 ** -8


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("B,S,ragged", [(1, 2, False), (1, 159, False), (2, 70, True), (2, 100, False),
                                        (2, 101, False)])
def test_short_prompts_by_one_native_call(B, S, ragged, dtype, monkeypatch):
    """The native call makes the launches that the layers make one by one: logits and cache to the
    bit, also for more rows than it takes, an off-cut weight and another row of the cache."""
    from neuronx_distributed_inference_amd.modules import fused_layer

    lm = _small_llama(dtype)
    ids = torch.randint(0, 512, (B, S), device="cuda")
    mask = torch.ones(B, S, dtype=torch.long, device="cuda")
    if ragged:
        mask[1, S // 3:] = 0
    seq = torch.arange(B, device="cuda").flip(0)
    calls = []
    native = fused_layer._short_prompt

    def run(rows):
        monkeypatch.setattr(fused_layer, "PROMPT_ROWS", rows)
        monkeypatch.setattr(fused_layer, "_short_prompt",
                            lambda *a: calls.append(native(*a)) or calls[-1])
        lm.reset()
        with torch.inference_mode():
            out = lm(input_ids=ids, attention_mask=mask, seq_ids=seq).logits.clone()
        return [out] + [t.data.clone() for i in range(2) for t in lm.model.kv_mgr.get_cache(i)]

    a, b = run(200), run(0)
    assert (calls[0] is not None) == (B * S <= 200) and calls[1] is None
    assert all(torch.equal(x, y) for x, y in zip(a, b))
    w = lm.model.layers[1].mlp.down_proj.weight
    off = torch.empty(w.numel() + 1, dtype=w.dtype, device="cuda")[1:].view_as(w).copy_(w.data)
    monkeypatch.setattr(w, "data", off)
    c = run(200)
    assert calls[2] is None
    assert all((x.float() - y.float()).norm() <= 0.03 * y.float().norm() for x, y in zip(c, a))


@pytest.mark.parametrize("E", [1, 8, 63, 64, 65, 128, 200, 257, 512, 513, 1000])
@pytest.mark.parametrize("kind", ["normal", "ties", "masked"])
def test_router_topk_of_any_width(E, kind):
    """Choices and their order against torch's stable sort, ties by the lowest index; masked logits
    (-inf, the type's lowest) are not chosen while others are left."""
    k = min(8, E)
    x = torch.randn(333, E, device="cuda")
    if kind == "ties":
        x = torch.randint(0, 3, (333, E), device="cuda").float()
    if kind == "masked":
        x[:, k:] = torch.where(torch.rand(333, E - k, device="cuda") < 0.5, x[:, k:],
                               torch.finfo(torch.float32).min)
        x[:, E - 1 if E > k else 0] = -float("inf") if E > k else x[:, 0]
    vals = torch.empty(333, k, device="cuda")
    idx = torch.empty(333, k, dtype=torch.long, device="cuda")
    ops._C.router_topk(vals, idx, x, k, 0, 0, 0)
    top, order = x.sort(dim=-1, descending=True, stable=True)
    assert torch.equal(idx, order[:, :k])
    want = torch.softmax(top[:, :k].double(), -1)
    assert ((vals - want).abs() < 1e-6).all()


@pytest.mark.parametrize("xd,yd", [(torch.bfloat16, torch.float32), (torch.float32, torch.bfloat16),
                                   (torch.float32, torch.float32)])
@pytest.mark.parametrize("taps,silu,residual,bias", [(2, False, True, False), (4, True, False, True), (7, False, False, False)])
def test_short_conv_of_single_tokens(taps, silu, residual, bias, xd, yd):
    """Conv and tail in one launch against the two: the same sums in the same order, to the bit;
    first tokens, padding rows and rows of other sequences among them."""
    from neuronx_distributed_inference_amd.ops import seqmix

    B, C = 9, 333
    x = torch.randn(B, 1, C + 7, device="cuda").to(xd)[..., 3:3 + C]
    w, tail = torch.randn(C, taps, device="cuda"), torch.randn(12, taps - 1, C, device="cuda")
    pos = torch.tensor([[0], [1], [2], [3], [50], [-1], [9], [2], [6]], device="cuda")
    seq = torch.tensor([3, 0, 11, 5, 4, 6, -1, 8, 9], device="cuda")
    step = seqmix.StepLayout(pos, seq)
    kw = dict(activation="silu" if silu else "none", residual=residual, out_dtype=yd,
              bias=torch.randn(C, device="cuda") if bias else None)
    t0 = tail.clone()
    want = seqmix.short_conv(x, w, t0, step, **kw)
    seqmix.short_conv_commit(x, t0, step)
    t1 = tail.clone()
    got = seqmix.short_conv_step(x, w, t1, step, **kw)
    assert torch.equal(got, want) and torch.equal(t0, t1)


def test_rows_of_8_bits_keep_the_roundings_on_the_way():
    """fp16 onto an 8-bit cache: a decoded token leaves the row that the modules one by one leave."""
    lm = _small_llama("float16", kv_cache_quant=True)
    ids = torch.randint(0, 512, (2, 40), device="cuda")
    step = torch.randint(0, 512, (2, 1), device="cuda")

    def run():
        lm.reset()
        with torch.inference_mode():
            lm(input_ids=ids)
            lm(input_ids=step, position_ids=torch.full((2, 1), 40, device="cuda"))
        return [t.data[:, :, 40].float() for i in range(2) for t in lm.model.kv_mgr.get_cache(i)]

    got = run()
    note = [m.register_forward_hook(lambda *a: None) for m in lm.model.modules()]
    want = run()
    for h in note:
        h.remove()
    for a, b in zip(got, want):
        assert (a != b).float().mean().item() <= 0.002


@pytest.mark.parametrize("moe", [False, True])
@pytest.mark.parametrize("what", ["layer class", "o_proj class", "layers' class", "norms' class",
                                  "linears' class", "o_projs' class", "attentions' class", "layer", "self_attn", "norm", "o_proj",
                                  "o_proj.o_proj", "qkv", "mlp", "down", "final", "embed_tokens",
                                  "embed", "prepare_hidden", "before_layer_run"])
def test_a_forward_of_its_own_is_called(what, moe, monkeypatch):
    """A module whose forward is not the one that the fused layers stand for (a subclass's, set on
    the instance or put in its class's place) is called, in the prompt and in the step after it, and its result counts."""
    if moe and what == "down":
        pytest.skip("no down projection")
    lm = _small_llama("bfloat16", moe=moe)
    model, layer = lm.model, lm.model.layers[1]
    attn, seen = layer.self_attn, []

    def halved(forward):
        def run(*a, **kw):
            seen.append(1)
            y = forward(*a, **kw)
            return (y[0] * 0.5, *y[1:]) if isinstance(y, tuple) else y * 0.5
        return run

    def run():
        lm.reset()
        with torch.inference_mode():
            a = lm(input_ids=ids, position_ids=pos).logits
            b = lm(input_ids=step, position_ids=torch.full((2, 1), 70, device="cuda")).logits
        return torch.cat([a, b], dim=1).float()

    ids, step = torch.randint(0, 512, (2, 70), device="cuda"), torch.randint(0, 512, (2, 1), device="cuda")
    pos = torch.arange(70, device="cuda").repeat(2, 1)
    start, starts = ops.step_start, []
    monkeypatch.setattr(ops, "step_start", lambda *a: starts.append(1) or start(*a))
    plain = run()
    assert len(starts) == 2                      # nothing here keeps the start kernel away
    if what.endswith("s' class"):
        mod = {"layers'": layer, "norms'": model.norm, "linears'": attn.o_proj.o_proj,
               "o_projs'": attn.o_proj, "attentions'": attn}[what[:-6]]
        monkeypatch.setattr(type(mod), "forward", halved(type(mod).forward))
    elif what.endswith(" class"):
        mod = layer if what == "layer class" else attn.o_proj
        base = type(mod)
        mod.__class__ = type("Own", (base,), {"forward": halved(base.forward)})
    elif what in ("embed", "prepare_hidden", "before_layer_run"):
        setattr(model, what, halved(getattr(model, what)))
    else:
        mod = {"layer": layer, "self_attn": attn, "norm": layer.post_attention_layernorm,
               "o_proj": attn.o_proj, "o_proj.o_proj": attn.o_proj.o_proj,
               "qkv": attn.qkv_proj.qkv, "mlp": layer.mlp,
               "down": getattr(layer.mlp, "down_proj", None), "final": model.norm,
               "embed_tokens": model.embed_tokens}[what]
        mod.forward = halved(mod.forward)
    own = run()
    assert len(seen) >= 2
    assert (own - plain).norm() > 0.05 * plain.norm()


@pytest.mark.parametrize("of_class", [False, True])
@pytest.mark.parametrize("rows", [1, 2])
def test_an_attend_fused_of_its_own_is_called(of_class, rows, monkeypatch):
    """With the arguments that it always had, in short and in ragged prompts and in steps."""
    lm = _small_llama("bfloat16")
    lm.enable_submodels()
    attn = lm.model.layers[1].self_attn
    ids = torch.randint(0, 512, (rows, 70), device="cuda")
    mask = torch.ones_like(ids)
    mask[-1, 60:] = 0

    def run():
        lm.reset()
        with torch.inference_mode():
            a = lm(input_ids=ids, attention_mask=mask).logits
            lm.reset()
            b = lm(input_ids=ids).logits
            c = lm(input_ids=ids[:, :1], position_ids=torch.full((rows, 1), 70, device="cuda")).logits
        return torch.stack([a, b, c]).float()

    plain, seen = run(), []
    inner = type(attn).attend_fused

    def own(self, hidden, cos, sin, kv_mgr, position_ids, phase, attention_mask=None, seq_ids=None,
            active_mask=None, sequence_parallel=False):
        seen.append(phase)
        return inner(self, hidden, cos, sin, kv_mgr, position_ids, phase, attention_mask, seq_ids,
                     active_mask, sequence_parallel) * 0.5

    if of_class:
        base = next(c for c in type(attn).__mro__ if "attend_fused" in vars(c))
        monkeypatch.setattr(base, "attend_fused", own)
    else:
        attn.attend_fused = own.__get__(attn)
    got = run()
    assert len(seen) == (6 if of_class else 3)
    assert ((got - plain).flatten(1).norm(dim=1) > 0.02 * plain.flatten(1).norm(dim=1)).all()


def test_hooks_of_all_modules_see_the_qkv_projection():
    lm = _small_llama("bfloat16")
    ids = torch.randint(0, 512, (2, 70), device="cuda")
    seen = []
    h = torch.nn.modules.module.register_module_forward_hook(lambda m, *a: seen.append(m))
    try:
        with torch.inference_mode():
            lm(input_ids=ids)
            lm(input_ids=ids[:, :1], position_ids=torch.full((2, 1), 70, device="cuda"))
    finally:
        h.remove()
    for layer in lm.model.layers:
        assert sum(m is layer.self_attn.qkv_proj.qkv for m in seen) == 2


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows_that_start_off_16_bytes(dtype):
    """Caches and rope rows that start off 16 bytes: what the kernels that take them give, in the
    step, in the prompt and in the native call, next to aligned ones."""
    lm = _small_llama(str(dtype)[6:])
    ids = torch.randint(0, 512, (2, 70), device="cuda")
    plain_cos_sin = lm.model.rotary.get_cos_sin

    def off(t):
        return torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")[1:].view_as(t).copy_(t)

    def run():
        lm.reset()
        with torch.inference_mode():
            a = lm(input_ids=ids).logits
            b = lm(input_ids=ids[:, :1], position_ids=torch.full((2, 1), 70, device="cuda")).logits
        return [a.float(), b.float()] + [t.data.float() for t in lm.model.kv_mgr.get_cache(1)]

    want = run()
    lm.model.rotary.get_cos_sin = lambda *a, **kw: tuple(map(off, plain_cos_sin(*a, **kw)))
    rope = run()
    lm.model.rotary.get_cos_sin = plain_cos_sin
    for i in range(2):
        for t in lm.model.kv_mgr.get_cache(i):
            t.data = off(t.data)
    cache = run()
    # 16-bit activations of two layers, rounded at other places
    tol = 0.03 if dtype == torch.bfloat16 else 0.004
    for got in (rope, cache):
        for a, b in zip(got, want):
            assert (a - b).norm() <= tol * b.norm()


@pytest.mark.parametrize("how", ["rows apart", "transposed", "off 16 bytes"])
def test_feed_forward_results_of_any_layout(how):
    """A feed-forward of the program's own may hand out rows apart, transposed or off 16 bytes."""
    lm = _small_llama("bfloat16")
    ids = torch.randint(0, 512, (2, 70), device="cuda")

    class Own(torch.nn.Module):
        def __init__(self, mlp):
            super().__init__()
            self.mlp = mlp

        def forward(self, x, sequence_parallel=False):
            y = self.mlp(x)
            B, S, H = y.shape
            if how == "rows apart":
                z = y.new_empty(B, S, 2 * H)[..., :H]
            elif how == "transposed":
                z = y.new_empty(H, S, B).permute(2, 1, 0)
            else:
                z = y.new_empty(y.numel() + 1)[1:].view(B, S, H)
            return z.copy_(y)

    def run():
        lm.reset()
        with torch.inference_mode():
            a = lm(input_ids=ids).logits
            b = lm(input_ids=ids[:, :1], position_ids=torch.full((2, 1), 70, device="cuda")).logits
        return a.float(), b.float()

    want = run()
    for layer in lm.model.layers:
        layer.mlp = Own(layer.mlp)
    for a, b in zip(run(), want):
        assert (a - b).norm() <= 0.03 * b.norm()


@pytest.mark.parametrize("switch", ["NXDI_DISABLE_SG5", "NXDI_DISABLE_HIPBLASLT"])
@pytest.mark.parametrize("moe", [False, True])
def test_switches_of_the_products_hold_in_fused_layers(switch, moe, monkeypatch):
    """Neither the tiled product nor the native prompt, which is made of it, under either switch."""
    lm = _small_llama("bfloat16", moe=moe)
    ids = torch.randint(0, 512, (2, 70), device="cuda")

    def run():
        lm.reset()
        with torch.inference_mode():
            a = lm(input_ids=ids).logits
            b = lm(input_ids=ids[:, :1], position_ids=torch.full((2, 1), 70, device="cuda")).logits
        return a.float(), b.float()

    want = run()
    calls = []
    for name in ("tile_gemm", "prompt_layers"):
        monkeypatch.setattr(ops._C, name, lambda *a, _n=name, **kw: calls.append(_n))
    monkeypatch.setitem(ops._lt_state, "enabled", None)
    monkeypatch.setenv(switch, "1")
    got = run()
    assert not calls
    for a, b in zip(got, want):
        assert (a - b).norm() <= 0.03 * b.norm()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("S", [70, 300])
def test_windowed_attention_under_steep_distances(S, D):
    """Portions under r2 of 1e5 and more: 1 + r2 * distance is one multiply-add of the whole distance. Made
    from a tile's first distance less a key's place in it, its sum cancels at the near keys, and
    what is lost is 59 * r2 of 2^-24: of a key's own 1, an eighth and more."""
    args = list(_windowed(S, 8, 2, D, 16, 40, dict(window=200)))
    args[-1] = dict(window=200, r1=torch.linspace(0.1, 0.4, 8), r2=torch.linspace(1e5, 2e5, 8))
    assert _windowed_error(tuple(args)) < 2.0 ** -8


def test_sequence_mixing_models_without_the_other_library(monkeypatch):
    """Step layouts, slots, page tables and the inputs of captured steps of models that load the
    sequence-mixing library only."""
    from neuronx_distributed_inference_amd.models.hybrid_base import HybridDecoderModel
    from neuronx_distributed_inference_amd.modules.kvcache.block_kv_cache_manager import (
        generate_slot_mapping)
    from neuronx_distributed_inference_amd.ops.seqmix import StepLayout
    from neuronx_distributed_inference_amd.runtime.graph_engine import GraphRunner

    monkeypatch.setattr(ops, "_C", None)
    pos, seq = torch.randint(-2, 90, (3, 5)), torch.tensor([2, -1, 0])
    table = torch.randint(-1, 40, (3, 6))
    model = type("M", (), {"max_blocks_per_seq": 7})()
    model.kv_mgr = type("K", (), {"num_blocks": 10 ** 6, "state": type("S", (), {"num_slots": 8})})()

    def run(dev):
        a = StepLayout(pos.to(dev), seq.to(dev))
        return [a.positions, a.seq_ids, a.nvalid,
                generate_slot_mapping(table.to(dev), pos.to(dev), 16, torch.int32),
                HybridDecoderModel.begin_step(model, pos.to(dev), seq.to(dev), None).long()]

    for a, b in zip(run("cuda"), run("cpu")):
        assert a.dtype == b.dtype and torch.equal(a.cpu(), b)
    step = GraphRunner(lambda x, y: x * 2 + y, (torch.zeros(4, device="cuda"), torch.zeros(4, device="cuda")))
    x, y = torch.arange(4.0, device="cuda"), torch.ones(4, device="cuda")
    assert torch.equal(step(x, y), x * 2 + y)


@pytest.mark.parametrize("T,E,k,H,I,f8", [(1, 8, 2, 4096, 1024, False), (1, 8, 2, 4096, 1024, True),
                                          (24, 64, 8, 2048, 512, False), (300, 8, 2, 4096, 1088, False)])
def test_moe_routed_room_for_shares_by_the_tiles(T, E, k, H, I, f8):
    """The down projection's shares take a place for each workgroup and each tile there can be, as
    long as those are few, and no more than that."""
    g = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn(T, H, device="cuda", generator=g).bfloat16()
    wt, idx = torch.softmax(torch.randn(T, E, device="cuda", generator=g), -1).topk(k, dim=-1)
    w = [(torch.randn(E, *s, device="cuda", generator=g) * 0.05).bfloat16() for s in ((I, H), (I, H), (H, I))]
    scales = None
    if f8:
        w, scales = zip(*[ops.fp8_moe_quantize(v) for v in w])
    mt = ops._moe_tile_rows(T * k, E, E, H, I, f8)
    tiles = (T * k + min(T * k, E) * (mt - 1)) // mt
    products = max(tiles * mt * H, (256 + min(512, tiles * -(-H // 256))) * mt * 256) * 4
    rest = tiles * mt * I * 2 + T * H * 2 + (1 + 2 * tiles + tiles * mt + T * k) * 4
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    ops.moe_routed_experts(x, wt, idx, *w, scales=scales, num_experts=E)
    # the allocator leaves up to 1 MB of a block with each of the large tensors (products, h, out)
    assert torch.cuda.max_memory_allocated() - before <= products + rest + (3 << 20)


def test_products_are_chosen_by_the_gpus_time(monkeypatch):
    """A library call that the host takes 50 us to launch and the GPU 8 to run stays the choice
    beside a kernel that takes the GPU 25 us or more and is launched at once: captured steps wait
    for the GPU only."""
    import time

    M, N, K = 48, 2048, 2048
    x, w, _, _ = _product(M, N, K, torch.bfloat16)
    lt, tiled = ops.lt_linear, ops._C.tile_gemm

    def slow_launch(*a):
        until = time.perf_counter() + 50e-6
        while time.perf_counter() < until:
            pass
        return lt(*a)

    def slow_kernel(*a, **kw):
        for _ in range(3):
            y = tiled(*a, **kw)
        return y

    monkeypatch.setattr(ops, "lt_linear", slow_launch)
    monkeypatch.setattr(ops._C, "tile_gemm", slow_kernel)
    monkeypatch.setitem(ops._sg5_state, "choice", {})
    assert ops._sg5_autotune((M, N, K, False, x.dtype), x, w, None) == 0


def _small_of(kind, dtype):
    """A two-layer model of the kinds that run_layers serves beside _small_llama's, random weights."""
    import importlib

    from neuronx_distributed_inference_amd.config import EngineConfig

    family, cls = {"llama": ("llama", "Llama"), "qwen2": ("qwen2", "Qwen2"), "qwen3": ("qwen3", "Qwen3"),
                   "qwen3moe": ("qwen3_moe", "Qwen3Moe")}[kind.split()[0]]
    mod = importlib.import_module(f"neuronx_distributed_inference_amd.models.{family}.modeling_{family}")
    paged = dict(is_block_kv_layout=True, pa_block_size=16, pa_num_blocks=24) if "paged" in kind else {}
    ec = EngineConfig(batch_size=2, max_batch_size=2, seq_len=160, max_length=160, torch_dtype=dtype,
                      tp_degree=1, output_logits=True, fused_qkv=True, fused_gate_up=True,
                      enable_batch_bucketing=False, **paged)
    sizes = dict(neuron_config=ec, hidden_size=512, intermediate_size=1024, num_hidden_layers=2,
                 num_attention_heads=8, num_key_value_heads=2, head_dim=64, vocab_size=512,
                 max_position_embeddings=320, rms_norm_eps=1e-5, rope_theta=10000.0, hidden_act="silu",
                 tie_word_embeddings=False)
    if family == "qwen3_moe":                     # all experts: no choice that rounding flips
        sizes.update(num_experts=4, num_experts_per_tok=4, moe_intermediate_size=512)
    with torch.device("cuda"):
        lm = getattr(mod, cls + "ForCausalLM")(getattr(mod, cls + "InferenceConfig")(**sizes)).eval()
    g = torch.Generator(device="cuda").manual_seed(0)
    for name, p in lm.model.named_parameters():
        p.data.uniform_(0.5, 1.5, generator=g) if "norm" in name else p.data.normal_(0, 0.05, generator=g)
    assert any("bias" in n for n, _ in lm.model.named_parameters()) == (family == "qwen2")
    return lm


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("kind", ["qwen2", "qwen3", "qwen3moe", "llama paged", "qwen2 paged", "qwen3 paged",
                                  "qwen3moe paged"])
def test_fused_layers_of_other_kinds(kind, dtype, monkeypatch):
    """q/k norms, q|k|v biases and pages (a first portion, a second onto its pages, a step): the
    fused layers against the chain of modules."""
    from neuronx_distributed_inference_amd.models import model_base

    lm = _small_of(kind, dtype)
    ids = torch.randint(0, 512, (2, 71), device="cuda")
    pos = torch.arange(71, device="cuda").repeat(2, 1)
    table = torch.randperm(24, device="cuda")[:20].view(2, 10)
    calls, run_layers = [], model_base.run_layers
    monkeypatch.setattr(model_base, "run_layers", lambda *a: calls.append(1) or run_layers(*a))

    def run():
        lm.reset()
        cuts, out = ([(0, 40), (40, 70), (70, 71)] if "paged" in kind else [(0, 70), (70, 71)]), []
        with torch.inference_mode():
            for a, b in cuts:
                kw = dict(block_table=table, phase="token_generation") if "paged" in kind else {}
                out.append(lm(input_ids=ids[:, a:b].contiguous(), position_ids=pos[:, a:b].contiguous(),
                              **kw).logits.float())
        return out + [t.data.float().clone() for i in range(2) for t in lm.model.kv_mgr.get_cache(i)]

    fused = run()
    assert len(calls) == len(fused) - 4
    hook = lm.model.norm.register_forward_hook(lambda *a: None)
    plain = run()
    hook.remove()
    assert len(calls) == len(fused) - 4
    # 16-bit activations of two layers, rounded at other places
    tol = 0.03 if dtype == "bfloat16" else 0.004
    for a, b in zip(fused, plain):
        assert b.norm() > 0 and (a - b).norm() <= tol * b.norm()


@pytest.mark.parametrize("mt,f8,rows,E,H,I,shared", [
    (32, False, 60, 4, 4096, 2048, True),      # second tiles, but 128 tiles: half a round
    (32, False, 70, 4, 4096, 2048, False),     # 192 of them
    (64, False, 50, 16, 2560, 2048, True),     # 160, a row tile an expert
    (48, True, 40, 24, 4096, 1536, True),      # 384 in two rounds, 18 steps a workgroup
    (48, True, 40, 24, 4096, 1280, False)])    # 15 steps
def test_moe_routed_shares_by_tiles_of_an_expert(mt, f8, rows, E, H, I, shared, monkeypatch):
    """On both sides of the rule for shares (mr_shares): even choices, sums against 64 bits."""
    ntn, nk, tiles = -(-H // 256), I // (128 if f8 else 64), E * -(-rows // mt)
    total = tiles * ntn
    assert total * 100 < -(-total // 256) * 256 * 85 and total * nk >= 2048
    assert shared == (total <= 128 or (total * nk >= 4096 and tiles * 8 < E * 9))
    monkeypatch.setattr(ops, "_moe_tile_rows", lambda *a: mt)
    g = torch.Generator(device="cuda").manual_seed(rows)
    T, k = rows * E // 2, 2
    x = torch.randn(T, H, device="cuda", generator=g).bfloat16()
    idx = torch.stack([torch.arange(T, device="cuda") % E, (torch.arange(T, device="cuda") + 1) % E], 1)
    wt = torch.rand(T, k, device="cuda", generator=g) + 0.1
    w = [(torch.randn(E, *s, device="cuda", generator=g) * 0.05).bfloat16() for s in ((I, H), (I, H), (H, I))]
    scales, ref = None, [v.to(F64) for v in w]
    if f8:
        w, scales = zip(*[ops.fp8_moe_quantize(v) for v in w])
        ref = [ops.fp8_moe_dequant(v, s).to(F64) for v, s in zip(w, scales)]
    want = torch.zeros(T, H, dtype=F64, device="cuda")
    for e in range(E):
        t, j = (idx == e).nonzero(as_tuple=True)
        xe = x[t].to(F64)
        h = torch.nn.functional.silu(xe @ ref[0][e].t()) * (xe @ ref[1][e].t())
        want.index_add_(0, t, (h @ ref[2][e].t()) * wt[t, j].to(F64).unsqueeze(1))
    got = ops.moe_routed_experts(x, wt, idx, *w, scales=scales, num_experts=E)
    assert (got.to(F64) - want).norm() < EPS16[torch.bfloat16] * want.norm()
    assert torch.equal(got, ops.moe_routed_experts(x, wt, idx, *w, scales=scales, num_experts=E))


@pytest.mark.parametrize("itype", [torch.int64, torch.int32])
@pytest.mark.parametrize("n_tok,E,k,first,El", [(1, 8, 2, 0, 8), (3, 4, 1, 2, 2), (64, 8, 8, 0, 8), (255, 130, 8, 1, 65),
                                                (256, 9, 8, 0, 9), (257, 64, 8, 0, 64), (1024, 8, 8, 3, 4),
                                                (1025, 300, 8, 0, 300), (5000, 8, 2, 0, 8)])
def test_moe_route_of_any_number_of_choices(n_tok, E, k, first, El, itype):
    """The table of rows against the same made on the CPU, to the bit: runs of choices that a wave
    reads once (up to 512 each of 4, then of 16 waves) and longer ones, other ranks' experts."""
    mt = 32
    idx = torch.randint(0, E, (n_tok, k), generator=torch.Generator().manual_seed(n_tok)).to(itype)
    n = idx.numel()
    most = (n + min(n, El) * (mt - 1)) // mt
    tiles, gather, inv = (torch.full((s,), -7, dtype=torch.int32, device="cuda")
                          for s in (1 + 2 * most, most * mt, n))
    ops._C.moe_route(tiles, gather, inv, idx.cuda(), El, first, mt)
    want_t, want_g, want_i = [], {}, [-1] * n
    flat = [int(e) - first for e in idx.flatten()]
    by = [[i for i, e in enumerate(flat) if e == x] for x in range(El)]
    for e, rows in enumerate(by):
        for a in range(0, len(rows), mt):
            for j, i in enumerate(rows[a:a + mt]):
                want_i[i] = len(want_t) * mt + j
                want_g[want_i[i]] = i // k
            want_t.append((e, len(rows[a:a + mt])))
    used = sum(bool(r) for r in by)
    crowded = len(want_t) * 8 >= used * 9
    t = tiles.tolist()
    assert t[0] == len(want_t) + (1 << 30) * crowded
    assert list(zip(t[1::2], t[2::2]))[:len(want_t)] == want_t
    assert inv.tolist() == want_i
    got = gather.tolist()
    assert all(got[r] == tok for r, tok in want_g.items())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,E,k,K", [(1, 1, 1, 8), (3, 8, 2, 4096), (7, 3, 3, 4104), (200, 9, 8, 1000),
                                     (511, 16, 4, 320), (512, 9, 2, 64), (1023, 5, 2, 512),
                                     (1030, 8, 8, 520), (5, 8, 2, 36)])
def test_router_of_few_experts(T, E, k, K, dtype):
    """Product and choice in one launch against the same in 64 bits: the chosen are the largest but
    for sums that lie within the rounding of 32 bits, their weights those of the chosen sums."""
    g = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn(T, K, device="cuda", generator=g).to(dtype)
    w = torch.randn(E, K, device="cuda", generator=g) * 0.1
    exact = x.to(F64) @ w.to(F64).t()
    slack = K * 2.0 ** -24 * (x.to(F64).abs() @ w.to(F64).abs().t()).max()
    for sigmoid, pre, norm in ((False, False, True), (False, True, False), (True, False, False)):
        vals, idx = ops.router_choice(x, w, k, sigmoid, pre, norm)
        assert vals.shape == idx.shape == (T, k) and vals.dtype == torch.float32
        assert (idx.sort(-1).values.diff() > 0).all() and 0 <= idx.min() and idx.max() < E
        chosen = exact.gather(1, idx)
        assert (chosen >= exact.topk(k, -1).values - 2 * slack).all()
        want = chosen.sigmoid() if sigmoid else \
            (exact.softmax(-1).gather(1, idx) if pre else chosen.softmax(-1))
        # exp of 32 bits, of sums that are off by the slack
        assert ((vals - want).abs() <= want * (4 * slack + 2.0 ** -18)).all()
    # a row that is not a number chooses as the rows of logits do
    x[0] = float("nan")
    got = ops.router_choice(x, w, k, False, False, True)
    ref = ops.router_topk(torch.nn.functional.linear(x.float(), w), k, False, False, True)
    assert torch.equal(got[1][:1], ref[1][:1])


def test_weights_in_host_memory_are_refused():
    x, w = torch.zeros(2, 512, device="cuda"), torch.zeros(8, 512)
    with pytest.raises(RuntimeError):
        ops.router_choice(x, w, 2, False, False, True)
    x, w = x.bfloat16(), torch.zeros(256, 512, dtype=torch.bfloat16)
    for call in (lambda: ops.linear_parts(x, w), lambda: ops.linear_silu_mul(x, w)):
        with pytest.raises(RuntimeError):
            call()
    q, cache = x[:1].view(1, 8, 1, 64), torch.zeros(1, 2, 600, 64, dtype=torch.bfloat16, device="cuda")
    pos = torch.tensor([[500]], device="cuda")
    with pytest.raises(RuntimeError):
        ops.attention_decode_product(q, cache, cache, pos, None, 1.0, 0, w)


@pytest.mark.parametrize("moe", [False, True])
def test_layers_are_asked_once_a_prompt(moe, monkeypatch):
    """Whether they run fused, also where they do not run without the prompt's padding."""
    from neuronx_distributed_inference_amd.models import model_base

    lm = _small_llama("bfloat16", moe=moe)
    lm.enable_submodels()
    ids = torch.randint(0, 512, (2, 70), device="cuda")
    asked, inner = [], model_base.fusable
    monkeypatch.setattr(model_base, "fusable", lambda *a: asked.append(inner(*a)) or asked[-1])
    with torch.inference_mode():
        lm(input_ids=ids, position_ids=torch.arange(70, device="cuda").repeat(2, 1))
    assert asked == [True]


@pytest.mark.parametrize("B,Hq,Hkv,S,D", [(1, 32, 8, 1024, 64), (1, 32, 8, 1025, 64), (1, 32, 8, 2048, 128),
                                          (3, 12, 3, 1791, 64), (100, 3, 3, 70, 64), (2, 8, 1, 2060, 128),
                                          (3, 32, 8, 1001, 128), (11, 32, 8, 255, 128)])
def test_prompts_of_one_round_of_workgroups(B, Hq, Hkv, S, D):
    """256 workgroups, 264, 512, 504 of 9 heads, more heads than CUs, 258 of 2 heads, 768 of waves with
    priority and 704 of short rows without: every row of the prompts, against 32-bit products: the result's rounding (2^-9) and as much for P's 16 bits."""
    g = torch.Generator(device="cuda").manual_seed(S)
    q, k, v = (torch.randn(B, h, S, D, device="cuda", generator=g).bfloat16() for h in (Hq, Hkv, Hkv))
    out = torch.full_like(q, float("nan"))
    ops._C.flash_prefill(out, q, k, v, D ** -0.5, 0, None)
    seen = torch.ones(S, S, dtype=torch.bool, device="cuda").tril()
    for b in range(B):
        kk, vv = (t[b].float().repeat_interleave(Hq // Hkv, 0) for t in (k, v))
        p = (q[b].float() @ kk.transpose(1, 2).contiguous() * D ** -0.5).masked_fill(~seen, float("-inf"))
        want = torch.softmax(p, -1) @ vv
        err = (out[b].float() - want).norm(dim=-1) / want.norm(dim=-1)
        assert out[b].isfinite().all() and err.max() < 2.0 ** -7 and err.square().mean().sqrt() < 2.0 ** -8


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,G,Dk,Dv,off,values", [
    (1, 1, 8, 8, 0, True), (700, 4, 128, 128, 0, True), (33, 2, 64, 64, 3, True), (70, 3, 12, 20, 0, True),
    (5, 1, 576, 0, 8, False), (9, 1, 7, 0, 0, False), (300, 2, 16, 32, 16, True)])
def test_paged_rows_are_written(N, G, Dk, Dv, off, values, dtype):
    """Whole 16 bytes and elements, rows that start off 16 bytes, no values, tokens without a slot:
    bit for bit."""
    from neuronx_distributed_inference_amd.ops import seqmix

    g = torch.Generator(device="cuda").manual_seed(N)
    rows = torch.randn(N, off + G * (Dk + Dv) + 8, device="cuda", generator=g).to(dtype)
    k, v = rows[:, off:off + G * Dk], rows[:, off + G * Dk:off + G * (Dk + Dv)]
    kc, vc = (torch.randn(N // 16 + 2, 16, G, d, device="cuda", generator=g).to(dtype) for d in (Dk, Dv))
    slots = torch.randperm(kc.shape[0] * 16, device="cuda", generator=g)[:N].to(torch.int32)
    if N > 2:                                        # (a token alone has one)
        slots[N // 2::3] = -1
        slots[N // 3:N // 3 + 1] = kc.shape[0] * 16
    want = kc.clone(), vc.clone()
    there = (slots >= 0) & (slots < kc.shape[0] * 16)
    assert there.any()
    for c, x, d in zip(want, (k, v), (Dk, Dv)):
        if d:
            c.view(-1, G * d)[slots[there].long()] = x[there]
    seqmix.paged_kv_write(kc, vc if values else None, k, v if values else None, slots)
    assert torch.equal(kc, want[0]) and torch.equal(vc, want[1])


@pytest.mark.parametrize("how", ["property", "instance", "deleted"])
@pytest.mark.parametrize("rows", [0, 200])
def test_feed_forwards_of_their_own_are_called(how, rows, monkeypatch):
    """A layer whose feed-forward a program has replaced, in a prompt and in a step: as the chain of
    modules, which calls it."""
    from neuronx_distributed_inference_amd.models import model_base
    from neuronx_distributed_inference_amd.modules import fused_layer

    monkeypatch.setattr(fused_layer, "PROMPT_ROWS", rows)
    lm = _small_llama("float16")
    layer, calls = lm.model.layers[1], []
    inner = layer.mlp

    def own(x, *a, **kw):
        calls.append(1)
        return -2.0 * inner(x, *a, **kw)

    if how == "property":
        layer.__class__ = type("Own", (type(layer),), {"mlp": property(lambda self: own)})
    elif how == "instance":
        layer.__dict__["mlp"] = own
    else:
        del layer.mlp
        layer.mlp = own
    ids = torch.randint(0, 512, (2, 70), device="cuda")
    step = torch.randint(0, 512, (2, 1), device="cuda")

    def run():
        lm.reset()
        with torch.inference_mode():
            return (lm(input_ids=ids).logits.float(),
                    lm(input_ids=step, position_ids=torch.full((2, 1), 70, device="cuda")).logits.float())

    got = run()
    assert len(calls) == 2
    monkeypatch.setattr(model_base, "fusable", lambda *a: False)
    # (16-bit activations of two layers, rounded at other places)
    assert all((a - b).norm() <= 0.004 * b.norm() for a, b in zip(got, run()))


def test_gate_of_windowed_portions_is_the_plain_sigmoid():
    """Rows that see one key, with values of 1: the result is the gate's sigmoid, 1 / (1 + exp(-x)) of 32
    bits rounded once, for every gate of 16 bits in which it is neither 0 nor 1, and for the others."""
    from neuronx_distributed_inference_amd.ops import seqmix

    S, H, D = 128, 4, 128
    gate = torch.arange(2 ** 16).to(torch.int16).view(torch.bfloat16).view(1, S, H * D).cuda()
    kc = torch.randn(S // 16, 16, 1, D, device="cuda").bfloat16()
    step = seqmix.StepLayout(torch.arange(S, device="cuda").view(1, S), torch.zeros(1, dtype=torch.long, device="cuda"))
    got = seqmix.paged_attention(torch.randn(1, S, H * D, device="cuda").bfloat16(), kc, torch.ones_like(kc), step,
                                 torch.arange(S // 16, device="cuda").view(1, -1).int(), D ** -0.5, H, window=1,
                                 gate=gate)
    want = (1 / (1 + torch.exp(-gate.float()))).bfloat16()
    same = (got == want) | (got.isnan() & want.isnan())
    assert same.all(), (int((~same).sum()), gate[~same][:8], got[~same][:8], want[~same][:8])


@pytest.mark.parametrize("Hq,Hkv,D,lens", [
    (32, 8, 128, (1001, 1001, 1001)), (32, 8, 128, (1001, 33, 700)), (8, 2, 128, (1100, 1100)),
    (32, 8, 64, (256, 256, 1, 255)), (32, 8, 128, (400,) + (40,) * 9), (16, 4, 128, (901, 900, 3, 128, 129))])
@pytest.mark.parametrize("window", [0, 300, -256])
def test_packed_prompts_of_any_lengths(Hq, Hkv, D, lens, window):
    """Prompts without padding, of one length (where the order and the priority of workgroups are those of
    padded ones) and of several: each as it is by itself, but for the order of 32-bit sums of one
    tile, which is the same: bit for bit."""
    g = torch.Generator(device="cuda").manual_seed(len(lens))
    rows, B, S = sum(lens), len(lens), max(lens)
    q = torch.randn(rows, Hq, 1, D, device="cuda", generator=g).bfloat16()
    kc, vc = (torch.randn(B + 2, Hkv, S + 5, D, device="cuda", generator=g).bfloat16() for _ in range(2))
    sid = torch.randperm(B + 2, device="cuda", generator=g)[:B].to(torch.int32)
    starts = torch.tensor((0,) + lens, device="cuda").cumsum(0).to(torch.int32)
    out = torch.full_like(q, float("nan"))
    ops._C.flash_prefill_packed(out, q, kc, vc, sid, starts, S, D ** -0.5, window)
    at = 0
    for b, n in enumerate(lens):
        one = q[at:at + n, :, 0].transpose(0, 1).unsqueeze(0).contiguous()
        want = torch.empty_like(one)
        ops._C.flash_prefill_cached(want, one, kc, vc, sid[b:b + 1], D ** -0.5, window, None)
        assert torch.equal(out[at:at + n, :, 0].transpose(0, 1), want[0]), (b, n)
        at += n
