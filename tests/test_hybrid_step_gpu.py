"""Single tokens of the hybrid decoder in fewer launches, against its modules one by one."""

import copy
import sys

import pytest
import torch

from neuronx_distributed_inference_amd import ops
from neuronx_distributed_inference_amd.config import EngineConfig
from neuronx_distributed_inference_amd.models.nabelix.modeling_nabelix import (
    NabelixForCausalLM,
    NabelixInferenceConfig,
)
from neuronx_distributed_inference_amd.ops import seqmix

sys.path.insert(0, __file__.rsplit("/", 1)[0])
from test_nabelix import layer_cfg, left_cfg, make_weights, model_cfg, right_cfg  # noqa: E402

pytestmark = pytest.mark.gpu
F64 = torch.float64
BF = torch.bfloat16


def _model(slots, taps=4, conv=4, width=512, dim=128, loop=None, ff=768, layers=2, heads=4):
    layer = layer_cfg(left_cfg(heads, 2, dim, dim, size=24, keep=3, scale=dim ** -0.5),
                      right_cfg(heads, heads, dim, dim, conv=conv, decay_rank=64, gate_rank=64), ff=ff)
    cfg = model_cfg([layer] * layers, width=width, vocab=96, taps=taps,
                    loop=loop or {"start": 0, "stop": 0, "times": 1})
    # a feed-forward every other layer where there is none in one
    if ff and layers > 1:
        cfg["layers"] = [copy.deepcopy(layer) for _ in range(layers)]
        cfg["layers"][0]["mlp"] = None
    ec = EngineConfig(batch_size=slots, max_batch_size=slots, kv_cache_batch_size=slots,
                      seq_len=64, max_length=64, torch_dtype="bfloat16", tp_degree=1,
                      is_block_kv_layout=True, pa_block_size=16, pa_num_blocks=4 * slots,
                      enable_hip_graphs=False)
    config = NabelixInferenceConfig(neuron_config=ec, **copy.deepcopy(cfg))
    lm = NabelixForCausalLM(config)
    sd = NabelixForCausalLM.convert_hf_to_native_state_dict(make_weights(cfg), config)
    lm.model.load_state_dict(sd, strict=False)
    return lm.cuda().eval()


def _everything(lm):
    mgr = lm.model.kv_mgr
    out = {n: t for n, t in mgr.named_buffers()}
    runs = len(lm.model.layer_runs())
    for i in range(runs):
        out.update({"k%d" % i: mgr.get_cache(i)[0].data, "v%d" % i: mgr.get_cache(i)[1].data})
        for n in ("canon", "conv", "mem"):
            out["%s%d" % (n, i)] = mgr.state.get("run%d.%s" % (i, n))
    return {n: t.detach() for n, t in out.items()}


def _steps(lm, B, pads=()):
    """Three steps from a state and cache of noise; logits, all that the steps leave behind, what was
    there before, and the rows' first positions and sequences."""
    g = torch.Generator(device="cuda").manual_seed(3)
    with torch.inference_mode():
        for n, t in _everything(lm).items():
            if t.is_floating_point():
                t.copy_(torch.empty(t.shape, device="cuda").normal_(0, 0.3, generator=g))
        pos = torch.randint(2, 60, (B, 1), generator=g, device="cuda")
        pos[0] = 0                                             # a sequence's first token
        seq = torch.arange(B, device="cuda")
        for b in pads:
            seq[b] = pos[b] = -1
        logits, noise = [], {n: t.clone() for n, t in _everything(lm).items()}
        for i in range(3):
            ids = torch.randint(0, 96, (B, 1), generator=g, device="cuda")
            logits.append(lm.model(ids, None, torch.where(pos < 0, pos, pos + i), seq)[1])
        after = {n: t.clone() for n, t in _everything(lm).items()}
        return torch.stack(logits), after, noise, pos.view(-1), seq


@pytest.mark.parametrize("B,kw", [
    (1, {}), (2, dict(taps=2, conv=3)), (16, dict(taps=3, conv=2, dim=64)), (17, dict(width=2112)),
    (33, dict(loop={"start": 0, "stop": 2, "times": 2})), (65, dict(width=4160, ff=256)),
    (130, dict(ff=0))])
def test_steps_in_fewer_launches(B, kw):
    lm = _model(B, **kw)
    pads = (1, B - 1) if B > 4 else ()
    # the modules' sums of two products and their activations are rounded to 16 bits on the way
    took = []
    inner = lm.model._steps_once
    lm.model._steps_once = lambda p: took.append(inner(p)) or took[-1]
    got, after, noise, pos, seq = _steps(lm, B, pads)
    assert took == [True] * 3
    lm.model._steps_once = lambda p: False
    want, before = _steps(lm, B, pads)[:2]
    live = [b for b in range(B) if b not in pads]
    assert (got[:, live] - want[:, live]).norm() <= 0.03 * want[:, live].norm()
    # cache rows and state slots of the live rows, one by one; all else stays as it was
    slots = seq[live].cpu()
    written = (slots.view(-1, 1) * 64 + pos[live].cpu().view(-1, 1) + torch.arange(3)).view(-1)
    runs = len(lm.model.layer_runs())
    rows = lambda t, n: t.flatten(0, 1) if n[0] in "kv" else t  # noqa: E731
    mine = {"%s%d" % (n, i) for i in range(runs) for n in ("k", "v", "canon", "conv", "mem")}
    for n in mine:
        own = written if n[0] in "kv" else slots
        x, y, z = (rows(d[n], n) for d in (after, before, noise))
        others = torch.ones(x.shape[0], dtype=torch.bool)
        others[own] = False
        assert others.sum() == x.shape[0] - len(own)
        assert torch.equal(x[others], z[others]), n
        x, y, z = (t[own].float().flatten(1) for t in (x, y, z))
        worst = ((x - y).norm(dim=1) / y.norm(dim=1)).max().item()
        # (two roundings of 2^-9 a product in each of up to four runs: 0.0064 at most)
        assert worst <= 0.02 and ((x != z).any(dim=1)).all(), (n, worst)
    # (the buffers are the same once more, under the modules' names)
    tensors = _everything(lm)
    places = {tensors[n].data_ptr() for n in mine}
    for n in set(tensors) - mine:
        assert tensors[n].data_ptr() in places or torch.equal(after[n], noise[n]), n


def test_hooks_keep_the_modules():
    lm = _model(2)
    for module in (lm.model.layers[0], lm.model.layers[1].mlp, lm.model.layers[0].mixer.right.conv,
                   lm.model.layers[1].mixer.in_proj, lm.model.norm):
        seen = []
        hook = module.register_forward_hook(lambda *a: seen.append(1))
        _steps(lm, 2)
        assert seen and not lm.model.kv_mgr.step.fused
        hook.remove()
    _steps(lm, 2)
    assert lm.model.kv_mgr.step.fused


@pytest.mark.parametrize("of", [lambda m: m.layers[1].norm1, lambda m: m.layers[0].canon,
                                lambda m: m.layers[1].norm2, lambda m: m.norm])
def test_small_weights_off_16_bytes_keep_the_modules(of):
    lm = _model(2)
    lm.model._steps_once = lambda p: False
    want = _steps(lm, 2)
    del lm.model._steps_once
    module = of(lm.model)
    flat = torch.empty(module.weight.numel() + 1, device="cuda")
    weight = flat[1:].view(module.weight.shape)
    weight.copy_(module.weight.detach())
    module.weight = torch.nn.Parameter(weight, requires_grad=False)
    assert module.weight.data_ptr() % 16
    got = _steps(lm, 2)
    assert not lm.model.kv_mgr.step.fused
    # the same modules: a norm without pieces adds up in another order, which now and then moves a
    # rounding to 16 bits
    for a, b in ((got[0], want[0]), *((got[1][n], t) for n, t in want[1].items())):
        assert (a.double() - b.double()).norm() <= 2.0 ** -8 * b.double().norm()


@pytest.mark.parametrize("C", [8, 2048, 2056, 4104, 8192])
@pytest.mark.parametrize("taps", [0, 2, 3, 4])
@pytest.mark.parametrize("na,nb", [(0, 0), (1, 0), (4, 5), (16, 3)])
def test_stream_step(C, taps, na, nb):
    B = 5
    g = torch.Generator(device="cuda").manual_seed(C + taps)
    rnd = lambda *s: torch.empty(*s, device="cuda").normal_(0, 1, generator=g)  # noqa: E731
    x, w = rnd(B, 1, C), rnd(C)
    pend = [(rnd(n, B, C), sc) for n, sc in ((na, 0.7), (nb, -1.3)) if n]
    step = seqmix.StepLayout(torch.tensor([[0], [1], [2], [-1], [9]], device="cuda"),
                             torch.tensor([2, 0, 5, 3, -1], device="cuda"))
    cw, tail = (rnd(C, taps), rnd(6, taps - 1, C)) if taps else (None, None)
    xw = x.to(F64) + sum((sc * p.to(F64).sum(0).view(B, 1, C) for p, sc in pend), torch.zeros((), device="cuda"))
    hn = torch.nn.functional.layer_norm(xw, (C,), w.to(F64), None, 1e-5)
    want = hn
    if taps:
        want, want_tail = hn.clone(), tail.clone()
        for b, (p, s) in enumerate([(0, 2), (1, 0), (2, 5), (-1, 3), (9, -1)]):
            if p < 0 or s < 0:
                want[b] = 0
                continue
            t = tail[s].to(F64)
            t[:max(0, taps - 1 - p)] = 0
            cols = torch.cat([t, hn[b]])
            want[b, 0] += (cols * cw.to(F64).t()).sum(0)
            want_tail[s] = cols[1:].float()
    got = seqmix.stream_step(x, pend, w, 1e-5, step, cw, tail)
    assert got.dtype == BF and got.shape == x.shape
    # 2^-8: a rounding to bf16; sums of up to 20 values of 32 bits, a norm and 5 products
    size = 4 * (xw.abs().amax() + 30)
    assert (x.to(F64) - xw).abs().amax() <= 2.0 ** -22 * size
    assert ((got.to(F64) - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -19 * size).all()
    if taps:
        assert (tail.to(F64) - want_tail).abs().amax() <= 2.0 ** -19 * size


@pytest.mark.parametrize("B,H,D,Dv,taps,per_head", [(1, 1, 128, 128, 4, False), (3, 4, 64, 72, 2, False),
                                                    (7, 2, 128, 16, 3, True), (5, 3, 64, 128, 4, True)])
def test_delta_step_with_its_convolution(B, H, D, Dv, taps, per_head):
    g = torch.Generator(device="cuda").manual_seed(B)
    rnd = lambda *s: torch.empty(*s, device="cuda").normal_(0, 1, generator=g)  # noqa: E731
    C = 2 * H * D + H * Dv
    wide = rnd(B, C + 32).to(BF)
    qkv, beta, a, gate = wide[:, 8:8 + C], rnd(B, H).to(BF), rnd(B, H if per_head else H * D).to(BF), \
        rnd(B, H * Dv).to(BF)
    cw, tail, state = rnd(C, taps), rnd(B + 2, taps - 1, C), 0.1 * rnd(B + 2, H, Dv, D)
    bias, a_log, nw = rnd(a.shape[1]), rnd(H), rnd(Dv)
    pos = torch.arange(B, device="cuda").view(B, 1) - int(B > 3)
    step = seqmix.StepLayout(pos, torch.arange(B, device="cuda").flip(0) + 1)
    t2, s2 = tail.clone(), state.clone()
    got = seqmix.gated_delta_conv(qkv, cw, tail, beta, a, bias, a_log, gate, nw, 1e-5, state, step, D, Dv)
    c = seqmix.short_conv_step(qkv.unsqueeze(1), cw, t2, step, "silu", False, torch.float32)
    want = seqmix.gated_delta_rule(c, beta.unsqueeze(1), a.unsqueeze(1), bias, a_log, gate.unsqueeze(1), nw,
                                   1e-5, s2, step, H, D, Dv, out_dtype=BF)
    # the same sums in the same order
    assert torch.equal(got, want[:, 0]) and torch.equal(tail, t2) and torch.equal(state, s2)


@pytest.mark.parametrize("B,H,G,D,page,bad,window", [
    (1, 2, 2, 128, 16, False, 33), (9, 8, 2, 64, 64, False, 33), (5, 40, 1, 128, 7, False, 33),
    (4, 4, 4, 128, 32, True, 33), (33, 16, 4, 128, 64, True, 700), (25, 8, 4, 64, 80, True, 510),
    # several workgroups a KV head, of which one writes the row that all of them see
    (4, 34, 2, 64, 16, True, 33), (5, 40, 1, 128, 7, True, 33), (34, 40, 1, 64, 80, True, 600)])
@pytest.mark.parametrize("writes", [True, False])
def test_window_attention_writes_its_rows(B, H, G, D, page, bad, window, writes):
    """Against the rows written by a launch of their own. A row without a place in the cache, or
    whose page is missing, counts with its own key and value all the same."""
    g = torch.Generator(device="cuda").manual_seed(D)
    rnd = lambda *s: torch.empty(*s, device="cuda").normal_(0, 1, generator=g).to(BF)  # noqa: E731
    pages = 8 * B
    kc, vc = rnd(pages, page, G, D), rnd(pages, page, G, D)
    q, k, v, gate = rnd(B, 1, H * D), rnd(B, G * D), rnd(B, G * D), rnd(B, 1, H * D)
    pos = torch.randint(0, 8 * page, (B, 1), generator=g, device="cuda")
    pos[0] = 0
    if B > 2:
        pos[2] = 3 * page                              # the first of its page
    if bad:
        v[0, 3] = float("inf")
        v[1, 5] = float("nan")
        v[2, 1] = float("-inf")
    seq = torch.arange(B, device="cuda")
    if B > 6:
        seq[3] = pos[3] = -1
    step = seqmix.StepLayout(pos, seq)
    table = torch.randperm(pages, generator=g, device="cuda").view(B, 8).int()
    slots = torch.where(pos < 0, -1, table.gather(1, pos.clamp(min=0) // page) * page + pos % page).view(-1)
    r1, r2 = torch.rand(H, device="cuda"), torch.rand(H, device="cuda")
    call = lambda kc, vc, table, **kw: seqmix.window_bias_attention(  # noqa: E731
        q, kc, vc, step, table, r1, r2, D ** -0.5, window, 2, H, gate=gate, **kw)
    k1, v1 = kc.clone(), vc.clone()
    assert seqmix.new_rows_taken(q, k, v, gate, kc, vc)
    if writes:
        got, after = call(k1, v1, table, new_rows=(k, v, slots)), (k1, v1)
    else:
        gone = table.clone()
        if B > 2:
            gone[2, 3] = -1
        before = k1.clone(), v1.clone()
        got, after = call(k1, v1, gone, new_rows=(k, v, torch.full_like(slots, -1))), None
        assert all(torch.equal(x.view(torch.int16), y.view(torch.int16)) for x, y in zip((k1, v1), before))
    seqmix.paged_kv_write(kc, vc, k, v, slots, step)
    want = call(kc, vc, table)
    live = seq >= 0
    for x, y in ((got[live], want[live]), *zip(after or (), (kc, vc))):
        assert torch.equal(x.view(torch.int16), y.view(torch.int16))


@pytest.mark.parametrize("B,H,G,D,page,pages,window", [
    (96, 4, 1, 128, 16, 32, 512), (24, 64, 4, 64, 64, 9, 10 ** 6), (13, 160, 8, 128, 100, 20, 700)])
def test_many_rows_through_lds_as_few_without(B, H, G, D, page, pages, window):
    """Many long rows at once take another way to the registers than two at a time do."""
    g = torch.Generator(device="cuda").manual_seed(D)
    rnd = lambda *s: torch.empty(*s, device="cuda").normal_(0, 1, generator=g).to(BF)  # noqa: E731
    kc, vc = rnd(B * pages, page, G, D), rnd(B * pages, page, G, D)
    vc[5, 3] = float("inf")
    q, r1, r2 = rnd(B, 1, H * D), torch.rand(H, device="cuda"), torch.rand(H, device="cuda")
    pos = torch.randint(0, pages * page, (B, 1), generator=g, device="cuda")
    pos[0] = pages * page - 1
    table = torch.randperm(B * pages, generator=g, device="cuda").view(B, pages).int()
    table[1, 1] = -1

    def call(rows):
        step = seqmix.StepLayout(pos[rows].contiguous(), torch.arange(pos[rows].shape[0], device="cuda"))
        return seqmix.window_bias_attention(q[rows], kc, vc, step, table[rows].contiguous(), r1, r2,
                                            D ** -0.5, window, 3, H)

    got = call(slice(0, B))
    want = torch.cat([call(slice(i, i + 1)) for i in range(B)])
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("M,N,K", [(1, 64, 128), (17, 4096, 128), (48, 11408, 2048), (64, 1000, 256),
                                   (100, 16384, 512), (129, 2048, 256)])
def test_products_of_whole_results(M, N, K):
    """Rows that lie apart, gelu, and two products in one launch."""
    g = torch.Generator(device="cuda").manual_seed(N)
    rnd = lambda *s: torch.empty(*s, device="cuda").normal_(0, 1, generator=g).to(BF)  # noqa: E731
    x, w, x2, w2 = rnd(M, K + 24)[:, 16:16 + K], rnd(N, K), rnd(M, K), rnd(N, K)
    d = lambda t: t.to(F64)  # noqa: E731
    e1, e2 = d(x) @ d(w).t(), d(x2) @ d(w2).t()
    s1, s2 = (K * 2.0 ** -24 * (d(a).abs() @ d(b).abs().t()) for a, b in ((x, w), (x2, w2)))
    assert ops._C.tile_gemm_splits(M, N, K, 0, True) >= 1
    y = ops._C.tile_gemm(x, w)
    assert ((d(y) - e1).abs() <= s1 + 2.0 ** -8 * e1.abs() + 1e-30).all()
    if K >= 256:
        parts = d(ops._C.tile_gemm_pair(x, w, x2, w2))
        n = parts.shape[0] // 2
        assert ((parts[:n].sum(0) - e1).abs() <= s1 + 1e-30).all()
        assert ((parts[n:].sum(0) - e2).abs() <= s2 + 1e-30).all()
        gate, up = e1[:, : N // 2], e1[:, N // 2:]
        want = torch.nn.functional.gelu(gate, approximate="tanh") * up
        y = ops._C.tile_gemm(x, w, glu=2)
        # the slope of gelu stays below 1.13; tanh of 32 bits beside one: 2^-22 of the gate
        limit = 1.13 * s1[:, : N // 2] * up.abs() + gate.abs() * s1[:, N // 2:] \
            + 2.0 ** -8 * want.abs() + 2.0 ** -21 * (gate * up).abs() + 1e-6
        assert ((d(y) - want).abs() <= limit).all()


@pytest.mark.parametrize("M,N,K", [(65, 32760, 320), (100, 22920, 2048), (128, 16376, 4096),
                                   (127, 23044, 128)])
def test_whole_products_of_full_chips(M, N, K):
    """Tiles of 128 columns where they, or two parts of them, take 180 CUs and more, and just less."""
    test_products_of_whole_results(M, N // 8 * 8, K)



@pytest.mark.parametrize("out", [BF, torch.float32])
@pytest.mark.parametrize("rows,C,summand", [(1, 8, None), (3, 2040, BF), (5, 2048, torch.float32),
                                            (2, 2056, BF), (7, 4104, BF), (2, 8192, torch.float32),
                                            (2, 8200, BF), (3, 37, BF)])
def test_sum_and_norm(rows, C, summand, out):
    """LayerNorm of a stream, alone and after its residual step: every count of pieces a thread
    holds, widths and addresses that go without pieces, infinities and NaN as they were."""
    g = torch.Generator(device="cuda").manual_seed(C)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    for offset in (0, 1):
        x = rnd(rows * C + 1)[offset:offset + rows * C].view(rows, C)
        w, bias = rnd(C), rnd(C)
        a, b = (None, None) if summand is None else (rnd(rows, C).to(summand) for _ in range(2))
        for second in (False, True) if summand else (False,):
            want = x.to(F64)
            got_x = x.clone() if not offset else torch.cat([x.new_zeros(1), x.flatten()])[1:].view(rows, C)
            if summand:
                want = want + 1.25 * a.to(F64) + (0.5 * b.to(F64) if second else 0)
                got = seqmix.residual_layer_norm(got_x, a, 1.25, b if second else None, 0.5, w, 1e-5,
                                                 out, bias)
                alone = seqmix.residual_add(x.clone(), a, 1.25, b if second else None, 0.5)
                assert (got_x - want).abs().max() <= 4 * 2.0 ** -24 * want.abs().max() + 1e-7
                assert (alone - want).abs().max() <= 4 * 2.0 ** -24 * want.abs().max() + 1e-7
            else:
                got = seqmix.layer_norm(got_x, w, 1e-5, out, bias)
                assert torch.equal(got_x, x)
            want = torch.nn.functional.layer_norm(want, (C,), w.to(F64), bias.to(F64), 1e-5)
            # rounding of the result, and 32-bit statistics of at most C / 256 terms in a chain
            tol = (2.0 ** -8 if out is BF else 0) + 2.0 ** -18
            assert ((got.to(F64) - want).abs() <= tol * (want.abs() + 1)).all()
    x = rnd(2, 64)
    x[0, 3], x[1, 5] = float("nan"), float("inf")
    assert seqmix.layer_norm(x, rnd(64), 1e-5, out).isnan().all()


@pytest.mark.parametrize("dtype", [BF, torch.float32])
@pytest.mark.parametrize("Dv", [64, 96, 128, 256])
def test_gated_norm_in_pieces(Dv, dtype):
    """Heads in 16-byte pieces against the same from a weight that lies across them; padded rows
    are zeros."""
    B, S, H, D = 3, 5, 3, 64
    g = torch.Generator(device="cuda").manual_seed(Dv)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    qkv = rnd(B, S, H * (2 * D + Dv))
    beta, a, gate = (rnd(B, S, n).to(dtype) for n in (H, H, H * Dv))
    weight = rnd(Dv + 1)
    weight[:Dv] = weight[1:].clone()
    pos = torch.arange(S, device="cuda").repeat(B, 1)
    pos[1, 3:] = -1
    step = seqmix.StepLayout(pos, torch.tensor([0, 1, -1], device="cuda"))
    for act in ("sigmoid", "silu"):
        res = []
        for nw in (weight[:Dv].clone(), torch.cat([weight[:1], weight[:Dv]])[1:]):
            state = torch.zeros(2, H, Dv, D, device="cuda")
            res.append(seqmix.gated_delta_rule(qkv, beta, a, torch.zeros(H, device="cuda"),
                                               torch.zeros(H, device="cuda"), gate, nw, 1e-5, state,
                                               step, H, D, Dv, dtype, act))
        assert res[1].abs().max() > 0.1 and not res[0][2].any() and not res[0][1, 3:].any()
        # the same value but for the order of a head's squares: one rounding of the result
        tol = 2.0 ** -8 if dtype is BF else 2.0 ** -20
        assert ((res[0] - res[1]).abs() <= tol * res[1].abs()).all()


def test_delta_rule_where_memory_is_short(monkeypatch):
    """Operands of fewer chunks at a time where there is no room for all, and in a capture: the same
    to the bit."""
    B, S, H, D = 16, 400, 16, 128                      # 220 MB of operands
    g = torch.Generator(device="cuda").manual_seed(0)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    qkv, beta, a, gate = rnd(B, S, 3 * H * D), rnd(B, S, H), rnd(B, S, H), rnd(B, S, H * D)
    bias, rate, w, first = rnd(H), rnd(H), rnd(D), rnd(B, H, D, D)
    step = seqmix.StepLayout(torch.arange(S, device="cuda").repeat(B, 1), torch.arange(B, device="cuda"))
    sizes, room = [], seqmix._delta_workspace
    monkeypatch.setattr(seqmix, "_delta_workspace", lambda *x: sizes.append(room(*x)) or sizes[-1])

    def run():
        state = first.clone()
        out = seqmix.gated_delta_rule(qkv, beta, a, bias, rate, gate, w, 1e-5, state, step, H, D, D)
        return out.cpu(), state.cpu(), sizes.pop().numel() * 4

    want = run()
    empty = torch.empty

    def short(*shape, **kw):
        if torch.Size(shape).numel() > 200 << 18:
            raise torch.cuda.OutOfMemoryError
        return empty(*shape, **kw)

    with monkeypatch.context() as m:
        m.setattr(torch, "empty", short)
        got = run()
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    captured = run()
    assert want[2] > 200 << 20 and got[2] == captured[2] <= 128 << 20
    for other in (got, captured):
        assert torch.equal(other[0], want[0]) and torch.equal(other[1], want[1])


@pytest.mark.parametrize("M,N,K,parts", [
    (16, 512, 256, 1), (16, 512, 512, 2), (1, 512, 1024, 4), (100, 1024, 1024, 4), (48, 1536, 1536, 4),
    (48, 1024, 2048, 4), (100, 2048, 2048, 4), (100, 2048, 4096, 5), (48, 4096, 2048, 2), (64, 16384, 512, 1)])
def test_parts_of_pairs_of_products(M, N, K, parts):
    """Parts that two products are taken in together, at both ends of what limits them, and their sums."""
    g = torch.Generator(device="cuda").manual_seed(K)
    x, w, x2, w2 = (torch.empty(*s, device="cuda").normal_(0, 1, generator=g).to(BF)
                    for s in ((M, K), (N, K)) * 2)
    got = ops._C.tile_gemm_pair(x, w, x2, w2)
    assert got.shape == (2 * parts, M, N)
    for y, a, b in ((got[:parts], x, w), (got[parts:], x2, w2)):
        limit = K * 2.0 ** -24 * (a.to(F64).abs() @ b.to(F64).abs().t())
        assert ((y.to(F64).sum(0) - a.to(F64) @ b.to(F64).t()).abs() <= limit + 1e-30).all()
