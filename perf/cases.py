"""The work that programs built on this package have it do: prompts encoded and
tokens decoded by whole models, through the same calls that a generation loop or
a serving engine makes.

Models are a few layers deep (the layer sizes are the real ones; a layer is the
unit that repeats) with random weights, over a vocabulary of 32000 (128256 in
one case, where the head weighs as much as it does in a model of full depth). ``run`` is one model step:

decode   one new token for each sequence of a batch, through the captured graph
prefill  whole prompts from an empty cache
extend   the next portion of prompts whose start is in the paged cache already

Outputs are the logits (and on-device tokens), and for prompts the written cache
as well; a decode step's own cache row is read by its own attention, so a wrong
one shows in the logits. Recurrent state that a step advances is returned whole.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

F64 = torch.float64
EPS = 1e-5
THETA = 500000.0

# layer sizes of bench.py's models
SIZES = {
    "1b": dict(width=2048, heads=32, kv_heads=8, dim=64, ff=8192),
    "8b": dict(width=4096, heads=32, kv_heads=8, dim=128, ff=14336),
    "70b": dict(width=8192, heads=64, kv_heads=8, dim=128, ff=28672),
    "mixtral": dict(width=4096, heads=32, kv_heads=8, dim=128, ff=14336, experts=8, top=2),
    "qwen3moe": dict(width=2048, heads=32, kv_heads=4, dim=128, ff=768, experts=128, top=8),
    "nabelix": dict(width=2048, heads=16, kv_heads=4, dim=128, ff=8192, window=1024, keep=4,
                    taps=4, rank=64),
}


def listed():
    return [
        # one user chatting with a small model: latency and launches
        _case("chat_1b_b1", "decode", "1b", layers=4, batch=1, ctx=700),
        # a loaded server in the middle of long conversations
        _case("serve_8b_b64", "decode", "8b", layers=8, batch=64, ctx=2048, vocab=128256),
        # throughput decoding of short conversations, the default bench.py batch
        _case("batch_8b_b256", "decode", "8b", layers=4, batch=256, ctx=168),
        # long documents on the largest dense model, 8-bit cache
        _case("long_70b_b13_kv8", "decode", "70b", layers=2, batch=13, ctx=8000, kv8=True),
        # time to first token of a one-line question, half precision
        _case("ask_1b_93", "prefill", "1b", layers=4, batch=1, tokens=93, dtype="float16"),
        # one long prompt
        _case("prompt_8b_8192", "prefill", "8b", layers=4, batch=1, tokens=8192),
        # a batch of unequal prompts, right-padded
        _case("prompts_8b_ragged", "prefill", "8b", layers=4, batch=5, tokens=777, ragged=True),
        # chunked prefill: the next 512 tokens of a prompt in the paged cache
        _case("chunk_8b_512", "extend", "8b", layers=4, batch=1, tokens=512, ctx=3500),
        # few-expert mixture, 8-bit expert weights, decoding
        _case("moe_mixtral_b128_fp8", "decode", "mixtral", layers=2, batch=128, ctx=512,
              quant="fp8"),
        # fine-grained mixture, a prompt
        _case("moe_qwen3_prompt", "prefill", "qwen3moe", layers=2, batch=1, tokens=2048),
        # hybrid decoder (windowed attention beside a gated delta rule), a prompt and decoding
        _case("hybrid_prompt_4000", "prefill", "nabelix", layers=2, batch=1, tokens=4000),
        _case("hybrid_b48", "decode", "nabelix", layers=4, batch=48, ctx=700),
    ]


def _case(name, step, size, layers, batch, tokens=1, ctx=0, vocab=32000, dtype="bfloat16",
          kv8=False, ragged=False, quant="none"):
    c = dict(step=step, size=size, layers=layers, batch=batch, tokens=tokens, ctx=ctx,
             vocab=vocab, dtype=dtype, kv8=kv8, ragged=ragged, quant=quant)
    return dict(c, name=name) if name else c


def draw(rng):
    def spread(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))

    kind = rng.choice(["decode"] * 5 + ["prefill"] * 3 + ["extend"] * 2 +
                      ["mixtral", "qwen3moe", "nabelix", "nabelix_decode"])
    dtype = rng.choice(["bfloat16"] * 3 + ["float16"])
    if kind == "decode":
        size = rng.choice(["1b", "8b", "8b", "70b"])
        batch = spread(1, 256)
        ctx = spread(64, min(8192, 131072 // batch))
        return _case(None, "decode", size, layers=2 if size == "70b" else 4, batch=batch, ctx=ctx,
                     dtype=dtype, kv8=rng.random() < 0.2)
    if kind == "prefill":
        size = rng.choice(["1b", "8b"])
        batch = rng.choice([1, 1, 2, 3, 6])
        return _case(None, "prefill", size, layers=4, batch=batch,
                     tokens=spread(16, 6000 // batch), dtype=dtype,
                     ragged=batch > 1 and rng.random() < 0.7)
    if kind == "extend":
        return _case(None, "extend", rng.choice(["1b", "8b"]), layers=4,
                     batch=rng.choice([1, 1, 2]), tokens=spread(32, 512), ctx=spread(128, 4000),
                     dtype=dtype)
    if kind == "mixtral":
        return _case(None, "decode", "mixtral", layers=2, batch=spread(16, 256),
                     ctx=spread(64, 512), quant=rng.choice(["none", "fp8", "mx4"]))
    if kind == "qwen3moe":
        return _case(None, "prefill", "qwen3moe", layers=2, batch=1, tokens=spread(64, 4096))
    if kind == "nabelix":
        return _case(None, "prefill", "nabelix", layers=2, batch=1, tokens=spread(32, 4096))
    return _case(None, "decode", "nabelix", layers=4, batch=spread(1, 128), ctx=spread(64, 1500))


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------
BLOCK = 64     # rows of a page of the paged caches


def _max_len(case):
    return case["ctx"] + case["tokens"] + 31


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _weights(case, g):
    """Weights under plain names. The head is a permutation of the embedding, so that the next
    token stands out as it does for a trained model; a mixture's router reads directions that
    the embedding of a token carries for its experts."""
    s, dt, V = SIZES[case["size"]], getattr(torch, case["dtype"]), case["vocab"]
    d, ff = s["width"], s["ff"]

    def normal(*shape, std=0.02, dtype=dt):
        return torch.empty(*shape, dtype=dtype, device="cuda").normal_(0, std, generator=g)

    def uniform(lo, hi, *shape):
        return torch.empty(*shape, device="cuda").uniform_(lo, hi, generator=g)

    W = {}
    if case["size"] == "nabelix":
        H, G, D = s["heads"], s["kv_heads"], s["dim"]
        W["embed"] = normal(V, d)
        for i in range(case["layers"]):
            p = "l%d." % i
            W[p + "canon"] = normal(d, s["taps"], std=0.3, dtype=torch.float32)
            W[p + "in"] = normal(2 * H * D + 2 * G * D + 3 * H * D + H + 2 * s["rank"], d)
            W[p + "r1"] = uniform(0.1, 1.0, H)
            W[p + "r2"] = uniform(0.05, 0.5, H)
            W[p + "left_o"] = normal(d, H * D)
            W[p + "right_o"] = normal(d, H * D)
            W[p + "conv"] = normal(3 * H * D, s["taps"], std=0.5, dtype=torch.float32)
            W[p + "a2"] = normal(H * D, s["rank"])
            W[p + "g2"] = normal(H * D, s["rank"])
            # decays between about exp(-1.6) and exp(-0.001) a token
            W[p + "A_log"] = uniform(1.0, 16.0, H).log()
            dt0 = torch.exp(uniform(math.log(1e-3), math.log(1e-1), H * D))
            W[p + "dt_bias"] = dt0 + torch.log(-torch.expm1(-dt0))
            W[p + "gate_up"] = normal(2 * ff, d)
            W[p + "down"] = normal(d, ff)
        return W
    W["embed"] = normal(V, d, std=1.0)
    perm = torch.randperm(V, device="cuda", generator=g)
    if "experts" in s:
        E, top = s["experts"], s["top"]
        dirs = F.normalize(normal(E, d, std=1.0, dtype=torch.float32), dim=-1)
        own = torch.rand(V, E, device="cuda", generator=g).topk(top, dim=-1).indices
        mark = torch.zeros(V, E, device="cuda").scatter_(1, own, 12.0 if top == 2 else 10.0)
        W["embed"] += (mark @ dirs).to(dt)
    W["head"] = W["embed"][perm] * 0.01
    qkv = (s["heads"] + 2 * s["kv_heads"]) * s["dim"]
    for i in range(case["layers"]):
        p = "l%d." % i
        W[p + "qkv"] = normal(qkv, d)
        W[p + "o"] = normal(d, s["heads"] * s["dim"])
        if "experts" in s:
            W[p + "router"] = 0.5 * dirs
            for n, shape in (("gate", (E, ff, d)), ("up", (E, ff, d)), ("down", (E, d, ff))):
                W[p + n] = normal(*shape)
        else:
            W[p + "gate_up"] = normal(2 * ff, d)
            W[p + "down"] = normal(d, ff)
    return W


def _inputs(case, g):
    """Token ids, positions (-1: padding) and, per layer, what earlier tokens left behind."""
    s, B, T = SIZES[case["size"]], case["batch"], case["tokens"]
    dt = getattr(torch, case["dtype"])
    ids = torch.randint(0, case["vocab"], (B, T), device="cuda", generator=g)
    past = torch.zeros(B, dtype=torch.long, device="cuda")
    if case["ctx"]:
        past = torch.randint(case["ctx"] // 2, case["ctx"] + 1, (B,), device="cuda", generator=g)
        past[0] = case["ctx"]
    pos = past.view(B, 1) + torch.arange(T, device="cuda").view(1, T)
    if case["ragged"]:
        n = torch.randint(T // 3 + 1, T + 1, (B,), device="cuda", generator=g)
        n[0] = T
        pad = torch.arange(T, device="cuda").view(1, T) >= n.view(B, 1)
        pos, ids = pos.masked_fill(pad, -1), ids.masked_fill(pad, 0)
    kv, state = [], []
    if case["ctx"]:
        L = _max_len(case)
        for _ in range(case["layers"]):
            pair = [torch.empty(B, s["kv_heads"], L, s["dim"], dtype=dt, device="cuda")
                    .normal_(0, 1.0, generator=g) for _ in range(2)]
            kv.append([t.to(torch.float8_e4m3fn) for t in pair] if case["kv8"] else pair)
            if case["size"] == "nabelix":
                H, D, t = s["heads"], s["dim"], s["taps"] - 1
                state.append({
                    n: torch.empty(shape, device="cuda").normal_(0, std, generator=g)
                    for n, shape, std in (("canon", (B, t, s["width"]), 1.0),
                                          ("conv", (B, t, (2 * H + H) * D), 1.0),
                                          ("mem", (B, H, D, D), 0.05))})
    return ids, pos, past, kv, state


# ---------------------------------------------------------------------------
# the program
# ---------------------------------------------------------------------------
def _engine(case, paged):
    from neuronx_distributed_inference_amd.config import EngineConfig, OnDeviceSamplingConfig

    sampling = None
    if case["size"] != "nabelix":
        sampling = OnDeviceSamplingConfig(top_k=1)
    B = case["batch"]
    return EngineConfig(
        batch_size=B, max_batch_size=B, seq_len=_max_len(case), max_length=_max_len(case),
        max_context_length=_max_len(case), torch_dtype=case["dtype"], tp_degree=1,
        on_device_sampling_config=sampling, output_logits=True, fused_qkv=True,
        fused_gate_up=True, enable_batch_bucketing=False, kv_cache_quant=case["kv8"],
        is_block_kv_layout=paged, pa_block_size=BLOCK,
        pa_num_blocks=B * -(-_max_len(case) // BLOCK) if paged else None)


def _model(case, W, paged):
    s, L = SIZES[case["size"]], case["layers"]
    ec = _engine(case, paged)
    common = dict(neuron_config=ec, hidden_size=s["width"], intermediate_size=s["ff"],
                  num_hidden_layers=L, num_attention_heads=s["heads"],
                  num_key_value_heads=s["kv_heads"], head_dim=s["dim"], vocab_size=case["vocab"],
                  max_position_embeddings=2 * _max_len(case), rms_norm_eps=EPS, rope_theta=THETA,
                  hidden_act="silu", tie_word_embeddings=False)
    if case["size"] == "nabelix":
        from neuronx_distributed_inference_amd.models.nabelix.modeling_nabelix import (
            NabelixForCausalLM as Model, NabelixInferenceConfig)

        H, G, D = s["heads"], s["kv_heads"], s["dim"]
        layer = {"type": "parallel", "mlp": {"kind": "dense", "ff": s["ff"]}, "mixer": {
            "left": {"heads": H, "kv_heads": G, "dim": D, "vdim": D, "scale": D ** -0.5,
                     "mask": {"size": s["window"], "keep_first": s["keep"]}},
            "right": {"heads": H, "kv_heads": H, "dim": D, "vdim": D, "conv": s["taps"],
                      "decay_rank": s["rank"], "gate_rank": s["rank"]},
            "left_scale": 1.0, "right_scale": 1.0}}
        cfg = NabelixInferenceConfig(
            neuron_config=ec, architecture="Nabelix", width=s["width"], vocab=case["vocab"],
            layers=[layer] * L, canon={"taps": s["taps"]}, norm={"eps": EPS},
            loop={"start": 0, "stop": 0, "times": 1}, logit_softcap=30.0)
        sd = {"embed_tokens.weight": W["embed"], "lm_head.weight": W["embed"]}
        for i in range(L):
            a, b = "layers.%d." % i, "l%d." % i
            for x, y in (("canon.weight", "canon"), ("mixer.in_proj.weight", "in"),
                         ("mixer.left.r1", "r1"), ("mixer.left.r2", "r2"),
                         ("mixer.left_o.weight", "left_o"), ("mixer.right_o.weight", "right_o"),
                         ("mixer.right.conv.weight", "conv"), ("mixer.right.A_log", "A_log"),
                         ("mixer.right.dt_bias", "dt_bias"),
                         ("mlp.gate_up_proj.weight", "gate_up"),
                         ("mlp.down_proj.weight", "down")):
                sd[a + x] = W[b + y]
            sd[a + "mixer.right.ag2.weight"] = torch.block_diag(W[b + "a2"], W[b + "g2"])
    else:
        if case["size"] == "mixtral":
            from neuronx_distributed_inference_amd.models.mixtral.modeling_mixtral import (
                MixtralForCausalLM as Model, MixtralInferenceConfig as Config)
            common.update(num_local_experts=s["experts"], num_experts_per_tok=s["top"])
        elif case["size"] == "qwen3moe":
            from neuronx_distributed_inference_amd.models.qwen3_moe.modeling_qwen3_moe import (
                Qwen3MoeForCausalLM as Model, Qwen3MoeInferenceConfig as Config)
            common.update(num_experts=s["experts"], num_experts_per_tok=s["top"],
                          moe_intermediate_size=s["ff"])
        else:
            from neuronx_distributed_inference_amd.models.llama.modeling_llama import (
                LlamaForCausalLM as Model, LlamaInferenceConfig as Config)
        cfg = Config(**common)
        sd = {"embed_tokens.weight": W["embed"], "lm_head.weight": W["head"]}
        for i in range(L):
            a, b = "layers.%d." % i, "l%d." % i
            sd[a + "self_attn.qkv_proj.qkv.weight"] = W[b + "qkv"]
            sd[a + "self_attn.o_proj.o_proj.weight"] = W[b + "o"]
            if "experts" in s:
                sd[a + "mlp.router.weight"] = W[b + "router"]
                for n in ("gate", "up", "down"):
                    sd[a + "mlp.experts.w_" + n] = W[b + n]
            else:
                sd[a + "mlp.gate_up_proj.weight"] = W[b + "gate_up"]
                sd[a + "mlp.down_proj.weight"] = W[b + "down"]
    with torch.device("cuda"):
        lm = Model(cfg).eval()
    lm.model.load_state_dict(sd, strict=False, assign=True)
    if case["quant"] != "none":
        for m in lm.model.modules():
            if type(m).__name__ == "ExpertMLPs":
                done = m.quantize_fp8() if case["quant"] == "fp8" else m.quantize_mx4()
                assert done
    return lm


def prepare(case, seed):
    g = _generator(seed)
    W = _weights(case, g)
    ids, pos, past, kv, state = _inputs(case, g)
    hybrid = case["size"] == "nabelix"
    paged = hybrid or case["step"] == "extend"
    B = case["batch"]
    with torch.inference_mode():
        lm = _model(case, W, paged)
        lm.enable_submodels()
        if case["step"] == "decode":
            lm.warmup()
        lm.reset()
        st = {"lm": lm, "ids": ids, "pos": pos, "seq": torch.arange(B, device="cuda"),
              "step": case["step"], "mask": (pos >= 0).long() if case["ragged"] else None}
        per = -(-_max_len(case) // BLOCK)
        table = torch.arange(B * per, device="cuda").view(B, per)
        if case["step"] == "extend":
            # pages are handed out in any order
            table = torch.randperm(B * per, device="cuda", generator=g).view(B, per)
            st["table"] = table
        for i, pair in enumerate(kv):
            for cache, rows in zip(lm.model.kv_mgr.get_cache(i), pair):
                if paged:
                    rows = F.pad(rows, (0, 0, 0, per * BLOCK - rows.shape[2]))
                    rows = rows.transpose(1, 2).reshape(B * per, BLOCK, rows.shape[1], -1)
                    cache.data[table.view(-1)] = rows
                else:
                    cache.data.copy_(rows)
        for i, values in enumerate(state):
            mgr = lm.model.kv_mgr.state
            for n, v in values.items():
                mgr.get("run%d.%s" % (i, n)).copy_(v.transpose(2, 3) if n == "mem" else v)
        lm.kv_cache_populated = case["ctx"] > 0
    if hybrid:
        st["state"] = [lm.model.kv_mgr.state.get("run%d.mem" % i) for i in range(case["layers"])]
    if case["step"] == "prefill":
        st["kv"] = [t.data for i in range(case["layers"]) for t in lm.model.kv_mgr.get_cache(i)]
    return st


def run(st):
    lm = st["lm"]
    with torch.inference_mode():
        if st["step"] == "prefill":
            lm.kv_cache_populated = False         # a new conversation
            out = lm(input_ids=st["ids"], attention_mask=st["mask"], position_ids=st["pos"],
                     seq_ids=st["seq"])
        elif st["step"] == "extend":
            out = lm(input_ids=st["ids"], position_ids=st["pos"], seq_ids=st["seq"],
                     block_table=st["table"], phase="token_generation")
        else:
            out = lm(input_ids=st["ids"], position_ids=st["pos"], seq_ids=st["seq"])
    got = {"logits": out.logits}
    if out.tokens is not None:
        got["tokens"] = out.tokens
    for n in ("kv", "state"):
        if n in st:
            got[n] = st[n]
    return got


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    s, B, T, L, V = (SIZES[case["size"]], case["batch"], case["tokens"], case["layers"],
                     case["vocab"])
    d, H, G, D, ff = s["width"], s["heads"], s["kv_heads"], s["dim"], s["ff"]
    hybrid = case["size"] == "nabelix"
    # rows and contexts are drawn uniformly: half to all of the declared context, a third to
    # all of a ragged prompt (the first row at the most)
    n = B * T if not case["ragged"] else T + (B - 1) * T * 2 // 3
    past = (case["ctx"] + (B - 1) * case["ctx"] * 3 // 4) / B
    keys = past + (T + 1) / 2 * (1 if not case["ragged"] else 0.8)
    if hybrid:
        window = s["window"] + s["keep"]
        keys = min(keys, window) if T == 1 else min(keys, window * (1 - window / (2 * max(T, window))))
    w_bytes = {"none": 2.0, "fp8": 1.0, "mx4": 17 / 32}[case["quant"]]
    if hybrid:
        mix = d * (2 * H * D + 2 * G * D + 3 * H * D + H + 2 * s["rank"]) + 2 * H * D * s["rank"] \
            + 2 * d * H * D
    else:
        mix = d * (H + 2 * G) * D + d * H * D
    if "experts" in s:
        hit = s["experts"] * (1 - (1 - s["top"] / s["experts"]) ** n)
        ffn_bytes, ffn_use = hit * 3 * d * ff * w_bytes, s["top"] * 3 * d * ff
    else:
        ffn_bytes, ffn_use = 3 * d * ff * 2, 3 * d * ff
    out_rows = B * T if case["step"] == "extend" else B
    kv_b = 1 if case["kv8"] else 2
    seen = past if not hybrid or T > 1 else min(past, s["window"] + s["keep"])
    byts = L * (mix * 2 + ffn_bytes + (B * seen + n) * 2 * G * D * kv_b) \
        + V * d * 2 + n * d * 2 + out_rows * V * (4 if hybrid else 2)
    flops = 2 * n * L * (mix + ffn_use) + L * 4 * n * keys * H * D + 2 * out_rows * V * d
    if hybrid:
        byts += L * 2 * B * H * D * D * 4
        flops += L * n * H * 6 * D * D
    return {"bytes": byts, "flops": flops}


def tolerance(case):
    # 16-bit weights and activations through two to eight layers: against 64 bits the outputs are
    # off by 0.003 to 0.016 in bfloat16 (later layers' cache rows and the logits the most) and by
    # 0.0003 to 0.0014 in float16
    if case["dtype"] == "float16":
        return {"rel": 0.005, "max": 0.05, "differ": 0.01}
    return {"rel": 0.03, "max": 0.3, "differ": 0.01}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def exact(case, seed):
    with torch.inference_mode():
        g = _generator(seed)
        W = _weights(case, g)
        ids, pos, past, kv, state = _inputs(case, g)
        if case["size"] == "nabelix":
            return _nabelix64(case, W, ids, pos, past, kv, state)
        return _llama64(case, W, ids, pos, past, kv)


def _mm(x, w):
    """x @ w^T in 64 bits, the weight widened a part at a time."""
    step = max(1, 2 ** 28 // w.shape[1])
    return torch.cat([x @ w[a:a + step].to(F64).t() for a in range(0, w.shape[0], step)], dim=-1)


def _rms(x):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)


def _rotate(x, pos):
    """Half-split rotation of (B, heads, T, D)."""
    D = x.shape[-1]
    f = THETA ** (-torch.arange(0, D, 2, dtype=F64, device=x.device) / D)
    a = pos.clamp(min=0).to(F64).unsqueeze(-1) * f
    c, s = a.cos().unsqueeze(1), a.sin().unsqueeze(1)
    u, v = x[..., : D // 2], x[..., D // 2:]
    return torch.cat([u * c - v * s, v * c + u * s], dim=-1)


def _attend(q, k, v, seen, scale, bias=None):
    """q (H, T, D), k and v (G, L, D), seen (T, L); bias(head) (T, L) is added to the scores."""
    per = q.shape[0] // k.shape[0]
    out = torch.empty(q.shape[0], q.shape[1], v.shape[-1], dtype=F64, device=q.device)
    for h in range(q.shape[0]):
        p = q[h] @ k[h // per].t() * scale
        if bias is not None:
            p += bias(h)
        p = torch.softmax(p.masked_fill_(~seen, -math.inf), dim=-1)
        out[h] = torch.nan_to_num_(p, nan=0.0) @ v[h // per]
    return out


def _fill(case, cache, new, pos):
    """The cache rows (in 64 bits) with the step's own at their positions."""
    for b in range(pos.shape[0]):
        ok = pos[b] >= 0
        cache[b, :, pos[b][ok]] = new[b][:, ok]
    return cache


def _expert_weights(case, w):
    """A stacked expert weight as its quantised form holds it."""
    if case["quant"] == "fp8":
        scale = w.float().abs().amax(-1, keepdim=True).clamp(min=1e-12) / 448.0
        q = (w.float() / scale).clamp(-448, 448).to(torch.float8_e4m3fn)
        return q.float(), scale.to(F64)
    if case["quant"] == "mx4":
        v = w.float().view(*w.shape[:-1], -1, 32)
        e = (torch.floor(torch.log2(v.abs().amax(-1, keepdim=True).clamp(min=1e-30))) - 2)
        scale = torch.pow(2.0, e.clamp(-127, 127))
        v = (v / scale).clamp(-6, 6)
        mids = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=w.device)
        grid = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0], device=w.device)
        v = grid[torch.bucketize(v.abs(), mids)] * v.sign() * scale
        return v.view(w.shape), None
    return w, None


def _experts64(case, W, p, x):
    s = SIZES[case["size"]]
    vals, idx = _mm(x, W[p + "router"]).topk(s["top"], dim=-1)
    vals = torch.softmax(vals, dim=-1)
    out = torch.zeros_like(x)
    for e in range(s["experts"]):
        row, at = (idx == e).nonzero(as_tuple=True)
        if not row.numel():
            continue

        def mm(v, name):
            w, scale = _expert_weights(case, W[p + name][e])
            y = _mm(v, w)
            return y if scale is None else y * scale.view(1, -1)

        y = mm(F.silu(mm(x[row], "gate")) * mm(x[row], "up"), "down")
        out.index_add_(0, row, y * vals[row, at].unsqueeze(-1))
    return out


def _llama64(case, W, ids, pos, past, kv):
    s, B, T = SIZES[case["size"]], case["batch"], case["tokens"]
    H, G, D = s["heads"], s["kv_heads"], s["dim"]
    L = _max_len(case)
    x = W["embed"][ids].to(F64)
    at = torch.arange(L, device=x.device)
    written = []
    for i in range(case["layers"]):
        p = "l%d." % i
        q, k, v = torch.split(_mm(_rms(x), W[p + "qkv"]).view(B, T, -1, D).transpose(1, 2),
                              [H, G, G], dim=1)
        if case["size"] == "qwen3moe":
            q, k = _rms(q), _rms(k)
        q, k = _rotate(q, pos), _rotate(k, pos)
        if case["kv8"]:
            k, v = (t.to(getattr(torch, case["dtype"])).to(torch.float8_e4m3fn).to(F64)
                    for t in (k, v))
        o = torch.empty(B, H, T, D, dtype=F64, device=x.device)
        full = []
        for b in range(B):
            rows = []
            for new, old in zip((k, v), kv[i] if kv else (None, None)):
                c = torch.zeros(1, G, L, D, dtype=F64, device=x.device) if old is None \
                    else old[b:b + 1].to(F64)
                rows.append(_fill(case, c, new[b:b + 1], pos[b:b + 1]))
            n = int(pos[b].max()) + 1
            seen = (at[:n].view(1, n) <= pos[b].view(T, 1))
            o[b] = _attend(q[b], rows[0][0, :, :n], rows[1][0, :, :n], seen, D ** -0.5)
            full.append(rows)
        if case["step"] == "prefill":
            written += [torch.cat([r[j] for r in full]) for j in (0, 1)]
        x = x + _mm(o.transpose(1, 2).reshape(B, T, -1), W[p + "o"])
        h = _rms(x).view(B * T, -1)
        if "experts" in s:
            y = _experts64(case, W, p, h)
        else:
            gate, up = _mm(h, W[p + "gate_up"]).chunk(2, dim=-1)
            y = _mm(F.silu(gate) * up, W[p + "down"])
        x = x + y.view(B, T, -1)
    if case["step"] == "prefill":
        last = (pos >= 0).sum(-1) - 1
        x = x[torch.arange(B, device=x.device), last].unsqueeze(1)
    out = {"logits": _mm(_rms(x), W["head"]), "tokens": None}
    if case["step"] == "prefill":
        out["kv"] = written
    return out


def _norm64(x):
    x = x - x.mean(-1, keepdim=True)
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)


def _conv64(x, w, tail):
    """x (B, T, C), w (C, taps), tail (B, taps - 1, C) or None."""
    taps = w.shape[1]
    tail = torch.zeros(x.shape[0], taps - 1, x.shape[2], dtype=F64, device=x.device) \
        if tail is None else tail.to(F64)
    ext = torch.cat([tail, x], dim=1)
    return sum(ext[:, j:j + x.shape[1]] * w[:, j].to(F64) for j in range(taps))


def _nabelix64(case, W, ids, pos, past, kv, state):
    s, B, T = SIZES[case["size"]], case["batch"], case["tokens"]
    H, G, D, r = s["heads"], s["kv_heads"], s["dim"], s["rank"]
    L = _max_len(case)
    x = W["embed"][ids].to(F64)
    mems, written = [], []
    for i in range(case["layers"]):
        p = "l%d." % i
        st = state[i] if state else {"canon": None, "conv": None, "mem": None}
        h = _norm64(x)
        h = h + _conv64(h, W[p + "canon"], st["canon"])
        y = _mm(h, W[p + "in"])
        q, k, v, gate, qkv, beta, low = torch.split(
            y, [H * D, G * D, G * D, H * D, 3 * H * D, H, 2 * r], dim=-1)
        heads = lambda t: t.view(B, T, -1, D).transpose(1, 2)  # noqa: E731
        q, k, v = heads(q), heads(k), heads(v)
        o = torch.empty(B, H, T, D, dtype=F64, device=x.device)
        r1, r2 = W[p + "r1"].to(F64), W[p + "r2"].to(F64)
        full = []
        for b in range(B):
            rows = []
            for new, old in zip((k, v), kv[i] if kv else (None, None)):
                c = torch.zeros(1, G, L, D, dtype=F64, device=x.device) if old is None \
                    else old[b:b + 1].to(F64)
                rows.append(_fill(case, c, new[b:b + 1], pos[b:b + 1]))
            n = int(pos[b].max()) + 1
            j = torch.arange(n, device=x.device).view(1, n)
            far = pos[b].view(T, 1) - j
            seen = (far >= 0) & ((far < s["window"]) | (j < s["keep"]))
            far = far.clamp(min=0).to(F64)
            o[b] = _attend(q[b], rows[0][0, :, :n], rows[1][0, :, :n], seen, D ** -0.5,
                           lambda hd: -r1[hd] * torch.log1p(r2[hd] * far))
            full.append(rows)
        if case["step"] == "prefill":
            # pages of 64 rows, as the paged cache holds them
            per = -(-L // BLOCK)
            for j in (0, 1):
                c = F.pad(torch.cat([f[j] for f in full]), (0, 0, 0, per * BLOCK - L))
                written.append(c.transpose(1, 2).reshape(B * per, BLOCK, G, D))
        left = o.transpose(1, 2).reshape(B, T, -1) * torch.sigmoid(gate)
        qd, kd, vd = torch.split(F.silu(_conv64(qkv, W[p + "conv"], st["conv"]))
                                 .view(B, T, 3 * H, D), [H, H, H], dim=2)
        qd = qd * torch.rsqrt(qd.square().sum(-1, keepdim=True) + 1e-6) * D ** -0.5
        kd = kd * torch.rsqrt(kd.square().sum(-1, keepdim=True) + 1e-6)
        a = (_mm(low[..., :r], W[p + "a2"]) + W[p + "dt_bias"].to(F64)).view(B, T, H, D)
        decay = torch.exp(-torch.exp(W[p + "A_log"].to(F64)).view(1, 1, H, 1) * F.softplus(a))
        beta = torch.sigmoid(beta)
        M = torch.zeros(B, H, D, D, dtype=F64, device=x.device) if st["mem"] is None \
            else st["mem"].to(F64)
        od = torch.empty(B, T, H, D, dtype=F64, device=x.device)
        for t in range(T):
            M = decay[:, t].unsqueeze(-1) * M
            u = beta[:, t].unsqueeze(-1) * (
                vd[:, t] - torch.matmul(kd[:, t].unsqueeze(-2), M).squeeze(-2))
            M = M + kd[:, t].unsqueeze(-1) * u.unsqueeze(-2)
            od[:, t] = torch.matmul(qd[:, t].unsqueeze(-2), M).squeeze(-2)
        mems.append(M.transpose(2, 3))
        right = (_rms(od).view(B, T, -1)) * torch.sigmoid(_mm(low[..., r:], W[p + "g2"]))
        x = x + _mm(left, W[p + "left_o"]) + _mm(right, W[p + "right_o"])
        gate, up = _mm(_norm64(x), W[p + "gate_up"]).chunk(2, dim=-1)
        x = x + _mm(F.gelu(gate, approximate="tanh") * up, W[p + "down"])
    if case["step"] == "prefill":
        x = x[:, -1:]
    out = {"logits": 30.0 * torch.tanh(_mm(_norm64(x), W["embed"]) / 30.0), "state": mems}
    if case["step"] == "prefill":
        out["kv"] = written
    return out
