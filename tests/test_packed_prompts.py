"""Batches of prompts without their padding, against the padded batch."""

import pytest
import torch

from neuronx_distributed_inference_amd import ops
from neuronx_distributed_inference_amd.config import EngineConfig, OnDeviceSamplingConfig
from neuronx_distributed_inference_amd.models.llama.modeling_llama import (
    LlamaForCausalLM,
    LlamaInferenceConfig,
)

pytestmark = pytest.mark.gpu


def _model(B, S, window=0, dtype="bfloat16"):
    ec = EngineConfig(
        batch_size=B, max_batch_size=B, seq_len=S, max_length=S, max_context_length=S,
        torch_dtype=dtype, tp_degree=1, fused_qkv=True, fused_gate_up=True, output_logits=True,
        on_device_sampling_config=OnDeviceSamplingConfig(top_k=1))
    cfg = LlamaInferenceConfig(
        neuron_config=ec, vocab_size=512, hidden_size=512, intermediate_size=1024,
        num_hidden_layers=2, num_attention_heads=8, num_key_value_heads=2, head_dim=64,
        max_position_embeddings=2 * S, rms_norm_eps=1e-5, rope_theta=10000.0, hidden_act="silu",
        tie_word_embeddings=False, sliding_window=window)
    torch.manual_seed(1)
    lm = LlamaForCausalLM(cfg).eval()
    for p in lm.parameters():
        torch.nn.init.normal_(p, std=0.05)
    lm = lm.cuda()
    lm.enable_submodels()
    return lm


def _lengths(mask, positions):
    got = ops.PromptLengths(mask, positions)
    assert got.all() == bool(mask.all())
    return got.get()


def _batch(lengths, S):
    g = torch.Generator().manual_seed(2)
    ids = torch.randint(0, 512, (len(lengths), S), generator=g)
    pos = torch.arange(S).expand(len(lengths), S).clone()
    mask = torch.zeros(len(lengths), S, dtype=torch.long)
    for b, n in enumerate(lengths):
        mask[b, :n] = 1
        pos[b, n:] = -1
    return ids.cuda(), pos.cuda(), mask.cuda()


def _run(lm, ids, pos, mask, seq_ids=None):
    B = ids.shape[0]
    lm.reset()
    with torch.inference_mode():
        out = lm(input_ids=ids, attention_mask=mask, position_ids=pos,
                 seq_ids=torch.arange(B, device="cuda") if seq_ids is None else seq_ids)
    kv = [t.data.clone() for i in range(2) for t in lm.model.kv_mgr.get_cache(i)]
    return out.logits.float(), out.tokens, kv


# a query tile is 32 tokens of 4 heads; 512 rows are the most that the tiled products take
@pytest.mark.parametrize("lengths,S,capacity", [
    ([1], 2, 40), ([93], 93, 124), ([31, 32, 33, 1, 70], 70, 101), ([300], 300, 300 + 31),
    ([129, 64, 1, 256, 97, 200], 256, 256), ([700, 1, 233], 700, 731), ([2, 800, 5], 801, 900)])
@pytest.mark.parametrize("window", [0, 50])
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
def test_packed_prompts(lengths, S, capacity, window, dtype):
    lm = _model(len(lengths), capacity, window, dtype)
    ids, pos, mask = _batch(lengths, S)
    took = []
    inner = lm.model.packed_prompts
    lm.model.packed_prompts = lambda *a: took.append(inner(*a)) or took[-1]
    got = _run(lm, ids, pos, None if min(lengths) == S else mask)
    assert (sum(lengths) < len(lengths) * capacity) == (took[0] is not None)
    lm.model.packed_prompts = lambda *a: None
    want = _run(lm, ids, pos, mask)
    # two layers of products that may be split at other places of K: a few roundings of 16 bits
    tol = 0.03 if dtype == "bfloat16" else 0.004
    assert (got[0] - want[0]).norm() <= tol * want[0].norm()
    for a, b in zip(got[2], want[2]):
        assert (a.float() - b.float()).norm() <= tol * b.float().norm()
        assert ((a == 0).all(-1) == (b == 0).all(-1)).all()       # the same rows are written


@pytest.mark.parametrize("lengths,S,seq_ids,batch", [
    ([93], 93, [2], 4), ([31, 1, 70], 70, [4, 0, 2], 5), ([64, 33], 64, [1, 0], 2), ([300, 350, 9], 350, [6, 1, 3], 8)])
@pytest.mark.parametrize("kind", [torch.int64, torch.int32])
@pytest.mark.parametrize("masked", [True, False])
def test_packed_prompts_of_other_cache_rows(lengths, S, seq_ids, batch, kind, masked):
    """A batch smaller than the model's, in cache rows that are not the prompts' own numbers."""
    lm = _model(batch, S + 7)
    if not masked:
        lengths = [S] * len(lengths)
    ids, pos, mask = _batch(lengths, S)
    seq = torch.tensor(seq_ids, device="cuda", dtype=kind)
    noise = torch.Generator(device="cuda").manual_seed(3)
    caches = [t.data for i in range(2) for t in lm.model.kv_mgr.get_cache(i)]
    lm.reset = lambda: [c.normal_(0, 1, generator=noise.manual_seed(3)) for c in caches]
    lm.kv_cache_populated = False
    took = []
    inner = lm.model.packed_prompts
    lm.model.packed_prompts = lambda *a: took.append(inner(*a)) or took[-1]
    got = _run(lm, ids, pos, mask if masked else None, seq)
    assert took[0] is not None
    lm.kv_cache_populated = False
    lm.model.packed_prompts = lambda *a: None
    want = _run(lm, ids, pos, mask if masked else None, seq)
    assert got[0].shape == want[0].shape and (got[0] - want[0]).norm() <= 0.03 * want[0].norm()
    lm.reset()
    for a, b, before in zip(got[2], want[2], caches):
        own = torch.zeros(a.shape[0], a.shape[2], dtype=torch.bool)
        for row, n in zip(seq_ids, lengths):
            own[row, :n] = True
        own = own.cuda()
        a, b, before = (t.transpose(1, 2) for t in (a, b, before))
        assert torch.equal(a[~own], before[~own])
        a, b = a[own].float().flatten(1), b[own].float().flatten(1)
        assert ((a - b).norm(dim=1) <= 0.03 * b.norm(dim=1)).all()
        assert (a != before[own].float().flatten(1)).any(dim=1).all()


@pytest.mark.parametrize("kind", [torch.int64, torch.int32, torch.bool])
@pytest.mark.parametrize("positions", [torch.int64, torch.int32])
def test_prompt_lengths(kind, positions):
    lengths = [1, 64, 255, 256, 257, 600]
    _, pos, mask = _batch(lengths, 600)
    pos, mask = pos.to(positions), mask.to(kind)
    assert _lengths(mask, pos) == lengths
    assert _lengths(torch.ones_like(mask), pos) == [600] * 6
    for b, j in ((0, 5), (3, 255), (4, 599)):
        other = mask.clone()
        other[b, j] = 1 - other[b, j].to(torch.int64)             # a hole, or a place without its token
        assert _lengths(other, pos) is None
    other = mask.clone()
    other[1] = 0
    assert _lengths(other, pos) is None                 # no token at all
    left = mask.flip(1).contiguous()
    assert _lengths(left, pos) is None
    later = pos.clone()
    later[2, 300] = 300                                           # padding with a place in the cache
    assert _lengths(mask, later) is None
    if kind != torch.bool:
        assert _lengths(mask * 2, pos) is None


def test_left_padding_keeps_the_mask():
    lm = _model(2, 64)
    ids, pos, mask = _batch([20, 40], 40)
    mask[0] = mask[0].flip(0)
    pos[0] = torch.cat([torch.full((20,), -1), torch.arange(20)]).cuda()
    took = []
    inner = lm.model.packed_prompts
    lm.model.packed_prompts = lambda *a: took.append(inner(*a))
    assert _run(lm, ids, pos, mask)[0].isfinite().all() and took == [None]


@pytest.mark.parametrize("masked", [True, False])
def test_captured_prompts_keep_the_padding(masked):
    """A captured call serves every later batch of its shape, by the mask that it is given then."""
    lm = _model(4, 101)
    ids, pos, mask = _batch([20, 33, 70], 70)
    sid, sampling = torch.arange(3, device="cuda"), torch.ones(3, 3, device="cuda")
    args = (ids, mask if masked else None, pos, sid, sampling)
    lm.model.packed_prompts = lambda *a: None
    side = torch.cuda.Stream()
    with torch.inference_mode():
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            lm.context_encoding_model(*args)
        torch.cuda.current_stream().wait_stream(side)
        del lm.model.packed_prompts
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            tokens, logits = lm.context_encoding_model(*args)
        for lengths in ([20, 33, 70], [70, 1, 5], [2, 69, 64]):
            new = _batch(lengths if masked else [70] * 3, 70)
            ids.copy_(new[0].flip(0))
            pos.copy_(new[1])
            mask.copy_(new[2])
            lm.model.packed_prompts = lambda *a: None
            want = lm.context_encoding_model(*args)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(tokens, want[0]) and torch.equal(logits, want[1])


def test_products_by_the_librarys_first_choice():
    """What packed prompts take: asked for once a shape, errors of the operands stay errors."""
    g = torch.Generator(device="cuda").manual_seed(0)
    x = torch.randn(700, 320, device="cuda", generator=g).bfloat16()
    w = torch.randn(96, 320, device="cuda", generator=g).bfloat16()
    want = x.double() @ w.double().t()
    slack = 2.0 ** -8 * want.abs() + 320 * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    for _ in range(3):
        y = torch.empty(700, 96, dtype=torch.bfloat16, device="cuda")
        assert ops._C.lt_linear(y, x, w, None, False) is True
        assert ((y.double() - want).abs() <= slack).all()
    for bad in (w[:, :319].contiguous(), w.t()):
        with pytest.raises(RuntimeError):
            ops._C.lt_linear(y, x, bad, None, False)
