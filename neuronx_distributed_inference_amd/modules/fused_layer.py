"""Decoder layers (norm, attention, residual, norm, feed-forward, residual) in fewer launches.

Between two products stands one kernel: the residual sum and the norm that follows take the parts
of K of the output and down projections (``ops.add_norm``), rope and cache write those of q|k|v,
and gate|up writes its activation. A step of few tokens is a chain of such launches, each waiting
for the last. The layer's modules keep the weights; they are not called, so a layer with hooks or a
forward of its own on any of them, biases, 8-bit weights, adapters or tensor parallelism keeps the
chain of modules.
"""

from __future__ import annotations

import torch
from torch.nn.modules import module as nn_module

from neuronx_distributed_inference_amd import ops
from neuronx_distributed_inference_amd.modules.attention.attention_base import (
    PHASE_CTE,
    PHASE_TKG,
    AttentionBase,
    _hooked,
)
from neuronx_distributed_inference_amd.modules.attention.gqa import GroupQueryAttentionO
from neuronx_distributed_inference_amd.modules.mlp import GatedMLP
from neuronx_distributed_inference_amd.modules.norm import RMSNorm
from neuronx_distributed_inference_amd.parallel.layers import entry, plain_linear


# what the loop does in their place, by heart: a class whose forward was replaced is not plain
_FORWARDS = {c: c.forward for c in (AttentionBase, GroupQueryAttentionO, GatedMLP, RMSNorm)}
_ATTEND = AttentionBase.attend_fused


def _plain(module, cls) -> bool:
    return type(module) is cls and cls.forward is _FORWARDS[cls] and not _hooked(module)


def _plain_norm(norm, h: torch.Tensor) -> bool:
    weight = norm._parameters.get("weight")
    return (_plain(norm, RMSNorm) and weight is not None and weight.dtype == h.dtype
            and weight.is_contiguous() and weight.data_ptr() % 16 == 0)


def _own_attend(attn) -> bool:
    """Whether a program has put an attend_fused of its own in place, which knows no `output`."""
    return type(attn).attend_fused is not _ATTEND or "attend_fused" in attn.__dict__


def fusable(layers, final_norm, h: torch.Tensor, attention_mask, phase: str) -> bool:
    """Whether :func:`run_layers` may stand for calling the layers and the final norm on h."""
    if not (layers and h.is_cuda and h.dtype in (torch.bfloat16, torch.float16) and h.shape[-1] % 8 == 0
            and h.shape[-1] <= 32768 and h.numel() and h.is_contiguous()
            and h.data_ptr() % 16 == 0):
        return False
    if nn_module._global_forward_hooks or nn_module._global_forward_pre_hooks:
        return False
    if attention_mask is not None and attention_mask.dim() == 4 and phase == PHASE_TKG:
        return False
    if not _plain_norm(final_norm, h):
        return False
    for layer in layers:
        # (a subclass with a forward of its own inherits fused_parts all the same)
        if getattr(type(layer), "fused_forward", None) is not type(layer).forward or _hooked(layer):
            return False
        attn, _ = layer.fused_parts()
        if not (isinstance(attn, AttentionBase)
                and type(attn).forward is _FORWARDS[AttentionBase]
                and type(attn).attend_fused is AttentionBase.attend_fused
                and not _hooked(attn)):
            return False
        out = entry(attn, "o_proj")
        if not (_plain(out, GroupQueryAttentionO)
                and plain_linear(entry(out, "o_proj"), h)
                and _plain_norm(entry(layer, "input_layernorm"), h)
                and _plain_norm(entry(layer, "post_attention_layernorm"), h)):
            return False
    return True


def _plain_mlp(mlp, x: torch.Tensor) -> bool:
    return (_plain(mlp, GatedMLP) and mlp.fused
            and mlp.act_mul_fused is ops.silu_mul_fused
            and plain_linear(entry(mlp, "gate_up_proj"), x) and plain_linear(entry(mlp, "down_proj"), x))


def _feed_forward(mlp, x: torch.Tensor) -> torch.Tensor:
    """Output of the feed-forward, or its parts of K."""
    if _plain_mlp(mlp, x):
        return ops.linear_parts(ops.linear_silu_mul(x, mlp.gate_up_proj.weight),
                                mlp.down_proj.weight)
    return mlp(x)


PROMPT_ROWS = ops.TILE_ROWS


def dense_layer(layer) -> bool:
    """Whether the layer's modules are of the kinds that :func:`prompt_operands` takes."""
    if getattr(type(layer), "fused_forward", None) is not type(layer).forward:
        return False
    attn, mlp = layer.fused_parts()
    return (isinstance(attn, AttentionBase) and attn.q_norm is None and attn.k_norm is None
            and type(mlp) is GatedMLP)


def prompt_operands(layers, final_norm, x, cos, kv_mgr, seq_ids):
    """What csrc/prompt_layers.cpp takes of dense layers without q/k norms, None for others."""
    if not ops.tiles_enabled():
        return None
    weights, sizes, numbers = [], [], []
    for layer, after in zip(layers, layers[1:] + [None]):
        attn, mlp = layer.fused_parts()
        if _own_attend(attn) or attn.q_norm is not None or attn.k_norm is not None:
            return None
        qkv = entry(attn, "qkv_proj")
        rows = attn.prompt_front(x, cos, kv_mgr, PHASE_CTE, seq_ids)
        if (rows is None or not attn.use_rope or attn.sinks is not None
                or _hooked(qkv) or not plain_linear(entry(qkv, "qkv"), x) or not _plain_mlp(mlp, x)):
            return None
        norm = entry(layer, "post_attention_layernorm")
        following = entry(after, "input_layernorm") if after is not None else final_norm
        weights += [m.weight for m in (
            entry(qkv, "qkv"), entry(entry(attn, "o_proj"), "o_proj"), norm, entry(mlp, "gate_up_proj"),
            entry(mlp, "down_proj"), following)]
        weights += rows
        sizes += [attn.num_heads_per_rank, attn.num_kv_heads_per_rank, int(attn.sliding_window)]
        numbers += [norm.variance_epsilon, following.variance_epsilon, float(attn.scale)]
    return weights, sizes, numbers


def _short_prompt(layers, final_norm, h, x, cos, sin, kv_mgr, position_ids, seq_ids):
    """What :func:`run_layers` gives for a short whole prompt of dense layers without q/k norms,
    its launches made by one native call (csrc/prompt_layers.cpp); None where that does not serve."""
    if h.numel() > PROMPT_ROWS * h.shape[-1] or not (cos.is_contiguous() and sin.is_contiguous()):
        return None
    operands = prompt_operands(layers, final_norm, x, cos, kv_mgr, seq_ids)
    if operands is None:
        return None
    return ops._require_ext("prompt_layers").prompt_layers(
        h, x, cos, sin, position_ids, seq_ids, *operands)


def packed_layers(operands, start, lengths):
    """Normed output (rows, 1, H) of the layers over prompts without their padding: `start` of
    ops.step_start_packed, operands of :func:`prompt_operands`. None, with nothing done, where that
    does not serve."""
    h, x, cos, sin, position_ids, rows, starts, prompts = start
    return ops._require_ext("prompt_layers").prompt_layers(
        h, x, cos, sin, position_ids, rows, *operands, starts=starts, prompt_sid=prompts,
        longest=max(lengths))


def run_layers(layers, final_norm, h: torch.Tensor, cos, sin, kv_mgr, position_ids, phase,
               attention_mask, seq_ids, x=None) -> torch.Tensor:
    """Normed output of the stack; h becomes the residual stream. x: the first layer's normed
    input, where that is there already."""
    layers = list(layers)
    if x is None:
        x = layers[0].input_layernorm(h)
    if (phase == PHASE_CTE and cos is not None and seq_ids is not None
            and position_ids.dtype == seq_ids.dtype == torch.int32
            and position_ids.is_contiguous() and seq_ids.is_contiguous()):
        y = _short_prompt(layers, final_norm, h, x, cos, sin, kv_mgr, position_ids, seq_ids)
        if y is not None:
            return y
    for layer, after in zip(layers, layers[1:] + [None]):
        attn, mlp = layer.fused_parts()
        args = (x, cos, sin, kv_mgr, position_ids, phase, attention_mask, seq_ids)
        if _own_attend(attn):
            y = attn.attend_fused(*args)
            y = y if y is None else ops.linear_parts(y, attn.o_proj.o_proj.weight)
        else:
            y = attn.attend_fused(*args, output=attn.o_proj.o_proj.weight)
        if y is None:
            y = attn(*args)
        norm = layer.post_attention_layernorm
        x = ops.add_norm(y, h, norm.weight, norm.variance_epsilon)
        y = _feed_forward(mlp, x)
        norm = final_norm if after is None else after.input_layernorm
        x = ops.add_norm(y, h, norm.weight, norm.variance_epsilon)
    return x
