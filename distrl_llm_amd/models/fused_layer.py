"""A decoder layer's two halves as single autograd nodes (GPU, bf16, LoRA
training): attention and feed-forward, each with its norm, its projections
with their adapters and its residual sum, backward written out.

The module-by-module layer launches ~200 kernels forward and backward, most
of them elementwise passes between the products (residual adds, adapter
scaling, gradient sums of projections that share an input, rotary steps,
head transposes), and short micro-batches are bound by launching them. A half
is 7 launches forward and 10 or 11 backward (attention) or 5 and 7 (feed-forward)
here, prepared in native code (ops/csrc/adapted_layer.cpp): products of our own
(ops/csrc/product.hip) take adapters as more of their projections' K, residuals,
the activation and its gradient with them. The library's products, where many
rows meet wide weights, have W laid out beside B for it; at ranks that ours don't
take large weights that few rows meet are taken as they lie, their adapters
joined to fp32 products. Adapter gradients are one launch and its sum
(ops/csrc/adapter_grads.hip).
"""

from __future__ import annotations

import torch
from torch.autograd.function import once_differentiable
from torch.nn.modules.module import _has_any_global_hook

from .lora import LoRALinear


def _hooked(module) -> bool:
    """Whether calling the module does more than its class's forward."""
    d = vars(module)
    return bool(d["_forward_hooks"] or d["_forward_pre_hooks"]
                or d["_backward_hooks"] or d["_backward_pre_hooks"]
                or "forward" in d)


def _trainable(mod: LoRALinear) -> bool:
    if type(mod) is not LoRALinear or mod.r <= 0:
        return False
    w, b, drop, bf16 = mod.weight, mod.bias, mod.lora_dropout, torch.bfloat16
    return (w.dtype == mod.lora_A.dtype == mod.lora_B.dtype == bf16
            and w.numel() > 0 and not w.requires_grad
            and (b is None or not b.requires_grad)
            and (isinstance(drop, torch.nn.Identity)
                 or not mod.training or drop.p == 0.0)
            and not _hooked(drop))


def usable(layer, x) -> bool:
    """Whether the layer's forward on x may take the fused nodes: everything
    else (CPU, other types, dropout, freed base weights, hooks on a part,
    parts of another class, no adapter, inference) stays with the modules."""
    if not (x.is_cuda and x.dtype == torch.bfloat16
            and torch.is_grad_enabled()) or _has_any_global_hook():
        return False
    from .model import MLP, Attention, RMSNorm
    at, mlp = layer.self_attn, layer.mlp
    if type(at) is not Attention or type(mlp) is not MLP:
        return False
    linears = (at.q_proj, at.k_proj, at.v_proj, at.o_proj,
               mlp.gate_proj, mlp.up_proj, mlp.down_proj)
    norms = [layer.input_layernorm, layer.post_attention_layernorm]
    if at.spec.qk_norm:
        norms += [at.q_norm, at.k_norm]
    return (at.spec.head_dim in (64, 128)
            and at.spec.hidden_size % 8 == at.spec.intermediate_size % 8 == 0
            and all(_trainable(m) for m in linears)
            and at.o_proj.bias is None and mlp.down_proj.bias is None
            and all(type(n) is RMSNorm and n.weight.dtype == torch.bfloat16
                    and not n.weight.requires_grad for n in norms)
            and not any(_hooked(m) for m in (*linears, *norms, at, mlp)))


def _ext():
    from ..ops.functional import _require_ext
    return _require_ext("fused decoder layer")


class _Attention(torch.autograd.Function):
    """x + o_proj(attention(qkv_proj(norm(x)))) over rows x (rows, hidden)."""

    @staticmethod
    def forward(ctx, x, rotary, at, norm, *adapters):
        pos, inv_freq, back_freq, cu, longest = rotary
        mods = (at.q_proj, at.k_proj, at.v_proj, at.o_proj)
        Ws, scales = [m.weight for m in mods], [m.scale for m in mods]
        As, Bs = list(adapters[0::2]), list(adapters[1::2])
        head_norms, eps = (None, None), (norm.eps, 0.0, 0.0)
        if at.spec.qk_norm:
            head_norms = at.q_norm.weight, at.k_norm.weight
            eps = norm.eps, at.q_norm.eps, at.k_norm.eps
        y, *own = _ext().attention_half_fwd(
            x, norm.weight, eps[0], Ws, [m.bias for m in mods[:3]], As, Bs,
            scales, *head_norms, *eps[1:], pos, inv_freq, cu, longest, at.scale,
            at.spec.head_dim)
        ctx.save_for_backward(x, norm.weight, *head_norms, pos, back_freq, cu,
                              *own, *Ws, *As, *Bs)
        ctx.scales, ctx.eps = scales, eps
        ctx.longest, ctx.scale = longest, at.scale
        return y

    @staticmethod
    @once_differentiable
    def backward(ctx, g):
        x, norm, q_norm, k_norm, pos, back_freq, cu, *rest = ctx.saved_tensors
        own, Ws, As, Bs = rest[:8], rest[8:12], rest[12:16], rest[16:]
        dx, *grads = _ext().attention_half_bwd(
            g, x, norm, ctx.eps[0], Ws, As, Bs, ctx.scales, q_norm, k_norm,
            *ctx.eps[1:], pos, back_freq, cu, ctx.longest, ctx.scale, *own,
            ctx.needs_input_grad[0])
        return (dx, None, None, None, *grads)


class _FeedForward(torch.autograd.Function):
    """x + down_proj(silu(gate_proj(norm(x))) * up_proj(norm(x)))."""

    @staticmethod
    def forward(ctx, x, mlp, norm, *adapters):
        mods = (mlp.gate_proj, mlp.up_proj, mlp.down_proj)
        Ws, scales = [m.weight for m in mods], [m.scale for m in mods]
        As, Bs = list(adapters[0::2]), list(adapters[1::2])
        y, *own = _ext().feed_forward_half_fwd(
            x, norm.weight, norm.eps, Ws, [m.bias for m in mods[:2]], As, Bs,
            scales)
        ctx.save_for_backward(x, norm.weight, *own, *Ws, *As, *Bs)
        ctx.scales, ctx.eps = scales, norm.eps
        return y

    @staticmethod
    @once_differentiable
    def backward(ctx, g):
        x, norm, hu, gu, au, *rest = ctx.saved_tensors
        dx, *grads = _ext().feed_forward_half_bwd(
            g, x, norm, ctx.eps, rest[:3], rest[3:6], rest[6:], ctx.scales, hu,
            gu, au, ctx.needs_input_grad[0])
        return (dx, None, None, *grads)


class Head(torch.autograd.Function):
    """x W^T of the frozen LM head; the input's gradient is a product of our own,
    whose sum over the vocabulary is cut into shares."""

    @staticmethod
    def forward(ctx, x, weight):
        ctx.save_for_backward(weight)
        return torch.nn.functional.linear(x, weight)

    @staticmethod
    @once_differentiable
    def backward(ctx, g):
        weight, = ctx.saved_tensors
        return _ext().product_rows(g, weight), None


def frozen_head(x, weight) -> bool:
    """Whether Head takes x (rows, hidden) and the LM head's weight."""
    bf16 = torch.bfloat16
    return (x.is_cuda and x.dim() == 2 and x.dtype == weight.dtype == bf16
            and weight.device == x.device and not weight.requires_grad
            and type(weight) in (torch.Tensor, torch.nn.Parameter))


def rotary(head_dim: int, theta: float, positions, cu, longest: int):
    """What the nodes need to know of the rows: int32 positions (rows,), fp32
    inverse frequencies and their negatives, the first row of every sequence
    and the end (int32), the most rows of one."""
    half = torch.arange(0, head_dim, 2, device=positions.device,
                        dtype=torch.float32)
    inv_freq = 1.0 / (theta ** (half / head_dim))
    return positions.to(torch.int32), inv_freq, -inv_freq, cu, longest


def forward(layer, x, rotary):
    """The layer on x, (B, T, hidden) or (rows, hidden); see rotary()."""
    at, mlp = layer.self_attn, layer.mlp
    shape = x.shape
    y = _Attention.apply(
        x.reshape(-1, shape[-1]).contiguous(), rotary, at,
        layer.input_layernorm,
        *(w for m in (at.q_proj, at.k_proj, at.v_proj, at.o_proj)
          for w in (m.lora_A, m.lora_B)))
    y = _FeedForward.apply(
        y, mlp, layer.post_attention_layernorm,
        *(w for m in (mlp.gate_proj, mlp.up_proj, mlp.down_proj)
          for w in (m.lora_A, m.lora_B)))
    return y.view(shape)
