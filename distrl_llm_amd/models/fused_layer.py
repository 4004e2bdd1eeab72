"""A decoder layer's two halves as single autograd nodes (GPU, bf16, LoRA
training): attention and feed-forward, each with its norm, its projections
with their adapters and its residual sum, backward written out.

The module-by-module layer launches ~200 kernels forward and backward, most
of them elementwise passes between the products (residual adds, adapter
scaling, gradient sums of projections that share an input, rotary steps,
head transposes), and short micro-batches are bound by launching them. Here
sums accumulate inside the products (beta = 1, in place), the adapters of
projections that share an input share one down product, and rotary, norm and
activation passes are one kernel each: ~65 launches.

A micro-batch of three short samples on a 24-layer 0.5B model: 58 ms to
28 ms (34 with the library adding the adapters); 16 x 1550 tokens on a
28-layer 1.5B model: 380 to 239 ms.
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
            and all(_trainable(m) for m in linears)
            and at.o_proj.bias is None and mlp.down_proj.bias is None
            and all(type(n) is RMSNorm and n.weight.dtype == torch.bfloat16
                    and not n.weight.requires_grad for n in norms)
            and not any(_hooked(m) for m in (*linears, *norms, at, mlp)))


def _ext():
    from ..ops.functional import _require_ext
    return _require_ext("fused decoder layer")


def _scaled_mm(a, b, scale, out=None):
    """scale * a @ b, the scale in the product's epilogue."""
    if out is None:
        out = a.new_empty(a.shape[0], b.shape[1])
    return torch.addmm(out, a, b, beta=0.0, alpha=scale, out=out)


def _add(y, u, m, scale=1.0):
    """y += scale * u m, in place; m as it lies or a transposed view."""
    return y if _ext().lora_add(y, u, m, scale) else y.addmm_(u, m, alpha=scale)


def _residual(res, x, u, weight, B, scale):
    """res + x W^T + scale * u B^T. The residual joins in the last sum: added
    in the product, it would be rounded at its own size twice."""
    y = x @ weight.t()
    if _ext().lora_add(y, u, B.t(), scale, res):
        return y
    return y.addmm_(u, B.t(), alpha=scale).add_(res)


def _project(x, u, weight, bias, B, scale):
    """x W^T + b + scale * u B^T."""
    y = x @ weight.t() if bias is None else torch.addmm(bias, x, weight.t())
    return _add(y, u, B.t(), scale)


class _Attention(torch.autograd.Function):
    """x + o_proj(attention(qkv_proj(norm(x)))) over rows x (rows, hidden)."""

    @staticmethod
    def forward(ctx, x, rotary, at, norm, Aq, Bq, Ak, Bk, Av, Bv, Ao, Bo):
        ext, s = _ext(), at.spec
        pos, inv_freq, back_freq, cu, longest = rotary
        h = ext.rmsnorm_fwd(x, norm.weight, norm.eps)
        A = torch.cat([Aq, Ak, Av])
        u = h @ A.t()
        uq, uk, uv = u.split([Aq.shape[0], Ak.shape[0], Av.shape[0]], 1)
        mods = (at.q_proj, at.k_proj, at.v_proj)
        q, k, v = (_project(h, p, m.weight, m.bias, b, m.scale)
                   for m, p, b in zip(mods, (uq, uk, uv), (Bq, Bk, Bv)))
        q = q.view(-1, s.num_heads, s.head_dim)
        k = k.view(-1, s.num_kv_heads, s.head_dim)
        q0 = k0 = None
        if s.qk_norm:
            q0, k0 = q, k
            q = ext.rmsnorm_fwd(q0, at.q_norm.weight, at.q_norm.eps)
            k = ext.rmsnorm_fwd(k0, at.k_norm.weight, at.k_norm.eps)
        ext.rope_inplace(q, k, pos, inv_freq)
        v = v.view(-1, s.num_kv_heads, s.head_dim)
        o, lse = ext.flash_varlen_fwd(q, k, v, cu, longest, at.scale)
        o2 = o.view(-1, s.q_size)
        uo = o2 @ Ao.t()
        y = _residual(x, o2, uo, at.o_proj.weight, Bo, at.o_proj.scale)
        head_norms = ((at.q_norm.weight, at.k_norm.weight) if s.qk_norm
                      else (None, None))
        ctx.save_for_backward(x, h, A, u, Bq, Bk, Bv, Ao, Bo, q, k, v, o, lse,
                              uo, pos, back_freq, cu, q0, k0, *head_norms,
                              norm.weight, at.o_proj.weight,
                              *(m.weight for m in mods))
        ctx.spec, ctx.longest, ctx.scale = s, longest, at.scale
        ctx.scales = [m.scale for m in (*mods, at.o_proj)]
        ctx.eps = (norm.eps, *((at.q_norm.eps, at.k_norm.eps) if s.qk_norm
                               else ()))
        return y

    @staticmethod
    @once_differentiable
    def backward(ctx, g):
        (x, h, A, u, Bq, Bk, Bv, Ao, Bo, q, k, v, o, lse, uo, pos, back_freq,
         cu, q0, k0, q_norm, k_norm, norm, Wo, *Ws) = ctx.saved_tensors
        ext, s = _ext(), ctx.spec
        *scales, scale_o = ctx.scales
        g = g.contiguous()
        rows = g.shape[0]
        o2 = o.view(rows, s.q_size)

        duo = _scaled_mm(g, Bo, scale_o)
        dAo, dBo = duo.t() @ o2, _scaled_mm(g.t(), uo, scale_o)
        do = _add(g @ Wo, duo, Ao)
        dq, dk, dv = ext.flash_varlen_bwd(do.view_as(o), q, k, v, o, lse, cu,
                                          ctx.longest, ctx.scale)
        # a rotation's gradient is the rotation by the negative angle
        ext.rope_inplace(dq, dk, pos, back_freq)
        if q0 is not None:
            dq = ext.rmsnorm_bwd(dq, q0, q_norm, ctx.eps[1])
            dk = ext.rmsnorm_bwd(dk, k0, k_norm, ctx.eps[2])
        dq, dk, dv = (t.reshape(rows, -1) for t in (dq, dk, dv))

        ranks = [Bq.shape[1], Bk.shape[1], Bv.shape[1]]
        du = g.new_empty(rows, sum(ranks))
        dBs = []
        for d, scale, b, p, part in zip(
                (dq, dk, dv), scales, (Bq, Bk, Bv), u.split(ranks, 1),
                du.split(ranks, 1)):
            _scaled_mm(d, b, scale, out=part)
            dBs.append(_scaled_mm(d.t(), p, scale))
        dAq, dAk, dAv = (du.t() @ h).split(ranks)
        dx = None
        if ctx.needs_input_grad[0]:
            dh = dq @ Ws[0]
            dh.addmm_(dk, Ws[1])
            dh.addmm_(dv, Ws[2])
            _add(dh, du, A)
            dx = ext.rmsnorm_bwd_add(dh, x, norm, g, ctx.eps[0])
        return (dx, None, None, None, dAq, dBs[0], dAk, dBs[1], dAv, dBs[2],
                dAo, dBo)


class _FeedForward(torch.autograd.Function):
    """x + down_proj(silu(gate_proj(norm(x))) * up_proj(norm(x)))."""

    @staticmethod
    def forward(ctx, x, mlp, norm, Ag, Bg, Au, Bu, Ad, Bd):
        ext = _ext()
        h = ext.rmsnorm_fwd(x, norm.weight, norm.eps)
        A = torch.cat([Ag, Au])
        u = h @ A.t()
        ug, uu = u.split([Ag.shape[0], Au.shape[0]], 1)
        gate = _project(h, ug, mlp.gate_proj.weight, mlp.gate_proj.bias, Bg,
                        mlp.gate_proj.scale)
        up = _project(h, uu, mlp.up_proj.weight, mlp.up_proj.bias, Bu,
                      mlp.up_proj.scale)
        act = ext.silu_mul_fwd(gate, up)
        ud = act @ Ad.t()
        y = _residual(x, act, ud, mlp.down_proj.weight, Bd,
                      mlp.down_proj.scale)
        mods = (mlp.gate_proj, mlp.up_proj, mlp.down_proj)
        ctx.save_for_backward(x, h, A, u, Bg, Bu, Ad, Bd, gate, up, act, ud,
                              norm.weight, *(m.weight for m in mods))
        ctx.scales, ctx.eps = [m.scale for m in mods], norm.eps
        return y

    @staticmethod
    @once_differentiable
    def backward(ctx, g):
        (x, h, A, u, Bg, Bu, Ad, Bd, gate, up, act, ud, norm, Wg, Wu,
         Wd) = ctx.saved_tensors
        ext, (scale_g, scale_u, scale_d) = _ext(), ctx.scales
        g = g.contiguous()
        dud = _scaled_mm(g, Bd, scale_d)
        dAd, dBd = dud.t() @ act, _scaled_mm(g.t(), ud, scale_d)
        dact = _add(g @ Wd, dud, Ad)
        dgate, dup = ext.silu_mul_bwd(dact, gate, up)
        ranks = [Bg.shape[1], Bu.shape[1]]
        du = g.new_empty(g.shape[0], sum(ranks))
        (ug, uu), (dug, duu) = u.split(ranks, 1), du.split(ranks, 1)
        _scaled_mm(dgate, Bg, scale_g, out=dug)
        _scaled_mm(dup, Bu, scale_u, out=duu)
        dBg = _scaled_mm(dgate.t(), ug, scale_g)
        dBu = _scaled_mm(dup.t(), uu, scale_u)
        dAg, dAu = (du.t() @ h).split(ranks)
        dx = None
        if ctx.needs_input_grad[0]:
            dh = dgate @ Wg
            dh.addmm_(dup, Wu)
            _add(dh, du, A)
            dx = ext.rmsnorm_bwd_add(dh, x, norm, g, ctx.eps)
        return dx, None, None, dAg, dBg, dAu, dBu, dAd, dBd


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
