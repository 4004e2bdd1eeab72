"""A decoder layer's two halves as single autograd nodes (GPU, bf16, LoRA
training): attention and feed-forward, each with its norm, its projections
with their adapters and its residual sum, backward written out.

The module-by-module layer launches ~200 kernels forward and backward, most
of them elementwise passes between the products (residual adds, adapter
scaling, gradient sums of projections that share an input, rotary steps,
head transposes), and short micro-batches are bound by launching them. Here
an adapter is more of its projection: u = scale * x A^T lies beside x in one
matrix, [x | u], and one product with [W | B] gives every projection of that
input, adapters and (beta = 1) the residual in its fp32 sums; backward is
[dY | du] [W; A]. Laying W out beside its adapter costs a copy of the weights,
37 us a layer of the 1.5B model forward and as long backward, where adding the
adapters' outputs to 18800 rows in passes of their own took 750. Adapter
gradients are one launch and its sum (ops/csrc/adapter_grads.hip). Rotary, norm
and activation passes are one kernel each: ~38 launches.
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


def _scaled_mm(a, b, scale, out=None):
    """scale * a @ b, the scale in the product's epilogue."""
    if out is None:
        out = a.new_empty(a.shape[0], b.shape[1])
    return torch.addmm(out, a, b, beta=0.0, alpha=scale, out=out)


def _padded(ranks) -> int:
    """Columns that adapters of such ranks get beside their input."""
    return (sum(ranks) + 7) // 8 * 8


def _beside(x, width: int):
    """A matrix of x's rows, `width` columns and some more; its two parts."""
    return x, x[:, :width], x[:, width:]


def _down(x, u, As, scales) -> None:
    """u <- the adapters' scaled inputs side by side, zeros in spare columns."""
    ranks = [a.shape[0] for a in As]
    A = torch.cat(As) if len(As) > 1 else As[0]
    if len(set(scales)) == 1:
        _scaled_mm(x, A.t(), scales[0], out=u[:, :sum(ranks)])
    else:
        for a, part, scale in zip(As, u[:, :sum(ranks)].split(ranks, 1), scales):
            _scaled_mm(x, a.t(), scale, out=part)
    if u.shape[1] > sum(ranks):
        u[:, sum(ranks):].zero_()


def _product(xu, W, mods):
    """xu W^T + the modules' biases."""
    if all(m.bias is None for m in mods):
        return xu @ W.t()
    return torch.addmm(torch.cat([
        m.bias if m.bias is not None else xu.new_zeros(m.out_features)
        for m in mods]), xu, W.t())


def _up(dys, us, Bs, scales) -> None:
    """us <- the gradients of the adapters' inputs."""
    for dy, u, b, scale in zip(dys, us, Bs, scales):
        _scaled_mm(dy, b, scale, out=u)


def _through(g, W, A, B, scale):
    """g W + du A with du = scale * g B, from one product of [g | du]; g and du
    as parts of that matrix."""
    (rows, N), r = g.shape, A.shape[0]
    pad = _padded([r])
    gd, g2, du = _beside(g.new_empty(rows, N + pad), N)
    g2.copy_(g)
    _scaled_mm(g, B, scale, out=du[:, :r])
    if pad > r:
        du[:, r:].zero_()
    return (gd @ _ext().stack_transposed([W, A], [0, N], N + pad).t(), g2,
            du[:, :r])


def _sums(jobs):
    """p^T y of every (y, p, transposed) over the rows: gradients of A, or of B
    (transposed). Ranks that the kernel does not take go through the library."""
    own = [i for i, (y, p, _) in enumerate(jobs)
           if p.shape[1] % 8 == 0 and 8 <= p.shape[1] <= 128
           and y.shape[1] % 8 == 0 and p.shape[0] > 0]
    out = [None] * len(jobs)
    if own:
        got = _ext().adapter_grads(*map(list, zip(*(jobs[i] for i in own))))
        for i, g in zip(own, got):
            out[i] = g
    for i, (y, p, transposed) in enumerate(jobs):
        if out[i] is None:
            out[i] = y.t() @ p if transposed else p.t() @ y
    return out


class _Attention(torch.autograd.Function):
    """x + o_proj(attention(qkv_proj(norm(x)))) over rows x (rows, hidden)."""

    @staticmethod
    def forward(ctx, x, rotary, at, norm, Aq, Bq, Ak, Bk, Av, Bv, Ao, Bo):
        ext, s = _ext(), at.spec
        pos, inv_freq, back_freq, cu, longest = rotary
        rows, hidden = x.shape
        mods = (at.q_proj, at.k_proj, at.v_proj)
        scales = [m.scale for m in (*mods, at.o_proj)]
        As, Bs, Ws = [Aq, Ak, Av], [Bq, Bk, Bv], [m.weight for m in mods]
        pad = _padded([a.shape[0] for a in As])
        hu, h, u = _beside(x.new_empty(rows, hidden + pad), hidden)
        ext.rmsnorm_fwd_into(x, norm.weight, norm.eps, h)
        _down(h, u, As, scales[:3])
        W = ext.adapted_weight(Ws, Bs, pad)
        qkv = _product(hu, W, mods)
        q, k, v = (t.unflatten(1, (-1, s.head_dim))
                   for t in qkv.split([s.q_size, s.kv_size, s.kv_size], 1))
        q0 = k0 = None
        if s.qk_norm:
            q0, k0 = q.contiguous(), k.contiguous()
            q = ext.rmsnorm_fwd(q0, at.q_norm.weight, at.q_norm.eps)
            k = ext.rmsnorm_fwd(k0, at.k_norm.weight, at.k_norm.eps)
        ext.rope_rows(q, k, pos, inv_freq)
        pad_o = _padded([Ao.shape[0]])
        ou, o, uo = _beside(x.new_empty(rows, s.q_size + pad_o), s.q_size)
        lse = ext.flash_varlen_fwd(q, k, v, cu, longest, at.scale,
                                   o.unflatten(1, (-1, s.head_dim)))[1]
        _down(o, uo, [Ao], scales[3:])
        Wo = at.o_proj.weight
        # the residual joins the product's sum: one rounding for all of it
        y = torch.addmm(x, ou, ext.adapted_weight([Wo], [Bo], pad_o).t())
        head_norms = ((at.q_norm.weight, at.k_norm.weight) if s.qk_norm
                      else (None, None))
        ctx.save_for_backward(x, hu, ou, q, k, v, lse, pos, back_freq, cu, q0,
                              k0, *head_norms, norm.weight, Ao, Bo, Wo,
                              *As, *Bs, *Ws)
        ctx.spec, ctx.longest, ctx.scale = s, longest, at.scale
        ctx.scales = scales
        ctx.eps = (norm.eps, *((at.q_norm.eps, at.k_norm.eps) if s.qk_norm
                               else ()))
        return y

    @staticmethod
    @once_differentiable
    def backward(ctx, g):
        (x, hu, ou, q, k, v, lse, pos, back_freq, cu, q0, k0, q_norm, k_norm,
         norm, Ao, Bo, Wo, *rest) = ctx.saved_tensors
        As, Bs, Ws = rest[:3], rest[3:6], rest[6:]
        ext, s = _ext(), ctx.spec
        *scales, scale_o = ctx.scales
        g = g.contiguous()
        rows, hidden = x.shape
        _, h, u = _beside(hu, hidden)
        _, o2, uo = _beside(ou, s.q_size)
        o = o2.unflatten(1, (-1, s.head_dim))

        do, g2, duo = _through(g, Wo, Ao, Bo, scale_o)
        do = do.view(rows, -1, s.head_dim)
        sizes, ranks = [s.q_size, s.kv_size, s.kv_size], [a.shape[0] for a in As]
        pad, width = _padded(ranks), sum(sizes)
        dyu, dy, du = _beside(x.new_empty(rows, width + pad), width)
        dys, dus = dy.split(sizes, 1), du[:, :sum(ranks)].split(ranks, 1)
        dq, dk, dv = (t.unflatten(1, (-1, s.head_dim)) for t in dys)
        ext.flash_varlen_bwd(do, q, k, v, o, lse, cu, ctx.longest, ctx.scale,
                             dq, dk, dv)
        # a rotation's gradient is the rotation by the negative angle
        ext.rope_rows(dq, dk, pos, back_freq)
        if q0 is not None:
            dq.copy_(ext.rmsnorm_bwd(dq.contiguous(), q0, q_norm, ctx.eps[1]))
            dk.copy_(ext.rmsnorm_bwd(dk.contiguous(), k0, k_norm, ctx.eps[2]))
        _up(dys, dus, Bs, scales)
        if pad > sum(ranks):
            du[:, sum(ranks):].zero_()
        us = u[:, :sum(ranks)].split(ranks, 1)
        dA, dAo, dBo, *dBs = _sums(
            [(h, du, False), (o2, duo, False), (g2, uo[:, :Ao.shape[0]], True),
             *((y, p, True) for y, p in zip(dys, us))])
        dAs = dA[:sum(ranks)].split(ranks)
        dx = None
        if ctx.needs_input_grad[0]:
            at = [sum(sizes[:i]) for i in range(3)]
            at += [width + sum(ranks[:i]) for i in range(3)]
            dh = dyu @ ext.stack_transposed([*Ws, *As], at, width + pad).t()
            dx = ext.rmsnorm_bwd_add(dh, x, norm, g, ctx.eps[0])
        return (dx, None, None, None, dAs[0], dBs[0], dAs[1], dBs[1], dAs[2],
                dBs[2], dAo, dBo)


class _FeedForward(torch.autograd.Function):
    """x + down_proj(silu(gate_proj(norm(x))) * up_proj(norm(x)))."""

    @staticmethod
    def forward(ctx, x, mlp, norm, Ag, Bg, Au, Bu, Ad, Bd):
        ext = _ext()
        rows, hidden = x.shape
        mods = (mlp.gate_proj, mlp.up_proj)
        scales = [m.scale for m in (*mods, mlp.down_proj)]
        As, Bs, Ws = [Ag, Au], [Bg, Bu], [m.weight for m in mods]
        pad = _padded([a.shape[0] for a in As])
        hu, h, u = _beside(x.new_empty(rows, hidden + pad), hidden)
        ext.rmsnorm_fwd_into(x, norm.weight, norm.eps, h)
        _down(h, u, As, scales[:2])
        W = ext.adapted_weight(Ws, Bs, pad)
        gu = _product(hu, W, mods)
        pad_d, inner = _padded([Ad.shape[0]]), gu.shape[1] // 2
        au, act, ud = _beside(x.new_empty(rows, inner + pad_d), inner)
        ext.silu_mul_packed_into(gu, act)
        _down(act, ud, [Ad], scales[2:])
        Wd = mlp.down_proj.weight
        y = torch.addmm(x, au, ext.adapted_weight([Wd], [Bd], pad_d).t())
        ctx.save_for_backward(x, hu, gu, au, norm.weight, Ad, Bd, Wd, *As, *Bs,
                              *Ws)
        ctx.scales, ctx.eps = scales, norm.eps
        return y

    @staticmethod
    @once_differentiable
    def backward(ctx, g):
        x, hu, gu, au, norm, Ad, Bd, Wd, *rest = ctx.saved_tensors
        As, Bs, Ws = rest[:2], rest[2:4], rest[4:]
        ext, (*scales, scale_d) = _ext(), ctx.scales
        rows, hidden = x.shape
        inner, ranks = gu.shape[1] // 2, [a.shape[0] for a in As]
        _, h, u = _beside(hu, hidden)
        _, act, ud = _beside(au, inner)

        g = g.contiguous()
        dact, g2, dud = _through(g, Wd, Ad, Bd, scale_d)
        # [dgate | du | dup]
        pad = _padded(ranks)
        dyu = x.new_empty(rows, 2 * inner + pad)
        dgate, du, dup = dyu.split([inner, pad, inner], 1)
        ext.silu_mul_bwd_packed(dact, gu, dgate, dup)
        dus = du[:, :sum(ranks)].split(ranks, 1)
        _up((dgate, dup), dus, Bs, scales)
        if pad > sum(ranks):
            du[:, sum(ranks):].zero_()
        us = u[:, :sum(ranks)].split(ranks, 1)
        dA, dAd, dBd, *dBs = _sums(
            [(h, du, False), (act, dud, False), (g2, ud[:, :Ad.shape[0]], True),
             *((y, p, True) for y, p in zip((dgate, dup), us))])
        dAs = dA[:sum(ranks)].split(ranks)
        dx = None
        if ctx.needs_input_grad[0]:
            at = [0, inner, inner + ranks[0], inner + pad]
            W = ext.stack_transposed([Ws[0], *As, Ws[1]], at, 2 * inner + pad)
            half = inner + ranks[0]
            if rows >= 8192 and hidden <= 2048 and half % 8 == 0:
                # few columns from many rows: the library's product of twice
                # the K takes up to three times as long (18793 x 17984 x 1536:
                # 1080 us, in two 790; from 4000 rows or for 2560 columns one
                # is the faster)
                dh = dyu[:, :half] @ W[:, :half].t()
                dh.addmm_(dyu[:, half:], W[:, half:].t())
            else:
                dh = dyu @ W.t()
            dx = ext.rmsnorm_bwd_add(dh, x, norm, g, ctx.eps)
        return dx, None, None, dAs[0], dBs[0], dAs[1], dBs[1], dAd, dBd


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
