"""Fused decode weights: per-layer merged (base + LoRA) projection tensors.

The decode hot loop must not pay 14 adapter GEMMs + 7 base GEMMs per layer
(measured ~10 ms/step at batch 160 on Qwen2.5-7B). LoRA only changes
between rounds, so the engine folds it once per weight-sync:

    W_eff = W_base + scale * (B @ A)

and lays the projections of a site (q|k|v, gate|up) out as one matrix, in the
tiles that the decode products read (ops/csrc/skinny_gemm.hip up to 16 rows,
stream_gemm.hip up to 160); row-major beside them only for what still goes to
the library: larger steps, and prompts whose operands our products don't take. A refresh
writes the projections' merged weights straight into their tiles, one kernel a
layer, once per generation round.

Replaces the reference's per-generate adapter hot-swap into vLLM
(``load_lora`` inside every fast_generate, reference
distributed_actor.py:148-150) — there the engine applies LoRA at runtime
per token; here the fold happens once per round, which 288 GB of HBM
makes free to cache.
"""

from __future__ import annotations

from typing import List

import torch


class LayerWeights:
    """One layer's decode weights, by site: qkv, o, gateup, down.

    ``tiles[site]``: the merged weight in the tiles that the decode products
    read (ops/csrc/stream_gemm.hip); ``tiles`` is None where the sizes do not
    tile.
    ``rows(site)``: the same row-major, for the library's products; laid out
    when first asked for and kept current by every later refresh, or for every
    call alone where there is no room beside the tiles. One weight without an
    adapter is the module's own; ``rows("base")`` is the down site's whatever
    its adapter."""

    __slots__ = ("layer", "tiles", "_rows", "_own", "_passing", "down_apart", "qkv_b", "in_norm", "post_norm",
                 # nf4 fragment packs (base, built once) + adapter fragment
                 # packs (rebuilt per refresh) for the fused nf4 GEMM path
                 "qkv_w4", "qkv_amax", "o_w4", "o_amax",
                 "gateup_w4", "gateup_amax", "down_w4", "down_amax",
                 "qkv_afrag", "qkv_bfrag", "o_afrag", "o_bfrag",
                 "gateup_afrag", "gateup_bfrag", "down_afrag", "down_bfrag",
                 "qkv_r", "o_r", "gateup_r", "down_r",
                 # the 4-bit down site beside its bf16 base image: the adapter
                 # (rank padded, scale folded into B), A as rows or in tiles,
                 # B as (hidden, r) and (r, hidden)
                 "down_a", "down_b", "down_bt")

    def __init__(self, layer):
        self.layer = layer
        self.tiles, self._rows = None, {}
        self._own = set()           # sites of one weight that is copied
        self._passing = set()       # sites without room, until the next refresh
        self.down_apart = False     # tiles["down"] without its adapter

    @property
    def mods(self):
        at, mlp = self.layer.self_attn, self.layer.mlp
        return {"qkv": (at.q_proj, at.k_proj, at.v_proj), "o": (at.o_proj,),
                "gateup": (mlp.gate_proj, mlp.up_proj),
                "down": (mlp.down_proj,)}

    def rows(self, site: str) -> torch.Tensor:
        if site not in self._rows and self._no_room(site):
            self._passing.add(site)     # a capture does as its warm-up did
            return _untiled(self.tiles[site], site == "gateup")
        if site not in self._rows:
            self._rows[site] = None
            self._fill_rows(site)
        return self._rows[site]

    def _no_room(self, site: str) -> bool:
        """Whether rows(site) must do without storage of its own: what was free
        when the engine was made may be a learner's by the first large step."""
        if site in self._passing:
            return True
        if (self.tiles is None or site == "base" or site == "down" and self.down_apart
                or len(self.mods[site]) == 1 and self.mods[site][0].r == 0):
            return False
        tiles = self.tiles[site]
        return not _room_for(tiles.numel() * tiles.element_size(), tiles.device)

    def refresh_rows(self) -> bool:
        """Whether rows lie elsewhere now: steps captured before are stale."""
        self._passing.clear()
        return any([self._fill_rows(site) for site in self._rows])

    def _fill_rows(self, site: str) -> bool:
        mods, out = self.mods["down" if site == "base" else site], self._rows[site]
        if site == "base" or len(mods) == 1 and mods[0].r == 0:
            return self._follow(site, mods[0].weight.detach())
        if out is None:
            out = self._rows[site] = mods[0].weight.new_empty(
                sum(m.out_features for m in mods), mods[0].in_features)
        # IN PLACE: captured decode steps hold these storages
        if self.tiles is not None and not (site == "down" and self.down_apart):
            out.copy_(_untiled(self.tiles[site], site == "gateup"))
            return False
        for m, rows in zip(mods, out.split([m.out_features for m in mods])):
            _merge_into(m, rows)
        return False

    def _follow(self, site: str, w: torch.Tensor) -> bool:
        """rows(site) <- the weight w itself, or what it holds."""
        out = self._rows[site]
        if site in self._own:
            out.copy_(w)
            return False
        if out is not None and out.data_ptr() == w.data_ptr() and w.is_contiguous():
            return False
        # first, or replaced: what was here before is the caller's, not written
        if not w.is_contiguous() or out is not None and out.dtype != w.dtype:
            self._own.add(site)
            w = w.to(w.dtype if out is None else out.dtype, copy=True,
                     memory_format=torch.contiguous_format)
        if out is None:
            self._rows[site] = w
            return False
        out.set_(w)
        return True


def _tiled(w: torch.Tensor, glu: bool = False) -> torch.Tensor:
    """(N, K) row-major -> tiles of 32 rows x 16 of K, [K half][row][8
    elements]; glu: [gate; up] as 16 gate and 16 up rows a tile."""
    N, K = w.shape
    if glu:
        w = w.view(2, N // 32, 16, K).transpose(0, 1)
    return w.reshape(N // 32, 32, K // 16, 2, 8).permute(0, 2, 3, 1, 4) \
        .reshape(N, K)


def _untiled(t: torch.Tensor, glu: bool = False) -> torch.Tensor:
    N, K = t.shape
    w = t.view(N // 32, K // 16, 2, 32, 8).permute(0, 3, 1, 2, 4)
    if glu:
        w = w.reshape(N // 32, 2, 16, K).transpose(0, 1)
    return w.reshape(N, K)


def _effective(mod) -> torch.Tensor:
    w = mod.weight
    if mod.r > 0:
        w = w + (mod.lora_B.to(torch.float32) @ mod.lora_A.to(torch.float32)
                 ).to(w.dtype) * mod.scale
    return w


def _merge_into(mod, out: torch.Tensor) -> None:
    """out <- the module's effective weight."""
    if mod.r > 0 and out.is_cuda and out.dtype == torch.bfloat16 \
            and mod.lora_A.dtype == out.dtype == mod.weight.dtype:
        from ..ops.functional import _require_ext
        if _require_ext("lora_merge").lora_merge(
                mod.weight.detach(), mod.lora_A.detach(),
                mod.lora_B.detach(), out, float(mod.scale)):
            return
    out.copy_(_effective(mod))


def _tile_jobs(mods, out: torch.Tensor, glu: bool, adapters: bool):
    """What brings the modules' weights, one below the other (glu: a SiLU*mul
    pair), with their adapters or without, into out's tiles."""
    row = 0
    for m in mods:
        a, b = ((m.lora_A.detach(), m.lora_B.detach())
                if adapters and m.r > 0 else (None, None))
        yield m.weight.detach(), out, row, glu, a, b, float(m.scale)
        row += 16 if glu else m.out_features


def _merge_tiles(sites) -> None:
    """Of each site (modules, out, glu, adapters): out, in tiles <- its weights."""
    from ..ops.functional import _require_ext
    ext = _require_ext("decode weights")

    def native(sites) -> bool:
        jobs = [job for site in sites for job in _tile_jobs(*site)]
        types = {t.dtype for w, _, _, _, a, b, _ in jobs
                 for t in (w, a, b) if t is not None}
        return types == {torch.bfloat16} and ext.weights_tiles(*map(list, zip(*jobs)))

    if native(sites):
        return
    for site in sites:
        if not native([site]):
            mods, out, glu, adapters = site
            out.copy_(_tiled(torch.cat(
                [_effective(m) if adapters else m.weight for m in mods]), glu))


def _room_for(size: int, device) -> bool:
    """Whether so many bytes can be allocated, a twentieth of the card left."""
    free, total = torch.cuda.mem_get_info(device)
    free += torch.cuda.memory_reserved(device) - torch.cuda.memory_allocated(device)
    return size <= free - total // 20


class FusedWeights:
    def __init__(self, model, use_nf4: bool = True):
        self.model = model
        self.layers: List[LayerWeights] = []
        self._built = False
        # nf4 fused-GEMM decode path: available when the model carries the
        # packed nf4 sidecars (load_in_4bit) and the kernels are built
        q0 = model.model.layers[0].self_attn.q_proj
        s = model.spec
        shapes_ok = (
            (s.q_size + 2 * s.kv_size) % 256 == 0
            and s.hidden_size % 256 == 0
            and (2 * s.intermediate_size) % 256 == 0
            and s.hidden_size % 64 == 0 and s.q_size % 64 == 0
            and s.intermediate_size % 64 == 0)
        # Both decode paths compute exactly nf4(W_base) + B@A: the merged
        # path pre-dequantizes that image into resident bf16 (288 GB HBM
        # makes the cache free) and currently measures faster at decode
        # batch sizes (10.8 vs 14.5 ms/step at batch 160); the fused nf4
        # GEMM path streams 4.3x fewer weight bytes and is selected with
        # DISTRL_DECODE_NF4=1 (kept fully tested).
        import os
        freed = (q0.weight_nf4 is not None and q0.weight.numel() == 0)
        env = os.environ.get("DISTRL_DECODE_NF4")
        if freed:
            # the bf16 base image was dropped (free_base_to_nf4_, big
            # models) — there is nothing to merge, the fused nf4 path is
            # the only decode path
            want_nf4 = True
        elif env is not None:
            want_nf4 = use_nf4 and env == "1"
        else:
            # default: merged cache for models whose bf16 copy is cheap;
            # fused nf4 path for very large models (e.g. 32B: a second
            # 65 GB merged copy is not worth the HBM)
            n_params = sum(p.numel() for p in model.parameters())
            want_nf4 = use_nf4 and n_params > 16e9
        self.nf4 = bool(want_nf4 and q0.weight_nf4 is not None
                        and q0.weight.is_cuda and shapes_ok)
        if freed and not self.nf4:
            raise RuntimeError(
                "base image freed but the fused nf4 decode path is "
                "unavailable for this shape — cannot fall back to merged")
        # hybrid: even when the merged-bf16 cache wins overall, the fused
        # nf4 kernel BEATS hipBLASLt on the deep-K down-projection
        # (61+13 vs 80 us/layer at decode batch 160) — steps that the
        # products on tiles do not take run just that site through it
        self.hybrid_down = bool(
            (not self.nf4) and q0.weight_nf4 is not None
            and q0.weight.is_cuda and shapes_ok
            and os.environ.get("DISTRL_HYBRID_DOWN", "1") == "1")
        self.lora_r = q0.r
        self.moves = 0      # refreshes after which captured steps are stale
        # the decode products read weights in tiles, where the tiles and the
        # row-major weights that prompts and larger steps read fit beside the
        # model (a 70B model without an adapter keeps row-major ones alone)
        self.tiled = bool(
            not self.nf4 and q0.weight.is_cuda
            and q0.weight.dtype == torch.bfloat16 and s.hidden_size % 64 == 0
            and s.q_size % 64 == 0 and s.kv_size % 32 == 0
            and s.intermediate_size % 64 == 0
            and _room_for(2 * s.num_layers * 2 * s.hidden_size * (
                2 * s.q_size + 2 * s.kv_size + 3 * s.intermediate_size),
                q0.weight.device))
        # whether the last-level cache (256 MB) holds the tiles from one step to
        # the next: steps of few rows then read them through it (one row, 96
        # tokens, ms, through and past the caches: 183 MB of layers 61.5 and
        # 63.1, 212 MB 35.0 and 35.5, 239 MB 28.7 and 28.4; 74.3 and 74.3)
        self.kept = 2 * s.num_layers * s.hidden_size * (
            2 * s.q_size + 2 * s.kv_size + 3 * s.intermediate_size) < 224e6
        # the 4-bit kernel's packs of the down site: only steps beyond the
        # streamed products' rows use them
        self._nf4_down = False

    @staticmethod
    def _nf4_cat(mods):
        """Concatenate the flat nf4 packs / absmax of modules along N
        (rows are K-contiguous, so flat concatenation is row concat)."""
        packed = torch.cat([m.weight_nf4 for m in mods])
        absmax = torch.cat([m.weight_absmax for m in mods])
        N = sum(m.out_features for m in mods)
        K = mods[0].in_features
        return packed, absmax, N, K

    def _build_nf4_base(self, lw: "LayerWeights", layer):
        from ..models.quant import prepack_nf4_fragments
        at, mlp = layer.self_attn, layer.mlp
        for name, mods in (("qkv", [at.q_proj, at.k_proj, at.v_proj]),
                           ("o", [at.o_proj]),
                           ("gateup", [mlp.gate_proj, mlp.up_proj]),
                           ("down", [mlp.down_proj])):
            packed, absmax, N, K = self._nf4_cat(mods)
            w4f, amaxf = prepack_nf4_fragments(packed, absmax, N, K)
            setattr(lw, f"{name}_w4", w4f)
            setattr(lw, f"{name}_amax", amaxf)

    def _refresh_nf4_adapters(self, lw: "LayerWeights", layer, sites=None):
        """Per-round: stack the A matrices and build the block-diagonal,
        scale-folded B matrix per fused site, prepacked into fragments."""
        if self.lora_r == 0:
            return
        from ..models.quant import prepack_bf16_fragments
        at, mlp = layer.self_attn, layer.mlp
        for name, mods in (("qkv", [at.q_proj, at.k_proj, at.v_proj]),
                           ("o", [at.o_proj]),
                           ("gateup", [mlp.gate_proj, mlp.up_proj]),
                           ("down", [mlp.down_proj])):
            if sites is not None and name not in sites:
                continue
            A = torch.cat([m.lora_A.detach() for m in mods], dim=0)  # (r_tot, K)
            r_tot = A.shape[0]
            r_pad = (r_tot + 31) // 32 * 32  # kernel needs rank % 32 == 0
            N = sum(m.out_features for m in mods)
            if r_pad != r_tot:
                A = torch.cat([A, A.new_zeros(r_pad - r_tot, A.shape[1])], 0)
            B = A.new_zeros(N, r_pad)
            n0, r0 = 0, 0
            for m in mods:
                B[n0:n0 + m.out_features, r0:r0 + m.r] = (
                    m.lora_B.detach() * m.scale)
                n0 += m.out_features
                r0 += m.r
            # IN-PLACE refresh: decode sessions capture hipGraphs that
            # reference these tensors, and the graph cache reuses those
            # graphs across generation rounds — a fresh allocation here
            # would leave every cached graph reading freed memory (at
            # single-size waves the allocator happens to hand the same
            # block back, which HID this; multi-wave rounds surfaced it
            # as NaN logits -> the sampler degenerating to token 0)
            af = prepack_bf16_fragments(A.to(torch.bfloat16))
            bf = prepack_bf16_fragments(B.to(torch.bfloat16))
            try:
                old_af = getattr(lw, f"{name}_afrag")
                old_bf = getattr(lw, f"{name}_bfrag")
            except AttributeError:
                old_af = old_bf = None
            if (old_af is not None and old_af.shape == af.shape
                    and old_bf.shape == bf.shape):
                old_af.copy_(af)
                old_bf.copy_(bf)
            else:
                setattr(lw, f"{name}_afrag", af)
                setattr(lw, f"{name}_bfrag", bf)
            setattr(lw, f"{name}_r", r_pad)

    def ensure_nf4_down(self):
        """The 4-bit kernel's packs of the down site, built when a step first
        needs them; every later refresh renews the adapter's."""
        if self._nf4_down:
            return
        from ..models.quant import prepack_nf4_fragments
        for layer, lw in zip(self.model.model.layers, self.layers):
            packed, absmax, N, K = self._nf4_cat([layer.mlp.down_proj])
            lw.down_w4, lw.down_amax = prepack_nf4_fragments(packed, absmax,
                                                             N, K)
            self._refresh_nf4_adapters(lw, layer, sites=("down",))
        self._nf4_down = True

    def _refresh_down_adapter(self, lw: "LayerWeights"):
        """The 4-bit down site's adapter beside the bf16 base image."""
        m, = lw.mods["down"]
        r_pad = (m.r + 31) // 32 * 32
        A = m.lora_A.detach().to(torch.bfloat16)
        B = (m.lora_B.detach() * m.scale).to(torch.bfloat16)
        if r_pad != m.r:
            A = torch.cat([A, A.new_zeros(r_pad - m.r, A.shape[1])])
            B = torch.cat([B, B.new_zeros(B.shape[0], r_pad - m.r)], 1)
        new = {"down_a": _tiled(A) if self.tiled else A, "down_b": B,
               "down_bt": B.t()}
        for name, t in new.items():
            # IN PLACE: captured decode steps hold these storages
            if hasattr(lw, name):
                getattr(lw, name).copy_(t)
            else:
                setattr(lw, name, t.contiguous().clone())

    @torch.no_grad()
    def refresh(self):
        """(Re)build the merged decode weights from the current base + LoRA
        tensors. Called once per weight sync, never inside the decode loop.

        nf4 mode: the quantized base fragments are built ONCE (frozen);
        only the adapter fragment packs (A stacks, block-diagonal scaled B)
        are rebuilt per refresh — the adapter stays exact bf16.
        """
        first, moved = not self._built, False
        for li, layer in enumerate(self.model.model.layers):
            at = layer.self_attn
            if first:
                lw = LayerWeights(layer)
                if at.q_proj.bias is not None:
                    lw.qkv_b = torch.cat([at.q_proj.bias, at.k_proj.bias,
                                          at.v_proj.bias]).contiguous()
                else:
                    lw.qkv_b = None
                lw.in_norm = layer.input_layernorm.weight
                lw.post_norm = layer.post_attention_layernorm.weight
                self.layers.append(lw)
            else:
                lw = self.layers[li]
                lw.layer = layer        # may be another one since
                if lw.qkv_b is not None:
                    torch.cat([at.q_proj.bias, at.k_proj.bias,
                               at.v_proj.bias], out=lw.qkv_b)
            if self.nf4:
                if first:
                    self._build_nf4_base(lw, layer)
                self._refresh_nf4_adapters(lw, layer)
                continue
            if self.tiled:
                self._refresh_tiles(lw)
            moved |= lw.refresh_rows()
            if self.hybrid_down:
                if self.lora_r > 0:
                    self._refresh_down_adapter(lw)
                if self._nf4_down:
                    self._refresh_nf4_adapters(lw, layer, sites=("down",))
        self.moves += moved
        self._built = True

    def _refresh_tiles(self, lw: "LayerWeights"):
        if lw.tiles is None:
            lw.tiles = {
                site: mods[0].weight.new_empty(
                    sum(m.out_features for m in mods), mods[0].in_features)
                for site, mods in lw.mods.items()}
            lw.down_apart = self.hybrid_down and self.lora_r > 0
        # IN PLACE: captured decode steps hold these storages
        _merge_tiles([(mods, lw.tiles[site], site == "gateup",
                       not (site == "down" and lw.down_apart))
                      for site, mods in lw.mods.items()])
