"""Row-major decode weights as they follow the model's tensors, on the CPU."""

import pytest
import torch

from distrl_llm_amd.engine import weights
from distrl_llm_amd.models import CausalLM, get_spec


def _model(lora_r=0):
    return CausalLM(get_spec("small-qwen2"), lora_r=lora_r, dtype=torch.float32).random_init(3)


def _rand(like, seed):
    return torch.randn(like.shape, generator=torch.Generator().manual_seed(seed), dtype=like.dtype)


@pytest.mark.parametrize("kind", ["plain", "strided", "other type"])
def test_replaced_weight_is_left_as_it_was(kind):
    """A weight without an adapter replaced by another tensor, and back: the
    rows follow, neither tensor is written, captured steps are given up."""
    model = _model()
    fused = weights.FusedWeights(model)
    fused.refresh()
    lin, lw = model.model.layers[0].self_attn.o_proj, fused.layers[0]
    first = lin.weight.data
    held, kept = lw.rows("o"), first.clone()
    assert fused.moves == 0
    other = _rand(first, 5)
    if kind == "strided":
        other = other.t().contiguous().t()
    elif kind == "other type":
        other = other.double()
    there = other.clone()
    for moves, data in ((1, other), (1 if kind != "plain" else 2, first), (None, other)):
        lin.weight.data = data
        fused.refresh()
        assert lw.rows("o") is held and torch.equal(held, lin.weight.to(held.dtype))
        assert torch.equal(first, kept) and torch.equal(other, there)
        assert moves is None or fused.moves == moves
        fused.refresh()
    if kind != "plain":     # a copy from the first that could not be held on
        other.add_(1.0)
        fused.refresh()
        assert torch.equal(held, other.to(held.dtype))


@pytest.mark.parametrize("lora_r", [0, 8])
def test_rows_without_room_are_laid_out_for_the_call(monkeypatch, lora_r):
    """No storage beside the tiles while the card is full; a capture does as its
    warm-up did; the next refresh looks again."""
    fused = weights.FusedWeights(_model(lora_r))
    fused.refresh()
    lw = fused.layers[0]
    want = {site: torch.cat([weights._effective(m) for m in mods]) for site, mods in lw.mods.items()}
    lw.tiles = {site: weights._tiled(w, site == "gateup") for site, w in want.items()}
    kept = {"qkv", "gateup"} | ({"o", "down"} if lora_r else set())
    for room in (False, True):
        monkeypatch.setattr(weights, "_room_for", lambda size, device: room)
        for site, w in want.items():
            assert torch.equal(lw.rows(site), w)
            assert (site in lw._rows) == (site not in kept)
    fused.refresh()
    for site, w in want.items():
        assert torch.equal(lw.rows(site), w) and site in lw._rows


def test_replaced_layer_is_followed():
    """Weights come from the model's layers as they are at the refresh."""
    model, other = _model(), _model()
    fused = weights.FusedWeights(model)
    fused.refresh()
    lw = fused.layers[0]
    held = {site: lw.rows(site) for site in ("qkv", "o", "gateup", "down")}
    for p in other.parameters():
        p.data = _rand(p, 7)
    model.model.layers[0] = other.model.layers[0]
    fused.refresh()
    for site, rows in held.items():
        assert lw.rows(site) is rows
        assert torch.equal(rows, torch.cat([m.weight for m in lw.mods[site]]))
        assert lw.mods[site][0] in set(model.model.layers[0].modules())
