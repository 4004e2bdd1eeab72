"""The measured work of this framework: one RL round of a dense model, in its
parts and as a whole, at the sizes of the model registry and of ``bench.py``.

A round generates candidates for a batch of prompts (``Engine.generate``:
prompt phase, fan-out, decode steps over paged K/V, sampling) and then trains
the LoRA adapter on them (``Learner.accumulate_gradients``: teacher-forced
forward, fused log-prob loss, backward). The server runs the same generation
for single requests. The kinds of case:

sample    one draw per sequence from the step's logits
attend    one decode step's attention over the paged K/V pool
flash     the learner's causal attention, forward and backward
loss      log-prob loss over the vocabulary, forward and backward
learn     one micro-batch through the learner: loss and adapter gradients
generate  a batch of prompts through the engine: tokens and K/V pages
"""

import math

import numpy as np
import torch
import torch.nn.functional as F

from distrl_llm_amd.config import EngineConfig, SamplingParams
from distrl_llm_amd.engine.engine import Engine
from distrl_llm_amd.models.model import CausalLM
from distrl_llm_amd.models.spec import get_spec
from distrl_llm_amd.ops import functional as OF
from distrl_llm_amd.train.learner import Learner
from distrl_llm_amd.utils.tokenizer import ByteTokenizer

DEVICE = "cuda"
PAGE = 16                    # tokens a K/V page holds (EngineConfig's default)
LORA_R, LORA_ALPHA = 32, 16.0


# ------------------------------------------------------------------ cases

def listed():
    return [
        # a server's request: one sequence, the vocabulary of the small
        # models, plain sampling (the API's defaults)
        {"name": "sample_request", "kind": "sample", "rows": 1, "vocab": 151936,
         "dtype": "bfloat16", "temperature": 1.0, "top_p": 1.0, "top_k": 0},
        # bench.py's decode step: 10 prompts x 16 candidates, its sampling
        {"name": "sample_round", "kind": "sample", "rows": 160, "vocab": 152064,
         "dtype": "bfloat16", "temperature": 1.2, "top_p": 0.95, "top_k": 0},
        # a few chats with long histories on the 0.5B model
        {"name": "attend_chats", "kind": "attend", "prompts": 3, "n": 1, "heads": 14,
         "kv_heads": 2, "dim": 64, "shortest": 911, "longest": 3777},
        # bench.py's decode step in mid-round on the 7B model: candidates
        # share their prompt's pages
        {"name": "attend_round", "kind": "attend", "prompts": 10, "n": 16, "heads": 28,
         "kv_heads": 4, "dim": 128, "shortest": 420, "longest": 1550},
        # a small micro-batch of ragged length on the 0.5B model
        {"name": "flash_short", "kind": "flash", "batch": 2, "heads": 14, "kv_heads": 2,
         "dim": 64, "tokens": 333},
        # bench.py's micro-batch of 16 on the 7B model
        {"name": "flash_round", "kind": "flash", "batch": 16, "heads": 28, "kv_heads": 4,
         "dim": 128, "tokens": 1550},
        # the answers of a micro-batch: 8 samples (the CLI's train_batch_size)
        {"name": "loss_answers", "kind": "loss", "batch": 8, "tokens": 301,
         "vocab": 152064},
        # debugging-scale run: three short samples on the 0.5B model, bf16
        {"name": "learn_short", "kind": "learn", "model": "qwen2.5-0.5b", "four_bit": False,
         "samples": 3, "prompt": 121, "answer": 187},
        # bench.py's micro-batch (16 samples, up to 350 + 1200 tokens) on the
        # 4-bit 1.5B model
        {"name": "learn_round", "kind": "learn", "model": "qwen2.5-1.5b", "four_bit": True,
         "samples": 16, "prompt": 350, "answer": 1200},
        # a server's single completion on the 0.5B model
        {"name": "generate_request", "kind": "generate", "model": "qwen2.5-0.5b",
         "four_bit": False, "lora": False, "prompts": 1, "n": 1, "shortest": 57,
         "longest": 57, "new": 48, "room": 2048, "temperature": 1.0, "top_p": 1.0},
        # the head of bench.py's round: the 4-bit 7B model with its adapter,
        # 10 prompts x 16 candidates
        {"name": "generate_round", "kind": "generate", "model": "qwen2.5-7b",
         "four_bit": True, "lora": True, "prompts": 10, "n": 16, "shortest": 180,
         "longest": 350, "new": 24, "room": 1550, "temperature": 1.2, "top_p": 0.95},
    ]


def _spread(rng, lo, hi):
    """A whole number, even over the logarithm of the range."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


#: (query heads, kv heads, head size) of the registry's models
HEADS = [(14, 2, 64), (12, 2, 128), (28, 4, 128), (40, 8, 128), (32, 8, 128), (64, 8, 128)]
VOCABS = [4096, 32003, 32768, 128256, 151936, 152064]


def draw(rng):
    kind = rng.choice(["sample", "attend", "flash", "loss", "learn", "generate"])
    if kind == "sample":
        return {"kind": kind, "rows": _spread(rng, 1, 320), "vocab": rng.choice(VOCABS),
                "dtype": rng.choice(["bfloat16", "bfloat16", "bfloat16", "float32"]),
                "temperature": round(rng.uniform(0.6, 1.3), 2),
                "top_p": rng.choice([1.0, 0.95, 0.95, 0.8]), "top_k": rng.choice([0, 0, 50])}
    if kind == "attend":
        heads, kv_heads, dim = rng.choice(HEADS)
        n = rng.choice([1, 1, 4, 8, 16])
        longest = _spread(rng, 24, 4000)
        most = 160 * 1550 // (longest * n)      # no more rows than the largest listed case
        return {"kind": kind, "prompts": _spread(rng, 1, max(1, min(32, most))), "n": n,
                "heads": heads, "kv_heads": kv_heads, "dim": dim,
                "shortest": rng.randint(1, longest), "longest": longest}
    if kind == "flash":
        heads, kv_heads, dim = rng.choice(HEADS)
        tokens = _spread(rng, 17, 2048)
        most = 16 * 28 * 1550 ** 2 // (heads * tokens ** 2)
        return {"kind": kind, "batch": _spread(rng, 1, max(1, min(16, most))), "heads": heads,
                "kv_heads": kv_heads, "dim": dim, "tokens": tokens}
    if kind == "loss":
        vocab = rng.choice(VOCABS)
        tokens = _spread(rng, 5, 600)
        most = 8 * 301 * 152064 // (tokens * vocab)
        return {"kind": kind, "batch": _spread(rng, 1, max(1, min(16, most))),
                "tokens": tokens, "vocab": vocab}
    if kind == "learn":
        small = rng.random() < 0.6
        return {"kind": kind, "model": "qwen2.5-0.5b" if small else "qwen2.5-1.5b",
                "four_bit": rng.random() < 0.5, "samples": rng.randint(1, 8),
                "prompt": _spread(rng, 20, 350), "answer": _spread(rng, 30, 700)}
    prompts, n = rng.choice([(1, 1), (5, 1), (3, 4), (4, 8), (2, 16), (19, 1)])
    longest = _spread(rng, 20, 400)
    return {"kind": kind, "model": rng.choice(["qwen2.5-0.5b", "qwen2.5-1.5b", "qwen3-4b"]),
            "four_bit": rng.random() < 0.5, "lora": rng.random() < 0.5,
            "prompts": prompts, "n": n, "shortest": rng.randint(max(4, longest // 2), longest),
            "longest": longest, "new": rng.randint(6, 40), "room": rng.choice([512, 1550, 2048]),
            "temperature": rng.choice([0.0, 0.7, 1.0, 1.2]), "top_p": rng.choice([1.0, 0.95])}


# ---------------------------------------------------------------- weights

def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _normal(g, shape, std=1.0, mean=0.0, dtype=torch.bfloat16):
    return torch.randn(shape, generator=g, device=DEVICE).mul_(std).add_(mean).to(dtype)


PROJECTIONS = ("q", "k", "v", "o", "gate", "up", "down")


def _shape(spec, name):
    h, f = spec.hidden_size, spec.intermediate_size
    return {"q": (spec.q_size, h), "k": (spec.kv_size, h), "v": (spec.kv_size, h),
            "o": (h, spec.q_size), "gate": (f, h), "up": (f, h), "down": (h, f)}[name]


def _layer_weights(spec, g, lora):
    """One layer's tensors by short name, in a fixed order of draws. The sizes
    keep the residual stream and the scores in a trained model's range."""
    w = {}
    for name in PROJECTIONS:
        rows, cols = _shape(spec, name)
        gain = 0.15 if name in ("o", "down") else 1.0
        w[name] = _normal(g, (rows, cols), gain / math.sqrt(cols))
        if spec.qkv_bias and name in ("q", "k", "v"):
            w[name + ".b"] = _normal(g, (rows,), 0.2)
        if lora:
            w[name + ".A"] = _normal(g, (LORA_R, cols), 0.6 / math.sqrt(cols))
            w[name + ".B"] = _normal(g, (rows, LORA_R), 0.3 * gain / math.sqrt(LORA_R))
    w["norm1"] = _normal(g, (spec.hidden_size,), 0.1, 1.0)
    w["norm2"] = _normal(g, (spec.hidden_size,), 0.1, 1.0)
    if spec.qk_norm:
        w["q.norm"] = _normal(g, (spec.head_dim,), 0.1, 1.0)
        w["k.norm"] = _normal(g, (spec.head_dim,), 0.1, 1.0)
    return w


def _outer_weights(spec, g, peaked):
    """(embedding, head or None where tied, final norm). ``peaked``: the head
    answers a token with a fixed successor by a wide margin, so that a
    generation's tokens do not hang on the last bits of its logits."""
    V, h = spec.vocab_size, spec.hidden_size
    embed = _normal(g, (V, h), 1.0 if peaked else 0.05)
    head = None
    if not spec.tie_word_embeddings:
        if peaked:
            head = torch.empty_like(embed)
            head[torch.randperm(V, generator=g, device=DEVICE)] = embed * (2.5 / math.sqrt(h))
        else:
            head = _normal(g, (V, h), 1.5 / math.sqrt(h))
    return embed, head, _normal(g, (h,), 0.1, 1.0)


def _modules(layer):
    at, mlp = layer.self_attn, layer.mlp
    return dict(zip(PROJECTIONS, (at.q_proj, at.k_proj, at.v_proj, at.o_proj,
                                  mlp.gate_proj, mlp.up_proj, mlp.down_proj)))


@torch.no_grad()
def _model(case, seed, lora, peaked):
    spec, g = get_spec(case["model"]), _generator(seed)
    model = CausalLM(spec, lora_r=LORA_R if lora else 0, lora_alpha=LORA_ALPHA,
                     dtype=torch.bfloat16, device=torch.device(DEVICE))
    embed, head, norm = _outer_weights(spec, g, peaked)
    model.model.embed_tokens.weight.copy_(embed)
    if head is not None:
        model.lm_head.weight.copy_(head)
    model.model.norm.weight.copy_(norm)
    for layer in model.model.layers:
        w = _layer_weights(spec, g, lora)
        for name, mod in _modules(layer).items():
            mod.weight.copy_(w[name])
            if mod.bias is not None:
                mod.bias.copy_(w[name + ".b"])
            if lora:
                mod.lora_A.copy_(w[name + ".A"])
                mod.lora_B.copy_(w[name + ".B"])
        layer.input_layernorm.weight.copy_(w["norm1"])
        layer.post_attention_layernorm.weight.copy_(w["norm2"])
        if spec.qk_norm:
            layer.self_attn.q_norm.weight.copy_(w["q.norm"])
            layer.self_attn.k_norm.weight.copy_(w["k.norm"])
    if case["four_bit"]:
        model.quantize_nf4_()
    return model


# ---------------------------------------------------------------- prepare

def _lengths(case, rng, count):
    return [int(v) for v in rng.integers(case["shortest"], case["longest"] + 1, count)]


def _pages(tokens):
    return (tokens + PAGE - 1) // PAGE


def _tables(case, seed):
    """Pages of a decode step's sequences: the n candidates of a prompt share
    the pages its prompt fills, the rest is their own; pages in random order."""
    rng = np.random.default_rng(seed)
    tables, lens = [], []
    for _ in range(case["prompts"]):
        ctx = _lengths(case, rng, case["n"])
        shared = min(min(ctx), int(rng.integers(1, 351))) // PAGE if case["n"] > 1 else 0
        common = [("p", len(lens), i) for i in range(shared)]
        for c in ctx:
            tables.append(common + [("c", len(lens), i) for i in range(shared, _pages(c))])
            lens.append(c)
    names = sorted({p for t in tables for p in t})
    order = rng.permutation(len(names))
    number = {p: int(order[i]) for i, p in enumerate(names)}
    table = np.zeros((len(tables), max(map(len, tables))), np.int32)
    for i, t in enumerate(tables):
        table[i, :len(t)] = [number[p] for p in t]
    return table, np.array(lens, np.int32), len(names)


def _text(rng, tokens):
    """Text of so many tokens (the tokenizer takes two bytes each), a few
    characters far more common than the others, as in worked sums."""
    chars = np.frombuffer(b" 0123=+4x-5(6)789y/.", dtype=np.uint8)
    often = 1.0 / np.arange(1, len(chars) + 1) ** 1.5
    return bytes(rng.choice(chars, 2 * tokens, p=often / often.sum())).decode()


def _samples(case, seed):
    rng = np.random.default_rng(seed)
    problems, answers = [], []
    for i in range(case["samples"]):
        problems.append(_text(rng, int(rng.integers(case["prompt"] // 2, case["prompt"] + 1))))
        # the first answer runs to the limit, as most do in a bench round
        answers.append(_text(rng, case["answer"] if i == 0 else
                             int(rng.integers(case["answer"] // 2, case["answer"] + 1))))
    return problems, answers, [float(v) for v in rng.uniform(0.1, 1.1, case["samples"])]


def _prompts(case, seed):
    rng = np.random.default_rng(seed)
    vocab = get_spec(case["model"]).vocab_size
    return [[int(t) for t in rng.integers(0, vocab, n)]
            for n in _lengths(case, rng, case["prompts"])]


def _pool_pages(case):
    """Pages for the batch at its longest (a full page may end anywhere)."""
    return 4 + case["prompts"] * (_pages(case["longest"])
                                  + case["n"] * (_pages(case["new"]) + 1))


def prepare(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    if kind == "sample":
        # a bulk of unlikely tokens and a few likely ones, differing by row
        B, V = case["rows"], case["vocab"]
        logits = torch.randn((B, V), generator=g, device=DEVICE).mul_(2.0)
        likely = torch.randint(0, V, (B, 40), generator=g, device=DEVICE)
        lift = torch.rand((B, 40), generator=g, device=DEVICE).mul_(16.0)
        logits.scatter_add_(1, likely, lift)
        return {"case": case, "logits": logits.to(getattr(torch, case["dtype"])),
                "seeds": torch.randint(0, 2 ** 31 - 1, (B,), generator=g, device=DEVICE),
                "step": torch.tensor([seed % 1000], device=DEVICE)}
    if kind == "attend":
        table, lens, pages = _tables(case, seed)
        shape = (pages, PAGE, case["kv_heads"], case["dim"])
        return {"case": case, "q": _normal(g, (len(lens), case["heads"], case["dim"]), 1.5),
                "key": _normal(g, shape, 1.2), "value": _normal(g, shape),
                "tables": torch.from_numpy(table).to(DEVICE),
                "lens": torch.from_numpy(lens).to(DEVICE)}
    if kind == "flash":
        B, H, G, T, D = (case[k] for k in ("batch", "heads", "kv_heads", "tokens", "dim"))
        q = _normal(g, (B, H, T, D), 1.5).requires_grad_()
        k = _normal(g, (B, G, T, D), 1.2).requires_grad_()
        v = _normal(g, (B, G, T, D)).requires_grad_()
        return {"case": case, "qkv": (q, k, v), "dout": _normal(g, (B, H, T, D), 0.01)}
    if kind == "loss":
        B, T, V = case["batch"], case["tokens"], case["vocab"]
        logits = _normal(g, (B, T, V), 2.0)
        targets = torch.randint(0, V, (B, T), generator=g, device=DEVICE)
        # the target is likely, as in text that the model wrote itself
        logits.scatter_add_(2, targets.unsqueeze(-1),
                            _normal(g, (B, T, 1), 3.0, 8.0))
        lens = torch.randint(T // 2, T + 1, (B, 1), generator=g, device=DEVICE)
        lens[0] = T
        mask = (torch.arange(T, device=DEVICE).unsqueeze(0) < lens).long()
        rewards = torch.rand((B,), generator=g, device=DEVICE).add_(0.1)
        return {"case": case, "logits": logits.requires_grad_(), "targets": targets,
                "mask": mask, "rewards": rewards}
    if kind == "learn":
        model = _model(case, seed, True, False)
        learner = Learner(model, ByteTokenizer(model.spec.vocab_size), lr=2e-5,
                          max_prompt_tokens=case["prompt"], max_new_tokens=case["answer"],
                          train_batch_size=case["samples"])
        return {"case": case, "learner": learner, "samples": _samples(case, seed)}
    model = _model(case, seed, case["lora"], True)
    prompts = _prompts(case, seed)
    engine = Engine(model, EngineConfig(max_seq_length=case["room"], kv_block_size=PAGE,
                                        num_kv_blocks=_pool_pages(case),
                                        max_num_seqs=256), seed=seed % 1000)
    return {"case": case, "engine": engine, "prompts": prompts,
            "params": SamplingParams(max_tokens=case["new"], n=case["n"],
                                     temperature=case["temperature"], top_p=case["top_p"])}


# -------------------------------------------------------------------- run

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "sample":
        return OF.sample_tokens(state["logits"], case["temperature"], case["top_p"],
                                case["top_k"], seeds=state["seeds"], step=state["step"])
    if kind == "attend":
        return OF.paged_attention_decode(state["q"], state["key"], state["value"],
                                         state["tables"], state["lens"], case["dim"] ** -0.5)
    if kind == "flash":
        q, k, v = state["qkv"]
        out = OF.flash_attention(q, k, v, case["dim"] ** -0.5)
        dq, dk, dv = torch.autograd.grad(out, (q, k, v), state["dout"])
        return {"out": out.detach(), "dq": dq, "dk": dk, "dv": dv}
    if kind == "loss":
        loss = OF.logprob_loss(state["logits"], state["targets"], state["mask"],
                               state["rewards"])
        grad, = torch.autograd.grad(loss, (state["logits"],))
        return {"loss": loss.detach(), "grad": grad}
    if kind == "learn":
        learner = state["learner"]
        loss = learner.accumulate_gradients(*state["samples"])
        # one flat buffer per matrix, as the learners' all-reduce takes them
        grads = [p.grad.reshape(-1) for p in learner.params]
        return {"loss": loss, "A": torch.cat(grads[0::2]), "B": torch.cat(grads[1::2])}
    engine = state["engine"]
    # every request is done: the next call gets the pool's pages in the same order
    engine.pool.allocator.reset()
    tokens = engine.generate(state["prompts"], state["params"])
    return {"tokens": np.array(tokens), "key": engine.pool.key, "value": engine.pool.value}


# ------------------------------------------------------- work, tolerances

def _params(spec, four_bit, lora):
    """(parameters in projections, bytes of them, bytes of the head)."""
    n = spec.num_layers * sum(math.prod(_shape(spec, p)) for p in PROJECTIONS)
    extra = (spec.num_layers * LORA_R * sum(sum(_shape(spec, p)) for p in PROJECTIONS)
             if lora else 0)
    # 4-bit: half a byte and a 32-bit scale per 64 weights
    return n, (n // 2 + n // 16 if four_bit else 2 * n) + 2 * extra, \
        2 * spec.vocab_size * spec.hidden_size


def work(case):
    kind = case["kind"]
    if kind == "sample":
        n = case["rows"] * case["vocab"]
        return {"bytes": n * (4 if case["dtype"] == "float32" else 2), "flops": 4 * n}
    if kind == "attend":
        _, lens, pages = _tables(case, 0)
        # shared pages once; q and the output beside them
        row = case["kv_heads"] * case["dim"] * 2 * 2
        return {"bytes": pages * PAGE * row + 4 * len(lens) * case["heads"] * case["dim"],
                "flops": 4 * int(lens.sum()) * case["heads"] * case["dim"]}
    if kind == "flash":
        B, H, G, T, D = (case[k] for k in ("batch", "heads", "kv_heads", "tokens", "dim"))
        # q, out, dout, dq and k, v, dk, dv; two products forward, five backward
        return {"bytes": 2 * B * T * D * (4 * H + 4 * G),
                "flops": 7 * 2 * B * H * D * T * (T + 1) // 2}
    if kind == "loss":
        n = case["batch"] * case["tokens"] * case["vocab"]
        return {"bytes": 4 * n, "flops": 8 * n}
    spec = get_spec(case["model"])
    attend = 4 * spec.num_layers * spec.q_size
    if kind == "learn":
        n, size, head = _params(spec, case["four_bit"], True)
        problems, answers, _ = _samples(case, 0)
        lens = [(len(p) + len(a)) // 2 for p, a in zip(problems, answers)]
        rows = sum(len(a) // 2 for a in answers)
        # forward and input gradients: twice the forward's products; the
        # attention's backward is two and a half of its forward
        return {"bytes": 2 * size + 2 * head + 4 * spec.num_layers * LORA_R
                * sum(sum(_shape(spec, p)) for p in PROJECTIONS),
                "flops": 4 * n * sum(lens) + 2 * head * rows
                + int(3.5 * attend * sum(t * (t + 1) // 2 for t in lens))}
    n, size, head = _params(spec, case["four_bit"], case["lora"])
    lens = [len(p) for p in _prompts(case, 0)]
    steps, rows = case["new"] - 1, case["prompts"] * case["n"]
    row = spec.num_layers * spec.kv_size * 2 * 2
    ctx = steps * case["n"] * sum(lens) + rows * steps * (steps + 1) // 2
    shared = steps * sum(lens) + rows * steps * (steps + 1) // 2
    return {"bytes": (steps + 1) * (size + head) + shared * row,
            "flops": 2 * n * (sum(lens) + steps * rows) + head * (len(lens) + steps * rows)
            + attend * (ctx + sum(t * (t + 1) // 2 for t in lens))}


def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        # a threshold that falls between two sums, or two keys in a tie
        return {"rel": 0.0, "differ": 0.005}
    if kind == "attend":
        return {"rel": 0.01, "max": 0.1}        # bf16 output
    if kind == "flash":
        return {"rel": 0.01, "max": 0.2}        # bf16 outputs and products
    if kind == "loss":
        return {"rel": 0.01, "max": 0.1}        # bf16 gradient
    if kind == "learn":
        return {"rel": 0.03, "max": 0.9}        # bf16 through every layer
    return {"rel": 0.02, "max": 0.9, "differ": 0.005}


# ------------------------------------------------------------------ exact

def _nf4(w):
    """bf16 image of a matrix in 4-bit normal-float blocks of 64."""
    code = torch.tensor([
        -1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453,
        -0.28444138169288635, -0.18477343022823334, -0.09105003625154495, 0.0,
        0.07958029955625534, 0.16093020141124725, 0.24611230194568634,
        0.33791524171829224, 0.44070982933044434, 0.5626170039176941,
        0.7229568362236023, 1.0], device=w.device)
    blocks = w.float().view(-1, 64)
    top = blocks.abs().amax(1, keepdim=True).clamp_min(1e-12)
    middle = (code[1:].double() + code[:-1].double()) / 2
    near = torch.bucketize((blocks / top).double(), middle)
    return (code[near] * top).view(w.shape).to(torch.bfloat16)


class _Exact:
    """The dense model in 64 bits, one sequence at a time."""

    def __init__(self, case, seed, lora, peaked):
        self.spec, self.lora = get_spec(case["model"]), lora
        g = _generator(seed)
        embed, head, norm = _outer_weights(self.spec, g, peaked)
        self.embed, self.norm = embed, norm.double()
        self.head = embed if head is None else head
        self.layers = [_layer_weights(self.spec, g, lora)
                       for _ in range(self.spec.num_layers)]
        if case["four_bit"]:
            for w in self.layers:
                for name in PROJECTIONS:
                    w[name] = _nf4(w[name])

    def rms(self, x, w):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + self.spec.rms_norm_eps) \
            * w.double()

    def linear(self, w, name, x):
        y = x @ w[name].double().t()
        if name + ".b" in w:
            y = y + w[name + ".b"].double()
        if self.lora:
            y = y + (x @ w[name + ".A"].double().t()) @ w[name + ".B"].double().t() \
                * (LORA_ALPHA / LORA_R)
        return y

    def rotate(self, x):
        half = self.spec.head_dim // 2
        freq = self.spec.rope_theta ** (-torch.arange(half, device=DEVICE).double() / half)
        at = torch.arange(x.shape[0], device=DEVICE).double()[:, None, None] * freq
        a, b = x[..., :half], x[..., half:]
        return torch.cat([a * at.cos() - b * at.sin(), b * at.cos() + a * at.sin()], -1)

    def layer(self, w, x):
        """One layer over a sequence from its first token: (x, k, v)."""
        s, T = self.spec, x.shape[0]
        h = self.rms(x, w["norm1"])
        q = self.linear(w, "q", h).view(T, s.num_heads, s.head_dim)
        k = self.linear(w, "k", h).view(T, s.num_kv_heads, s.head_dim)
        v = self.linear(w, "v", h).view(T, s.num_kv_heads, s.head_dim)
        if s.qk_norm:
            q, k = self.rms(q, w["q.norm"]), self.rms(k, w["k.norm"])
        q, k = self.rotate(q), self.rotate(k)
        o = _attention(q.transpose(0, 1), k.transpose(0, 1), v.transpose(0, 1))
        x = x + self.linear(w, "o", o.transpose(0, 1).reshape(T, s.q_size))
        h = self.rms(x, w["norm2"])
        x = x + self.linear(w, "down", F.silu(self.linear(w, "gate", h))
                            * self.linear(w, "up", h))
        return x, k, v


def _attention(q, k, v):
    """Causal attention in 64 bits, q [H, T, D] at the end of k, v [G, S, D]."""
    G, S = k.shape[:2]
    q = q.reshape(G, -1, q.shape[1], q.shape[2])            # [G, H/G, T, D]
    T = q.shape[2]
    s = (q.flatten(1, 2) @ k.transpose(1, 2)).view(G, -1, T, S) * q.shape[3] ** -0.5
    hidden = torch.ones(T, S, dtype=torch.bool, device=q.device).triu(S - T + 1)
    p = s.masked_fill(hidden, -math.inf).softmax(-1)
    return (p.flatten(1, 2) @ v).view(-1, T, v.shape[2])


def _exact_learn(case, seed):
    net = _Exact(case, seed, True, False)
    for w in net.layers:
        for name in PROJECTIONS:
            for m in (".A", ".B"):
                w[name + m] = w[name + m].double().requires_grad_()
    tok = ByteTokenizer(net.spec.vocab_size)
    total = 0.0
    for problem, answer, reward in zip(*_samples(case, seed)):
        ids = torch.tensor(tok.encode(problem) + tok.encode(answer), device=DEVICE)
        n = len(tok.encode(answer))
        x = net.embed[ids].double()
        for w in net.layers:
            x = net.layer(w, x)[0]
        hidden = net.rms(x, net.norm)[len(ids) - n - 1:-1]
        logp = (hidden @ net.head.double().t()).log_softmax(-1)
        loss = -logp.gather(1, ids[-n:, None]).mean() * reward / case["samples"]
        loss.backward()
        total += float(loss)
    grads = {m: torch.cat([w[name + m].grad.reshape(-1) for w in net.layers
                           for name in PROJECTIONS]) for m in (".A", ".B")}
    return {"loss": total, "A": grads[".A"], "B": grads[".B"]}


def _exact_generate(case, seed):
    net, s = _Exact(case, seed, case["lora"], True), get_spec(case["model"])
    prompts, n, new = _prompts(case, seed), case["n"], case["new"]

    def follow(prompt):
        """(tokens, keys per layer, values per layer) of the prompt and its answer."""
        full = prompt + _successors(net, prompt[-1], new - 1)
        x, keys, values = net.embed[torch.tensor(full, device=DEVICE)].double(), [], []
        for w in net.layers:
            x, k, v = net.layer(w, x)
            keys.append(k)
            values.append(v)
        hidden = net.rms(x[len(prompt) - 1:], net.norm).float()
        return (hidden @ net.head.float().t()).argmax(-1).tolist(), keys, values

    streams = [follow(p) for p in prompts]
    pages = _pool_pages(case)
    shape = (s.num_layers, pages, PAGE, s.num_kv_heads, s.head_dim)
    key, value = (torch.zeros(shape, dtype=torch.float64, device=DEVICE) for _ in range(2))

    def put(table, first, last, keys, values):
        at = torch.arange(first, last, device=DEVICE)
        page, row = torch.tensor(table, device=DEVICE)[at // PAGE], at % PAGE
        for i in range(s.num_layers):
            key[i, page, row] = keys[i][first:last]
            value[i, page, row] = values[i][first:last]

    # pages as the pool hands them out: prompts, then each prompt's candidates
    # (full pages shared, the last one copied), a spare page where the batch is
    # padded, then the candidates' further pages
    free = list(range(pages - 1, -1, -1))
    tables = []
    for p, (_, keys, values) in zip(prompts, streams):
        tables.append([free.pop() for _ in range(_pages(len(p)))])
        put(tables[-1], 0, len(p), keys, values)
    lanes = []
    for p, table, stream in zip(prompts, tables, streams):
        full = len(p) // PAGE
        for _ in range(n):
            own = table[:full]
            if full < len(table):
                own = own + [free.pop()]
                key[:, own[-1]] = key[:, table[full]]
                value[:, own[-1]] = value[:, table[full]]
            lanes.append((own, p, stream))
        if full < len(table):
            free.append(table[full])
    padded = 8 if len(lanes) <= 8 else (len(lanes) + 15) // 16 * 16
    if padded > len(lanes):
        spare = [free.pop()]
        x = net.embed[:1].double()
        for i, w in enumerate(net.layers):
            x, k, v = net.layer(w, x)
            key[i, spare[0], 0], value[i, spare[0], 0] = k[0], v[0]
    for own, p, _ in lanes:
        while len(own) < _pages(len(p) + new):
            own.append(free.pop())
    for own, p, (_, keys, values) in lanes:
        put(own, len(p), len(p) + new - 1, keys, values)
    tokens = np.array([[t] * n for t, _, _ in streams])
    return {"tokens": tokens, "key": key, "value": value}


def _successors(net, token, count):
    """The peaked head's answers, from the embedding alone."""
    out = []
    for _ in range(count):
        token = int((net.head.float() @ (net.embed[token].float() * net.norm.float())).argmax())
        out.append(token)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        return None                     # whole numbers, drawn by the framework's own hash
    if kind == "learn":
        return _exact_learn(case, seed)
    if kind == "generate":
        with torch.no_grad():
            return _exact_generate(case, seed)
    state = prepare(case, seed)
    if kind == "attend":
        out = torch.empty(state["q"].shape, dtype=torch.float64, device=DEVICE)
        for i, c in enumerate(state["lens"].tolist()):
            pages = state["tables"][i, :_pages(c)].long()
            k, v = (state[x][pages].flatten(0, 1)[:c].double().transpose(0, 1)
                    for x in ("key", "value"))
            out[i] = _attention(state["q"][i][:, None].double(), k, v)[:, 0]
        return out
    if kind == "flash":
        q, k, v = (t.detach().double() for t in state["qkv"])
        grads = [torch.empty_like(t) for t in (q, k, v)]
        out = torch.empty_like(q)
        for b in range(q.shape[0]):
            for j in range(k.shape[1]):          # a kv head with its query heads
                hs = slice(j * q.shape[1] // k.shape[1], (j + 1) * q.shape[1] // k.shape[1])
                part = [q[b, hs], k[b, j:j + 1], v[b, j:j + 1]]
                part = [t.clone().requires_grad_() for t in part]
                o = _attention(*part)
                gs = torch.autograd.grad(o, part, state["dout"][b, hs].double())
                out[b, hs], grads[0][b, hs] = o.detach(), gs[0]
                grads[1][b, j:j + 1], grads[2][b, j:j + 1] = gs[1], gs[2]
        return {"out": out, "dq": grads[0], "dk": grads[1], "dv": grads[2]}
    logits = state["logits"].detach()
    weight = state["mask"].double() / state["mask"].sum(-1, keepdim=True) \
        * state["rewards"].double()[:, None] / logits.shape[0]
    loss, grad = 0.0, torch.empty(logits.shape, dtype=torch.float64, device=DEVICE)
    for b in range(logits.shape[0]):
        logp = logits[b].double().log_softmax(-1)
        target = state["targets"][b][:, None]
        loss = loss - (logp.gather(1, target)[:, 0] * weight[b]).sum()
        grad[b] = logp.exp_() * weight[b][:, None]
        grad[b].scatter_add_(1, target, -weight[b][:, None])
    return {"loss": loss, "grad": grad}
