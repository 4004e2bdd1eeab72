"""Decode products on weights in tiles and the kernels that join their partial
sums, at the edges of their tiles and splits, against fp64 torch."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ext():
    from distrl_llm_amd.ops.build import build
    return build()


def _rand(shape, seed, std=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * std).to("cuda", torch.bfloat16)


def _rel(x, ref):
    return float((x.double() - ref.double()).norm() / ref.double().norm().clamp_min(1e-30))


def _tiles(ext, *ws, glu=False):
    out = torch.empty(sum(w.shape[0] for w in ws), ws[0].shape[1], dtype=torch.bfloat16,
                      device="cuda")
    row = 0
    for w in ws:
        assert ext.weight_tiles(w, out, row, glu)
        row += 16 if glu else w.shape[0]
    return out


@pytest.mark.parametrize("N1,N2,K", [(32, 32, 32), (64, 96, 288), (256, 32, 1056)])
@pytest.mark.parametrize("r", [0, 8, 40])
def test_weight_tiles(ext, N1, N2, K, r):
    """Tiles of two matrices one below the other, with an adapter and without,
    are the torch permutation of the row-major kernel's results, and back."""
    from distrl_llm_amd.engine.weights import _tiled, _untiled
    ws, out = [_rand((N, K), i) for i, N in enumerate((N1, N2))], _rand((N1 + N2, K), 9)
    row, rows = 0, []
    for i, w in enumerate(ws):
        a, b = _rand((r, K), 3 + i, 0.1), _rand((w.shape[0], r), 5 + i, 0.1)
        rows.append(w.clone())
        if r:
            assert ext.lora_merge(w, a, b, rows[-1], 0.5)
        assert ext.weight_tiles(w, out, row, False, *((a, b, 0.5) if r else ()))
        row += w.shape[0]
    rows = torch.cat(rows)
    assert torch.equal(out, _tiled(rows)) and torch.equal(_untiled(out), rows)
    if N1 % 32 == 0 and N1 == N2:
        assert torch.equal(_tiles(ext, *ws, glu=True), _tiled(torch.cat(ws), True))
        assert torch.equal(_untiled(_tiles(ext, *ws, glu=True), True), torch.cat(ws))
    # refused: a row-major matrix that 16 B loads can't walk
    assert not ext.weight_tiles(_rand((N1, K + 2), 1)[:, 1:K + 1], out, 0, False)


@pytest.mark.parametrize("n", [1, 7, 8, 9, 17])
def test_weights_tiles(ext, n):
    """Weights of several shapes and ranks a launch, as one a launch; one that is refused
    leaves all as they were."""
    shapes = [((32, 32, 0), (256, 1056, 8), (64, 288, 128), (96, 1280, 40))[i % 4] for i in range(n)]
    ws = [_rand((N, K), i) for i, (N, K, _) in enumerate(shapes)]
    a = [_rand((r, K), 30 + i, 0.1) if r else None for i, (_, K, r) in enumerate(shapes)]
    b = [_rand((N, r), 60 + i, 0.1) if r else None for i, (N, _, r) in enumerate(shapes)]
    glu, scale = [i % 3 == 2 for i in range(n)], [0.5 + i for i in range(n)]
    outs = [torch.full((N * (2 if g else 1) + 32, K), 3.0, dtype=torch.bfloat16, device="cuda")[:-32]
            for (N, K, _), g in zip(shapes, glu)]
    row, want = [16 if g else 0 for g in glu], [o.clone() for o in outs]
    for i in range(n):
        assert ext.weight_tiles(ws[i], want[i], row[i], glu[i], a[i], b[i], scale[i])
    refused = ws[:-1] + [_rand((shapes[-1][0], shapes[-1][1] + 2), 1)[:, 1:-1]]
    assert not ext.weights_tiles(refused, outs, row, glu, a, b, scale)
    assert all(bool((o == 3).all()) for o in outs)
    assert ext.weights_tiles(ws, outs, row, glu, a, b, scale)
    assert all(torch.equal(o, w) for o, w in zip(outs, want))


@pytest.mark.parametrize("N,K", [(18944, 3584), (3584, 18944)])
def test_weights_tiles_of_all_sizes(ext, N, K):
    """A weight of whose rows a workgroup takes 256, between small ones of whose it takes
    64, in one launch: each is what torch makes of W + s B A, rounded once (sums in fp32
    of products that are exact), and what lies beside it stays."""
    from distrl_llm_amd.engine.weights import _untiled
    jobs = []
    for i, (n, k, r, row) in enumerate(((96, 1056, 40, 0), (N, K, 32, 16), (256, 288, 8, 32), (N, K, 0, 0),
                                        (32, 32, 128, 0), (N, K, 16, 32))):
        g = torch.Generator("cuda").manual_seed(i)
        rand = lambda *s, std=1.0: torch.randn(s, generator=g, device="cuda").mul_(std).bfloat16()
        glu = row == 16
        out = torch.full((n * (2 if glu else 1) + 64 * (not glu), k), 3.0, dtype=torch.bfloat16, device="cuda")
        jobs.append((rand(n, k), out, row, glu, rand(r, k, std=0.1) if r else None,
                     rand(n, r, std=0.1) if r else None, 0.5 + i))
    assert ext.weights_tiles(*map(list, zip(*jobs)))
    for w, out, row, glu, a, b, scale in jobs:
        got, first = _untiled(out, glu), len(w) if glu else row
        there = got[first:first + len(w)]
        assert bool((got[:first] == 3).all()) and bool((got[first + len(w):] == 3).all())
        if a is None:
            assert torch.equal(there, w)
        else:
            ref = w.double().addmm_(b.double(), a.double(), alpha=scale)
            assert float(((there.double() - ref).abs() / ref.abs().clamp_min(2.0 ** -6)).max()) < 2.0 ** -8


@pytest.mark.parametrize("M", [1, 17, 32, 33, 96, 128, 129, 160])
@pytest.mark.parametrize("N,K", [(32, 64), (96, 192), (1152, 896), (2048, 1536), (160, 8960)])
def test_stream_gemm(ext, M, N, K):
    """Every row tile and cut, ragged last workgroups, more rows of W behind;
    SiLU*mul. Bounds: fp32 sums (some K roundings of 2^-24); one rounding of
    the activation's result."""
    x, w, a = _rand((M, K), 1), _rand((N, K), 2, K ** -0.5), _rand((32, K), 3)
    xd, ref = x.double(), x.double() @ w.double().t()
    got = ext.stream_gemm(x, _tiles(ext, w))
    assert got.shape[1:] == (M, N) and _rel(got.sum(0), ref) < 1e-5
    got = ext.stream_gemm(x, _tiles(ext, w), _tiles(ext, a)).sum(0)
    assert _rel(got[:, :N], ref) < 1e-5 and _rel(got[:, N:], xd @ a.double().t()) < 1e-5
    up = _rand((N, K), 4, K ** -0.5)
    ref = torch.nn.functional.silu(ref) * (xd @ up.double().t())
    assert _rel(ext.stream_glu(x, _tiles(ext, w, up, glu=True)), ref) < 2.0 ** -8
    assert not ext.stream_gemm_takes(161, N, K)         # one row further


@pytest.mark.parametrize("M", [1, 8, 17, 32])
@pytest.mark.parametrize("N,K", [(32, 512), (896, 896), (2080, 544), (4128, 4864)])
def test_skinny_gemm_tiles(ext, M, N, K):
    """The same results from tiles as from rows."""
    x, w, b = _rand((M, K), 1), _rand((2 * N, K), 2, K ** -0.5), _rand((N,), 3)
    res, u, ub = _rand((M, N), 4), _rand((M, 64), 5), _rand((N, 64), 6, 0.1)
    kw = {"norm_w": _rand((K,), 7, 0.1) + 1, "eps": 1e-6}
    half = w[:N].contiguous()
    t, tg = _tiles(ext, half), _tiles(ext, half, w[N:], glu=True)
    for mode, rows, tiles, args in (
            (0, half, t, {"bias": b}), (0, half, t, {"bias": b, **kw}),
            (1, half, t, {"res": res, "u": u, "ub": ub}), (2, w, tg, {}), (2, w, tg, kw)):
        want = ext.skinny_gemm(x, rows, mode, **args)
        for kept in (False, True):
            assert torch.equal(ext.skinny_gemm(x, tiles, mode, tiles=True, kept=kept, **args), want)


@pytest.mark.parametrize("M", [1, 7, 8])
@pytest.mark.parametrize("N,K,R", [(16, 512, 32), (896, 896, 0), (1152, 1024, 96), (2048, 1088, 64),
                                   (2064, 576, 32), (32, 4864, 0), (2080, 8960, 32), (64, 2560, 0),
                                   (48, 3584, 32), (2048, 4608, 0), (2064, 1536, 32), (2560, 4096, 0),
                                   (2080, 4608, 0), (8960, 1536, 0), (9728, 2560, 0), (4608, 3584, 32)])
def test_skinny_gemm_few_rows(ext, M, N, K, R):
    """Up to 8 rows: two steps of K side by side, every number of them that a wave has in
    flight (1, 3, 5, 7, 9, 10, with SiLU*mul 2 for 1; more rows of W: 2 to 5, to 4). Sums in fp32 of
    products that are exact: what is left is the output's rounding, and of gate and up
    each their own, whose errors silu at most doubles."""
    x, w, b = _rand((M, K), 1), _rand((2 * N, K), 2, K ** -0.5), _rand((N,), 3)
    res, kw = _rand((M, N), 4), {"norm_w": _rand((K,), 7, 0.1) + 1, "eps": 1e-6}
    half = w[:N].contiguous()
    xd, wd = x.double(), half.double()
    n = (xd * kw["norm_w"].double()).to(torch.bfloat16).double() \
        * (xd.pow(2).mean(-1, keepdim=True) + 1e-6).rsqrt()
    assert _rel(ext.skinny_gemm(x, half, 0, b, **kw), n @ wd.t() + b.double()) < 2.0 ** -8
    y = xd @ wd.t() + res.double()
    assert _rel(ext.skinny_gemm(x, half, 1, res=res), y) < 2.0 ** -8
    if R:
        u, ub = _rand((M, R), 5), _rand((N, R), 6, 0.1)
        got = ext.skinny_gemm(x, half, 1, res=res, u=u, ub=ub)
        assert _rel(got, y + u.double() @ ub.double().t()) < 2.0 ** -8
    gate, up = (n @ w.double().t()).split(N, 1)
    assert _rel(ext.skinny_gemm(x, w, 2, **kw), torch.nn.functional.silu(gate) * up) < 2.0 ** -6
    # a row that is no number stays by itself
    x[0, 0] = float("inf")
    assert ext.skinny_gemm(x, half, 1, res=res)[1:].isfinite().all()
    assert ext.skinny_gemm(x, half, 0, **kw)[1:].isfinite().all()


@pytest.mark.parametrize("model,n,tiled,skinny", [
    ("qwen2.5-0.5b", 16, True, True), ("qwen2.5-0.5b", 17, True, False),
    ("qwen2.5-0.5b", 32, False, True), ("qwen2.5-0.5b", 33, False, False),
    ("small-qwen2", 32, True, True), ("qwen2.5-1.5b", 17, False, False)])
def test_steps_on_skinny_products(model, n, tiled, skinny):
    """The decode steps that take them, as measured."""
    from types import SimpleNamespace
    from distrl_llm_amd.engine import Engine
    from distrl_llm_amd.models import get_spec
    engine = SimpleNamespace(spec=get_spec(model), dtype=torch.bfloat16, _streamed=lambda n: tiled)
    assert Engine._skinny(engine, n) == skinny


@pytest.mark.parametrize("S", [1, 3, 4, 9])
@pytest.mark.parametrize("rows,hidden,r", [(1, 64, 0), (5, 896, 32), (33, 4096, 64), (2, 4160, 128),
                                           (3, 8192, 0)])
def test_add_rmsnorm_join(ext, S, rows, hidden, r):
    """Bounds: the residual rounded once, its norm from the rounded values."""
    g = torch.Generator(device="cuda").manual_seed(S)
    parts = torch.randn((S, rows, hidden + r), generator=g, device="cuda")
    res, w, bt = _rand((rows, hidden), 1), _rand((hidden,), 2, 0.1) + 1, _rand((r, hidden), 3, 0.1)
    y, out = ext.add_rmsnorm_join(parts, res, w, 1e-6, bt if r else None)
    total = parts.double().sum(0)
    ref = res.double() + total[:, :hidden] + total[:, hidden:] @ bt.double()
    assert _rel(out, ref) < 2.0 ** -8
    assert _rel(y, ref * torch.rsqrt((ref * ref).mean(-1, keepdim=True) + 1e-6) * w.double()) \
        < 2.0 ** -7


@pytest.mark.parametrize("H,KV,D", [(14, 2, 64), (28, 4, 128), (8, 8, 64), (64, 8, 128)])
@pytest.mark.parametrize("N,longest,bs", [(1, 1, 16), (5, 40, 16), (3, 2500, 16), (9, 700, 24),
                                          (130, 90, 16)])
@pytest.mark.parametrize("S,bias,norms", [(0, False, False), (1, True, False), (5, False, True)])
def test_paged_decode_packed(ext, H, KV, D, N, longest, bs, S, bias, norms):
    """Against rotation with cache write and attention as two calls on the
    summed rows (their inputs rounded to bf16: a few roundings more): one slice
    and several, more than once with the same counters, a row of the cache that
    holds no number before it is written, a token without a slot."""
    width, g = (H + 2 * KV) * D, torch.Generator(device="cuda").manual_seed(N)
    lens = torch.randint(1, longest + 1, (N,), generator=g, device="cuda", dtype=torch.int32)
    lens[0] = longest
    nb = (longest + bs - 1) // bs
    pages = torch.randperm(N * nb, generator=g, device="cuda").view(N, nb).int()
    pos = (lens - 1).int()
    slots = pages.gather(1, (pos // bs).long()[:, None])[:, 0].long() * bs + pos % bs
    cache = [_rand((N * nb, bs, KV, D), 4 + i) for i in range(2)]
    for c in cache:
        c.view(-1, KV, D)[slots] = float("nan")
    parts = torch.randn((max(S, 1), N, width), generator=g, device="cuda")
    b = _rand((width,), 1) if bias else None
    nw = (_rand((D,), 2, 0.1) + 1, _rand((D,), 3, 0.1) + 1, 1e-6) if norms else ()
    inv = 1.0 / 1e4 ** (torch.arange(0, D, 2, device="cuda").float() / D)
    rows = (parts.sum(0) + (b.float() if bias else 0)).to(torch.bfloat16)
    arrived = torch.zeros(N * KV, dtype=torch.int32, device="cuda")
    ref_cache, ref_rows = [c.clone() for c in cache], rows.clone()
    ext.rope_scatter_qkv(ref_rows, pos, slots, inv, *ref_cache, H, KV, D, *nw)
    queries = ref_rows[:, :H * D].reshape(N, H, D).contiguous()
    ref = ext.paged_attention_decode(queries, *ref_cache, pages, lens,
                                     D ** -0.5).flatten(1)
    for _ in range(2):
        got = [c.clone() for c in cache]
        out = ext.paged_decode_packed(parts if S else rows, b if S else None, pos, slots, inv, *got,
                                      pages, lens, arrived, H, D ** -0.5, *nw)
        assert _rel(out, ref) < (5e-3 if longest == 1 else 0.02)
        for x, y in zip(got, ref_cache):
            assert _rel(x, y) < 3 * 2.0 ** -9
        assert not arrived.any()
    slots[-1] = -1
    got = [c.clone() for c in cache]
    ext.paged_decode_packed(parts if S else rows, b if S else None, pos, slots, inv, *got, pages,
                            lens, arrived, H, D ** -0.5, *nw)
    assert got[0].isnan().any(-1).sum() == KV


@pytest.mark.parametrize("S", [2, 3, 4])
def test_paged_decode_packed_few_partial_sums(ext, S):
    """As many as a workgroup of four waves with rows of 64 fetches ahead, and more."""
    test_paged_decode_packed(ext, 8, 8, 64, 130, 90, 16, S, True, False)


def test_paged_decode_packed_refuses(ext):
    """Operands in host memory, and ones that do not lie on end."""
    D, N = 64, 3
    qkv, cache = _rand((N, 4 * D), 1), [_rand((4, 16, 1, D), 2 + i) for i in range(2)]
    args = [torch.zeros(N, dtype=torch.int32, device="cuda"),
            torch.zeros(N, dtype=torch.long, device="cuda"), torch.ones(D // 2, device="cuda"),
            *cache, torch.zeros(N, 2, dtype=torch.int32, device="cuda"),
            torch.ones(N, dtype=torch.int32, device="cuda"),
            torch.zeros(N, dtype=torch.int32, device="cuda")]
    ext.paged_decode_packed(qkv, None, *args, 2, 0.125)
    for i, t in enumerate(args):
        for bad in (t.cpu(), t[:1].expand(t.shape)):
            with pytest.raises(RuntimeError):
                ext.paged_decode_packed(qkv, None, *args[:i], bad, *args[i + 1:], 2, 0.125)


@pytest.mark.parametrize("H,KV,D,N,cs", [(28, 4, 128, 16, 4), (28, 4, 128, 32, 2), (14, 2, 64, 32, 4)])
@pytest.mark.parametrize("S", [0, 2])
def test_paged_decode_packed_behind_a_slice_end(ext, monkeypatch, H, KV, D, N, cs, S):
    """Contexts that end 1 to 32 tokens behind a slice whose end is no multiple
    of 32, after a call that leaves numbers that are none in LDS: the slice does
    not take the new token, which another one has. Against the same call in one
    slice; both round to bf16."""
    bs, nb, width = 16, 97, (H + 2 * KV) * D
    room = bs * nb
    end = (room + cs - 1) // cs
    assert end % 32
    behind = [z * end + d for z in range(1, cs) for d in (1, 2, 16, 27, 28, 29, 32)]
    lens = torch.tensor((behind * N)[:N - 1] + [room], device="cuda", dtype=torch.int32)
    pages = torch.randperm(N * nb, generator=torch.Generator().manual_seed(N)).view(N, nb)
    pages = pages.to("cuda", torch.int32)
    pos = lens - 1
    slots = pages.gather(1, (pos // bs).long()[:, None])[:, 0].long() * bs + pos % bs
    cache = [_rand((N * nb, bs, KV, D), 4 + i) for i in range(2)]
    inv = 1.0 / 1e4 ** (torch.arange(0, D, 2, device="cuda").float() / D)
    rows = _rand((S, N, width), 1).float() if S else _rand((N, width), 1)
    arrived = torch.zeros(256, dtype=torch.int32, device="cuda")
    most = 255 // KV

    def call(qkv, at, slots, tables, lens):
        return ext.paged_decode_packed(qkv, None, at, slots, inv, *cache, tables, lens, arrived, H,
                                       D ** -0.5)

    def full(value, dtype):
        return torch.full((most,), value, dtype=dtype, device="cuda")

    monkeypatch.setenv("DISTRL_PAGED_CS", "1")
    ref = call(rows, pos, slots, pages, lens)
    call(torch.full((most, width), float("nan"), dtype=torch.bfloat16, device="cuda"),
         full(room - 1, torch.int32), full(-1, torch.long), pages[torch.arange(most) % N].contiguous(),
         full(room, torch.int32))
    monkeypatch.delenv("DISTRL_PAGED_CS")
    out = call(rows, pos, slots, pages, lens)
    assert bool(out.isfinite().all()) and _rel(out, ref) < 2.0 ** -8
    assert not arrived.any()


@pytest.mark.parametrize("name,four_bit,lora_r", [("small-qwen2", False, 8), ("small-qwen2", True, 8),
                                                  ("small-qwen3", True, 0), ("small-qwen3", False, 12)])
@pytest.mark.parametrize("n", [3, 40, 161])
def test_decode_step_matches_modules(name, four_bit, lora_r, n):
    """Steps of few, of tens and of more sequences after a changed adapter, twice
    through the cached graph: the cache rows they write against a teacher-forced
    pass of the modules (two bf16 paths of the same products: 3 %)."""
    from distrl_llm_amd.config import EngineConfig, SamplingParams
    from distrl_llm_amd.engine import Engine
    from distrl_llm_amd.models import CausalLM, get_spec
    model = CausalLM(get_spec(name), lora_r=lora_r, dtype=torch.bfloat16,
                     device=torch.device("cuda")).random_init(3).eval()
    if four_bit:
        model.quantize_nf4_()
    eng = Engine(model, EngineConfig(max_seq_length=64, num_kv_blocks=2 * n + 8, max_num_seqs=256))
    prompt, sp = [5, 6, 7, 8, 9], SamplingParams(max_tokens=4, temperature=0.0, n=n)
    for seed in (7, 8):
        with torch.no_grad():
            for key, p in model.named_parameters():
                if key.endswith(("lora_B", "bias")):
                    p.copy_(_rand(p.shape, seed, 0.05))
        eng.pool.allocator.reset()
        tokens = eng.generate([prompt], sp)[0][0]
        ids, ref = torch.tensor([prompt + tokens[:3]], device="cuda"), []
        hooks = [l.self_attn.v_proj.register_forward_hook(lambda m, i, o: ref.append(o[0].detach()))
                 for l in model.model.layers]
        with torch.no_grad():
            model(ids)
        for h in hooks:
            h.remove()
        # the first candidate's page: the prompt's rows, then three steps'
        rows = [v.flatten(1) for v in eng.pool.value.flatten(1, 2)]
        for layer, want in zip(rows, ref):
            at = (layer[:, None, :] - want[0]).abs().sum(-1).argmin().item()
            assert _rel(layer[at:at + 8], want) < 0.03


def test_replaced_weight_reaches_row_major_storage():
    """A weight without an adapter that is another tensor at the next refresh:
    the storage that captured steps hold follows it."""
    from distrl_llm_amd.engine.weights import FusedWeights
    from distrl_llm_amd.models import CausalLM, get_spec
    model = CausalLM(get_spec("small-qwen2"), dtype=torch.bfloat16,
                     device=torch.device("cuda")).random_init(3)
    fused = FusedWeights(model)
    fused.refresh()
    at, lw = model.model.layers[0].self_attn, fused.layers[0]
    held = lw.rows("o")
    at.o_proj.weight.data = _rand(at.o_proj.weight.shape, 5)
    fused.refresh()
    assert lw.rows("o") is held and torch.equal(held, at.o_proj.weight)


def _cache_rows(eng, n, tokens=4):
    """What a generation of n candidates leaves in the cache."""
    from distrl_llm_amd.config import SamplingParams
    eng.pool.allocator.reset()
    for rows in (eng.pool.key, eng.pool.value):
        rows.zero_()
    eng.generate([[5, 6, 7, 8]], SamplingParams(max_tokens=tokens, temperature=0.0, n=n))
    return torch.stack([eng.pool.key, eng.pool.value])


def test_four_bit_waves_are_padded_within_their_pool(monkeypatch):
    """As many sequences as the engine takes, a wave padded beyond them: the
    adapter inputs of the padding stay out of the next layer's. Against an
    engine with room (atomic fp32 sums in another order: 2 %)."""
    from distrl_llm_amd.config import EngineConfig
    from distrl_llm_amd.engine import Engine
    from distrl_llm_amd.models import CausalLM, get_spec
    monkeypatch.setenv("DISTRL_DECODE_NF4", "1")
    model = CausalLM(get_spec("small-qwen2"), lora_r=8, dtype=torch.bfloat16,
                     device=torch.device("cuda")).random_init(3).eval()
    with torch.no_grad():
        for name, p in model.named_parameters():
            if name.endswith("lora_B"):
                p.copy_(_rand(p.shape, 7, 0.05))
    model.quantize_nf4_()
    pools = []
    for most in (20, 64):
        eng = Engine(model, EngineConfig(max_seq_length=64, num_kv_blocks=64, max_num_seqs=most))
        assert eng.fused.nf4
        pools.append(_cache_rows(eng, 20, 2))
    assert _rel(*pools) < 0.02


@pytest.mark.parametrize("lora_r", [0, 8])
def test_large_steps_on_a_full_card(monkeypatch, lora_r):
    """Steps of more sequences than the streamed products take, the row-major
    weights laid out within the step, twice through the captured graph: the
    cache rows of an engine with room."""
    from distrl_llm_amd.config import EngineConfig
    from distrl_llm_amd.engine import Engine, weights
    from distrl_llm_amd.models import CausalLM, get_spec
    model = CausalLM(get_spec("small-qwen2"), lora_r=lora_r, dtype=torch.bfloat16,
                     device=torch.device("cuda")).random_init(3).eval()
    pools = []
    for room in (True, False):
        eng = Engine(model, EngineConfig(max_seq_length=64, num_kv_blocks=400, max_num_seqs=256))
        assert eng.fused.tiled
        with monkeypatch.context() as m:
            m.setattr(weights, "_room_for", lambda size, device: room)
            pools += [_cache_rows(eng, 161) for _ in range(2)][1:]
        assert ("gateup" in eng.fused.layers[0]._rows) == room
    assert torch.equal(*pools)


@pytest.mark.parametrize("lora_r,four_bit", [(0, False), (8, True)])
def test_replaced_weight_reaches_captured_steps(monkeypatch, lora_r, four_bit):
    """Row-major steps captured before a weight is another tensor: the cache
    rows that they write next are a fresh engine's."""
    from distrl_llm_amd.config import EngineConfig
    from distrl_llm_amd.engine import Engine, weights
    from distrl_llm_amd.models import CausalLM, get_spec
    monkeypatch.setattr(weights, "_room_for", lambda size, device: False)
    model = CausalLM(get_spec("small-qwen2"), lora_r=lora_r, dtype=torch.bfloat16,
                     device=torch.device("cuda")).random_init(3).eval()
    if four_bit:
        model.quantize_nf4_()
    cfg = EngineConfig(max_seq_length=64, num_kv_blocks=32, max_num_seqs=8)
    eng = Engine(model, cfg)
    before = _cache_rows(eng, 3)
    for layer in model.model.layers:
        for lin in (layer.self_attn.o_proj, layer.mlp.down_proj):
            lin.weight.data = _rand(lin.weight.shape, 5, 0.05)
    after = _cache_rows(eng, 3)
    assert not torch.equal(before, after) and torch.equal(after, _cache_rows(Engine(model, cfg), 3))


def test_no_tiles_without_room(monkeypatch):
    """Where a second copy of the weights does not fit, steps run row-major."""
    from distrl_llm_amd.config import EngineConfig, SamplingParams
    from distrl_llm_amd.engine import Engine, weights
    from distrl_llm_amd.models import CausalLM, get_spec
    model = CausalLM(get_spec("small-qwen2"), dtype=torch.bfloat16,
                     device=torch.device("cuda")).random_init(3).eval()
    tokens = []
    for room in (True, False):
        monkeypatch.setattr(weights, "_room_for", lambda size, device: room)
        eng = Engine(model, EngineConfig(max_seq_length=64, num_kv_blocks=96, max_num_seqs=64))
        assert eng.fused.tiled == room
        tokens.append([eng.generate([[5, 6, 7]], SamplingParams(max_tokens=2, temperature=0.0, n=n))
                       for n in (3, 40)])
        assert (eng.fused.layers[0].tiles is None) != room
    assert len(tokens[0][1][0]) == len(tokens[1][1][0]) == 40


@pytest.mark.parametrize("N,bs,eos", [(1, 16, None), (8, 16, 3), (300, 24, 3)])
def test_decode_state(ext, N, bs, eos):
    """Three steps against the same in torch operations: sequences that end at
    their limit, with eos, and long before."""
    g = torch.Generator(device="cuda").manual_seed(N)

    def ints(hi, *shape):
        return torch.randint(0, hi, shape, generator=g, device="cuda")

    tables, pos = ints(1000, N, 9).int(), ints(8 * bs, N)
    limits, fin = pos + ints(4, N), ints(3, N) == 0
    state = [ints(5, N), pos.clone(), pos.int() + 1, limits, fin.clone(),
             torch.zeros(1, dtype=torch.long, device="cuda"), torch.zeros(4, N, dtype=torch.long, device="cuda")]
    tok, ctx, out = state[0].clone(), state[2].clone(), state[6].clone()
    for step in range(3):
        slots, pos32 = ext.decode_slots(state[1], tables, bs)
        assert torch.equal(slots, tables.gather(1, (pos // bs)[:, None])[:, 0].long() * bs + pos % bs)
        assert pos32.dtype == torch.int32 and torch.equal(pos32, pos.int())
        new = ints(5, N)
        ext.decode_advance(new, *state, eos)
        out[step], go = new, ~fin
        fin = fin | (pos + 1 >= limits) | ((new == eos) if eos is not None else False)
        tok, pos, ctx = torch.where(go, new, tok), pos + go, ctx + go.int()
        for a, b in zip(state, (tok, pos, ctx, limits, fin, torch.tensor([step + 1], device="cuda"), out)):
            assert torch.equal(a, b)


@pytest.mark.parametrize("N,H,KV", [(128, 28, 4), (129, 28, 4), (257, 4, 2)])
def test_paged_decode_many_sequences(ext, N, H, KV):
    """512 workgroups, one more a kv head and 514: workgroups of four and of two
    waves, contexts of one token to several chunks; bf16 output."""
    D, bs, g = 128, 16, torch.Generator(device="cuda").manual_seed(N)
    lens = torch.randint(1, 300, (N,), generator=g, device="cuda", dtype=torch.int32)
    lens[:6] = torch.tensor([1, 32, 33, 64, 65, 299], device="cuda")
    nb = (300 + bs - 1) // bs
    pages = torch.randperm(N * nb, generator=g, device="cuda").view(N, nb).int()
    q, key, value = _rand((N, H, D), 1), _rand((N * nb, bs, KV, D), 2), _rand((N * nb, bs, KV, D), 3)
    out = ext.paged_attention_decode(q, key, value, pages, lens, D ** -0.5).double()
    for i in [*range(6), N - 1]:
        c = int(lens[i])
        k, v = (t[pages[i].long()].flatten(0, 1)[:c].double().repeat_interleave(H // KV, 1)
                for t in (key, value))
        p = (torch.einsum("hd,chd->hc", q[i].double(), k) * D ** -0.5).softmax(-1)
        assert _rel(out[i], torch.einsum("hc,chd->hd", p, v)) < 2.0 ** -8
