"""Kernels at the edges of their tiles, splits and layouts, against plain
fp32 or fp64 torch."""

import numpy as np
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


# ------------------------------------------------------------------ flash
# Bound: weights, dS and the outputs are each rounded to bf16 (2^-9 of the
# value at most), everything else is fp32: three roundings, 3 * 2^-9 < 0.6 %.
FLASH_REL = 3 * 2.0 ** -9


def _flash_reference(q, k, v, dout, scale):
    q, k, v = (t.detach().float().requires_grad_() for t in (q, k, v))
    group, T = q.shape[1] // k.shape[1], q.shape[2]
    s = q @ k.repeat_interleave(group, 1).transpose(2, 3).contiguous() * scale
    s = s.masked_fill(torch.ones(T, T, dtype=torch.bool, device=q.device).triu(1), float("-inf"))
    o = s.softmax(-1) @ v.repeat_interleave(group, 1)
    return (o.detach(), *torch.autograd.grad(o, (q, k, v), dout.float()))


@pytest.mark.parametrize("B,Hq,Hkv,T,D", [
    (1, 1, 1, 1, 64), (1, 2, 1, 31, 128), (2, 7, 1, 32, 64), (1, 4, 2, 33, 128),
    (1, 3, 3, 64, 64), (2, 10, 2, 65, 128), (1, 28, 4, 127, 128), (1, 14, 2, 129, 64),
    (3, 6, 2, 257, 128), (12, 28, 4, 193, 128), (20, 14, 2, 300, 64)])
@pytest.mark.parametrize("layout", ["heads_first", "tokens_first", "sliced"])
def test_flash_edges(B, Hq, Hkv, T, D, layout):
    """Row blocks of 64 and 128 rows, key tiles of 32 and 64, ragged ends, a
    head split with partial sums (few key blocks) and without; contiguous
    operands, transposed projections, and rows cut out of a wider one at an
    offset that is not a multiple of 16 bytes."""
    from distrl_llm_amd.ops import functional as OF

    def make(H, seed):
        if layout == "heads_first":
            return _rand((B, H, T, D), seed)
        if layout == "tokens_first":
            return _rand((B, T, H, D), seed).transpose(1, 2)
        return _rand((B, T, H * D + 6), seed)[..., 3:3 + H * D].unflatten(2, (H, D)).transpose(1, 2)

    q, k, v, dout = (make(H, i) for i, H in enumerate((Hq, Hkv, Hkv, Hq)))
    scale = 1.3 * D ** -0.5
    ref = _flash_reference(q, k, v, dout, scale)
    leaves = [t.detach().requires_grad_() for t in (q, k, v)]
    o = OF.flash_attention(*leaves, scale)
    got = (o.detach(), *torch.autograd.grad(o, leaves, dout))
    for name, x, r in zip(("o", "dq", "dk", "dv"), got, ref):
        if name in ("dq", "dk") and T == 1:
            # one key: the gradient is zero up to delta's fp32 rounding
            assert float(x.float().abs().max()) < 1e-5
            continue
        assert _rel(x, r) < FLASH_REL, name


def test_flash_scale_signs_and_far_scores():
    """Scores hundreds below the maximum (forward: a saturated softmax's
    gradients cancel, which the bound does not cover), negative and zero scale."""
    from distrl_llm_amd.ops import functional as OF
    q, k, v, dout = (_rand((1, 2, 150, 64), i, 2.0 if i < 2 else 1.0) for i in range(4))
    for scale in (8.0, -8.0):
        ref = _flash_reference(q, k, v, dout, scale)[0]
        assert _rel(OF.flash_attention(q, k, v, scale), ref) < FLASH_REL
    for scale in (-0.125, 0.0, 0.125):
        ref = _flash_reference(q, k, v, dout, scale)
        leaves = [t.detach().requires_grad_() for t in (q, k, v)]
        o = OF.flash_attention(*leaves, scale)
        got = (o.detach(), *torch.autograd.grad(o, leaves, dout))
        for x, r in zip(got, ref):
            if float(r.abs().max()) == 0.0:
                assert float(x.float().abs().max()) == 0.0
            else:
                assert _rel(x, r) < FLASH_REL


@pytest.mark.parametrize("B,H,D", [(1, 2, 64), (1, 2, 128), (300, 2, 64), (300, 2, 128)])
def test_flash_leading_weight(B, H, D):
    """A key that takes the lead in a later tile, by 0..8 in log2 over the 64
    before it, and the only one with a value: its weight carries no rounding, so
    the output has only its own (2^-8 of the value; 2^-16 for the fp32 sums)."""
    from distrl_llm_amd.ops import functional as OF
    T, lead = 160, 64
    q, k, v = (torch.zeros(B, H, T, D, dtype=torch.bfloat16, device="cuda") for _ in range(3))
    # scores q[0] * 1 / 8 against zeros
    q[..., 0] = torch.linspace(0.1, 44.0, B * H * T, device="cuda").view(B, H, T)
    k[:, :, lead, 0] = 1.0
    v[:, :, lead] = 1.0
    out = OF.flash_attention(q, k, v, 0.125)[:, :, lead:].double()
    s = (q[:, :, lead:, 0].double() * 0.125).exp()
    ref = (s / (s + torch.arange(lead, T, device="cuda").double()))[..., None]
    assert float(((out - ref).abs() / ref).max()) < 2.0 ** -8 + 2.0 ** -16


@pytest.mark.parametrize("lens", [[1], [5, 64, 65, 1, 200], [130, 3]])
@pytest.mark.parametrize("H,KV,D", [(4, 2, 64), (7, 1, 128)])
def test_flash_varlen(ext, lens, H, KV, D):
    q, k, v = (_rand((sum(lens), h, D), i) for i, h in enumerate((H, KV, KV)))
    cu = torch.tensor([0] + lens, dtype=torch.int32).cumsum(0).to(torch.int32).cuda()
    out = ext.flash_attn_varlen(q, k, v, cu, max(lens), D ** -0.5)
    at = 0
    for n in lens:
        part = [t[at:at + n].transpose(0, 1).unsqueeze(0).contiguous() for t in (q, k, v)]
        ref = _flash_reference(*part, torch.zeros_like(part[0]), D ** -0.5)[0][0].transpose(0, 1)
        assert _rel(out[at:at + n], ref) < FLASH_REL
        at += n


# ---------------------------------------------------------------- sampler

def _splitmix64(x):
    with np.errstate(over="ignore"):
        x = x + np.uint64(0x9E3779B97F4A7C15)
        x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return x ^ (x >> np.uint64(31))


def _sampled(logits, temperature, top_p, top_k, seeds, step):
    """The sampler's definition, row by row in numpy: whole bins of 1/32 down
    to the threshold, then the largest z - log(-log u)."""
    V, out = logits.shape[1], []
    for row, seed in zip(logits.float().cpu().numpy(), seeds.tolist()):
        z = (row - row.max()) * (np.float32(1) / np.float32(temperature))
        inside = z > -32
        bins = np.minimum(1023, (np.where(inside, -z, 0) * 32).astype(np.int64))
        p = np.bincount(bins[inside], np.exp(z[inside].astype(np.float64)), 1024).cumsum()
        c = np.bincount(bins[inside], minlength=1024).cumsum()
        thr = 1023
        if top_p < 1:
            thr = min(thr, int(np.argmax(p >= top_p * p[-1])))
        if 0 < top_k < V and c[-1] >= top_k:
            thr = min(thr, int(np.argmax(c >= top_k)))
        base = np.uint64(seed) ^ _splitmix64(np.uint64(0x5D21 + step))
        h = _splitmix64(base ^ _splitmix64(np.arange(V, dtype=np.uint64)))
        u = np.minimum((h >> np.uint64(40)).astype(np.float64) + 1, 2 ** 24 - 1) / 2 ** 24
        kept = np.where(inside, bins <= thr, thr == 1023)
        key = np.where(kept, z - np.log(-np.log(u)), -np.inf)
        out.append(int(key.argmax()))
    return out


@pytest.mark.parametrize("B,V,dtype", [
    (3, 8, "bfloat16"), (2, 4096, "bfloat16"), (2, 8200, "bfloat16"), (2, 32768, "bfloat16"),
    (2, 65536, "bfloat16"), (2, 128256, "bfloat16"), (2, 152064, "bfloat16"),
    (1, 160000, "bfloat16"), (2, 32003, "bfloat16"), (2, 32003, "float32"),
    (2, 151936, "float32"), (1200, 40, "float32"), (300, 2056, "bfloat16")])
@pytest.mark.parametrize("temperature,top_p,top_k", [
    (1.0, 1.0, 0), (1.2, 0.95, 0), (0.7, 0.8, 50), (1.0, 1.0, 7)])
def test_sampler_draws_as_defined(ext, B, V, dtype, temperature, top_p, top_k):
    """One slice and several, aligned rows and others, each threshold, each
    draw against the definition. The inputs put no cumulative sum within
    rounding of top_p."""
    g = torch.Generator().manual_seed(V + B)
    logits = torch.randn(B, V, generator=g) * 2.5
    logits[:, 3] += 9.0
    logits = logits.to("cuda", getattr(torch, dtype))
    seeds = torch.randint(0, 2 ** 31 - 1, (B,), generator=g)
    got = ext.sample_tokens(logits, temperature, top_p, top_k, seeds.cuda(),
                            torch.tensor([11], device="cuda"))
    assert got.tolist() == _sampled(logits, temperature, top_p, top_k, seeds, 11)


@pytest.mark.parametrize("B,V,dtype", [
    (640, 2048, "bfloat16"), (640, 2056, "bfloat16"), (641, 20480, "bfloat16"),
    (320, 20488, "bfloat16"), (200, 20479, "float32"), (33, 61440, "bfloat16"),
    (12, 163841, "bfloat16"), (1, 300000, "float32")])
@pytest.mark.parametrize("spread,temperature,top_p,top_k", [
    (3.0, 0.6, 1.0, 0), (0.5, 1.0, 0.9, 0), (3.0, 1.3, 0.97, 0), (2.0, 1.0, 0.9, 300)])
def test_sampler_long_slices(ext, B, V, dtype, spread, temperature, top_p, top_k):
    """Slices as long as a workgroup's registers hold, one element more and
    less, a row in one and in more than 64; thresholds just below the maximum
    and deep, flat rows of which most is drawn."""
    g = torch.Generator().manual_seed(V + B)
    logits = torch.randn(B, V, generator=g) * spread
    logits[:, V // 3] += 4.0 * spread
    logits = logits.to("cuda", getattr(torch, dtype))
    seeds = torch.randint(0, 2 ** 31 - 1, (B,), generator=g)
    got = ext.sample_tokens(logits, temperature, top_p, top_k, seeds.cuda(),
                            torch.tensor([3], device="cuda")).tolist()
    for at in range(0, B, max(1, B // 12)):
        row = slice(at, at + 1)
        assert got[row] == _sampled(logits[row], temperature, top_p, top_k, seeds[row], 3)


def test_sampler_odd_places_and_values(ext):
    """A matrix that does not start on 16 bytes, rows with -inf, and a row
    with nothing finite below its maximum."""
    B, V = 4, 4096
    g = torch.Generator().manual_seed(1)
    flat = (torch.randn(B * V + 1, generator=g) * 2).to("cuda", torch.bfloat16)
    logits = flat[1:].view(B, V)
    logits[1, ::2] = float("-inf")
    logits[2] = float("-inf")
    logits[2, 77] = 1.0
    seeds, step = torch.arange(B), torch.tensor([5], device="cuda")
    for top_p in (1.0, 0.9):
        for x in (logits, logits.clone()):
            got = ext.sample_tokens(x, 1.0, top_p, 0, seeds.cuda(), step).tolist()
            assert got == _sampled(logits, 1.0, top_p, 0, seeds, 5)
            assert got[1] % 2 == 1 and got[2] == 77


def test_sampler_largest_variate(ext):
    """Index 39387 of this row hashes to the largest 24 bits there are. Its key
    is z + 16.64 and not infinite: at z = -18 it does not win over the maximum."""
    V, at = 152064, 39387
    h = _splitmix64(np.uint64(203) ^ _splitmix64(np.uint64(0x5D21)) ^ _splitmix64(np.uint64(at)))
    assert int(h >> np.uint64(40)) == 2 ** 24 - 1
    logits = torch.full((1, V), -40.0)
    logits[0, 7], logits[0, at] = 0.0, -18.0
    logits, seeds = logits.to("cuda", torch.bfloat16), torch.tensor([203])
    for top_k in (0, 2):
        got = ext.sample_tokens(logits, 1.0, 1.0, top_k, seeds.cuda(), torch.tensor([0], device="cuda"))
        assert got.tolist() == _sampled(logits, 1.0, 1.0, top_k, seeds, 0) == [7]
    # and does where its probability allows it: -0.5 + 16.64
    logits[0, at] = -0.5
    got = ext.sample_tokens(logits, 1.0, 1.0, 0, seeds.cuda(), torch.tensor([0], device="cuda"))
    assert got.tolist() == [at]


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_sampler_threshold_on_a_bin_edge(ext, dtype):
    """Logits whose distance from the maximum is a whole number of bins: an
    entry on the threshold bin's lower edge belongs to the next bin, dropped."""
    B, V = 64, 4096
    logits = torch.full((B, V), -20.0)
    logits[:, 5], logits[:, 9], logits[:, 11] = 7.5, 7.46875, 7.4375
    logits, seeds = logits.to("cuda", getattr(torch, dtype)), torch.arange(B)
    step = torch.tensor([0], device="cuda")
    for top_p, top_k, kept in ((1.0, 1, {5}), (0.2, 0, {5}), (1.0, 2, {5, 9}), (0.5, 0, {5, 9}),
                               (0.9, 0, {5, 9, 11})):
        got = ext.sample_tokens(logits, 1.0, top_p, top_k, seeds.cuda(), step).tolist()
        assert set(got) == kept
        assert got == _sampled(logits, 1.0, top_p, top_k, seeds, 0)


def test_sampler_repeats_itself(ext):
    """64 equal rows with one seed draw one token, also where a cumulative
    probability falls on top_p within rounding: slices finish in any order."""
    V, step = 32768, torch.tensor([0], device="cuda")
    for i in range(20):
        row = torch.randn(1, V, generator=torch.Generator().manual_seed(i)) * 2
        z = (row[0] - row[0].max()).double()
        p = torch.bincount((-z * 32).long().clamp(max=1023), z.exp()).cumsum(0)
        rows, top_p = row.cuda().expand(64, -1).contiguous(), float((p[150 + i] / p[-1]).float())
        for seed in range(100):
            seeds = torch.full((64,), seed, device="cuda")
            assert len(set(ext.sample_tokens(rows, 1.0, top_p, 0, seeds, step).tolist())) == 1


def test_sampler_total_of_many_slices(ext):
    """The total that top_p is a share of counts what single slices add little
    to: 73 of them add e^-9.875 to 1368 each, less than half of what fp32 resolves there, and
    with an eighth of that missing the first group alone would reach top_p. Every
    sum here is good to 1e-7, the eighth is 3.4e-7 of it."""
    V = 151936
    logits = torch.full((1, V), -40.0)
    logits[0, :1000], logits[0, 1000:2000] = 0.0, -1.0
    logits[0, 2057::2056] = -9.875
    small = int((logits == -9.875).sum()) * np.exp(-9.875)
    total = 1000 + 1000 * np.exp(-1.0) + small
    top_p, logits = float(np.float32(1000 / (total - small / 8))), logits.cuda()
    got = []
    for seed in range(40):
        seeds = torch.tensor([seed])
        got += ext.sample_tokens(logits, 1.0, top_p, 0, seeds.cuda(),
                                 torch.tensor([0], device="cuda")).tolist()
        assert got[-1:] == _sampled(logits, 1.0, top_p, 0, seeds, 0)
    assert max(got) >= 1000


def test_sampler_sums_small_probabilities(ext):
    """100000 elements of probability 3000.55 * 2^-32, each: a sum that rounds them to
    whole 2^-32 first is 0.45 * 2^-32 * 100000 = 1e-5 too large, reaches a top_p that is
    half of that above the group's share, and drops the group below."""
    V, n = 152064, 100000
    logits = torch.full((160, V), -40.0)
    logits[:, 0] = 0.0
    logits[:, 1:n + 1] = float(np.log(3000.55) - 32 * np.log(2.0))
    logits[:, n + 1:n + 50001] = -14.7
    p = logits[0].double().exp()
    top_p = float((1 + p[1:n + 1].sum() + 0.22 * n * 2.0 ** -32) / p.sum())
    logits, seeds = logits.cuda(), torch.arange(160)
    got = ext.sample_tokens(logits, 1.0, top_p, 0, seeds.cuda(),
                            torch.tensor([3], device="cuda")).tolist()
    assert max(got) > n
    at = [i for i, x in enumerate(got) if x > n] + list(range(4))
    assert [got[i] for i in at] == _sampled(logits[at], 1.0, top_p, 0, seeds[at], 3)


def test_sampler_draw_does_not_hang_on_the_slices(ext):
    """Alone a row is cut into 148 slices, among 640 into eight, and draws the
    same where two keys are next to each other: the logit of one is raised to the
    last value at which it is not drawn and the next one, at which it is. Higher
    elements lie beside it in a short slice and in a long one."""
    B, V, at, temperature = 640, 151936, 1500, 0.7
    seeds, step = torch.arange(B, device="cuda"), torch.zeros(1, dtype=torch.int64, device="cuda")
    logits = torch.full((B, V), -30.0, device="cuda")
    logits[:, 100], logits[:, 1600], logits[:, 9000] = 0.3, 1.1, 1.7
    low, high = (torch.full((B,), x, device="cuda") for x in (-20.0, 20.0))
    for _ in range(60):
        logits[:, at] = (low + high) / 2
        drawn = ext.sample_tokens(logits, temperature, 1.0, 0, seeds, step) == at
        low, high = torch.where(drawn, low, logits[:, at]), torch.where(drawn, logits[:, at], high)
    assert torch.equal(torch.nextafter(low, high), high)
    for x, drawn in ((low, False), (high, True)):
        logits[:, at] = x
        among = ext.sample_tokens(logits, temperature, 1.0, 0, seeds, step).tolist()
        assert all((t == at) == drawn for t in among)
        assert among == [ext.sample_tokens(logits[r:r + 1], temperature, 1.0, 0, seeds[r:r + 1],
                                           step).item() for r in range(B)]


def test_sampler_without_a_finite_maximum(ext):
    """A row with an infinite logit, or none above the lowest finite one, has no
    element that is drawn, and answers 0, however it is cut."""
    V = 32768
    logits = torch.randn(3, V, generator=torch.Generator().manual_seed(1))
    logits[0, 20000] = float("inf")
    logits[1] = torch.finfo(torch.bfloat16).min
    logits = logits.to("cuda", torch.bfloat16)
    step = torch.tensor([0], device="cuda")
    for rows in (logits, logits.repeat(200, 1)):
        for top_p in (1.0, 0.9):
            got = ext.sample_tokens(rows, 1.0, top_p, 0, torch.arange(len(rows), device="cuda"), step)
            assert not got.view(-1, 3)[:, :2].any() and got.view(-1, 3)[:, 2].all()


def test_sampler_in_a_graph(ext):
    """Replays draw anew with the device step and match eager draws."""
    logits = _rand((5, 32768), 2, 3.0)
    seeds, step = torch.arange(5, device="cuda"), torch.zeros(1, dtype=torch.int64, device="cuda")
    for top_p in (1.0, 0.9):
        step.zero_()
        ext.sample_tokens(logits, 1.0, top_p, 0, seeds, step)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = ext.sample_tokens(logits, 1.0, top_p, 0, seeds, step)
        for i in range(4):
            step.fill_(i)
            graph.replay()
            got = out.clone()
            assert torch.equal(got, ext.sample_tokens(logits, 1.0, top_p, 0, seeds, step))


# --------------------------------------------------- paged decode attention
# Bound: the output's rounding, 2^-9 of each value at most; scores and sums are
# fp32 and the weights carry 17 bits.
DECODE_REL = 2.0 ** -8


@pytest.mark.parametrize("H,KV,D", [(28, 4, 128), (5, 5, 128), (10, 2, 128), (14, 2, 64), (8, 8, 64)])
@pytest.mark.parametrize("ctxs,width,bs", [
    ([1, 2, 15, 16, 17, 31, 32, 33], 40, 16), ([100, 255, 256, 257, 511, 512, 513], 520, 16),
    ([2048, 1, 1025], 2048, 16), ([5000, 3, 2049, 257], 5000, 16), ([77, 300], 333, 12),
    ([400 + i for i in range(130)], 560, 16), ([60], 64, 1)])
def test_paged_decode_edges(ext, H, KV, D, ctxs, width, bs):
    """Chunk ends, one and several slices (also empty ones), eight and four
    waves, page sizes that are no power of two; pages in random order, some
    shared, and NaN in every row that no sequence holds."""
    g = torch.Generator().manual_seed(len(ctxs) + H)
    nb = (width + bs - 1) // bs
    pages = nb * len(ctxs)
    bt = torch.randperm(pages, generator=g).view(len(ctxs), nb).int()
    bt[:, 0] = bt[0, 0]
    q, kc, vc = (_rand(s, i) for i, s in enumerate(
        ((len(ctxs), H, D), (pages, bs, KV, D), (pages, bs, KV, D))))
    used = torch.zeros(pages, bs, dtype=torch.bool)
    for i, n in enumerate(ctxs):
        t = torch.arange(n)
        used[bt[i, t // bs].long(), t % bs] = True
    kc[~used.cuda()] = float("nan")
    vc[~used.cuda()] = float("nan")
    lens = torch.tensor(ctxs, dtype=torch.int32)
    for scale in (D ** -0.5, -1.0):
        out = ext.paged_attention_decode(q, kc, vc, bt.cuda(), lens.cuda(), scale)
        for i, n in enumerate(ctxs):
            t = torch.arange(n)
            k, v = (c[bt[i, t // bs].long().cuda(), (t % bs).cuda()].double().transpose(0, 1)
                    .repeat_interleave(H // KV, 0) for c in (kc, vc))
            p = ((k @ q[i].double().unsqueeze(2)).squeeze(2) * scale).softmax(-1)
            assert _rel(out[i], (p.unsqueeze(1) @ v).squeeze(1)) < DECODE_REL, (i, n)


@pytest.mark.parametrize("N,nb", [(3, 5), (3, 129), (300, 9)])
def test_paged_decode_stays_in_its_table(ext, N, nb):
    """A context length beyond the block table counts as the table's end, with
    one slice and with several."""
    H, KV, D, bs = 8, 2, 128, 16
    kc, vc = _rand((nb + 1, bs, KV, D), 1), _rand((nb + 1, bs, KV, D), 2)
    bt = torch.randperm(nb, generator=torch.Generator().manual_seed(N)).int().expand(N, -1)
    bt, q = bt.contiguous().cuda(), _rand((N, H, D), 3)
    lens = torch.full((N,), nb * bs, dtype=torch.int32, device="cuda")
    ref = ext.paged_attention_decode(q, kc, vc, bt, lens, 0.1)
    lens[::2] += 3 * bs * nb + 5
    assert torch.equal(ext.paged_attention_decode(q, kc, vc, bt, lens, 0.1), ref)


def test_paged_decode_slices_in_a_graph(ext):
    """Slices of a context find each other in every replay of a capture."""
    H, KV, D, bs, nb = 8, 2, 64, 16, 130
    kc, vc = (_rand((3 * nb, bs, KV, D), i) for i in (1, 2))
    q = _rand((3, H, D), 3)
    bt = torch.randperm(3 * nb, generator=torch.Generator().manual_seed(0)).view(3, nb).int().cuda()
    lens = torch.tensor([2080, 1, 1300], dtype=torch.int32, device="cuda")
    ref = ext.paged_attention_decode(q, kc, vc, bt, lens, 0.125)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ext.paged_attention_decode(q, kc, vc, bt, lens, 0.125)
    for _ in range(5):
        out.zero_()
        graph.replay()
        assert torch.equal(out, ref)
        assert torch.equal(ext.paged_attention_decode(q, kc, vc, bt, lens, 0.125), ref)


def test_paged_decode_reads_packed_rows(ext):
    """Query heads at the head of wider rows, at any alignment."""
    H, KV, D, N = 14, 2, 64, 3
    kc, vc = _rand((9, 16, KV, D), 1), _rand((9, 16, KV, D), 2)
    bt = torch.arange(9, dtype=torch.int32).view(3, 3).cuda()
    lens = torch.tensor([48, 7, 33], dtype=torch.int32, device="cuda")
    q = _rand((N, H, D), 3)
    ref = ext.paged_attention_decode(q, kc, vc, bt, lens, 0.125)
    for stride in (H * D + 2 * KV * D, H * D + 3):
        flat = torch.zeros(N * stride + 1, dtype=torch.bfloat16, device="cuda")
        for off in (0, 1):
            rows = flat[off:off + N * stride].view(N, stride)
            rows[:, :H * D] = q.view(N, -1)
            out = ext.paged_attention_decode_strided(rows, H, D, stride, kc, vc, bt, lens, 0.125)
            assert torch.equal(out, ref)


# ----------------------------------------------------- fused layer, rotary

def _train_model(name, lora_r=8, **kw):
    from distrl_llm_amd.models import CausalLM, get_spec
    model = CausalLM(get_spec(name) if isinstance(name, str) else name, lora_r=lora_r,
                     lora_alpha=16, dtype=torch.bfloat16, device=torch.device("cuda"),
                     **kw).random_init(3)
    g = torch.Generator(device="cuda").manual_seed(5)
    with torch.no_grad():
        for n, p in model.named_parameters():
            if n.endswith(("lora_B", "bias")):
                p.copy_(torch.randn(p.shape, generator=g, device="cuda") * 0.05)
            elif "norm" in n:
                p.copy_(1 + 0.1 * torch.randn(p.shape, generator=g, device="cuda"))
    return model.train()


def _kernels(call):
    """What the call returns, and how often a kernel of a name ran in it."""
    from torch.profiler import ProfilerActivity, profile
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        out = call()
        torch.cuda.synchronize()
    counts = [(e.key, e.count) for e in prof.key_averages()]
    assert counts
    return out, lambda name: sum(n for key, n in counts if name in key)


def _grads(model, ids, mask, dout):
    out = model.forward_hidden(ids, mask)
    params = [p for p in model.parameters() if p.requires_grad]
    return [out.detach(), *torch.autograd.grad(out, params, dout)]


@pytest.mark.parametrize("name", ["small-qwen2", "small-qwen3"])
@pytest.mark.parametrize("B,T", [(1, 1), (2, 77), (3, 200)])
@pytest.mark.parametrize("lora_r", [8, 32, 64])
def test_fused_layer_matches_modules(name, B, T, lora_r):
    """Hidden states and adapter gradients against the same model in fp64 on
    the CPU: no further off than the module path (1.3 times leaves room for
    other roundings of the same size), with padding at the ends; at a rank that
    the library's products take and at two that ours do."""
    from distrl_llm_amd.models import CausalLM, fused_layer
    model = _train_model(name, lora_r=lora_r)
    g = torch.Generator().manual_seed(T)
    ids = torch.randint(0, model.spec.vocab_size, (B, T), generator=g).cuda()
    lens = torch.randint(max(1, T // 2), T + 1, (B,), generator=g)
    mask = (torch.arange(T)[None] < lens[:, None]).long().cuda()
    dout = _rand((B, T, model.spec.hidden_size), 9) * mask.unsqueeze(-1)
    exact = CausalLM(model.spec, lora_r=lora_r, lora_alpha=16, dtype=torch.float64)
    exact.load_state_dict({k: v.double().cpu() for k, v in model.state_dict().items()})
    ref = _grads(exact.train(), ids.cpu(), mask.cpu(), dout.double().cpu())
    real = mask.bool().cpu()
    (fused, ran) = _kernels(lambda: _grads(model, ids, mask, dout))
    # a layer: q|k|v, o, gate|up, down and back, but to the embedding
    assert ran("product_kernel") == (0 if lora_r % 32 else 8 * model.spec.num_layers - 1)
    usable = fused_layer.usable
    fused_layer.usable = lambda layer, x: False
    try:
        plain = _grads(model, ids, mask, dout)
    finally:
        fused_layer.usable = usable
    fused, plain, ref = ([x.double().cpu() for x in xs] for xs in (fused, plain, ref))
    fused[0], plain[0], ref[0] = (xs[0][real] for xs in (fused, plain, ref))
    assert _rel(fused[0], ref[0]) < 1.3 * _rel(plain[0], ref[0]) + 2.0 ** -9
    # the adapters' gradients together: one tensor's alone, from few tokens, is
    # a single rounding or two of luck
    fused, plain, ref = (torch.cat([x.reshape(-1) for x in xs[1:]]) for xs in (fused, plain, ref))
    assert _rel(fused, ref) < 1.3 * _rel(plain, ref) + 2.0 ** -9


@pytest.mark.parametrize("B,T", [(1, 1), (2, 77)])
@pytest.mark.parametrize("lora_r,norms", [(8, False), (12, True), (32, False), (96, False)])
def test_fused_layer_takes_large_weights_as_they_lie(B, T, lora_r, norms):
    """Few rows of a layer whose products are all past the size where weights
    are no longer laid out beside their adapters, at ranks that the joining
    kernel takes and that it does not, and at two that go through our own products:
    against fp64, as above."""
    from distrl_llm_amd.models import CausalLM, fused_layer
    from distrl_llm_amd.models.spec import ModelSpec
    spec = ModelSpec("wide", 64, 4096, 8192, 1, 64, 8, 128, 1e6, 1e-6, True, not norms,
                     qk_norm=norms)
    model = _train_model(spec, lora_r=lora_r)
    g = torch.Generator().manual_seed(T)
    ids = torch.randint(0, 64, (B, T), generator=g).cuda()
    mask, dout = torch.ones_like(ids), _rand((B, T, 4096), 9)
    exact = CausalLM(spec, lora_r=lora_r, lora_alpha=16, dtype=torch.float64)
    exact.load_state_dict({k: v.double().cpu() for k, v in model.state_dict().items()})
    ref = _grads(exact.train(), ids.cpu(), mask.cpu(), dout.double().cpu())
    fused, ran = _kernels(lambda: _grads(model, ids, mask, dout))
    assert ran("product_kernel") == (0 if lora_r % 32 else 7)
    usable = fused_layer.usable
    fused_layer.usable = lambda layer, x: False
    try:
        plain = _grads(model, ids, mask, dout)
    finally:
        fused_layer.usable = usable
    for part in (slice(0, 1), slice(1, None)):
        got, base, want = (torch.cat([x.double().cpu().reshape(-1) for x in xs[part]])
                           for xs in (fused, plain, ref))
        assert _rel(got, want) < 1.3 * _rel(base, want) + 2.0 ** -9


def test_fused_layer_steps_aside():
    """Hooks, dropout, inference and frozen shapes keep the modules."""
    from distrl_llm_amd.models import fused_layer
    model = _train_model("small-qwen2")
    layer = model.model.layers[0]
    x = _rand((1, 5, model.spec.hidden_size), 1)
    assert fused_layer.usable(layer, x)
    with torch.no_grad():
        assert not fused_layer.usable(layer, x)
    assert not fused_layer.usable(layer, x.float())
    seen = []
    handle = layer.mlp.up_proj.register_forward_hook(lambda m, i, o: seen.append(o))
    model.forward_hidden(torch.zeros(1, 5, dtype=torch.long, device="cuda"))
    assert len(seen) == 1
    handle.remove()
    assert fused_layer.usable(layer, x)
    handle = torch.nn.modules.module.register_module_forward_hook(
        lambda m, i, o: seen.append(m) if m is layer.mlp.up_proj else None)
    model.forward_hidden(torch.zeros(1, 5, dtype=torch.long, device="cuda"))
    handle.remove()
    assert len(seen) == 2
    norm, layer.input_layernorm = layer.input_layernorm, torch.nn.Identity()
    assert not fused_layer.usable(layer, x)
    layer.input_layernorm = norm
    layer.mlp.down_proj.bias = torch.nn.Parameter(x[0, 0].clone(), requires_grad=False)
    assert not fused_layer.usable(layer, x)
    layer.mlp.down_proj.bias = None
    layer.mlp.forward = lambda y: y
    assert not fused_layer.usable(layer, x)
    del layer.mlp.forward
    assert fused_layer.usable(layer, x)
    dropped = _train_model("small-qwen2", lora_dropout=0.1).model.layers[0]
    assert not fused_layer.usable(dropped, x)
    assert fused_layer.usable(dropped.eval(), x)


@pytest.mark.parametrize("part", ["self_attn.k_proj", "self_attn.o_proj", "mlp.up_proj",
                                  "mlp.down_proj", "input_layernorm", "post_attention_layernorm"])
def test_fused_layer_notices_changed_weights(part):
    """A weight written in place between the passes: an error, as with the
    modules, not the gradient of another weight."""
    model = _train_model("small-qwen2")
    out = model.forward_hidden(torch.zeros(1, 5, dtype=torch.long, device="cuda"))
    with torch.no_grad():
        model.model.layers[1].get_submodule(part).weight.mul_(2.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.float().sum().backward()


@pytest.mark.parametrize("T,H,KV,D", [(1, 1, 1, 16), (5, 14, 2, 64), (9, 28, 4, 128), (7, 3, 1, 24),
                                      (6, 4, 2, 48)])
def test_rope_inplace_units(ext, T, H, KV, D):
    """Vector and element rotation at odd head counts and sizes. Bound: one
    bf16 rounding, and the fast sine's 2^-10 at these angles."""
    q, k = _rand((T, H, D), 1), _rand((T, KV, D), 2)
    pos = torch.randint(0, 3000, (T,), dtype=torch.int32, device="cuda")
    inv = 1.0 / (1e4 ** (torch.arange(0, D, 2, device="cuda").float() / D))
    a = (pos.double()[:, None] * inv.double())[:, None]
    ref = []
    for x in (q, k):
        x1, x2 = x.double().chunk(2, -1)
        ref.append(torch.cat([x1 * a.cos() - x2 * a.sin(), x2 * a.cos() + x1 * a.sin()], -1))
    ext.rope_inplace(q, k, pos, inv)
    assert _rel(q, ref[0]) < 2.0 ** -8 and _rel(k, ref[1]) < 2.0 ** -8


@pytest.mark.parametrize("rows,hidden", [(1, 8), (3, 896), (2, 2056)])
def test_rmsnorm_bwd_add(ext, rows, hidden):
    """One rounding of the sum instead of two."""
    x, dy, g = (_rand((rows, hidden), i) for i in range(3))
    w = _rand((hidden,), 4)
    xr = x.double().requires_grad_()
    y = xr * torch.rsqrt((xr * xr).mean(-1, keepdim=True) + 1e-6) * w.double()
    ref = g.double() + torch.autograd.grad(y, xr, dy.double())[0]
    assert _rel(ext.rmsnorm_bwd_add(dy, x, w, g, 1e-6), ref) < 2.0 ** -9


# ------------------------------------------------------------ skinny products

@pytest.mark.parametrize("M", [1, 8, 15, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(16, 512), (896, 896), (2064, 544), (4112, 4864), (256, 8960)])
def test_skinny_gemm(ext, M, N, K):
    """Every wave count and row tile, K that does not divide among the waves;
    bias, residual with an adapter, SiLU*mul, with and without the norm.
    Bounds: one rounding of the result (2^-9) over fp32 sums; the norm rounds
    its output first, SiLU*mul its two inputs."""
    x, w, b = _rand((M, K), 1), _rand((2 * N, K), 2, K ** -0.5), _rand((N,), 3)
    res, u, ub = _rand((M, N), 4), _rand((M, 64), 5), _rand((N, 64), 6, 0.1)
    nw = _rand((K,), 7, 0.1) + 1
    xd, wd = x.double(), w[:N].contiguous()
    assert _rel(ext.skinny_gemm(x, wd, 0), xd @ wd.double().t()) < 2.0 ** -8
    assert _rel(ext.skinny_gemm(x, wd, 0, b), xd @ wd.double().t() + b.double()) < 2.0 ** -8
    ref = res.double() + xd @ wd.double().t()
    assert _rel(ext.skinny_gemm(x, wd, 1, res=res), ref) < 2.0 ** -8
    assert _rel(ext.skinny_gemm(x, wd, 1, res=res, u=u, ub=ub),
                ref + u.double() @ ub.double().t()) < 2.0 ** -8
    assert not ext.skinny_gemm_takes(33, N, K)          # one row further
    normed = xd * torch.rsqrt((xd * xd).mean(-1, keepdim=True) + 1e-6) * nw.double()
    for inp, kw, bound in ((xd, {}, 2.0 ** -7), (normed, {"norm_w": nw, "eps": 1e-6}, 2.0 ** -6)):
        gate, up = (inp @ w.double().t()).chunk(2, -1)
        assert _rel(ext.skinny_gemm(x, w, 2, **kw), torch.nn.functional.silu(gate) * up) < bound
        assert _rel(ext.skinny_gemm(x, wd, 0, b, **kw),
                    inp @ wd.double().t() + b.double()) < bound


def test_skinny_gemm_operands_anywhere(ext):
    """Each operand in turn at an odd element of a buffer: the same results."""
    M, N, K, R = 5, 64, 512, 32

    def odd(t):
        flat = t.new_empty(t.numel() + 1)
        flat[1:] = t.reshape(-1)
        return flat[1:].view(t.shape)

    ops = {"x": _rand((M, K), 1), "w": _rand((N, K), 2, 0.05), "bias": _rand((N,), 3),
           "norm_w": _rand((K,), 4), "res": _rand((M, N), 5), "u": _rand((M, R), 6),
           "ub": _rand((N, R), 7)}
    for mode, names in ((0, ("x", "w", "bias", "norm_w")), (1, ("x", "w", "res", "u", "ub"))):
        ref = ext.skinny_gemm(mode=mode, eps=1e-6, **{n: ops[n] for n in names})
        for name in names:
            args = {n: odd(ops[n]) if n == name else ops[n] for n in names}
            assert torch.equal(ext.skinny_gemm(mode=mode, eps=1e-6, **args), ref), name


@pytest.mark.parametrize("V,dtype", [(24000, torch.bfloat16), (20481, torch.float32), (4100, torch.bfloat16)])
@pytest.mark.parametrize("top_p,top_k", [(1.0, 0), (0.5, 0), (1.0, 1)])
def test_draws_at_chunk_edges(ext, V, dtype, top_p, top_k):
    """The one likely element of each of 700 rows, which are slices of up to ten chunks,
    at the edges of threads' pieces and of chunks, where nearly all of them keep none."""
    places = [p for e in range(0, V, 2048) for p in (e - 1, e, e + 7, e + 8, e + 511) if 0 <= p < V] + [V - 1]
    at = torch.tensor([places[i % len(places)] for i in range(700)], device="cuda")
    logits = torch.zeros(700, V, dtype=dtype, device="cuda")
    logits.scatter_(1, at[:, None], 40.0)
    for seed in range(3):
        seeds = torch.arange(700, device="cuda") + 1000 * seed
        step = torch.tensor([seed], device="cuda")
        assert torch.equal(ext.sample_tokens(logits, 1.0, top_p, top_k, seeds, step), at)


@pytest.mark.parametrize("n", [1, 60, 61, 125])
@pytest.mark.parametrize("page,dtype", [((16, 4, 128), torch.bfloat16), ((1, 1, 8), torch.bfloat16),
                                        ((5, 3, 20), torch.float32), ((1, 1, 4), torch.bfloat16)])
def test_page_copies(n, page, dtype):
    """One page of every layer to n others, past what one launch takes; a page of 8 bytes,
    which is copied by torch."""
    from distrl_llm_amd.engine.kvcache import KVCachePool
    pool = KVCachePool(3, 130, *page, dtype, "cuda")
    pool.key.normal_()
    pool.value.normal_()
    want = pool.key.clone(), pool.value.clone()
    dsts = [d for d in torch.randperm(130, generator=torch.Generator().manual_seed(n)).tolist() if d != 7][:n]
    for t in want:
        t[:, dsts] = t[:, 7:8]
    pool.copy_to(7, dsts)
    assert torch.equal(pool.key, want[0]) and torch.equal(pool.value, want[1])
    if page != (1, 1, 4):
        with pytest.raises(RuntimeError, match="no such page"):
            pool.copy_to(7, [130])


@pytest.mark.parametrize("D,H,KV", [(64, 3, 1), (128, 28, 4)])
def test_rope_scatter_norms(ext, D, H, KV):
    """Per-head norms, rotation and cache write of packed projections, a
    skipped slot among them, against the separate kernels."""
    T = 5
    qkv, wq, wk = _rand((T, (H + 2 * KV) * D), 1), _rand((D,), 2, 0.1) + 1, _rand((D,), 3, 0.1) + 1
    pos = torch.randint(0, 2000, (T,), dtype=torch.int32, device="cuda")
    slots = torch.tensor([3, -1, 40, 0, 17], device="cuda")
    inv = 1.0 / (1e4 ** (torch.arange(0, D, 2, device="cuda").float() / D))
    for norms in ((), (wq, wk, 1e-6)):
        q, k, v = (t.reshape(T, -1, D).contiguous()
                   for t in qkv.split([H * D, KV * D, KV * D], 1))
        if norms:
            q, k = ext.rmsnorm_fwd(q, wq, 1e-6), ext.rmsnorm_fwd(k, wk, 1e-6)
        ext.rope_inplace(q, k, pos, inv)
        kc, vc = torch.zeros(2, 3, 16, KV, D, dtype=torch.bfloat16, device="cuda")
        ext.kv_cache_scatter(k, v, kc, vc, slots.int())
        packed, kc2, vc2 = qkv.clone(), torch.zeros_like(kc), torch.zeros_like(vc)
        ext.rope_scatter_qkv(packed, pos, slots, inv, kc2, vc2, H, KV, D, *norms)
        # norm sums in another order: the last bit may differ
        assert _rel(packed[:, :H * D].reshape(q.shape), q) < 2.0 ** -9
        assert _rel(kc2, kc) < 2.0 ** -9
        assert torch.equal(vc2, vc)


# ---------------------------------------------- merged weights, prompt phase

@pytest.mark.parametrize("N,K,r", [(1, 32, 8), (17, 288, 8), (130, 256, 32), (128, 1056, 40),
                                   (70, 544, 128)])
def test_lora_merge(ext, N, K, r):
    """Row and column remainders, ranks that do not fill a product step. One
    rounding of an fp32 sum."""
    w, a, b = _rand((N, K), 1), _rand((r, K), 2, 0.3), _rand((N, r), 3, 0.3)
    out = torch.full((N + 1, K), float("nan"), dtype=torch.bfloat16, device="cuda")
    assert ext.lora_merge(w, a, b, out[:N], 0.5)
    assert _rel(out[:N], w.double() + 0.5 * b.double() @ a.double()) < 2.0 ** -9
    assert bool(out[N].isnan().all())


@pytest.mark.parametrize("M,N,r", [(1, 32, 8), (17, 288, 8), (130, 256, 32), (129, 1056, 40),
                                   (70, 544, 96), (33, 64, 128)])
def test_lora_add(ext, M, N, r):
    """In place on rows cut out of wider ones, the matrix in both layouts."""
    wide, uw, m = _rand((M, N + 64), 1), _rand((M, r + 32), 2), _rand((r, N), 3, 0.3)
    before = wide.clone()
    ref = before[:, 32:32 + N].double() + 0.5 * uw[:, 16:16 + r].double() @ m.double()
    for mat in (m, m.t().contiguous().t()):
        wide.copy_(before)
        assert ext.lora_add(wide[:, 32:32 + N], uw[:, 16:16 + r], mat, 0.5)
        assert _rel(wide[:, 32:32 + N], ref) < 2.0 ** -8
        assert torch.equal(wide[:, :32], before[:, :32])
        assert torch.equal(wide[:, 32 + N:], before[:, 32 + N:])
    wide.copy_(before)
    res = _rand((M, N + 32), 4)[:, 16:16 + N]
    assert ext.lora_add(wide[:, 32:32 + N], uw[:, 16:16 + r], m, 0.5, res)
    assert _rel(wide[:, 32:32 + N], ref + res.double()) < 2.0 ** -8
    # refused, nothing written: unaligned rows, strided columns, other types
    assert not ext.lora_add(wide[:, 4:4 + N], uw[:, 16:16 + r], m, 0.5)
    assert not ext.lora_add(wide[:, :N], uw[:, 4:4 + r], m, 0.5)
    assert not ext.lora_add(wide[:, :N], uw[:, :r].float(), m, 0.5)
    assert not ext.lora_add(wide[:, :N], uw[:, :r], m.flip(0)[:, ::2], 0.5)
    if M > 1:
        same, over = _rand((1, N), 5).expand(M, N), _rand((M * 32 + N,), 6).as_strided((M, N), (16, 1))
        for y in (same, over):
            assert not ext.lora_add(y, uw[:, 16:16 + r], m, 0.5)
    assert torch.equal(wide[:, :32], before[:, :32])


@pytest.mark.parametrize("name", ["small-qwen2", "small-qwen3"])
@pytest.mark.parametrize("lora_r,four_bit", [(0, False), (8, False), (8, True), (12, False),
                                             (32, False), (64, True)])
def test_packed_prefill_matches_modules(ext, monkeypatch, name, lora_r, four_bit):
    """Logits and cache rows of a ragged batch against the module path (two
    bf16 paths of the same products: 2 %), and the merged weights against
    W + scale * B A at a rank the kernel takes and one it does not."""
    from distrl_llm_amd.config import EngineConfig
    from distrl_llm_amd.engine import Engine
    from distrl_llm_amd.engine.kvcache import Sequence
    from distrl_llm_amd.models import CausalLM, get_spec
    model = CausalLM(get_spec(name), lora_r=lora_r, lora_alpha=16, dtype=torch.bfloat16,
                     device=torch.device("cuda")).random_init(3).eval()
    with torch.no_grad():
        for n, p in model.named_parameters():
            if n.endswith(("lora_B", "bias")):
                p.copy_(_rand(p.shape, 7, 0.05))
    if four_bit:
        model.quantize_nf4_()
    g = torch.Generator().manual_seed(1)
    prompts = [torch.randint(0, 4096, (n,), generator=g).tolist() for n in (3, 64, 129, 1)]
    got, own = [], []
    for f in ("adapted_projection", "adapted_activation"):
        monkeypatch.setattr(ext, f, lambda *a, _f=getattr(ext, f): own.append(_f(*a)) or own[-1])
    for packs in (True, False):
        eng = Engine(model, EngineConfig(max_seq_length=256, num_kv_blocks=32, max_num_seqs=8))
        eng.fused.refresh()
        if not packs:
            eng._prefill_packs = lambda: False
        logits = eng._prefill_batch([Sequence(i, p, i) for i, p in enumerate(prompts)])
        got.append((logits, eng.pool.key, eng.pool.value))
    for x, y in zip(*got):
        assert _rel(x, y) < 0.02
    # every site through our products, or through the library's
    assert len(own) == 4 * model.spec.num_layers
    assert all((x is None) == (lora_r % 32 != 0) for x in own)
    at = model.model.layers[1].self_attn
    w = at.k_proj.weight.double()
    if lora_r:
        w = w + at.k_proj.scale * at.k_proj.lora_B.double() @ at.k_proj.lora_A.double()
    q = model.spec.q_size
    assert _rel(eng.fused.layers[1].rows("qkv")[q:q + model.spec.kv_size], w) < 2.0 ** -8


def test_packed_prefill_after_a_changed_bias():
    """Weights and biases written in place between two generations."""
    from distrl_llm_amd.config import EngineConfig
    from distrl_llm_amd.engine import Engine
    from distrl_llm_amd.engine.kvcache import Sequence
    from distrl_llm_amd.models import CausalLM, get_spec
    model = CausalLM(get_spec("small-qwen2"), dtype=torch.bfloat16,
                     device=torch.device("cuda")).random_init(3).eval()
    eng = Engine(model, EngineConfig(max_seq_length=64, num_kv_blocks=32, max_num_seqs=8))
    eng.fused.refresh()
    at = model.model.layers[0].self_attn
    with torch.no_grad():
        at.k_proj.bias.add_(3.0)
        at.v_proj.weight.mul_(-1.0)
    eng.fused.refresh()
    logits = [eng._prefill_batch([Sequence(0, [5, 6, 7], 0)])]
    key = eng.pool.key.clone()
    eng._prefill_packs = lambda: False
    eng.pool.allocator.reset()
    logits.append(eng._prefill_batch([Sequence(1, [5, 6, 7], 1)]))
    assert _rel(*logits) < 0.02 and _rel(key, eng.pool.key) < 0.02


@pytest.mark.parametrize("part", ["layers.1.self_attn.q_proj", "layers.0.mlp.down_proj", "norm",
                                  "layers.1.input_layernorm", None])
def test_packed_prefill_leaves_hooks_their_modules(part):
    """A hook on a module, or on all of them, sees the prompt's rows."""
    from distrl_llm_amd.config import EngineConfig, SamplingParams
    from distrl_llm_amd.engine import Engine
    from distrl_llm_amd.models import CausalLM, get_spec
    model = CausalLM(get_spec("small-qwen2"), lora_r=8, dtype=torch.bfloat16,
                     device=torch.device("cuda")).random_init(3).eval()
    eng = Engine(model, EngineConfig(max_seq_length=64, num_kv_blocks=32, max_num_seqs=8))
    mod, seen = model.model.get_submodule(part or "layers.0.mlp.gate_proj"), []

    def hook(m, i, o):
        if m is mod:
            seen.append(o.shape[0])

    handle = (mod.register_forward_hook(hook) if part
              else torch.nn.modules.module.register_module_forward_hook(hook))
    try:
        eng.generate([[5, 6, 7]], SamplingParams(max_tokens=2, temperature=0.0))
    finally:
        handle.remove()
    assert seen == [3]
    assert eng._prefill_packs()


@pytest.mark.parametrize("env", [("DISTRL_HYBRID_DOWN", "1"), ("DISTRL_DECODE_NF4", "1")])
@pytest.mark.parametrize("n", [1, 40])
def test_four_bit_decode_without_adapter(monkeypatch, env, n):
    """A 4-bit model with no adapter through the 4-bit kernels (few rows and
    many) against its bf16 image: the cache rows that a decode step writes (two
    bf16 paths of the same products: 2 %)."""
    from distrl_llm_amd.config import EngineConfig, SamplingParams
    from distrl_llm_amd.engine import Engine
    from distrl_llm_amd.models import CausalLM, get_spec
    model = CausalLM(get_spec("small-qwen2"), dtype=torch.bfloat16,
                     device=torch.device("cuda")).random_init(3).eval()
    model.quantize_nf4_()
    pools = []
    for name, value in (env, ("DISTRL_HYBRID_DOWN", "0")):
        with monkeypatch.context() as m:
            m.setenv(name, value)
            eng = Engine(model, EngineConfig(max_seq_length=64, num_kv_blocks=128, max_num_seqs=64))
            assert (eng.fused.nf4 or eng.fused.hybrid_down) == (value == "1")
            eng.generate([[1, 2, 3, 4, 5]], SamplingParams(max_tokens=2, temperature=0.0, n=n))
            pools.append(torch.stack([eng.pool.key, eng.pool.value]))
    assert _rel(*pools) < 0.02


# ------------------------------------------------------------------- loss

@pytest.mark.parametrize("B,T,V,dtype", [
    (1, 1, 8, "bfloat16"), (2, 3, 4095, "bfloat16"), (17, 5, 4104, "bfloat16"),
    (3, 70, 6000, "float32"), (2, 2, 152064, "bfloat16")])
@pytest.mark.parametrize("mask_dtype", [torch.int64, torch.bool, torch.float32])
def test_loss_edges(B, T, V, dtype, mask_dtype):
    """Vector remainders and odd row places, more sequences than waves, empty
    masks, each mask type, a scaled loss. fp32 sums: 1e-5 of the largest term;
    the gradient is rounded to the logits' type once."""
    from distrl_llm_amd.ops import functional as OF
    g = torch.Generator().manual_seed(V)
    logits = (torch.randn(B, T, V, generator=g) * 3).to("cuda", getattr(torch, dtype))
    logits[..., 1] = float("-inf")
    targets = torch.randint(2, V, (B, T), generator=g).cuda()
    mask = (torch.rand(B, T, generator=g) < 0.7).to(mask_dtype).cuda()
    mask[-1] = 0
    rewards = torch.randn(B, generator=g).cuda()
    leaf = logits.detach().requires_grad_()
    loss = OF.logprob_loss(leaf, targets, mask, rewards, 0.25)
    grad, = torch.autograd.grad(loss * 3.0, leaf)
    exact = logits.double().requires_grad_()
    m = mask.double()
    tok = exact.log_softmax(-1).gather(-1, targets.unsqueeze(-1)).squeeze(-1)
    ref = -((tok * m).sum(-1) / m.sum(-1).clamp_min(1) * rewards.double()).mean() * 0.25
    ref_grad, = torch.autograd.grad(ref * 3.0, exact)
    ref_grad = ref_grad.nan_to_num(0.0)
    loss, ref, tok = loss.detach(), ref.detach(), tok.detach()
    assert abs(float(loss) - float(ref)) < 1e-5 * float((tok * m).abs().max() * rewards.abs().max()
                                                        + 1e-30)
    if float(ref_grad.norm()) == 0.0:
        assert float(grad.float().abs().max()) == 0.0
    else:
        assert _rel(grad, ref_grad) < (2.0 ** -8 if dtype == "bfloat16" else 1e-5)


@pytest.mark.parametrize("B,T,V", [(3, 1300, 301), (1, 20000, 64), (2, 2600, 513), (41, 60, 8192),
                                   (300, 6, 4097), (2, 150, 40000), (290, 1, 70001), (3, 3, 152065),
                                   (2, 1500, 20000), (2, 1200, 40000)])
@pytest.mark.parametrize("mask_dtype", [torch.int64, torch.float32])
def test_masked_loss_gradients_made_forward(B, T, V, mask_dtype):
    """Losses large enough for the gradient to be made in the forward pass: an empty mask,
    parts of a token, more tokens than a workgroup has threads and fewer, weights made of
    a row's mask and ahead, rows that walk, of every number of threads, a target that is no word (its gradient is the softmax alone).
    What forward made, what is made anew behind it in a kept graph and what is made of a
    scaled loss. The first two have the same weights: a first token of 2^24 that swallows
    others' ones makes its sequence's sum hang on the order, and each 2^-24 by which weights
    differ moves 2^-16 of the values over a bf16 edge. Loss sums in fp32, the gradient
    rounds to bf16 once."""
    from distrl_llm_amd.ops import functional as OF
    g = torch.Generator().manual_seed(V)
    gd = torch.Generator("cuda").manual_seed(V)
    leaf = torch.randn(B, T, V, generator=gd, device="cuda").mul_(3).bfloat16()
    leaf[..., 1] = float("-inf")
    targets = torch.randint(2, V, (B, T), generator=g).cuda()
    targets[0, 0] = -100
    mask = torch.rand(B, T, generator=g).mul_(1.2)
    mask = (mask if mask_dtype == torch.float32 else mask < 0.8).to(mask_dtype).cuda()
    if mask_dtype == torch.float32:
        mask[:, 0] = 2.0 ** 24
    mask[1:][-1:] = 0
    rewards = torch.randn(B, generator=g).cuda()
    leaf.requires_grad_()
    assert leaf.numel() >= 1 << 20
    loss = OF.logprob_loss(leaf, targets, mask, rewards, 0.25)
    first, = torch.autograd.grad(loss, leaf, retain_graph=True)
    second, = torch.autograd.grad(loss, leaf, retain_graph=True)
    assert float((first != second).float().mean()) < 2.0 ** -14
    scaled, = torch.autograd.grad(loss * 3.0, leaf)
    m = mask.double()
    w = m * (-rewards.double() / m.sum(-1).clamp_min(1) / B * 0.25)[:, None]
    tok, bad, size = 0.0, 0.0, 0.0
    for b in range(B):                                  # fp64 of one sequence at a time
        logp = leaf[b].detach().double().log_softmax(-1)
        hot = torch.zeros_like(logp)
        there = (targets[b] >= 0).nonzero()[:, 0]
        hot[there, targets[b, there]] = 1.0
        ref = w[b][:, None] * (hot - logp.exp())
        lse = leaf[b].detach().double().logsumexp(-1)
        t = torch.where(targets[b] >= 0, logp.gather(-1, targets[b].clamp_min(0)[:, None])[:, 0], -lse)
        tok += float((w[b] * t).sum())
        bad += float((first[b].double() - ref).square().sum())
        bad += float((scaled[b].double() / 3 - ref).square().sum())
        size += 2 * float(ref.square().sum())
        if mask[b].count_nonzero() == 0:
            assert first[b].count_nonzero() == 0 and scaled[b].count_nonzero() == 0
    assert (bad / max(size, 1e-60)) ** 0.5 < 2.0 ** -8 or size == 0
    assert abs(float(loss) - tok) < 1e-5 * float((w.abs() * 20).sum() + 1e-30)


@pytest.mark.parametrize("off,V", [(1, 4096), (3, 4103), (0, 32003), (1, 7)])
def test_loss_rows_at_any_element(ext, off, V):
    """A matrix that starts inside another and rows of an odd vocabulary give
    what aligned ones do, forward bit for bit; the gradient rounds once."""
    rows = 5
    flat = _rand((rows * V + off,), V, 3.0)
    logits, targets = flat[off:].view(rows, V), torch.arange(rows, device="cuda")
    w = torch.linspace(0.0, 1.0, rows, device="cuda")
    tok, lse = ext.logprob_lse_fwd(logits, targets)
    grad = ext.logprob_loss_bwd(logits, targets, w, lse)
    logp = logits.double().log_softmax(-1)
    ref = w.double()[:, None] * (torch.nn.functional.one_hot(targets, V) - logp.exp())
    assert torch.allclose(tok.double(), logp[torch.arange(rows), targets], rtol=0, atol=1e-5)
    assert _rel(grad, ref) < 2.0 ** -8
    aligned = logits.clone()
    assert all(torch.equal(a, b) for a, b in zip((tok, lse), ext.logprob_lse_fwd(aligned, targets)))


@pytest.mark.parametrize("off,V", [(1, 32767), (0, 32768), (3, 32775), (2, 65539)])
def test_loss_long_rows_at_any_element(ext, off, V):
    """Either side of the gradient's rule for 1024 threads a row."""
    test_loss_rows_at_any_element(ext, off, V)


@pytest.mark.parametrize("lead,mask_shape,reward_shape,host", [
    ((6,), (6,), (), False), ((6,), (6,), (1,), False), ((3, 6), (3, 6), (), False),
    ((3, 6), (3, 6), (1,), False), ((3, 6), (1, 6), (3,), False), ((3, 6), (6,), (3,), False),
    ((3, 6), (3, 1), (3,), False), ((3, 6), (3, 6), (), True), ((2, 3, 6), (3, 6), (2, 3), False)])
def test_loss_broadcasts(lead, mask_shape, reward_shape, host):
    """Shapes that torch broadcasts, against the formula in fp64 (fp32 sums,
    the gradient rounded to bf16 once)."""
    from distrl_llm_amd.ops import functional as OF
    V = 40
    logits = _rand((*lead, V), 1, 2.0).requires_grad_()
    targets = torch.randint(0, V, lead, generator=torch.Generator().manual_seed(2)).cuda()
    mask = (_rand(mask_shape, 3) > -0.5).long()
    rewards = torch.randn(reward_shape, generator=torch.Generator().manual_seed(4))
    rewards = rewards if host else rewards.cuda()
    loss = OF.logprob_loss(logits, targets, mask, rewards, 0.5)
    grad, = torch.autograd.grad(loss, logits)
    x = logits.detach().double().requires_grad_()
    tok = x.log_softmax(-1).gather(-1, targets.unsqueeze(-1)).squeeze(-1)
    m = mask.double()
    ref = ((tok * m).sum(-1) * (-rewards.cuda().double() / m.sum(-1).clamp_min(1) / lead[0] * 0.5)).sum()
    assert float((loss - ref).detach().abs()) < 1e-5 * float(tok.detach().abs().max())
    assert _rel(grad, torch.autograd.grad(ref, x)[0]) < 2.0 ** -8


# ------------------------------------------------- training without padding

@pytest.mark.parametrize("lens", [[1], [33, 1, 64, 65], [200, 5, 129]])
@pytest.mark.parametrize("H,KV,D", [(4, 2, 64), (7, 1, 128), (14, 2, 64)])
@pytest.mark.parametrize("packed", [False, True])
def test_flash_varlen_backward(ext, lens, H, KV, D, packed):
    """Each sequence of a flat batch against itself alone; rows of their own
    and cut out of wider ones."""
    T = sum(lens)
    rows = _rand((T, (H + 2 * KV) * D), 1)
    q, k, v = (t.unflatten(1, (-1, D)) for t in rows.split([H * D, KV * D, KV * D], 1))
    if not packed:
        q, k, v = (t.contiguous() for t in (q, k, v))
    dout = _rand((T, H, D), 2, 0.1)
    cu = torch.tensor([0, *lens]).cumsum(0).to("cuda", torch.int32)
    o, lse = ext.flash_varlen_fwd(q, k, v, cu, max(lens), D ** -0.5)
    wide = torch.full((T, (H + 2 * KV) * D + 8), 7.0, dtype=torch.bfloat16, device="cuda")
    grads = [t.unflatten(1, (-1, D)) for t in wide[:, :-8].split([H * D, KV * D, KV * D], 1)]
    if not packed:
        grads = [torch.empty_like(t) for t in (q, k, v)]
    else:       # the output into a wider matrix too
        room = torch.empty((T, H * D + 8), dtype=torch.bfloat16, device="cuda")
        ext.flash_varlen_fwd(q, k, v, cu, max(lens), D ** -0.5,
                             room[:, :H * D].unflatten(1, (H, D)))
        assert torch.equal(room[:, :H * D], o.flatten(1))
        o = room[:, :H * D].unflatten(1, (H, D))
    ext.flash_varlen_bwd(dout, q, k, v, o, lse, cu, max(lens), D ** -0.5, *grads)
    assert (wide[:, -8:] == 7).all()
    got, start = (o, *grads), 0
    for n in lens:
        part = [t[start:start + n].transpose(0, 1).unsqueeze(0) for t in (q, k, v, dout)]
        for x, y in zip(got, _flash_reference(*part, D ** -0.5)):
            # a single row's dq and dk are 0: fp32 roundings of terms of dout's size
            off = (x[start:start + n].transpose(0, 1).double() - y[0].double()).norm()
            assert off < FLASH_REL * y.double().norm() + 2.0 ** -18 * dout.double().norm()
        start += n


@pytest.mark.parametrize("rows", [1, 63, 64, 65, 700, 5000])
@pytest.mark.parametrize("shapes", [[(8, 8)], [(128, 32), (136, 40), (1000, 64), (256, 96), (64, 128),
                                               (1536, 32)]])
def test_adapter_grads(ext, rows, shapes):
    """Ends of the row steps, column blocks and rank tiles, several operands at
    once, in place and cut out of wider rows; both layouts of the output. Bound:
    fp32 sums, one rounding."""
    ys, ps = [], []
    for i, (N, r) in enumerate(shapes):
        ys.append(_rand((rows, N + 8), 2 * i)[:, 8:] if i % 2 else _rand((rows, N), 2 * i))
        ps.append(_rand((rows, r + 3), 2 * i + 1)[:, 3:] if i % 3 == 2 else
                  _rand((rows, r), 2 * i + 1))
    for flip in (0, 1):
        by_col = [(i + flip) % 2 for i in range(len(shapes))]
        for y, p, c, got in zip(ys, ps, by_col, ext.adapter_grads(ys, ps, by_col)):
            ref = p.double().t() @ y.double()
            assert _rel(got, ref.t() if c else ref) < 2.0 ** -8
    assert all((t == 0).all() for t in ext.adapter_grads([ys[0][:0]], [ps[0][:0]], [0]))


@pytest.mark.parametrize("rows", [1, 31, 33, 700, 17000])
@pytest.mark.parametrize("K,ranks,pad", [(8, (8,), 8), (136, (32, 32, 32), 96), (896, (8, 24), 40),
                                         (1000, (64,), 64), (264, (40, 48, 40), 128),
                                         (4864, (32,), 32)])
def test_adapter_input(ext, rows, K, ranks, pad):
    """Ends of the row, K and column tiles, adapters side by side with a scale
    each, zeros in spare columns, cut out of wider rows, both layouts of the
    adapter. Bound: fp32 sums, one rounding."""
    if rows * K > 2e7:
        K = 392
    x = _rand((rows, K + 8), 1)[:, 8:]
    ms, scales = [_rand((r, K), 2 + i) for i, r in enumerate(ranks)], [0.5 + i for i in range(len(ranks))]
    wide = torch.full((rows, pad + 16), 7.0, dtype=torch.bfloat16, device="cuda")
    out = wide[:, 8:8 + pad]
    ref = x.double() @ torch.cat([m.double() * s for m, s in zip(ms, scales)]).t()
    assert ext.adapter_input(x, ms, scales, out, False)
    assert _rel(out[:, :sum(ranks)], ref) < 2.0 ** -8
    assert (out[:, sum(ranks):] == 0).all() and (wide[:, :8] == 7).all() and (wide[:, 8 + pad:] == 7).all()
    out.fill_(7.0)
    assert ext.adapter_input(x, [torch.cat(ms).t().contiguous()], [2.0], out, True)
    assert _rel(out[:, :sum(ranks)], x.double() @ torch.cat(ms).double().t() * 2) < 2.0 ** -8
    assert (out[:, sum(ranks):] == 0).all() and (wide[:, :8] == 7).all() and (wide[:, 8 + pad:] == 7).all()


def test_adapter_input_refuses(ext):
    """What 16 B accesses or the tiles can't take is left to the caller."""
    x, m, out = _rand((5, 64), 1), _rand((8, 64), 2), _rand((5, 8), 3)
    assert ext.adapter_input(x, [m], [1.0], out, False)
    assert not ext.adapter_input(x[:, 1:57], [m[:, :56].contiguous()], [1.0], out, False)
    assert not ext.adapter_input(x, [m[:5].contiguous()], [1.0], out, False)
    assert not ext.adapter_input(x, [m], [1.0], out[:1].expand(5, 8), False)
    assert not ext.adapter_input(x, [_rand((136, 64), 4)], [1.0], _rand((5, 136), 5), False)
    assert not ext.adapter_input(x.float(), [m], [1.0], out, False)
    wide = torch.full((5, 16), 7.0, dtype=torch.bfloat16, device="cuda")
    assert not ext.adapter_input(x, [m], [1.0], wide[:, :10], False)    # a part of four
    assert (wide == 7).all()


@pytest.mark.parametrize("N,K,ranks,pad", [((16, 8, 24), 64, (8, 8, 8), 24), ((40, 24), 136, (5, 12), 24),
                                           ((64,), 8, (32,), 32)])
def test_adapted_weight(ext, N, K, ranks, pad):
    ws, As, Bs = ([_rand(s, i) for i, s in enumerate(shapes)] for shapes in (
        [(n, K) for n in N], [(r, K) for r in ranks], list(zip(N, ranks))))
    odd = ws[0].new_empty(ws[0].numel() + 1)[1:].view(ws[0].shape).copy_(ws[0])
    beside = torch.block_diag(*Bs, ws[0].new_zeros(0, pad - sum(ranks)))
    for w0 in (ws[0], odd):
        w = [w0, *ws[1:]]
        assert torch.equal(ext.adapted_weight(w, Bs, pad), torch.cat([torch.cat(ws), beside], 1))
        # a gap of zeros between the first matrix and the rest
        stack, at = [w0, *As, *ws[1:]], [0]
        for t in stack[:-1]:
            at.append(at[-1] + t.shape[0] + (8 if len(at) == 1 else 0))
        cols = (at[-1] + stack[-1].shape[0] + 7) // 8 * 8
        ref = torch.zeros(cols, K, device="cuda", dtype=torch.bfloat16)
        for t, i in zip(stack, at):
            ref[i:i + t.shape[0]] = t
        assert torch.equal(ext.stack_transposed(stack, at, cols), ref.t())


@pytest.mark.parametrize("rows,F", [(1, 8), (5, 2056), (33, 4864)])
def test_activation_and_norm_into_wider_rows(ext, rows, F):
    """The same numbers as into matrices of their own, nothing beside them."""
    gu, dy, w = _rand((rows, 2 * F), 1), _rand((rows, F), 2), _rand((F,), 3)
    gate, up = (t.contiguous() for t in gu.chunk(2, 1))
    act, back = (torch.full((rows, n + 8), 7.0, dtype=torch.bfloat16, device="cuda")
                 for n in (F, 2 * F))
    ext.silu_mul_packed_into(gu, act[:, :F])
    ext.silu_mul_bwd_packed(dy, gu, back[:, :F], back[:, F + 8:])
    assert torch.equal(act[:, :F], ext.silu_mul_fwd(gate, up))
    ref = ext.silu_mul_bwd(dy, gate, up)
    assert torch.equal(back[:, :F], ref[0]) and torch.equal(back[:, F + 8:], ref[1])
    ext.rmsnorm_fwd_into(dy, w, 1e-6, act[:, :F])
    assert torch.equal(act[:, :F], ext.rmsnorm_fwd(dy, w, 1e-6))
    assert (act[:, F:] == 7).all() and (back[:, F:F + 8] == 7).all()


@pytest.mark.parametrize("T,H,KV,D", [(1, 1, 1, 64), (9, 14, 2, 64), (5, 12, 2, 128)])
def test_rope_rows(ext, T, H, KV, D):
    wide = _rand((T, (H + 2 * KV) * D + 8), 1)
    q, k = (t.unflatten(1, (-1, D)) for t in wide[:, :(H + KV) * D].split([H * D, KV * D], 1))
    pos = torch.arange(T, dtype=torch.int32, device="cuda") * 37
    inv = 1.0 / 1e4 ** (torch.arange(0, D, 2, device="cuda").float() / D)
    ref, rest = [q.contiguous(), k.contiguous()], wide[:, (H + KV) * D:].clone()
    ext.rope_inplace(*ref, pos, inv)
    ext.rope_rows(q, k, pos, inv)
    assert torch.equal(q, ref[0]) and torch.equal(k, ref[1])
    assert torch.equal(wide[:, (H + KV) * D:], rest)


@pytest.mark.parametrize("rows,V", [(1, 7), (3, 4103), (1500, 4096)])
def test_logprob_rows(ext, rows, V):
    """Value and gradient against fp64; rows of weight zero. Bounds: bf16
    gradient, and for the value as many fp32 roundings as there are rows."""
    from distrl_llm_amd.ops import functional as OF
    logits, g = _rand((rows, V), 1, 2.0).requires_grad_(), torch.Generator().manual_seed(2)
    targets = torch.randint(0, V, (rows,), generator=g).cuda()
    w = torch.randn(rows, generator=g).cuda() * (torch.arange(rows, device="cuda") % 3 != 1)
    loss = OF.logprob_rows(logits, targets, w)
    grad, = torch.autograd.grad(loss * 2, logits)
    x = logits.detach().double().requires_grad_()
    terms = x.log_softmax(-1).gather(1, targets[:, None])[:, 0] * w.double()
    ref, = torch.autograd.grad(terms.sum() * 2, x)
    assert abs(float(loss) - float(terms.sum())) < 1e-5 * float(terms.abs().sum())
    assert _rel(grad, ref) < 2.0 ** -8


@pytest.mark.parametrize("rows,V", [(5, 8), (131073, 8), (255, 4096), (256, 4096), (700, 4104), (65, 16384),
                                    (64, 16391), (530, 32768), (17, 65544), (17, 62000), (9, 131079),
                                    (9, 131072), (259, 155648), (9, 155656)])
def test_loss_gradients_made_forward(ext, rows, V):
    """Rows at the edges of what is held in registers, rows beyond and few rows: one backward,
    those behind it in a kept graph (what the first gave out is overwritten) and one
    that is scaled give what the two passes apart do, up to the log-sum-exp's rounding
    (some 1e-6, which moves few values over a bf16 rounding edge)."""
    from distrl_llm_amd.ops import functional as OF
    logits, g = _rand((rows, V), V, 2.0), torch.Generator().manual_seed(2)
    logits[0, 1] = float("-inf")
    targets = torch.randint(2, V, (rows,), generator=g).cuda()
    w = torch.randn(rows, generator=g).cuda() * (torch.arange(rows, device="cuda") % 3 != 1)
    tok, lse = ext.logprob_lse_fwd(logits, targets)
    leaf = logits.clone().requires_grad_()
    loss = OF.logprob_rows(leaf, targets, w)
    assert abs(float(loss.detach()) - float((tok * w).sum())) < 1e-5 * float((tok * w).abs().sum() + 1e-30)
    for scale in (1.0, 1.0, 3.0):
        got, = torch.autograd.grad(loss * scale, leaf, retain_graph=True)
        want = ext.logprob_loss_bwd(logits, targets, w * scale, lse)
        assert _rel(got, want) < 1e-5
        got.fill_(7.0)
    once, = torch.autograd.grad(OF.logprob_rows(leaf, targets, w) * 3.0, leaf)
    assert _rel(once, ext.logprob_loss_bwd(logits, targets, w * 3.0, lse)) < 1e-5
    leaf.requires_grad_(False)                  # no gradient is wanted: none is made
    assert not OF.logprob_rows(leaf, targets, w).requires_grad


@pytest.mark.parametrize("threads,pieces", [(256, k) for k in range(1, 9)] + [(512, k) for k in range(5, 9)]
                         + [(1024, k) for k in range(5, 20)])
def test_loss_gradients_by_pieces(ext, threads, pieces):
    """The narrowest and the widest row of every number of pieces that a workgroup's threads
    hold, one row more than workgroups: as the two passes apart (as above)."""
    from distrl_llm_amd.ops import functional as OF
    rows = 256 * (8 * 256 // threads) + 1
    for V in (threads * 8 * (pieces - 1) + 9, threads * 8 * pieces):
        if rows * V < 1 << 20:
            continue
        g = torch.Generator("cuda").manual_seed(V)
        leaf = torch.randn(rows, V, generator=g, device="cuda").mul_(2).bfloat16().requires_grad_()
        targets = torch.randint(0, V, (rows,), generator=g, device="cuda")
        targets[:2] = torch.tensor([V - 1, 0])
        w = torch.randn(rows, generator=g, device="cuda")
        tok, lse = ext.logprob_lse_fwd(leaf.detach(), targets)
        loss = OF.logprob_rows(leaf, targets, w)
        assert abs(float(loss.detach()) - float((tok * w).sum())) < 1e-5 * float((tok * w).abs().sum())
        got, = torch.autograd.grad(loss, leaf)
        assert _rel(got, ext.logprob_loss_bwd(leaf.detach(), targets, w, lse)) < 1e-5


@pytest.mark.parametrize("V,dtype", [(40, torch.bfloat16), (41, torch.float32), (32777, torch.bfloat16),
                                     (66000, torch.bfloat16)])
def test_targets_that_are_no_word(V, dtype):
    """Targets below a row and past it, by all of their 64 bits: the loss has no logit of
    theirs and the gradient is the softmax alone."""
    from distrl_llm_amd.ops import functional as OF
    targets = torch.tensor([-1, -100, V, 2 ** 31 + 3, 2 ** 32 + 5, 2 ** 35 + 9, 2 ** 40 + V - 1, -2 ** 32 + 4,
                            -2 ** 63, 2 ** 63 - 1, V - 1, 5], device="cuda").repeat(3)
    leaf = _rand((len(targets), V), V, 2.0).to(dtype).requires_grad_()
    w = torch.linspace(0.5, 1.5, len(targets), device="cuda")
    exact = leaf.detach().double().requires_grad_()
    there = (targets >= 0) & (targets < V)
    tok = torch.where(there, exact.gather(1, targets.where(there, 0)[:, None])[:, 0], 0.0) - exact.logsumexp(-1)
    ref, = torch.autograd.grad((tok * w).sum(), exact)
    for scale in (1.0, 3.0):
        loss = OF.logprob_rows(leaf, targets, w)
        assert abs(float(loss.detach()) - float((tok * w).sum().detach())) < 1e-5 * float((tok * w).abs().sum().detach())
        grad, = torch.autograd.grad(loss * scale, leaf)
        assert _rel(grad, ref * scale) < 2.0 ** -8


@pytest.mark.parametrize("B,T,V", [(3, 700, 512), (2, 300, 16391), (1, 40, 152064), (1, 20000, 64),
                                   (2, 1200, 33000)])
def test_masked_loss_in_a_graph(B, T, V):
    """A captured loss and its gradient, made forward, replayed on other values with eager
    ones in between: the workgroups' sums meet anew each time, in the same order."""
    from distrl_llm_amd.ops import functional as OF
    g = torch.Generator("cuda").manual_seed(V)
    leaf = torch.randn(B, T, V, generator=g, device="cuda").bfloat16().requires_grad_()
    targets = torch.randint(0, V, (B, T), generator=g, device="cuda")
    mask = (torch.rand(B, T, generator=g, device="cuda") < 0.8).long()
    rewards = torch.randn(B, generator=g, device="cuda")

    def call():
        loss = OF.logprob_loss(leaf, targets, mask, rewards, 0.5)
        return loss.detach(), torch.autograd.grad(loss, leaf, torch.ones_like(loss))[0]

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for _ in range(4):
        with torch.no_grad():
            leaf.copy_(torch.randn(B, T, V, generator=g, device="cuda"))
            rewards.normal_(generator=g)
        graph.replay()
        torch.cuda.synchronize()
        got = [t.clone() for t in out]
        want = call()
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("masked", [False, True])
def test_loss_without_room_for_a_gradient(masked):
    """A loss is had, with gradients enabled, where memory holds no gradient of its logits
    yet, and its backward once there is room."""
    from distrl_llm_amd.ops import functional as OF
    leaf = _rand((1024, 16384), 1, 2.0).requires_grad_()
    targets, r = torch.arange(1024, device="cuda"), torch.rand(1024, device="cuda")

    def loss_of(x):
        if masked:
            return OF.logprob_loss(x[None], targets[None], r[None], r[:1], 0.5)
        return OF.logprob_rows(x, targets, r)

    want = loss_of(leaf)
    ref, = torch.autograd.grad(want, leaf)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total, rest = torch.cuda.get_device_properties(0).total_memory, []
    try:
        torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() / total)
        with pytest.raises(torch.OutOfMemoryError):
            while True:
                rest.append(torch.empty(8 << 20, dtype=torch.uint8, device="cuda"))
        loss = loss_of(leaf)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert abs(float(loss - want)) < 1e-5 * abs(float(want))
    assert _rel(torch.autograd.grad(loss, leaf)[0], ref) < 1e-5


@pytest.mark.parametrize("masked", [False, True])
def test_loss_under_saved_tensor_hooks(masked):
    """A loss that is checkpointed, or whose saved tensors go to the host, holds nothing
    of its logits' size on the GPU until its backward; its gradient is the same."""
    from torch.utils.checkpoint import checkpoint
    from distrl_llm_amd.ops import functional as OF
    x, w = _rand((512, 64), 1), _rand((64, 8192), 2, 0.3)
    targets, r = torch.arange(512, device="cuda"), torch.rand(512, device="cuda")
    size = 512 * 8192 * 2

    def loss_of(x):
        logits = x @ w
        if masked:
            return OF.logprob_loss(logits[None], targets[None], r[None], r[:1], 0.5)
        return OF.logprob_rows(logits, targets, r)

    grads = []
    for how in ("plain", "checkpoint", "host"):
        leaf = x.clone().requires_grad_()
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        if how == "checkpoint":
            loss = checkpoint(loss_of, leaf, use_reentrant=False)
        elif how == "host":
            with torch.autograd.graph.save_on_cpu():
                loss = loss_of(leaf)
        else:
            loss = loss_of(leaf)
        held = torch.cuda.memory_allocated() - before
        assert how == "plain" or held < size // 2, (how, held)
        grads.append(torch.autograd.grad(loss, leaf)[0])
    assert all(_rel(g, grads[0]) < 2.0 ** -8 for g in grads[1:])


@pytest.mark.parametrize("rows", [4096, 4097, 6145, 8200])
def test_feed_forward_half_in_waves(ext, rows):
    """Input gradients of rows whose tiles fill the chip once, of one row more,
    of half a wave and a row more, and of three runs, against fp64: the bf16 rounding of each value on the way
    (activation, its gradient, the sum: some 2^-9 each)."""
    h, f, r = 4096, 64, 8
    x, g, norm = _rand((rows, h), 1), _rand((rows, h), 2), _rand((h,), 3, 0.1) + 1
    Ws = [_rand(s, 4 + i, 0.1) for i, s in enumerate(((f, h), (f, h), (h, f)))]
    As = [_rand((r, w.shape[1]), 7 + i, 0.02) for i, w in enumerate(Ws)]
    Bs = [_rand((w.shape[0], r), 10 + i, 0.1) for i, w in enumerate(Ws)]
    scales = [0.5, 2.0, 1.0]
    y, hu, gu, au = ext.feed_forward_half_fwd(x, norm, 1e-6, Ws, [None, None], As, Bs, scales)
    dx = ext.feed_forward_half_bwd(g, x, norm, 1e-6, Ws, As, Bs, scales, hu, gu, au, True)[0]
    xd = x.double().requires_grad_()
    n = xd * torch.rsqrt((xd * xd).mean(-1, keepdim=True) + 1e-6) * norm.double()
    wg, wu, wd = (w.double() + s * b.double() @ a.double()
                  for w, a, b, s in zip(Ws, As, Bs, scales))
    ref = xd + (torch.nn.functional.silu(n @ wg.t()) * (n @ wu.t())) @ wd.t()
    want, = torch.autograd.grad(ref, xd, g.double())
    assert _rel(y, ref.detach()) < 2.0 ** -7
    for at in (slice(None), slice(0, 1), slice(4095, 4097), slice(rows - 1, rows)):
        assert _rel(dx[at], want[at]) < 2.0 ** -6


@pytest.mark.parametrize("rows,h,f", [(70, 128, 256), (8200, 128, 256), (8200, 8192, 64)])
@pytest.mark.parametrize("r", [8, 32, 64])
@pytest.mark.parametrize("biased", [False, True])
def test_feed_forward_half(ext, rows, h, f, r, biased):
    """Output, input gradient and every adapter's gradients of one half against fp64, each
    adapter a scale of its own and some tenth of its projection, rows and widths on
    either side of the rules for our products and the library's. Bounds: the
    bf16 rounding of each value on the way (adapter inputs, activation, its
    gradient, the sum), some 2^-9 each."""
    x, g, norm = _rand((rows, h), 1), _rand((rows, h), 2), _rand((h,), 3, 0.1) + 1
    Ws = [_rand(s, 4 + i, s[1] ** -0.5) for i, s in enumerate(((f, h), (f, h), (h, f)))]
    As = [_rand((r, w.shape[1]), 7 + i, w.shape[1] ** -0.5) for i, w in enumerate(Ws)]
    Bs = [_rand((w.shape[0], r), 10 + i, 0.3 * r ** -0.5) for i, w in enumerate(Ws)]
    scales, bias = [0.5, 2.0, 1.0], [_rand((f,), 13 + i) if biased else None for i in range(2)]
    (y, hu, gu, au), ran = _kernels(
        lambda: ext.feed_forward_half_fwd(x, norm, 1e-6, Ws, bias, As, Bs, scales))
    own, wide = r % 32 == 0, rows > 8192 and h >= 8192      # as the rules have it
    # gate|up with their activation, and down
    assert ran("product_kernel") == (2 if own and not wide else 0)
    assert ran("activation_inputs_kernel") == (1 if rows >= 8192 and (wide or not own) else 0)
    (dx, *got), ran = _kernels(
        lambda: ext.feed_forward_half_bwd(g, x, norm, 1e-6, Ws, As, Bs, scales, hu, gu, au, True))
    assert ran("product_kernel") == (2 if own and not wide else 0)
    leaves = [t.double().requires_grad_() for t in (x, *(m for ab in zip(As, Bs) for m in ab))]
    xd, Ad, Bd = leaves[0], leaves[1::2], leaves[2::2]
    n = xd * torch.rsqrt((xd * xd).mean(-1, keepdim=True) + 1e-6) * norm.double()

    def proj(i, t):
        return t @ Ws[i].double().t() + scales[i] * (t @ Ad[i].t()) @ Bd[i].t()

    gate, up = (proj(i, n) + (bias[i].double() if biased else 0.0) for i in range(2))
    ref = xd + proj(2, torch.nn.functional.silu(gate) * up)
    want = torch.autograd.grad(ref, leaves, g.double())
    assert _rel(gu, torch.cat([gate, up], 1).detach()) < 2.0 ** -7
    for at in (slice(None), slice(0, 1), slice(rows - 1, rows)):
        assert _rel(y[at], ref[at].detach()) < 2.0 ** -7
        assert _rel(dx[at], want[0][at]) < 2.0 ** -6
    for x, t in zip(got, want[1:]):
        assert _rel(x, t) < 2.0 ** -6


@pytest.mark.parametrize("r", [8, 16, 32])
def test_halves_take_adapter_inputs_once(ext, r):
    """Whatever products a rank goes through, the inputs of the adapters on one
    matrix are one launch: those on x, then on the second product's operand, and
    the same of the gradients."""
    rows, h, D, f = 64, 128, 64, 256
    x, g, norm = _rand((rows, h), 1), _rand((rows, h), 2), _rand((h,), 3, 0.1) + 1

    def adapted(*shapes):
        Ws = [_rand(s, 4 + i, 0.1) for i, s in enumerate(shapes)]
        return (Ws, [_rand((r, w.shape[1]), 8 + i, 0.1) for i, w in enumerate(Ws)],
                [_rand((w.shape[0], r), 12 + i, 0.1) for i, w in enumerate(Ws)])

    Ws, As, Bs = adapted((h, h), (D, h), (D, h), (h, h))
    pos = torch.arange(rows, dtype=torch.int32, device="cuda")
    inv = 1.0 / 1e4 ** (torch.arange(0, D, 2, device="cuda").float() / D)
    cu = torch.tensor([0, rows], dtype=torch.int32, device="cuda")
    (y, *own), ran = _kernels(lambda: ext.attention_half_fwd(
        x, norm, 1e-6, Ws, [None] * 3, As, Bs, [1.0] * 4, None, None, 0.0, 0.0, pos, inv, cu, rows,
        D ** -0.5, D))
    assert ran("adapter_inputs_kernel") == 2
    _, ran = _kernels(lambda: ext.attention_half_bwd(
        g, x, norm, 1e-6, Ws, As, Bs, [1.0] * 4, None, None, 0.0, 0.0, pos, -inv, cu, rows,
        D ** -0.5, *own, True))
    assert ran("adapter_inputs_kernel") == 2
    Ws, As, Bs = adapted((f, h), (f, h), (h, f))
    (y, *own), ran = _kernels(lambda: ext.feed_forward_half_fwd(
        x, norm, 1e-6, Ws, [None] * 2, As, Bs, [1.0] * 3))
    assert ran("adapter_inputs_kernel") == 2
    _, ran = _kernels(lambda: ext.feed_forward_half_bwd(
        g, x, norm, 1e-6, Ws, As, Bs, [1.0] * 3, *own, True))
    assert ran("adapter_inputs_kernel") == 2


@pytest.mark.parametrize("tied", [True, False])
@pytest.mark.parametrize("V,own", [(4096, 0), (32768, 1), (65544, 0), (70016, 1)])
def test_rows_logits(tied, V, own):
    """Logits of rows and their gradient on either side of the LM head's line to products
    of our own, a vocabulary that they don't take, a gradient that is laid out by columns
    (the library's). Sums in fp32, rounded to bf16 once."""
    import dataclasses
    from distrl_llm_amd.models import get_spec
    model = _train_model(dataclasses.replace(get_spec("small-qwen2"), vocab_size=V, tie_word_embeddings=tied))
    weight = (model.model.embed_tokens if tied else model.lm_head).weight
    assert not weight.requires_grad
    hidden, g = _rand((37, 512), 1).requires_grad_(), _rand((37, V), 2, 0.1)
    logits = model.rows_logits(hidden)
    assert torch.equal(logits, model.logits(hidden))
    (grad,), ran = _kernels(lambda: torch.autograd.grad(logits, hidden, g, retain_graph=True))
    assert (ran("product_kernel") > 0) == bool(own)
    ref = g.double() @ weight.double()
    assert _rel(logits, hidden.detach().double() @ weight.double().t()) < 2.0 ** -8
    assert _rel(grad, ref) < 2.0 ** -8
    other, = torch.autograd.grad(logits, hidden, g.t().contiguous().t())
    assert _rel(other, ref) < 2.0 ** -8


@pytest.mark.parametrize("prompts,answers", [([9, 30, 1], [40, 7, 100]), ([0, 5, 3], [4, 0, 6]),
                                             ([3], [1]), ([4, 2], [0, 0])])
def test_learner_rows_match_padding(prompts, answers):
    """Loss and adapter gradients without padding against the padded batch (two
    bf16 paths of the same sums: 1 %), with empty prompts and answers; a hook
    on a part keeps the padded batch."""
    from distrl_llm_amd.train.learner import Learner
    from distrl_llm_amd.utils.tokenizer import ByteTokenizer
    model = _train_model("small-qwen2")
    learner = Learner(model, ByteTokenizer(model.spec.vocab_size), lr=1e-4, max_prompt_tokens=64,
                      max_new_tokens=128, train_batch_size=4)
    enc = [([5 + i] * p, [7 + i + j % 9 for j in range(a)])
           for i, (p, a) in enumerate(zip(prompts, answers))]
    learner._encode = lambda problems, answers: enc
    rewards, got = torch.tensor([0.5, -1.0, 0.8][:len(enc)], device="cuda"), []
    for rows in (True, False):
        if not rows:
            handle = model.model.norm.register_forward_hook(lambda m, i, o: None)
        assert model.takes_rows() == rows
        loss = learner._micro_loss(enc, enc, rewards, 0.5)
        grads = torch.autograd.grad(loss, learner.params, allow_unused=True)
        got.append((loss.detach(), torch.cat([g.reshape(-1).double() for g in grads])))
    handle.remove()
    assert abs(float(got[0][0]) - float(got[1][0])) < 0.01 * abs(float(got[1][0])) + 1e-6
    assert _rel(got[0][1], got[1][1]) < 0.01 or not any(answers)
