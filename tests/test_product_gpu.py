"""Products on matrix cores (ops/csrc/product.hip) at the edges of their
tiles, shares of K and terms, against plain fp32 torch."""

import pytest
import torch

pytestmark = pytest.mark.gpu

# Bounds, of every output: operands are exact in bf16, so an output is off by its own
# rounding to 8 significant bits, 2^-8 of it at most, and by its fp32 sum, n terms in
# whatever order: n 2^-24 of the sum of their magnitudes.
REL = 2.0 ** -8
SENTINEL = 7.0
TILES = [0, 8, 7, 6, 5, 4, 128, 64, 64 + 512, 128 + 768, 64 + 2048]


@pytest.fixture(scope="module")
def ext():
    from distrl_llm_amd.ops.build import build
    return build()


def _make(seed):
    g = torch.Generator().manual_seed(seed)

    def rand(*shape, spare=0):
        x = torch.randn(*shape[:-1], shape[-1] + spare, generator=g).to("cuda", torch.bfloat16)
        return x[..., :shape[-1]]
    return rand


def _close(x, ref):
    assert float((x.float() - ref).norm() / ref.norm()) < REL


def _each_close(x, ref, off):
    """off: what else than its rounding an output may be off by, of every one."""
    assert bool(((x.double() - ref).abs() <= REL * ref.abs() + 2 * off).all())


def _sum(pairs, rows_of_b=False):
    """Sums of products in fp64, and how far an fp32 sum of them may be off."""
    pairs = [(x.double(), y.double() if rows_of_b else y.double().t()) for x, y in pairs]
    return (sum(x @ y for x, y in pairs),
            sum(x.abs() @ y.abs() for x, y in pairs) * (sum(x.shape[1] for x, _ in pairs) + 2) * 2.0 ** -24)


def _room(M, width, spare):
    """(rows to write into, whether what stands around them is untouched)"""
    room = torch.full((M + 2, width + spare + 8), SENTINEL, dtype=torch.bfloat16, device="cuda")
    out = room[1:-1, :width]

    def untouched():
        around = room.clone()
        around[1:-1, :width] = SENTINEL
        return bool((around == SENTINEL).all())
    return out, untouched


@pytest.mark.parametrize("M,widths,deep,spare", [
    (1, (8,), (32,), 0), (63, (64, 8), (32, 32), 8), (65, (72, 128, 64), (96, 32), 0),
    (129, (136,), (64, 32, 160), 64), (257, (256, 40), (224, 64), 0), (300, (520,), (1024,), 8),
    (513, (264, 8, 8), (320, 32), 0)])
@pytest.mark.parametrize("tile", TILES)
def test_sums_of_products(ext, M, widths, deep, spare, tile):
    """Blocks of columns with their bias or a residual, terms of different
    depths, rows further apart than they are long; b as (width, k) and (k, width)."""
    rand = _make(M)
    for what in ("columns", "rows"):
        a = [[rand(M, k, spare=spare) for k in deep] for _ in widths]
        b = [[rand(w, k, spare=spare) if what == "columns" else rand(k, w, spare=spare)
              for k in deep] for w in widths]
        bias = [rand(w) if i != 1 else None for i, w in enumerate(widths)]
        sums = [_sum(zip(xs, ys), what == "rows") for xs, ys in zip(a, b)]
        ref = torch.cat([r if c is None else r + c.double() for (r, _), c in zip(sums, bias)], 1)
        off = torch.cat([o for _, o in sums], 1)
        for res in (None, rand(M, sum(widths), spare=spare)):
            out, untouched = _room(M, sum(widths), spare)
            assert ext.product(a, b, bias, widths, what, [out], res, tile)
            want = ref if res is None else ref + res.double()
            _each_close(out, want, off + 2.0 ** -23 * (ref.abs() + want.abs()))
            assert untouched()


@pytest.mark.parametrize("M,N,steps,spare", [(1, 8, 3, 0), (127, 264, 7, 8), (129, 248, 40, 0),
                                             (257, 520, 11, 64)])
@pytest.mark.parametrize("rows,shares", [(4, 2), (5, 3), (6, 7), (7, 64), (8, 5)])
@pytest.mark.parametrize("what", ["rows", "columns"])
def test_large_tiles_in_shares(ext, M, N, steps, spare, rows, shares, what):
    """Shares of K of large tiles: of one step, of less than the ring, more of them than steps."""
    rand, K = _make(M + shares), steps * 32
    a = rand(M, K, spare=spare)
    b = rand(K, N, spare=spare) if what == "rows" else rand(N, K, spare=spare)
    out, untouched = _room(M, N, spare)
    assert ext.product([[a]], [[b]], [None], [N], what, [out], None, rows | shares << 8)
    _each_close(out, *_sum([(a, b)], what == "rows"))
    assert untouched()


@pytest.mark.parametrize("M,V,N", [(1, 65536, 64), (37, 65568, 96), (300, 70016, 264), (9, 32003, 64),
                                   (0, 65536, 64), (700, 32768, 520), (1200, 32800, 8), (2408, 32768, 1024)])
def test_head_input_gradient(ext, M, V, N):
    """Sums long enough for shares by the rule, and what goes to the library."""
    rand = _make(M)
    g, w = rand(M, V), rand(V, N)
    _each_close(ext.product_rows(g, w), *_sum([(g, w)], True))


def test_head_input_gradient_without_room(ext):
    """Shares whose partial sums no memory is left for: the same product, without them."""
    rand = _make(1)
    g, w = rand(561, 65536), rand(65536, 896)
    want = ext.product_rows(g, w)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    room = torch.empty_like(want)                           # of the result, kept by the allocator
    total, rest = torch.cuda.get_device_properties(0).total_memory, []
    try:
        torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() / total)
        with pytest.raises(torch.OutOfMemoryError):
            while True:
                rest.append(torch.empty(16 << 20, dtype=torch.uint8, device="cuda"))
        del room
        got = ext.product_rows(g, w)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    _each_close(got, *_sum([(g, w)], True))
    assert float((got.float() - want.float()).norm() / want.float().norm()) < 2.0 ** -8


@pytest.mark.parametrize("M,F,K,r", [(1, 8, 32, 32), (70, 40, 96, 32), (130, 136, 64, 64),
                                     (300, 264, 160, 32)])
@pytest.mark.parametrize("tile", TILES)
def test_activation(ext, M, F, K, r, tile):
    """gate and up with an adapter each, and the activation's gradient: the
    activation of what was rounded into [gate | up]."""
    rand = _make(F)
    x, ug, uu = rand(M, K), rand(M, r), rand(M, r)
    wg, wu, bg, bu = rand(F, K), rand(F, K), rand(F, r), rand(F, r)
    bias = [rand(F), None]
    (gu, gu_alone), (act, act_alone) = _room(M, 2 * F, 0), _room(M, F, 24)
    assert ext.product([[x, ug, uu]] * 2, [[wg, bg, None], [wu, None, bu]], bias, [F, F], "glu",
                       [gu, act], None, tile)
    (gate, gate_off), (up, up_off) = _sum([(x, wg), (ug, bg)]), _sum([(x, wu), (uu, bu)])
    gate = gate + bias[0].double()
    _each_close(gu, torch.cat([gate, up], 1),
                torch.cat([gate_off + 2.0 ** -23 * gate.abs(), up_off], 1))
    gate, up = gu.double().split(F, 1)
    sig = gate.sigmoid()
    # the fast exponential and reciprocal: some 2^-22 of the result
    _each_close(act, gate * sig * up, 2.0 ** -20 * (gate * sig * up).abs())
    assert gu_alone() and act_alone()

    g, w, du, a = rand(M, K), rand(K, F), rand(M, r), rand(r, F)
    d, alone = _room(M, 2 * F, 0)
    assert ext.product([[g, du]], [[w, a]], [None], [F], "glu_bwd", list(d.split(F, 1)), gu, tile)
    dact, off = _sum([(g, w), (du, a)], True)
    slope = 1 + gate * (1 - sig)
    # the slope passes zero: its two terms are good to 2^-20 of their own
    fast = 2.0 ** -20 * (dact * up * sig).abs() * (1 + gate.abs())
    _each_close(d, torch.cat([dact * up * sig * slope, dact * gate * sig], 1),
                torch.cat([off * (up * sig * slope).abs() + fast,
                           off * (gate * sig).abs() + 2.0 ** -20 * (dact * gate * sig).abs()], 1))
    assert alone()


@pytest.mark.parametrize("M,F", [(1, 8), (31, 120), (33, 128), (64, 136), (100, 400), (70, 1032)])
@pytest.mark.parametrize("r,spare", [((32, 32), 0), ((8, 24), 4), ((64, 40), 0)])
def test_activation_with_adapter_inputs(ext, M, F, r, spare):
    """Edges of 32 rows and steps of 128 columns; the products are those of
    what was rounded and written, spare columns zero."""
    rand = _make(M + F)
    gu, m = rand(M, 2 * F), rand(r[0], F)
    (act, act_alone), (out, out_alone) = _room(M, F, 16), _room(M, r[0] + spare, 12)
    assert ext.silu_mul_inputs(gu, act, m, 0.5, out)
    gate, up = gu.double().split(F, 1)
    sig = gate.sigmoid()
    _each_close(act, gate * sig * up, 2.0 ** -20 * (gate * sig * up).abs())
    ref, off = _sum([(act, m)])
    _each_close(out[:, :r[0]], ref * 0.5, off * 0.5)
    assert not out[:, r[0]:].any() and act_alone() and out_alone()

    dact, (d, d_alone), (du, du_alone) = rand(M, F), _room(M, 2 * F, 0), _room(M, sum(r) + spare, 4)
    dgate, dup = d[:, :F], d[:, F:]
    b = [rand(F, x) for x in r]
    assert ext.silu_mul_bwd_inputs(dact, gu, dgate, dup, b, [0.5, 2.0], du)
    dact = dact.double()
    _each_close(dgate, dact * up * sig * (1 + gate * (1 - sig)),
                2.0 ** -20 * (dact * up * sig).abs() * (1 + gate.abs()))
    _each_close(dup, dact * gate * sig, 2.0 ** -20 * (dact * gate * sig).abs())
    for x, y, scale, at in ((dgate, b[0], 0.5, slice(0, r[0])), (dup, b[1], 2.0, slice(r[0], sum(r)))):
        ref, off = _sum([(x, y)], True)
        _each_close(du[:, at], ref * scale, off * scale)
    assert not du[:, sum(r):].any() and d_alone() and du_alone()


@pytest.mark.parametrize("M", [1, 57, 300])
@pytest.mark.parametrize("r", [0, 32, 64])
def test_adapted_projection_and_activation(ext, M, r):
    """A layer's projections with adapters or without, bias or residual."""
    rand, K, widths = _make(M + r), 160, (96, 40, 40)
    x, res, n = rand(M, K), rand(M, sum(widths)), len(widths) if r else 0
    w, bias = [rand(k, K) for k in widths], [rand(k) for k in widths]
    a, b = [rand(r, K) for _ in range(n)], [rand(k, r) for k in widths[:n]]
    # the adapters' inputs as they are rounded: their error is not this one's
    u = [(x.float() @ y.float().t() * 0.25).to(torch.bfloat16).float() for y in a]
    y = [x.float() @ v.float().t() for v in w]
    y = [v + u[i] @ b[i].float().t() if r else v for i, v in enumerate(y)]
    # 1e-3: of u, 2^-8 at most, a few land on the other side of a rounding
    out = ext.adapted_projection(x, w, bias, a, b, [0.25] * n)
    ref = torch.cat([v + c.float() for v, c in zip(y, bias)], 1)
    assert float((out.float() - ref).norm() / ref.norm()) < REL + 1e-3
    out = ext.adapted_projection(x, w, [None] * 3, a, b, [0.25] * n, res)
    ref = torch.cat(y, 1) + res.float()
    assert float((out.float() - ref).norm() / ref.norm()) < REL + 1e-3
    act = ext.adapted_activation(x, w[1:], a[1:], b[1:], [0.25] * max(n - 1, 0))
    gate, up = (v.to(torch.bfloat16).float() for v in y[1:])
    ref = torch.nn.functional.silu(gate) * up
    assert float((act.float() - ref).norm() / ref.norm()) < 3 * REL   # gate, up, act


def test_adapted_projection_leaves_the_rest(ext):
    rand = _make(5)
    x, w = rand(40, 64), rand(64, 64)
    for a, b in ((rand(16, 64), rand(64, 16)), (rand(32, 64).float(), rand(64, 32).float())):
        assert ext.adapted_projection(x, [w], [None], [a], [b], [1.0]) is None
        assert ext.adapted_activation(x, [w, w], [a, a], [b, b], [1.0, 1.0]) is None
    assert ext.adapted_projection(x[:0], [w], [None], [], [], []) is None
    assert ext.adapted_projection(x.float(), [w], [None], [], [], []) is None


def test_repeats_itself_in_a_graph(ext):
    """Shares of K meet in their order, also when a captured launch runs again."""
    rand = _make(3)
    a, b, out = rand(200, 4096), rand(96, 4096), rand(200, 96)

    def run(tile):
        assert ext.product([[a]], [[b]], [None], [96], "columns", [out], None, tile)
        return out.clone()

    for tile in (64 + 2048, 128 + 1024):
        first = run(tile)
        _close(first, a.float() @ b.float().t())
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            again = run(tile)
        for _ in range(5):
            out.zero_()
            graph.replay()
            assert torch.equal(again, first) and torch.equal(run(tile), first)


def test_refuses_what_it_cannot_walk(ext):
    rand = _make(4)
    out = rand(64, 64)

    def takes(a, b, out=out, width=64):
        return ext.product([[a]], [[b]], [None], [width], "columns", [out])

    assert takes(rand(64, 64), rand(64, 64))
    assert not takes(rand(64, 48), rand(64, 48))              # K no multiple of 32
    assert not takes(rand(64, 64, spare=4), rand(64, 64))     # rows not on 16 bytes
    assert not takes(rand(64, 65)[:, 1:], rand(64, 64))       # start not on 16 bytes
    assert not takes(rand(64, 64).float(), rand(64, 64))
    assert not takes(rand(64, 64), rand(64, 96))              # other K
    assert not takes(rand(64, 64).t(), rand(64, 64))          # columns on end
    assert not takes(rand(64, 64), rand(60, 64), rand(64, 60), 60)
    assert not takes(rand(64, 64).cpu(), rand(64, 64))


def test_refuses_a_residual_where_it_writes(ext):
    """Shares of K may be joined twice: what is added lies clear of the output."""
    rand = _make(6)
    a, b, wide = rand(64, 64), rand(64, 64), rand(130, 72)
    before = wide.clone()
    for out, res in ((wide[:64, :64], wide[:64, :64]), (wide[:64, :64], wide[63:127, :64])):
        assert not ext.product([[a]], [[b]], [None], [64], "columns", [out], res)
        gu = wide.view(-1)[:64 * 128].view(64, 128)
        assert not ext.product([[a]], [[b]], [None], [64], "glu_bwd", [out, out], gu)
    assert torch.equal(wide, before)
    assert ext.product([[a]], [[b]], [None], [64], "columns", [wide[:64, :64]], wide[64:128, :64])
    _close(wide[:64, :64], a.float() @ b.float().t() + before[64:128, :64].float())
