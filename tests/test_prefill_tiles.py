"""Prompt attention at the edges of its tiles of 64 keys: last tiles of every kind, pages of other sizes, tree rows that
start anywhere in a tile; against 64 bits."""
import math

import pytest
import torch

from dgi import ops
from dgi.ops import mix

pytestmark = pytest.mark.gpu


def _case(nh, nkv, hd, page, qlens, ctxs, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def rand(*shape):
        return torch.randn(*shape, device="cuda", generator=g).bfloat16()

    width = max(-(-c // page) for c in ctxs) + 1
    pages = len(ctxs) * width
    kc, vc = rand(pages, nkv, page, hd), rand(pages, nkv, page, hd)
    table = torch.randperm(pages, device="cuda", generator=g).int().view(len(ctxs), width)
    for b, c in enumerate(ctxs):                       # what lies past a sequence's end is never part of a result
        for p in range(c // page, width):
            kc[table[b, p], :, c - p * page if p == c // page else 0:] = float("nan")
            vc[table[b, p], :, c - p * page if p == c // page else 0:] = float("nan")
    cu = torch.tensor([sum(qlens[:i]) for i in range(len(qlens) + 1)], dtype=torch.int32, device="cuda")
    return rand(sum(qlens), nh * hd), kc, vc, table, cu, torch.tensor(ctxs, dtype=torch.int32, device="cuda")


def _check(out, q, kc, vc, table, cu, ctx, nh, nkv, hd, visible):
    """|error| <= 2^-8 (sum p |v| + |o|): weights and results are rounded to bf16 (2^-9 each), the rest is fp32."""
    page, scale = kc.shape[2], hd ** -0.5
    for b in range(len(ctx)):
        n, lo, hi = int(ctx[b]), int(cu[b]), int(cu[b + 1])
        rows = torch.arange(n, device="cuda")
        k, v = (c[table[b].long()[rows // page], :, rows % page].double().repeat_interleave(nh // nkv, 1) for c in (kc, vc))
        s = torch.einsum("qhd,khd->hqk", q[lo:hi].double().view(-1, nh, hd), k) * scale
        p = torch.softmax(s.masked_fill(~visible(b, hi - lo, n)[None], -math.inf), -1)
        want, size = torch.einsum("hqk,khd->qhd", p, v), torch.einsum("hqk,khd->qhd", p, v.abs())
        off = (out[lo:hi].double().view(-1, nh, hd) - want).abs()
        assert bool((off <= 2.0 ** -8 * (size + want.abs())).all()), (b, float(off.max()))


def _causal(_, m, n):
    return torch.arange(n, device="cuda")[None] <= torch.arange(n - m, n, device="cuda")[:, None]


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("page", [8, 16, 32])
@pytest.mark.parametrize("tile", [128, 256])
def test_ends_of_tiles(hd, page, tile, monkeypatch):
    monkeypatch.setattr(ops, "PREFILL_TILE", tile)
    qlens, ctxs = [1, 63, 64, 65, 128, 129, 33, 300], [1, 63, 64, 65, 128, 129, 190, 449]
    case = _case(6, 3, hd, page, qlens, ctxs, 5)
    _check(ops.paged_prefill(*case, 6, 3, hd ** -0.5), *case, 6, 3, hd, _causal)


@pytest.mark.parametrize("ctx", [64, 65, 96, 100, 127, 128, 131, 160, 200])
def test_tree_rows_anywhere_in_a_tile(ctx):
    """64 tree rows, the last ones of a sequence, whose keys begin at any offset of a tile and of a lane's keys."""
    hd, n = 128, 64
    par = torch.tensor([[-1] + [(i - 1) // 2 if i % 3 else max(0, i - 5) for i in range(1, n)]] * 2, dtype=torch.int32)
    anc, _ = ops.tree_mask_ref(par)
    case = _case(4, 2, hd, 16, [n, n], [ctx, ctx + 7], ctx)
    out = ops.paged_prefill(*case, 4, 2, hd ** -0.5, tree_mask=anc.cuda(), tree_n=n)

    def visible(b, m, keys):
        see = torch.ones(m, keys, dtype=torch.bool)
        for i in range(n):
            bits = int(anc[b, i]) & (1 << 64) - 1
            see[i, keys - n:] = torch.tensor([bool(bits >> j & 1) for j in range(n)])
        return see.cuda() & _causal(b, m, keys)

    _check(out, *case, 4, 2, hd, visible)


@pytest.mark.parametrize("window,block", [(1, 0), (31, 0), (64, 0), (65, 0), (0, 1), (0, 32), (0, 100)])
def test_first_keys_anywhere_in_a_tile(window, block):
    hd = 64
    case = _case(4, 2, hd, 16, [200, 70], [200, 333], 9)
    out = mix.paged_prefill_masked(*case, 4, 2, hd ** -0.5, block, None, window=window)

    def visible(b, m, n):
        p, j = torch.arange(n - m, n, device="cuda")[:, None], torch.arange(n, device="cuda")[None]
        return (j <= p) & (j > p - window if window else j >= p // block * block)

    _check(out, *case, 4, 2, hd, visible)


@pytest.mark.parametrize("hd,vd", [(64, 64), (128, 128), (96, 40)])
@pytest.mark.parametrize("page", [2, 8, 64, 256])
def test_pages_of_any_size(hd, vd, page):
    """A wave's rows of a tile have several pages, or lie anywhere in one; ends in the middle of a wave's rows and before them."""
    q, kc, vc, table, cu, ctx = _case(4, 2, hd, page, [1, 40, 129, 200], [300, 40, 263, 500], 3)
    out = mix.paged_prefill_masked(q, kc, vc[..., :vd].contiguous(), table, cu, ctx, 4, 2, hd ** -0.5, 0, None)
    padded = torch.zeros(*out.shape[:-1], 4 * hd, dtype=out.dtype, device="cuda").view(-1, 4, hd)
    padded[..., :vd] = out.view(-1, 4, vd)
    vc[..., vd:] = torch.where(vc[..., vd:].isnan(), vc[..., vd:], 0)
    _check(padded.view(-1, 4 * hd), q, kc, vc, table, cu, ctx, 4, 2, hd, _causal)


@pytest.mark.parametrize("page", [8, 32, 64])
def test_pages_cost_the_same(page):
    """Blocks' ids are there before the rows they name are asked for: pages of other sizes take little longer than those of 16 (half as long
    again where every load waits for its own id)."""
    def best(page):
        case = _case(32, 8, 128, page, [2000], [4000], 1)
        tiles = torch.from_numpy(ops.order_prefill_tiles([0, 2000], [4000])).cuda()
        times = []
        for i in range(8):
            e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            e[0].record()
            for _ in range(10):
                ops.paged_prefill(*case, 32, 8, 128 ** -0.5, tiles=tiles)
            e[1].record()
            e[1].synchronize()
            times.append(e[0].elapsed_time(e[1]))
        return min(times)

    assert best(page) <= 1.25 * best(16)


@pytest.mark.parametrize("form", ["plain", "masked"])
def test_caches_off_sixteen_bytes(form):
    """Caches that start between two 16-byte boundaries, which loads straight to LDS cannot take."""
    case = list(_case(4, 2, 64, 16, [70, 200], [100, 200], 7))

    def call(c):
        if form == "plain":
            return ops.paged_prefill(*c, 4, 2, 0.125)
        return mix.paged_prefill_masked(*c, 4, 2, 0.125, 0, None)

    want = call(case)
    for i in (1, 2):
        x = torch.empty(case[i].numel() + 8, dtype=torch.bfloat16, device="cuda")[i:][: case[i].numel()].view(case[i].shape)
        assert x.data_ptr() % 16 and x.is_contiguous()
        x.copy_(case[i])
        case[i] = x
    assert torch.equal(call(case), want)


@pytest.mark.parametrize("D", [64, 80, 128])
@pytest.mark.parametrize("cap,scale", [(0.0, 0.1), (0.5, 1.0), (30.0, 0.1), (1e4, 0.1)])
def test_caps_factors_and_gates(D, cap, scale):
    """Caps far below the scores, about them and far above, heads with factors below, at and above zero, sinks on both sides of the capped
    scores, gates from shut to open; rows behind a prefix and a last tile that ends early."""
    g = torch.Generator().manual_seed(D)
    H, G, lens, pre, bs = 6, 2, [150, 37], 70, 16
    cu, ctx = [0, 150, 187], [x + pre for x in lens]
    width = -(-max(ctx) // bs)
    table = (torch.randperm(2 * width, generator=g) + 1).view(2, width).int()
    k, v = (torch.randn(2 * width + 1, G, bs, D, generator=g).to(torch.bfloat16) for _ in range(2))
    q = torch.randn(187, H * D, generator=g).to(torch.bfloat16)
    gate = (40.0 * torch.randn(187, H * D, generator=g)).to(torch.bfloat16)
    sinks, factor = torch.linspace(-6, 9, H), torch.tensor([-1.5, -0.2, 0.0, 0.3, 1.0, 2.0])
    i32 = lambda x: torch.tensor(x, dtype=torch.int32)  # noqa: E731

    def run(dev, dt):
        to = lambda x: x.to(dev, dt)  # noqa: E731
        return mix.paged_prefill_masked(to(q), to(k), to(v), table.to(dev), i32(cu).to(dev), i32(ctx).to(dev), H, G, scale, 100, to(gate),
                                        softcap=cap, sinks=sinks.to(dev), head_scale=factor.to(dev)).float().cpu()

    got, want = run("cuda", torch.bfloat16), run("cpu", torch.float32)
    # each weight is rounded to bf16 once, as is the result; a cap adds the rounding of its quotient near 1/2, times twice the cap
    open_ = torch.sigmoid(gate.float())
    slack = open_ * v.float().abs().max() * (2.0 ** -8 + 2 * cap * 2.0 ** -23) + 2.0 ** -8 * want.abs() + 1e-6
    assert torch.isfinite(got).all() and ((got - want).abs() <= slack).all(), ((got - want).abs() / slack).max()


def test_element_gates_to_the_last_bits():
    """A row that sees its own key alone is its value times the gate's sigmoid: exp, sum, quotient and product are off by 4 x 2^-24 at most (two and a half measured for
    the sigmoid over all gates, half a unit of the product's), so a result is not the nearest bf16 number only where two are as near as that."""
    n, nh, hd = 512, 16, 128
    g = torch.Generator(device="cuda").manual_seed(9)
    kc = torch.zeros(n, nh, 16, hd, device="cuda", dtype=torch.bfloat16)
    vc = torch.randn(n, nh, 16, hd, device="cuda", generator=g).bfloat16()
    gate = ((torch.rand(n, nh * hd, device="cuda", generator=g) * 2 - 1) * 30).bfloat16()
    i32 = dict(device="cuda", dtype=torch.int32)
    out = mix.paged_prefill_masked(torch.zeros(n, nh * hd, device="cuda", dtype=torch.bfloat16), kc, vc, torch.arange(n, **i32)[:, None].contiguous(),
                                   torch.arange(n + 1, **i32), torch.ones(n, **i32), nh, nh, 1.0, 1024, gate)
    want = vc[:, :, 0].reshape(n, -1).double() * torch.sigmoid(gate.double())
    near = want.float().bfloat16()
    wrong = out != near
    middle = (out.double() + near.double()) / 2
    assert bool(((want - middle).abs() <= 4 * 2.0 ** -24 * want.abs())[wrong].all())
    assert wrong.float().mean() <= 4 * 2 * 2.0 ** -24 * 2 ** 8      # that near lie at most so many
