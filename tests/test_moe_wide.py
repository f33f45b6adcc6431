"""Grouped expert products on tiles of 256 places: experts of no, few and many places, edges of the weight tiles, the
shortest inner sizes, widths that fall back to the smaller tile, against the products in 64 bits."""
import pytest
import torch

from dgi.ops import moe

F64 = torch.float64
BF16 = torch.bfloat16

# places per expert around the tile's sizes: whole tiles, one place more, blocks of 64 and of 16
COUNTS = [0, 1, 16, 63, 64, 65, 128, 130, 192, 200, 255, 256, 257, 512, 513, 0, 700]


def draw(*shape, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(BF16)


def exact(h, idx, w, gu, dn, act, limit, weigh):
    """The weighed sum in 64 bits, and the sum of its terms' magnitudes."""
    h, gu, dn, w = h.to(F64), gu.to(F64), dn.to(F64), w.to(F64)
    y, mag = torch.zeros_like(h), torch.zeros_like(h)
    for e in range(gu.shape[0]):
        t, k = torch.nonzero(idx == e, as_tuple=True)
        ws = w[t, k][:, None]
        z = (h[t] * ws if weigh == "input" else h[t]) @ gu[e].t()
        g, u = z.chunk(2, dim=1)
        if act == "clamped":
            g, u = g.clamp(max=limit), u.clamp(-limit, limit)
            mid = g * torch.sigmoid(1.702 * g) * (u + 1.0)
        else:
            mid = torch.nn.functional.silu(g) * u
        f = 1.0 if weigh == "input" else ws
        y.index_add_(0, t, f * (mid @ dn[e].t()))
        mag.index_add_(0, t, f * (mid.abs() @ dn[e].abs().t()))
    return y, mag


@pytest.mark.gpu
@pytest.mark.parametrize("act,weigh", [("silu", "output"), ("clamped", "input")])
@pytest.mark.parametrize("W,ff", [(128, 128), (256, 72), (384, 640), (72, 256)])
def test_wide_tiles(monkeypatch, W, ff, act, weigh):
    E, top = len(COUNTS), 2
    g = torch.Generator().manual_seed(7)
    flat = torch.cat([torch.full((c,), e) for e, c in enumerate(COUNTS)])
    flat = flat[torch.randperm(flat.numel(), generator=g)]
    flat = flat[: flat.numel() // top * top]
    idx = flat.reshape(-1, top).to(torch.int32)
    T = idx.shape[0]
    h = draw(T, W, seed=1)
    gu, dn = draw(E, 2 * ff, W, seed=2, scale=W ** -0.5), draw(E, W, ff, seed=3, scale=ff ** -0.5)
    w = torch.rand(T, top, generator=g)
    monkeypatch.setattr(moe, "group_tile", lambda *a: 256)
    got = moe.moe_experts(h.cuda(), idx.cuda(), w.cuda(), gu.cuda(), dn.cuda(), None, act=act, limit=0.8, weigh=weigh)
    y, mag = exact(h, idx, w, gu, dn, act, 0.8, weigh)
    # three roundings to bf16 (at most 2^-8 of the value): each term's activation, each expert's row, the sum; fp32 elsewhere
    bound = 2.0 ** -8 * (2 * mag + y.abs()) + 1e-5 * (1 + mag)
    worst = ((got.cpu().to(F64) - y).abs() / bound).max().item()
    assert worst <= 1.0, worst


def run(counts, W, ff, tile, monkeypatch):
    E = len(counts)
    g = torch.Generator().manual_seed(9)
    idx = torch.cat([torch.full((c,), e) for e, c in enumerate(counts)])
    idx = idx[torch.randperm(idx.numel(), generator=g)].reshape(-1, 1).to(torch.int32)
    h = draw(idx.shape[0], W, seed=1)
    gu, dn = draw(E, 2 * ff, W, seed=2, scale=W ** -0.5), draw(E, W, ff, seed=3, scale=ff ** -0.5)
    w = torch.rand(idx.shape[0], 1, generator=g)
    monkeypatch.setattr(moe, "group_tile", lambda *a: tile)
    got = moe.moe_experts(h.cuda(), idx.cuda(), w.cuda(), gu.cuda(), dn.cuda())
    y, mag = exact(h, idx, w, gu, dn, "silu", 0.8, "output")
    bound = 2.0 ** -8 * (2 * mag + y.abs()) + 1e-5 * (1 + mag)      # as above
    assert ((got.cpu().to(F64) - y).abs() / bound).max().item() <= 1.0


@pytest.mark.gpu
@pytest.mark.parametrize("counts,W", [([200], 2048), ([256], 16384), ([130, 60], 9216), ([256], 32768), ([65], 34816), ([250], 67584), ([600, 1], 2304),
                                      ([1], 256)], ids=str)
def test_tiles_that_are_cut(monkeypatch, counts, W):
    """1, 8, 9, 16, 17 and 1 more than 32 tiles an XCD in the down product, several of them of one expert, fewer than there are XCDs."""
    run(counts, W, 128, 256, monkeypatch)


@pytest.mark.gpu
@pytest.mark.parametrize("counts,W,ff", [([50, 40, 66, 3], 2048, 1024), ([60, 64, 30, 53], 2048, 1024), ([30, 80], 1024, 512), ([70, 80], 1024, 512), ([100, 28], 136, 1024)],
                         ids=str)
def test_middling_experts(monkeypatch, counts, W, ff):
    """Tiles of 128 asked for: streamed ones of 64, wide ones or those, as means and widths say."""
    run(counts, W, ff, 128, monkeypatch)


@pytest.mark.gpu
@pytest.mark.parametrize("T,E,top,K", [(1, 16, 2, 4096), (17, 16, 16, 2048), (33, 9, 4, 6144), (5, 32, 3, 4160), (20, 64, 5, 2080), (2, 40, 2, 12288)])
def test_router_widths(T, E, top, K):
    """Routes of widths whose steps a wave takes eight, four or two at a time, some past the end: scores against 64 bits; rows of equal scores
    take the lowest experts; a row that is not a number gets experts that there are, each once."""
    from dgi.ops import moe
    g = torch.Generator().manual_seed(K + T)
    h = torch.randn(T + 2, K, generator=g).to(torch.bfloat16)
    h[T], h[T + 1] = 0.0, float("nan")
    router = (torch.randn(E, K, generator=g) * K ** -0.5).to(torch.bfloat16)
    idx, w = moe.moe_router(h.cuda(), router.float().cuda(), router.cuda(), top, False, 1.0)
    idx, w = idx.cpu().long(), w.cpu()
    score = torch.sigmoid(h.double() @ router.double().t())
    best = torch.sort(score[:T], 1, descending=True).values[:, :top]
    # fp32 sums of K products of about K ** -0.5 each: 1e-5 of a logit leaves room for every order
    assert ((w[:T] - best).abs() < 1e-5).all() and ((score[:T].gather(1, idx[:T]) - best).abs() < 1e-5).all()
    assert idx[T].tolist() == list(range(top)) and (w[T] == 0.5).all()
    assert all(len(set(r)) == top and 0 <= min(r) and max(r) < E for r in idx.tolist())
