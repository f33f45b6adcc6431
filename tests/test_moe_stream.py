"""Grouped expert products that stream the weights (dgi/csrc/mix/moe_group.hip: moe_group_stream_kernel, moe_group_rows_kernel): tiles of
16, 32 and 64 places, blocks of weights that end inside 16 rows, inner sizes around what eight waves share, and too long or ragged for
the rows of A to stay in registers, against the products in 64 bits."""
import pytest
import torch

from dgi.ops import moe
from test_moe_wide import BF16, F64, draw, exact

COUNTS = [0, 1, 15, 16, 17, 0, 31, 33, 64, 65, 7, 0]


def run(monkeypatch, tile, W, ff, counts, act="silu", weigh="output", top=2):
    E = len(counts)
    g = torch.Generator().manual_seed(7)
    flat = torch.cat([torch.full((c,), e) for e, c in enumerate(counts)])
    flat = flat[torch.randperm(flat.numel(), generator=g)]
    flat = flat[: flat.numel() // top * top]
    idx = flat.reshape(-1, top).to(torch.int32)
    T = idx.shape[0]
    h = draw(T, W, seed=1)
    gu, dn = draw(E, 2 * ff, W, seed=2, scale=W ** -0.5), draw(E, W, ff, seed=3, scale=ff ** -0.5)
    w = torch.rand(T, top, generator=g)
    monkeypatch.setattr(moe, "group_tile", lambda *a: tile)
    got = moe.moe_experts(h.cuda(), idx.cuda(), w.cuda(), gu.cuda(), dn.cuda(), None, act=act, limit=0.8, weigh=weigh)
    y, mag = exact(h, idx, w, gu, dn, act, 0.8, weigh)
    # three roundings to bf16 (at most 2^-8 of the value): each term's activation, each expert's row, the sum; fp32 elsewhere
    bound = 2.0 ** -8 * (2 * mag + y.abs()) + 1e-5 * (1 + mag)
    worst = ((got.cpu().to(F64) - y).abs() / bound).max().item()
    assert worst <= 1.0, worst


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [16, 32, 64])
@pytest.mark.parametrize("W,ff", [(64, 128), (576, 72), (1088, 200), (2048, 64), (72, 104), (8, 16)])
def test_streamed_experts(monkeypatch, W, ff, tile):
    """72, 104, 8 and 200 are no multiples of 64 (the other kernel); 576 = 9 stages leave waves without any."""
    run(monkeypatch, tile, W, ff, COUNTS)
    run(monkeypatch, tile, W, ff, COUNTS, "clamped", "input")


@pytest.mark.gpu
@pytest.mark.parametrize("tile,W,ff", [(16, 8192, 64), (16, 8256, 128), (32, 4096, 64), (32, 4160, 64), (64, 2112, 64), (16, 2560, 1088)])
def test_rows_around_what_the_registers_hold(monkeypatch, tile, W, ff):
    run(monkeypatch, tile, W, ff, [3, 0, 20, 1, 35])


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [16, 32, 64])
def test_one_row_and_more_shares_than_blocks(monkeypatch, tile):
    run(monkeypatch, tile, 128, 64, [1, 0, 1])
    run(monkeypatch, tile, 128, 64, [0] * 70 + [5] + [0] * 40 + [70, 3])       # more experts than lanes


def test_tiles_by_the_mean_rows_of_an_expert():
    big, small = 1 << 24, 1 << 19
    assert [moe.group_tile(16 * m, 16, big) for m in (1, 4, 5, 20, 21, 40, 41, 95, 96)] == [16, 16, 32, 32, 64, 64, 128, 128, 256]
    assert [moe.group_tile(16 * m, 16, small) for m in (40, 41, 255, 256)] == [64, 128, 128, 256]
    assert [moe.group_tile(64 * m, 64, small) for m in (12, 13)] == [32, 128]


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [16, 32, 64])
@pytest.mark.parametrize("T,top,E", [(1, 1, 1), (1, 2, 16), (31, 2, 3), (32, 2, 16), (63, 1, 64), (128, 4, 64), (171, 3, 64), (129, 4, 16), (40, 2, 65)])
def test_pairs_sorted_by_the_product(T, top, E, tile):
    """Up to 512 pairs and 64 experts the gate-up product sorts the pairs itself: the plan that ``moe_plan`` makes, identity routes
    (E and beyond) left out, and the same product."""
    from dgi.ops import _call
    W, ff = 128, 72
    g = torch.Generator().manual_seed(T + E)
    idx = torch.randint(0, E + 2, (T, top), generator=g, dtype=torch.int32).cuda()
    h, gu = draw(T, W, seed=4).cuda(), draw(E, 2 * ff, W, seed=5, scale=W ** -0.5).cuda()
    scale = torch.rand(T * top, generator=g).cuda()
    P = T * top
    for weights in (None, scale):
        made = []
        for fused in (False, True):
            order, where, seg = (torch.full((n,), -7, dtype=torch.int32, device="cuda") for n in (P, P, E + 1))
            out = torch.full((P, ff), 3.0, dtype=BF16, device="cuda")
            if fused:
                _call("moe_plan_group", out, order, where, seg, idx, h, gu, weights, top, 0, 0.0, 0.0, tile)
            else:
                _call("moe_plan", order, where, seg, idx)
                _call("moe_group", out, h, gu, seg, order, weights, top, 0, 0.0, 0.0, tile)
            made.append((order, where, seg, out))
        for a, b in zip(*made):
            assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("skip", [0, 1])
@pytest.mark.parametrize("P,E", [(1, 1), (3, 5), (4, 2), (1023, 16), (1024, 16), (1025, 3), (4096, 64), (4097, 65), (8190, 16), (20000, 130)])
def test_plan_of_many_pairs(P, E, skip):
    """The places of the pairs by expert in their order, identity routes left out, also from an index at no 16-byte boundary."""
    from dgi.ops import _call
    idx = torch.randint(-1, E + 1, (P + skip,), generator=torch.Generator().manual_seed(P), dtype=torch.int32).cuda()[skip:]
    order, where, seg = (torch.full((n,), -7, dtype=torch.int32, device="cuda") for n in (P, P, E + 1))
    _call("moe_plan", order, where, seg, idx)
    i = idx.cpu().long()
    pairs = torch.nonzero((i >= 0) & (i < E))[:, 0]
    pairs = pairs[torch.argsort(i[pairs], stable=True)]
    counts = torch.bincount(i[pairs], minlength=E)
    assert seg.tolist() == [0] + counts.cumsum(0).tolist()
    n = pairs.numel()
    assert torch.equal(order[:n].cpu().long(), pairs) and (order[n:] == -7).all()
    assert torch.equal(where.cpu().long()[pairs], torch.arange(n))


def test_tiles_of_ragged_widths():
    assert [moe.expert_tile(16 * m, 16, 2040, 2040) for m in (20, 24, 25, 40, 41)] == [32, 64, 128, 128, 128]
    assert [moe.expert_tile(16 * m, 16, 2048, 2048) for m in (24, 25, 40, 41)] == [64, 64, 64, 128]
    assert moe.expert_tile(16 * 36, 16, 1000, 1000) == moe.expert_tile(4 * 36, 4, 1032, 4104) == 64
    assert moe.expert_tile(8 * 36, 8, 4104, 3592) == moe.expert_tile(8 * 36, 8, 4096, 4104) == 128
