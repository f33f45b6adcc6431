"""Prompt attention: every (tile, head) pair of the flat grid, for head counts that are no multiple of the XCDs' and for
rows whose first tiles leave half of a wave's lanes without a visible key."""
import pytest
import torch

from dgi import ops


@pytest.mark.gpu
@pytest.mark.parametrize("nh,nkv", [(1, 1), (5, 1), (6, 3), (12, 4), (10, 10)])
@pytest.mark.parametrize("hd", [64, 128])
def test_heads_and_tiles(nh, nkv, hd):
    qlens, ctxs = [1, 2, 5, 33, 130, 300], [1, 2, 5, 97, 130, 365]
    g = torch.Generator().manual_seed(nh * hd)
    bs, per = 16, [-(-c // 16) for c in ctxs]
    perm = torch.randperm(sum(per) + 2, generator=g)
    bt = torch.zeros(len(per), max(per), dtype=torch.int32)
    at = 0
    for i, n in enumerate(per):
        bt[i, :n] = perm[at:at + n]
        at += n
    kc, vc = (torch.randn(sum(per) + 2, nkv, bs, hd, generator=g).to(torch.bfloat16) for _ in range(2))
    q = torch.randn(sum(qlens), nh * hd, generator=g).to(torch.bfloat16)
    cu = torch.tensor([0] + qlens).cumsum(0).to(torch.int32)
    ctx = torch.tensor(ctxs, dtype=torch.int32)
    got = ops.paged_prefill(q.cuda(), kc.cuda(), vc.cuda(), bt.cuda(), cu.cuda(), ctx.cuda(), nh, nkv, hd ** -0.5).cpu().double()
    for b, (n, c) in enumerate(zip(qlens, ctxs)):
        keys = torch.arange(c)
        kk, vv = (t[bt[b][keys // bs].long(), :, keys % bs].double().repeat_interleave(nh // nkv, 1) for t in (kc, vc))
        rows = slice(int(cu[b]), int(cu[b + 1]))
        s = torch.einsum("thd,khd->htk", q[rows].double().view(n, nh, hd), kk) * hd ** -0.5
        s = s.masked_fill(keys[None, None] > (torch.arange(n) + c - n)[None, :, None], float("-inf"))
        w = torch.softmax(s, -1)
        want, mag = (torch.einsum("htk,khd->thd", w, v).reshape(n, -1) for v in (vv, vv.abs()))
        # weights and results are rounded to bf16, at most 2^-8 of their size each
        assert ((got[rows] - want).abs() <= 2.0 ** -8 * (mag + want.abs()) + 1e-4).all()
