"""Latent attention on shared tiles (512 + 64 dims, bf16): runs without keys, tiles of one key, windows that start inside a
tile, head groups that are not full, rows of portions, against softmax attention in 64 bits."""
import pytest
import torch

from dgi.ops import latent

F64, BF16, I32 = torch.float64, torch.bfloat16, torch.int32
KR, RD, DIM = 512, 64, 24


@pytest.mark.gpu
@pytest.mark.parametrize("H", [1, 16, 17, 32, 40])
@pytest.mark.parametrize("window,bs", [(0, 16), (70, 16), (200, 5)])
@pytest.mark.parametrize("dims,inter", [(64, True), (32, False), (0, False)])
def test_latent_tiles(H, window, bs, dims, inter):
    g = torch.Generator().manual_seed(H + window)
    N = 460
    queries = [459, 400, 255, 256, 129, 128, 127, 64, 63, 32, 31, 1, 0]
    T = len(queries)
    nblk = -(-N // bs)
    perm = torch.randperm(nblk + 3, generator=g)[:nblk].to(I32)
    rows = torch.randn(N, KR + RD, generator=g).to(BF16)
    cache = torch.full((nblk + 3, 1, bs, KR + RD), float("nan"), dtype=BF16)      # nothing but the listed keys may be read
    for j in range(N):
        cache[int(perm[j // bs]), 0, j % bs] = rows[j]
    q = torch.randn(T, H * (DIM + RD), generator=g).to(BF16)
    q_lat = (torch.randn(H, T, KR, generator=g) * 0.3).to(BF16)
    sinks = torch.randn(H, generator=g)
    ang = torch.arange(512, dtype=F64)[:, None] * torch.exp(-torch.arange(max(dims, 2) // 2, dtype=F64) / 8)
    cs = torch.cat([ang.cos(), ang.sin()], 1).float() if dims else None
    scale = (DIM + RD) ** -0.5
    want, slack = torch.zeros(H, T, KR, dtype=F64), torch.zeros(H, T, KR, dtype=F64)
    qr = q.view(T, H, DIM + RD)[:, :, DIM:].float()
    if dims:
        qr = latent.rotate_ref(qr, cs[torch.tensor(queries)], dims, inter)
    qr = qr.to(BF16).to(F64)                                                       # the rotated part is rounded once
    for t, p in enumerate(queries):
        lo = max(0, p - window + 1) if window else 0
        c, r = rows[lo:p + 1, :KR].to(F64), rows[lo:p + 1, KR:].to(F64)
        s = (q_lat[:, t].to(F64) @ c.t() + qr[t] @ r.t()) * scale
        w = torch.softmax(torch.cat([s, sinks.to(F64)[:, None]], 1), 1)[:, :-1]
        want[:, t] = w @ c
        # weights and results are rounded to bf16, 2^-8 of their size each.  Where a rotated value (a fused or a plain sum of
        # two products) lies at the edge of two bf16 numbers it may be rounded either way: at most 2^-7 of each rotated term
        # of a score, which moves a weight by that much and the weights' sum by the mean of it
        ds = (qr[t].abs() @ r.abs().t()) * scale * (2.0 ** -7 if dims else 0.0)
        slack[:, t] = 2.0 ** -8 * (w @ c.abs()) + (w * (ds + (w * ds).sum(1, keepdim=True))) @ c.abs() + 1e-5
    dev = "cuda"
    tables = perm[None, :].repeat(T, 1).contiguous().to(dev)
    pos = torch.tensor(queries, dtype=I32, device=dev)
    args = (H, DIM, RD, KR, scale, window, None if cs is None else cs.to(dev), inter)

    def check(got, order=slice(None)):
        worst = ((got.cpu().to(F64) - want[:, order]).abs() / (slack[:, order] + 2.0 ** -8 * want[:, order].abs())).max().item()
        assert worst <= 1.0, worst

    qd, ql, cd, sd = q.to(dev), q_lat.to(dev), cache.to(dev), sinks.to(dev)
    for max_keys in (0, N, 1 << 14):
        out = torch.full((H, T, KR), 7.0, dtype=BF16, device=dev)
        latent.latent_attn_rows(qd, ql, cd, tables, None, pos, *args, out, max_keys=max_keys, sinks=sd)
        check(out)
    # odd strides (no wide accesses of queries or results), and the rows as portions of two sequences on the same pages
    wide = torch.zeros(H, T, KR + 6, dtype=BF16, device=dev)
    wide[:, :, 3:KR + 3] = ql
    out = torch.full((H, T, KR + 2), 7.0, dtype=BF16, device=dev)[:, :, 1:KR + 1]
    latent.latent_attn_rows(qd, wide[:, :, 3:KR + 3], cd, tables, None, pos, *args, out, sinks=sd)
    check(out)
    order = sorted(range(T), key=lambda i: queries[i])
    cu = torch.tensor([0, 4, T], dtype=I32, device=dev)
    out = torch.full((H, T, KR), 7.0, dtype=BF16, device=dev)
    latent.latent_attn_rows(qd[order].contiguous(), ql[:, order].contiguous(), cd, tables[:2].contiguous(), cu,
                            pos[order].contiguous(), *args, out, sinks=sd)
    check(out, order)


@pytest.mark.gpu
@pytest.mark.parametrize("kr,rd,dtype", [(512, 64, BF16), (128, 64, BF16), (512, 32, BF16), (64, 20, torch.float32)])
@pytest.mark.parametrize("sinks", [False, True])
def test_rows_without_a_position(kr, rd, dtype, sinks):
    """A negative position (a row that pads a step): no key, results of zero in every form, the rows beside it as without it."""
    g = torch.Generator().manual_seed(kr + rd)
    H, T, bs, N, dev = 5, 4, 16, 700, "cuda"
    pos = [699, -1, 300, -70]
    cache = torch.randn(N // bs + 1, 1, bs, kr + rd, generator=g).to(dtype)
    tables = torch.arange(N // bs + 1, dtype=I32)[None, :].repeat(T, 1).contiguous()
    q, q_lat = torch.randn(T, H * (32 + rd), generator=g).to(dtype), (torch.randn(H, T, kr, generator=g) * 0.3).to(dtype)
    cs = torch.randn(N, rd, generator=g)
    sk = torch.randn(H, generator=g) if sinks else None

    def run(rows, max_keys, device):
        o = torch.full((H, len(rows), kr), 7.0, dtype=dtype, device=device)
        to = lambda t: None if t is None else t.to(device)  # noqa: E731
        latent.latent_attn_rows(to(q[rows].contiguous()), to(q_lat[:, rows].contiguous()), to(cache), to(tables[rows]), None,
                                torch.tensor([pos[i] for i in rows], dtype=I32, device=device), H, 32, rd, kr, 0.1, 0, to(cs), True, o,
                                max_keys=max_keys, sinks=to(sk))
        return o.cpu().float()

    want = run([0, 2], 0, "cpu")
    for max_keys in (0, 1 << 14):
        got = run([0, 1, 2, 3], max_keys, dev)
        assert (got[:, [1, 3]] == 0).all()
        # bf16: the query's rotated part, weights and results are rounded, 2^-8 each, and a score is a few units large
        assert (got[:, [0, 2]] - want).abs().max() <= (2.0 ** -6 if dtype == BF16 else 1e-4) * want.abs().max()


@pytest.mark.gpu
@pytest.mark.parametrize("H,n,max_keys", [(32, 90, 0), (17, 900, 0), (32, 900, 1 << 11)])
def test_weights_keep_their_precision(monkeypatch, H, n, max_keys):
    """No further from 64 bits than the form that holds the weights in fp32: what both round is the result.  Two such errors over 2e5
    values differ by under one per cent; weights rounded to bf16 add two fifths."""
    g = torch.Generator().manual_seed(H + n)
    T, bs, dev = 12, 16, "cuda"
    nblk = -(-n // bs)
    cache = torch.randn(nblk, 1, bs, KR + RD, generator=g).to(BF16)
    q, q_lat = torch.randn(T, H * (DIM + RD), generator=g).to(BF16), (torch.randn(H, T, KR, generator=g) * 0.3).to(BF16)
    pos = torch.tensor([n - 1 - 3 * t for t in range(T)], dtype=I32)
    scale = (DIM + RD) ** -0.5
    rows = cache.view(-1, KR + RD).to(F64)
    want = torch.empty(H, T, KR, dtype=F64)
    for t, p in enumerate(pos.tolist()):
        s = torch.cat([q_lat[:, t].to(F64), q[t].to(F64).view(H, DIM + RD)[:, DIM:]], 1) @ rows[:p + 1].t() * scale
        want[:, t] = torch.softmax(s, 1) @ rows[:p + 1, :KR]
    tables = torch.arange(nblk, dtype=I32)[None, :].repeat(T, 1).contiguous().to(dev)

    def error():
        out = torch.empty(H, T, KR, dtype=BF16, device=dev)
        latent.latent_attn_rows(q.to(dev), q_lat.to(dev), cache.to(dev), tables, None, pos.to(dev), H, DIM, RD, KR, scale, 0, None, True,
                                out, max_keys=max_keys)
        return ((out.cpu().to(F64) - want).norm() / want.norm()).item()

    tiles = error()
    monkeypatch.setattr(latent, "MFMA_ROWS", False)
    assert tiles <= 1.05 * error()
