"""Decode rows on cached latents, the whole layer part (latent_decode_heads: fold, attention in runs, values with gates) against
64 bits: one row, rows around sixteen and many, one run and up to 64, query and value sizes, gates, strided queries, windows, rotation."""
from types import SimpleNamespace

import pytest
import torch

from dgi.models import latent_mixer
from dgi.ops import latent

F64, BF16, I32 = torch.float64, torch.bfloat16, torch.int32
KR, RD, BS = 512, 64, 16


def compare(T, H, dim, vdim, gated, keys=(0, 1 << 12), window=0, dims=0, inter=True, N=330, layer=False, pos=None):
    """latent_decode_heads (or the layer around it) against 64 bits for rows at positions spread over N."""
    g = torch.Generator().manual_seed(T * H)
    qk = dim + RD
    rows = torch.randn(N, KR + RD, generator=g).to(BF16)
    nblk = -(-N // BS)
    perm = torch.randperm(nblk, generator=g).to(I32)
    cache = torch.zeros(nblk, 1, BS, KR + RD, dtype=BF16)
    for j in range(N):
        cache[int(perm[j // BS]), 0, j % BS] = rows[j]
    wide = torch.randn(T, H * qk + 8, generator=g).to(BF16)
    q = wide[:, :H * qk]
    uk, uv = ((torch.randn(H, n, KR, generator=g) * KR ** -0.5).to(BF16) for n in (dim, vdim))
    sinks = torch.randn(H, generator=g)
    gate = None if gated is None else torch.randn(T, H if gated == "head" else H * vdim, generator=g).to(BF16)
    pos = [(37 * t + 5) % N for t in range(T)] if pos is None else pos
    ang = torch.arange(N, dtype=F64)[:, None] * torch.exp(-torch.arange(max(dims, 2) // 2, dtype=F64) / 8)
    cs = torch.cat([ang.cos(), ang.sin()], 1).float() if dims else None
    scale = qk ** -0.5
    qr = q.view(T, H, qk)[:, :, dim:].float()
    if dims:
        qr = latent.rotate_ref(qr, cs[torch.tensor(pos)], dims, inter)
    qr = qr.to(BF16).to(F64)                                 # the rotated part is rounded once
    want, slack = torch.zeros(T, H * vdim, dtype=F64), torch.zeros(T, H * vdim, dtype=F64)
    e = 2.0 ** -8                                            # a rounding to bf16, at most, of a number's size
    for t, p in enumerate(pos):
        lo = max(0, p - window + 1) if window else 0
        c, r = rows[lo:p + 1, :KR].to(F64), rows[lo:p + 1, KR:].to(F64)
        ql = torch.einsum("hd,hdk->hk", q[t].to(F64).view(H, qk)[:, :dim], uk.to(F64))
        s = (ql @ c.t() + qr[t] @ r.t()) * scale
        w = torch.softmax(torch.cat([s, sinks.to(F64)[:, None]], 1), 1)[:, :-1]
        ds = (ql.abs() @ c.abs().t()) * scale * e            # the folded query is rounded: a score moves by this at most
        if dims:                                             # a rotated value between two bf16 numbers may go either way
            ds = ds + (qr[t].abs() @ r.abs().t()) * scale * 2 * e
        o, om = w @ c, (w * (e + ds + (w * ds).sum(1, keepdim=True))) @ c.abs()
        y = torch.einsum("hk,hvk->hv", o, uv.to(F64))
        ym = torch.einsum("hk,hvk->hv", om + e * o.abs(), uv.to(F64).abs()) + e * y.abs()
        f = torch.ones(H, vdim, dtype=F64)
        if gated is not None:
            f = torch.sigmoid(gate[t].to(F64)).view(H, -1).expand(H, vdim)
        want[t], slack[t] = (y * f).reshape(-1), (ym * f).reshape(-1) + 1e-5
    dev = "cuda"
    assert latent.decode_heads_ok(wide.to(dev)[:, :H * qk], T, dim, RD, KR, vdim, gate)
    to = lambda x: None if x is None else x.to(dev)  # noqa: E731
    tables = perm[None, :].repeat(T, 1).contiguous().to(dev)
    positions = torch.tensor(pos, dtype=I32, device=dev)
    qd = wide.to(dev)[:, :H * qk]
    for max_keys in keys:
        out = torch.full((T, H * vdim), 7.0, dtype=BF16, device=dev)
        if layer:
            m = SimpleNamespace(heads=H, dim=dim, rot_dim=RD, kv_rank=KR, vdim=vdim, qk_dim=qk, scale=scale, window=window, gate=gated,
                                rot=SimpleNamespace(layout="interleaved" if inter else "half"), o_size=H * vdim, cache_dim=KR + RD)
            wt = torch.zeros(T, -(-max(max_keys, N) // BS), dtype=I32, device=dev)
            wt[:, :nblk] = tables
            meta = SimpleNamespace(num_decode=T, num_prefill_tokens=0, dec_block_tables=wt, positions=positions)
            out = latent_mixer.latent_heads(m, SimpleNamespace(uk=to(uk), uv=to(uv)), qd, to(cache), meta, to(cs), to(gate), to(sinks))
        else:
            latent.latent_decode_heads(qd, to(uk), to(uv), to(cache), tables, positions, RD, scale, window, to(cs), inter, out, max_keys,
                                       to(sinks), to(gate), gated == "head")
        worst = ((out.cpu().to(F64) - want).abs() / slack).max().item()
        assert worst <= 1.0, worst


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 15, 16, 17, 40])
@pytest.mark.parametrize("H,dim,vdim,gated", [(4, 64, 128, None), (3, 32, 16, "head"), (33, 96, 48, "element"), (2, 128, 112, None)])
def test_decode_heads(T, H, dim, vdim, gated):
    compare(T, H, dim, vdim, gated)


@pytest.mark.gpu
@pytest.mark.parametrize("T,H", [(96, 32), (90, 32), (128, 32), (129, 33), (250, 32), (256, 17)])
def test_decode_heads_rows_per_workgroup(T, H):
    """Steps whose value product takes eight and sixteen rows a workgroup, the last of them full and not."""
    compare(T, H, 32, 32, "head")


@pytest.mark.gpu
@pytest.mark.parametrize("T,max_keys", [(1, 1 << 13), (3, 1 << 14), (7, 1 << 13)])
def test_decode_heads_many_runs(T, max_keys):
    """64 runs of keys (the most there are), some and most of them empty, and a number of runs that is no multiple of four."""
    assert latent.tile_runs(T, 20, max_keys) == {1: 64, 3: 64, 7: 36}[T]
    compare(T, 20, 64, 48, None, keys=(max_keys,), N=330 if T > 1 else 6)
    compare(T, 20, 64, 48, None, keys=(max_keys,), N=5000, pos=[4999 - 611 * t for t in range(T)])


@pytest.mark.gpu
@pytest.mark.parametrize("T,vdim", [(1, 128), (2, 80), (3, 128), (5, 64), (6, 96), (11, 128)])
def test_decode_heads_rows_that_share_threads(T, vdim):
    """Values: one row, two and four at a time, whose threads share its runs, in fewer and more than a batch; a workgroup's value dims from 16 to all."""
    compare(T, 20, 64, vdim, "element", keys=(128, 1 << 10, 1 << 12))


@pytest.mark.gpu
@pytest.mark.parametrize("T", [5, 100])
@pytest.mark.parametrize("window,dims,inter,gated", [(0, 64, True, None), (100, 64, False, "head"), (70, 32, True, "element"), (33, 0, True, None)])
def test_layer_with_windows_and_rotation(T, window, dims, inter, gated):
    """The layer's part as a model calls it: windows, rotations of all and of some dims in both layouts, tables wider than the contexts."""
    compare(T, 18, 64, 32, gated, keys=(0, 1 << 12), window=window, dims=dims, inter=inter, layer=True)

@pytest.mark.gpu
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("max_keys", [0, 1 << 13])
def test_rows_without_a_position(gated, max_keys):
    """A negative position: no key, head outputs of zero, with one run of keys and with several."""
    g = torch.Generator().manual_seed(5)
    T, H, dim, vdim, dev = 3, 4, 64, 32, "cuda"
    cache = torch.randn(20, 1, BS, KR + RD, generator=g).to(BF16).to(dev)
    q = torch.randn(T, H * (dim + RD), generator=g).to(BF16).to(dev)
    uk, uv = (torch.randn(H, n, KR, generator=g).to(BF16).to(dev) for n in (dim, vdim))
    gate = torch.randn(T, H, generator=g).to(BF16).to(dev) if gated else None
    out = torch.full((T, H * vdim), 7.0, dtype=BF16, device=dev)
    latent.latent_decode_heads(q, uk, uv, cache, torch.arange(20, dtype=I32, device=dev)[None, :].repeat(T, 1).contiguous(),
                               torch.tensor([-1, 300, -70], dtype=I32, device=dev), RD, 0.1, 0, torch.randn(320, RD, generator=g).to(dev),
                               True, out, max_keys, None, gate, True)
    assert (out[[0, 2]] == 0).all() and torch.isfinite(out).all() and (out[1] != 0).any()


@pytest.mark.gpu
@pytest.mark.parametrize("H", [4, 32])
def test_contexts_around_the_tiles(H):
    """Contexts around tiles of 32 keys and what is loaded ahead of them, runs without keys, and rows without a position whose pages are
    nobody's, against the same rows one by one in a single run, and those against 64 bits."""
    g = torch.Generator().manual_seed(H)
    pos = [0, 14, 30, 31, 32, 62, 63, 64, 95, 96, 127, 128, 300, -1, 2049]
    T, dim, vdim, dev = len(pos), 64, 32, "cuda"
    cols = 2100 // BS + 1
    cache = torch.randn(cols, 1, BS, KR + RD, generator=g).to(BF16).to(dev)
    tables = torch.stack([torch.randperm(cols, generator=g) if p >= 0 else torch.full((cols,), 1 << 30) for p in pos]).to(I32).to(dev)
    q = torch.randn(T, H * (dim + RD), generator=g).to(BF16).to(dev)
    uk, uv = ((torch.randn(H, n, KR, generator=g) * KR ** -0.5).to(BF16).to(dev) for n in (dim, vdim))
    cs = torch.randn(2100, RD, generator=g).to(dev)
    positions = torch.tensor(pos, dtype=I32, device=dev)

    def run(rows, max_keys):
        out = torch.full((len(rows), H * vdim), 7.0, dtype=BF16, device=dev)
        latent.latent_decode_heads(q[rows].contiguous(), uk, uv, cache, tables[rows].contiguous(), positions[rows].contiguous(), RD, 0.08, 0, cs,
                                   True, out, max_keys, None, None, False)
        return out.float()

    many = run(list(range(T)), 1 << 14)
    wide, kinds = cache.cpu(), [x.cpu().to(F64) for x in (uk, uv)]
    for i, p in enumerate(pos):
        if p < 0:
            assert (many[i] == 0).all()
            continue
        one = run([i], 0)[0]
        # weights relative to another maximum, sums and the head's value rounded to bf16
        assert (many[i] - one).abs().max() <= 2.0 ** -7 * one.abs().max()
        rows = wide[tables[i].long().cpu(), 0].reshape(-1, KR + RD)[: p + 1].to(F64)
        qi = q[i].cpu().view(H, dim + RD)
        qr = latent.rotate_ref(qi[None, :, dim:].float(), cs[p: p + 1].cpu(), RD, True)[0].to(BF16).to(F64)
        folded = torch.einsum("hd,hdk->hk", qi[:, :dim].to(F64), kinds[0]).to(BF16).to(F64)
        w = torch.softmax((folded @ rows[:, :KR].t() + qr @ rows[:, KR:].t()) * 0.08, 1)
        want = torch.einsum("hk,hvk->hv", w @ rows[:, :KR], kinds[1]).reshape(-1)
        # both roundings that move a score (the folded query, a rotated value between two bf16 numbers) are the reference's up to their ties; the
        # values and the result are rounded once each
        assert ((one.cpu().to(F64) - want).norm() / want.norm()) <= 2.0 ** -6, p


@pytest.mark.gpu
@pytest.mark.parametrize("T,H,pos", [(64, 32, None), (70, 16, None), (129, 16, None), (17, 32, None), (256, 32, 100)])
def test_many_rows(T, H, pos):
    """Rows of several workgroups each way: no runs, two (four rows of a group at once), three and four (two at once), and folds of 32 and 64 rows."""
    for keys in (1 << 7, 250, 400, 600):
        compare(T, H, 64, 128, None if keys == 250 else "element", keys=(keys,), pos=None if pos is None else [t % pos for t in range(T)])


def test_runs_of_keys_cpu():
    """At most what fills the chip, at least 64 keys each; fewer for many rows, where writing a run's sums costs more than it saves."""
    for rows in (0, 1, 7, 32, 64, 100, 128, 300):
        for heads in (1, 16, 32, 64):
            last = 1
            for bound in (0, 100, 191, 192, 300, 700, 3000, 30000, 1 << 20):
                n = latent.decode_runs(rows, heads, bound)
                assert 1 <= n <= max(1, min(64, bound // 64)) and n * max(rows, 1) <= max(256, rows) and n >= last
                last = n
    assert [latent.decode_runs(64, 32, b) for b in (192, 240, 320, 480, 576, 1312)] == [1, 2, 2, 3, 4, 4]
    assert latent.decode_runs(60, 32, 512) == 4 and latent.decode_runs(32, 32, 240) == 3      # four take less than three from about 450 keys on
    assert [latent.decode_runs(128, h, 384) for h in (16, 32)] == [2, 1] and latent.decode_runs(32, 32, 2564) == 8
