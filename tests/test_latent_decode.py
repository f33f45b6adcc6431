"""Decode rows on cached latents, the whole layer part (latent_decode_heads: fold, attention in runs, values with gates) against
64 bits: one row, rows around sixteen, one run and several, query and value sizes, gates, strided queries."""
import pytest
import torch

from dgi.ops import latent

F64, BF16, I32 = torch.float64, torch.bfloat16, torch.int32
KR, RD, BS = 512, 64, 16


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 15, 16, 17, 40])
@pytest.mark.parametrize("H,dim,vdim,gated", [(4, 64, 128, None), (3, 32, 16, "head"), (33, 96, 48, "element"), (2, 128, 112, None)])
def test_decode_heads(T, H, dim, vdim, gated):
    g = torch.Generator().manual_seed(T * H)
    N, qk = 330, dim + RD
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
    pos = [(37 * t + 5) % N for t in range(T)]
    scale = qk ** -0.5
    want, slack = torch.zeros(T, H * vdim, dtype=F64), torch.zeros(T, H * vdim, dtype=F64)
    e = 2.0 ** -8                                            # a rounding to bf16, at most, of a number's size
    for t, p in enumerate(pos):
        c, r = rows[:p + 1, :KR].to(F64), rows[:p + 1, KR:].to(F64)
        qq = q[t].to(F64).view(H, qk)
        ql = torch.einsum("hd,hdk->hk", qq[:, :dim], uk.to(F64))
        s = (ql @ c.t() + qq[:, dim:] @ r.t()) * scale
        w = torch.softmax(torch.cat([s, sinks.to(F64)[:, None]], 1), 1)[:, :-1]
        ds = (ql.abs() @ c.abs().t()) * scale * e            # the folded query is rounded: a score moves by this at most
        o, om = w @ c, (w * (e + ds + (w * ds).sum(1, keepdim=True))) @ c.abs()
        y = torch.einsum("hk,hvk->hv", o, uv.to(F64))
        ym = torch.einsum("hk,hvk->hv", om + e * o.abs(), uv.to(F64).abs()) + e * y.abs()
        f = torch.ones(H, vdim, dtype=F64)
        if gated is not None:
            f = torch.sigmoid(gate[t].to(F64)).view(H, -1).expand(H, vdim)
        want[t], slack[t] = (y * f).reshape(-1), (ym * f).reshape(-1) + 1e-5
    dev = "cuda"
    assert latent.decode_heads_ok(wide.to(dev)[:, :H * qk], T, dim, RD, KR, vdim, gate)
    tables = perm[None, :].repeat(T, 1).contiguous().to(dev)
    for max_keys in (0, 1 << 12):
        out = torch.full((T, H * vdim), 7.0, dtype=BF16, device=dev)
        latent.latent_decode_heads(wide.to(dev)[:, :H * qk], uk.to(dev), uv.to(dev), cache.to(dev), tables,
                                   torch.tensor(pos, dtype=I32, device=dev), RD, scale, 0, None, True, out, max_keys, sinks.to(dev),
                                   None if gate is None else gate.to(dev), gated == "head")
        worst = ((out.cpu().to(F64) - want).abs() / slack).max().item()
        assert worst <= 1.0, worst


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
