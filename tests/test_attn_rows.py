"""Masked attention of single rows in bf16 (dgi/csrc/mix/masked_attention.hip: masked_attn_tiles_kernel) against the fp32 reference:
edges of the 64-key tiles and of the waves' turns, head sizes around the 32-dim products, group sizes, runs, masks that start inside a page."""
import pytest
import torch

from dgi.ops import mix

I32, BF16 = torch.int32, torch.bfloat16


def case(ctx, H, G, dk, dv, bs, seed):
    g = torch.Generator().manual_seed(seed)
    need = [-(-n // bs) for n in ctx]
    pages = sum(need) + 1
    perm = (torch.randperm(pages - 1, generator=g) + 1).to(I32)
    table = torch.zeros(len(ctx), max(need), dtype=I32)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = perm[at:at + n]
        at += n
    # page 0 belongs to no row: reading it shows
    kc, vc = (torch.randn(pages, G, bs, d, generator=g).to(BF16) for d in (dk, dv))
    kc[0], vc[0] = 50.0, 50.0
    q = torch.randn(len(ctx), H * dk + 3, generator=g).to(BF16)        # rows at odd strides
    gate = torch.randn(len(ctx), H * dv + 5, generator=g).to(BF16)
    return q, kc, vc, table, torch.tensor([n - 1 for n in ctx], dtype=I32), gate


def check(q, kc, vc, table, pos, H, G, mask=0, gate=None, runs=1, **opt):
    scale = kc.shape[3] ** -0.5
    want = mix.masked_attn_rows_ref(q.float(), kc.float(), vc.float(), table, None, pos, H, G, scale, mask,
                                    None if gate is None else gate.float(), **opt)
    dev = {k: v.cuda() if torch.is_tensor(v) else v for k, v in opt.items()}
    old = mix.masked_split_runs
    mix.masked_split_runs = lambda *a: runs
    try:
        got = mix.masked_attn_rows(q.cuda(), kc.cuda(), vc.cuda(), table.cuda(), None, pos.cuda(), H, G, scale, mask,
                                   None if gate is None else gate.cuda(), **dev)
    finally:
        mix.masked_split_runs = old
    # the result is rounded to bf16 once (2^-9 of it); scores and sums in fp32 over at most 3000 keys add some 1e-5 of the largest value (5)
    err = (got.float().cpu() - want).abs()
    assert (err <= 2 ** -8 * want.abs() + 1e-4).all(), float((err - 2 ** -8 * want.abs()).max())


@pytest.mark.gpu
@pytest.mark.parametrize("runs", [1, 3])
@pytest.mark.parametrize("H,G,dk,dv", [(8, 2, 128, 128), (2, 2, 64, 64), (6, 2, 24, 72), (16, 2, 128, 104), (5, 1, 8, 8), (2, 1, 120, 40)])
def test_rows_at_the_edges_of_tiles(H, G, dk, dv, runs):
    ctx = [1, 15, 16, 17, 63, 64, 65, 128, 511, 512, 513, 577, 1025, 1600]
    q, kc, vc, table, pos, gate = case(ctx, H, G, dk, dv, 16, 5)
    check(q, kc, vc, table, pos, H, G, runs=runs)
    check(q, kc, vc, table, pos, H, G, 100, gate, runs=runs, softcap=20.0, sinks=torch.linspace(-2.0, 3.0, H))
    check(q, kc, vc, table, pos, H, G, 0, gate[:, :H], runs=runs, window=77, head_scale=torch.linspace(-1.5, 2.0, H), gate_heads=True)


@pytest.mark.gpu
@pytest.mark.parametrize("dk", [64, 128])
def test_four_waves_a_workgroup(dk):
    """More workgroups than compute units: four waves take the tiles in turn; pages of four and a distance bias."""
    ctx = [1 + (37 * i) % 700 for i in range(300)]
    q, kc, vc, table, pos, gate = case(ctx, 4, 1, dk, dk, 4, 6)
    check(q, kc, vc, table, pos, 4, 1, 0, gate, dist_bias=torch.randn(90, 4, generator=torch.Generator().manual_seed(7)))


@pytest.mark.gpu
def test_an_infinite_key_and_value_stay_theirs():
    """A key's infinity makes its own weight 0 (scores of minus infinity) in heads that look away from it; its value is multiplied by that zero
    only where the row sees it."""
    q, kc, vc, table, pos, _ = case([200, 90], 2, 1, 40, 40, 16, 8)
    q[:, :80] = q[:, :80].abs() + 0.1
    kc[int(table[0, 5]), 0, 3, 7] = -float("inf")        # position 83 of row 0
    vc[int(table[1, 5]), 0, 10:] = float("inf")          # positions 90 on of row 1: past its end
    check(q, kc, vc, table, pos, 2, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("runs", [1, 3])
def test_rows_without_a_position(runs):
    """Position -1: no key is read, the result is zero; the rows beside it keep theirs."""
    q, kc, vc, table, pos, gate = case([700, 1, 33], 4, 2, 64, 64, 16, 9)
    pos[1] = -1
    check(q, kc, vc, table, pos, 4, 2, gate=gate, runs=runs)
    check(q, kc, vc, table, pos, 4, 2, runs=runs, sinks=torch.linspace(-2.0, 3.0, 4), window=20)
    kept = [0, 2]
    want = mix.masked_attn_rows(q.cuda()[kept], kc.cuda(), vc.cuda(), table.cuda()[kept], None, pos.cuda()[kept], 4, 2, 0.125, 1)
    got = mix.masked_attn_rows(q.cuda(), kc.cuda(), vc.cuda(), table.cuda(), None, pos.cuda(), 4, 2, 0.125, 1)
    assert torch.equal(got[kept], want) and not got[1].any()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 32, 33, 63, 64, 96, 600])
def test_an_infinite_value_at_the_row_s_own_position(n):
    """What stands in for keys past the last one is that key: its infinite value must not meet their zero weights."""
    q, kc, vc, table, pos, _ = case([n, 20], 2, 1, 64, 64, 16, 10)
    vc[int(table[0, (n - 1) // 16]), 0, (n - 1) % 16, 5] = float("inf")
    args = (table.cuda(), None, pos.cuda(), 2, 1, 0.125)
    got = mix.masked_attn_rows(q.cuda(), kc.cuda(), vc.cuda(), *args)
    assert torch.isposinf(got.view(2, 2, 64)[0, :, 5]).all() and int(torch.isfinite(got).sum()) == got.numel() - 2


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [119, 120, 128, 129, 223, 224])
def test_workgroups_around_the_lines_of_the_launch(rows):
    """Two groups: 238 to 448 workgroups, of eight waves and four, cached rows marked as read once and not."""
    ctx = [1 + (53 * i) % 260 for i in range(rows)]
    q, kc, vc, table, pos, gate = case(ctx, 8, 2, 64, 64, 16, rows)
    check(q, kc, vc, table, pos, 8, 2, 0, gate)


@pytest.mark.gpu
@pytest.mark.parametrize("runs", [2, 8, 9, 31, 64, 65, 130])
@pytest.mark.parametrize("H,G,dk,dv", [(4, 2, 64, 64), (4, 1, 128, 120), (2, 2, 96, 136)])
def test_numbers_of_runs(H, G, dk, dv, runs):
    """Runs around a batch of eight and a wave of 64, most of them without keys; values of one round of threads and of two."""
    q, kc, vc, table, pos, gate = case([1, 70, 700, 2900], H, G, dk, dv, 16, runs)
    check(q, kc, vc, table, pos, H, G, runs=runs)
    check(q, kc, vc, table, pos, H, G, 0, gate, runs=runs, softcap=20.0, sinks=torch.linspace(-2.0, 3.0, H))
