"""Decode attention's tiles of 32 cached tokens: contexts at the edges of tiles, pages and splits, with no numbers in the
cache past each context's end; and the plan of the splits."""
import math

import pytest
import torch

from dgi import ops

CTX = [1, 15, 16, 17, 31, 32, 33, 64, 127, 129, 255, 257, 289, 640, 1025, 2049]


@pytest.mark.gpu
@pytest.mark.parametrize("bs", [16, 32])
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("nh,nkv", [(8, 2), (64, 8), (16, 16)])
@pytest.mark.parametrize("splits,part", [(1, 1 << 20), (3, -128), (20, -64), (8, -2048), (17, 128)])
def test_contexts_at_edges(bs, hd, nh, nkv, splits, part):
    g = torch.Generator().manual_seed(bs + hd + nh)
    need = [-(-c // bs) for c in CTX]
    pages = sum(need) + 1
    perm = torch.randperm(pages - 1, generator=g) + 1
    bt = torch.zeros(len(CTX), max(need), dtype=torch.int32)
    cache = torch.randn(2, pages, nkv, bs, hd, generator=g).bfloat16()
    cache[:, 0] = math.nan                                     # nobody's page
    at = 0
    for i, (c, n) in enumerate(zip(CTX, need)):
        bt[i, :n] = perm[at: at + n]
        at += n
        if c % bs:
            cache[:, bt[i, n - 1].long(), :, c % bs:] = math.nan
    q = torch.randn(len(CTX), nh * hd, generator=g).bfloat16()
    cache, bt, q = cache.cuda(), bt.cuda(), q.cuda()
    ctx = torch.tensor(CTX, dtype=torch.int32, device="cuda")
    scale = hd ** -0.5
    ref = ops.paged_decode_ref(q, cache[0], cache[1], bt, ctx, nh, nkv, scale)
    out = ops.paged_decode(q, cache[0], cache[1], bt, ctx, nh, nkv, scale, splits, part)
    # weights and results are rounded to bf16 (2^-9 each) against values of unit size
    torch.testing.assert_close(out.float(), ref.float(), atol=2e-2, rtol=2e-2)
    if splits > 1:
        ws = (torch.empty(len(CTX) * nh * splits * hd, device="cuda"), torch.empty(len(CTX) * nh * splits, device="cuda"))
        again = ops.paged_decode(q, cache[0], cache[1], bt, ctx, nh, nkv, scale, splits, part, workspace=ws)
        torch.testing.assert_close(again.float(), ref.float(), atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("batch,ctx,nkv", [(1, 1, 8), (1, 8000, 8), (2, 600, 8), (8, 4000, 8), (12, 900, 8), (17, 9000, 8), (64, 1024, 8),
                                           (350, 40000, 8), (300, 100, 1), (1, 1 << 17, 1), (3, 5000, 7)])
def test_plan_of_splits(batch, ctx, nkv):
    """At least one split, none that a longest context would leave empty, a workspace of 128-token parts holds them, and no
    more than one workgroup per unit but for long contexts of many rows."""
    splits, part = ops.decode_split_plan(batch, ctx, nkv)
    assert part < 0 and part % 32 == 0
    assert 1 <= splits <= max(1, -(-ctx // 128))
    if splits > 1:
        assert (splits - 1) * -part < ctx
    if batch * nkv * splits > 256:
        assert splits <= 8 and (splits == 1 or ctx > 2048)


def live_splits(ctx, splits, part):
    """Splits of one context as the kernel's device-side plan makes them."""
    n = max(1, min(splits, -(-ctx // -part)))
    part = -(-(-(-ctx // n)) // 32) * 32
    return -(-ctx // part)


@pytest.mark.parametrize("nkv", [4, 8])
@pytest.mark.parametrize("limit", [4096, 8192, 32768])
def test_plans_keep_the_units_busy(nkv, limit):
    """Steps of up to a workgroup per unit, which run one at a time on each: long contexts take rounds of the chip that are two
    thirds full at least, whatever the longest context that may come."""
    for seqs in range(96, 257, nkv):
        splits, part = ops.decode_split_plan(seqs // nkv, limit, nkv)
        for ctx in (3400, 4096):
            n = seqs * live_splits(ctx, splits, part)
            assert n / (-(-n // 256) * 256) >= 0.66, (seqs, ctx)


def test_captured_plans_serve_short_contexts(monkeypatch):
    """A bucket's plan is that of the longest context that may come.  Where it would split contexts that are best left whole, or leave a second
    kernel to combine nothing, a graph of whole rows goes with it."""
    from types import SimpleNamespace
    from dgi.runtime.model_runner import GraphRunner
    for name in ("DGI_DECODE_DYNAMIC", "DGI_DECODE_MIN_PART"):
        monkeypatch.delenv(name, raising=False)
    for limit in (1024, 2048, 8192, 131072):
        r = GraphRunner.__new__(GraphRunner)
        cfg = SimpleNamespace(num_kv_heads=8, head_dim=128)
        r.r = SimpleNamespace(model=SimpleNamespace(cfg=cfg, decode_splits=True), num_cus=256, max_model_len=limit, ws_splits=limit // 128)
        r.short_ctx, r.short_max_b = 384, 8
        assert [r.short_limit(b) for b in (1, 8, 9, 16)] == [384, 384, 0, 0]
        for b in (17, 24, 32, 40, 48, 64, 512):
            splits, part = r.split_plan(b)
            whole = ops.decode_whole(b, 8)
            assert whole in (1024, 2048, 8192) and (splits > 1) == (limit > whole)
            assert r.short_limit(b) == (whole if splits > 1 else 0)
            assert ops.decode_split_plan(b, whole, 8)[0] == 1 and ops.decode_split_plan(b, whole + 1, 8)[0] > 1
        r.r.model.decode_splits = False                  # models whose attention has no such plan
        assert [r.short_limit(b) for b in (8, 24, 64)] == [384, 0, 0]
        r.short_ctx = 0
        assert not any(r.short_limit(b) for b in (1, 24, 64))


@pytest.mark.gpu
def test_both_graphs_of_a_large_bucket(monkeypatch):
    """Contexts that grow past the line between the two graphs of a bucket: the same tokens as with one graph."""
    from dgi.engine import EngineConfig, LLMEngine
    from dgi.models.config import get_config
    from dgi.models.llama import LlamaModel
    from dgi.runtime.model_runner import GraphRunner
    from dgi.sched.request import SamplingParams
    monkeypatch.setattr(ops, "decode_whole", lambda b, nkv, num_cus=256: 64)
    cfg = get_config("llama3-8b@L2")
    cfg.hidden_size, cfg.intermediate_size, cfg.num_heads, cfg.num_kv_heads, cfg.vocab_size = 1024, 1024, 8, 8, 1024
    m = LlamaModel(cfg, "cuda", torch.bfloat16, init="random", seed=5)
    keys, outs = [], []
    launch = GraphRunner.launch
    monkeypatch.setattr(GraphRunner, "launch", lambda self, *a, **k: (launch(self, *a, **k), keys.append(self.last_key))[0])
    for short in ("384", "0"):
        monkeypatch.setenv("DGI_DECODE_SHORT_CTX", short)
        eng = LLMEngine(EngineConfig(model=cfg.name, device="cuda", num_blocks=256, max_num_seqs=40, max_model_len=4096,
                                     max_num_batched_tokens=512, graph_buckets=(40,)), model_cfg=cfg, model=m)
        reqs = eng.generate([[(7 * i + j) % 1000 for j in range(52 + i)] for i in range(3)],
                            SamplingParams(max_tokens=20, temperature=0.0, ignore_eos=True))
        outs.append([r.output for r in reqs])
        assert {k for k in keys} == ({(40, True), (40, False)} if short != "0" else {(40, False)})
        keys.clear()
    assert outs[0] == outs[1]
