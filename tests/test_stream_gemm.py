"""Streaming products of few rows (dgi/csrc/stream_gemm.hip): edges of the row blocks, of the 128-output tiles and of the parts of K,
and the kernels that read the parts, against plain references; the Llama layers that are made of them against the other layers."""
import pytest
import torch

from dgi import ops
from dgi.models.config import get_config
from dgi.models.llama import LlamaLayerWeights, LlamaModel
from dgi.runtime.batch import AttnMeta

BF16, F64 = torch.bfloat16, torch.float64


def rnd(*shape, seed=0, scale=1.0):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale).to(BF16)


def product(x, w):
    """(x w^T in 64 bits, the sums of its terms' magnitudes)."""
    x, w = x.to(F64), w.to(F64)
    return x @ w.t(), x.abs() @ w.abs().t()


def test_parts_fill_the_chip_and_none_is_empty():
    for N in (8, 128, 2048, 4096, 6144, 8192, 10240, 28672, 128256):
        for K in (64, 128, 320, 2048, 4096, 8192, 14336, 28672):
            p = ops.stream_part_count(N, K)
            per = -(-(K // 64) // p)
            assert p >= 1 and (p - 1) * per < K // 64 and (p == 1 or per >= 4) and p * -(-N // 128) <= max(256, -(-N // 128))
    assert [ops.stream_part_count(n, 4096) for n in (4096, 6144, 28672)] == [8, 5, 1]


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 15, 16, 17, 32, 33, 48, 49, 64, 65, 96, 97, 128])
@pytest.mark.parametrize("N,K", [(136, 64), (128, 576), (1000, 1024), (40064, 128)])
def test_rows_and_parts(M, N, K):
    ops.load_native(True)
    x, w, b = rnd(M, K + 8, seed=1), rnd(N, K, seed=2, scale=K ** -0.5), rnd(N, seed=3)
    xd, wd, bd = x.cuda()[:, :K], w.cuda(), b.cuda()
    y, mag = product(x[:, :K], w)
    assert (M == 1 or xd.stride(0) == K + 8) and ops.stream_ok(xd, wd)
    out = torch.full((M, N + 8), 7.0, dtype=BF16, device="cuda")
    ops._call("stream_gemm", out[:, :N], xd, wd, bd, 0)
    # one rounding to bf16; K products summed in fp32: at most K roundings of 2^-24 of the magnitudes
    err = (out[:, :N].cpu().to(F64) - (y + b.to(F64))).abs()
    assert (err <= 2 ** -8 * (y + b.to(F64)).abs() + K * 2.0 ** -24 * (mag + b.to(F64).abs())).all()
    assert (out[:, N:] == 7.0).all()
    stages = K // 64
    for parts in sorted({1, min(2, stages), stages, ops.stream_part_count(N, K)}):
        if (parts - 1) * -(-stages // parts) >= stages:
            continue
        got = torch.empty(parts, M, N, device="cuda")
        ops._call("stream_gemm", got, xd, wd, None, 2)
        assert ((got.cpu().to(F64).sum(0) - y).abs() <= K * 2.0 ** -24 * mag + 1e-30).all()
        s = ops.sum_parts(got, bd)
        want = got.cpu().to(F64).sum(0) + b.to(F64)
        assert ((s.cpu().to(F64) - want).abs() <= 2 ** -8 * want.abs() + 1e-5).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,I,K", [(1, 8, 64), (17, 72, 128), (64, 1000, 320), (128, 20544, 64), (80, 64, 4160)])
def test_swiglu(M, I, K):
    x, w = rnd(M, K, seed=4), rnd(2 * I, K, seed=5, scale=K ** -0.5)
    got = ops.stream_glu(x.cuda(), w.cuda()).cpu().to(F64)
    y, _ = product(x, w)
    g, u = y[:, :I], y[:, I:]
    want = torch.nn.functional.silu(g) * u
    # gate and up are rounded to bf16 first, as between two kernels: 2^-9 each, the activation's slope is at most 1.1
    bound = 2 ** -8 * (1.1 * g.abs() * u.abs() + want.abs() + want.abs()) + 1e-5 * (1 + u.abs())
    assert ((got - want).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("T,H,parts", [(1, 64, 1), (5, 2048, 3), (33, 4096, 8), (128, 8192, 4), (2, 16384, 2)])
def test_norm_of_parts(T, H, parts):
    p = torch.randn(parts, T, H, generator=torch.Generator().manual_seed(6))
    res, g = rnd(T, H, seed=7), (1 + 0.1 * torch.randn(H, generator=torch.Generator().manual_seed(8))).to(BF16)
    rd = res.cuda()
    out = ops.add_rmsnorm_parts(p.cuda(), rd, g.cuda(), 1e-5)
    # the same parts in fp32, part 0 first, and the plain kernel on their sum
    s = p[0].clone()
    for i in range(1, parts):
        s += p[i]
    x, r2 = s.to(BF16).cuda(), res.cuda()
    ops.fused_add_rmsnorm(x, r2, g.cuda(), 1e-5)
    assert torch.equal(rd, r2) and torch.equal(out, x)


@pytest.mark.gpu
@pytest.mark.parametrize("nh,nkv,hd,rd,mode,bias", [(4, 2, 128, 128, 0, False), (3, 1, 64, 64, 0, True), (8, 2, 128, 64, 1, True),
                                                    (2, 2, 64, 32, 0, False), (32, 8, 128, 128, 0, True)])
def test_rotary_of_parts(nh, nkv, hd, rd, mode, bias):
    T, parts, bs, W = 37, 3, 16, (nh + 2 * nkv) * hd
    p = torch.randn(parts, T, W, generator=torch.Generator().manual_seed(9))
    b = rnd(W, seed=10) if bias else None
    pos = torch.randint(0, 500, (T,), generator=torch.Generator().manual_seed(11)).to(torch.int32)
    slots = torch.randperm(20 * bs, generator=torch.Generator().manual_seed(12))[:T].to(torch.int32)
    slots[5] = slots[30] = -1
    cs = ops.rope_cos_sin(rd, 500, 10000.0)
    s = p[0] + p[1] + p[2]
    qkv = (s + b.float() if bias else s).to(BF16).cuda()
    kc, vc = (torch.full((20, nkv, bs, hd), 3.0, dtype=BF16, device="cuda") for _ in range(2))
    k2, v2 = kc.clone(), vc.clone()
    ops.rope_cache(qkv, pos.cuda(), cs.cuda(), nh, nkv, hd, slots.cuda(), kc, vc, mode)
    q = ops.rope_cache_parts(p.cuda(), b.cuda() if bias else None, pos.cuda(), cs.cuda(), nh, nkv, hd, slots.cuda(), k2, v2, mode)
    assert torch.equal(vc, v2)
    for a, b in ((kc, k2), (qkv[:, : nh * hd], q)):
        # the rotation's two products are contracted in one order or the other: the last bit of bf16 (2^-8 of the value) may differ, and where
        # they cancel 2^-23 of the products, which are below 32
        assert ((a.float() - b.float()).abs() <= 2 ** -7 * a.float().abs() + 2.0 ** -18).all()


@pytest.mark.gpu
def test_linear_takes_them_where_they_are_the_faster(monkeypatch):
    calls = []
    real = ops._call
    monkeypatch.setattr(ops, "_call", lambda name, *a: (calls.append(name), real(name, *a))[1])
    for M, N, K, bias, want in [(17, 32768, 512, False, ["stream_gemm"]), (96, 20480, 64, True, ["stream_gemm"]), (97, 20480, 64, False, []),
                                (128, 4096, 12288, True, ["stream_gemm", "sum_parts"]), (64, 4096, 4096, False, []), (129, 4096, 12288, False, []),
                                (20, 20484, 64, False, []), (20, 32768, 72, False, [])]:
        x, w, b = rnd(M, K, seed=13), rnd(N, K, seed=14, scale=K ** -0.5), rnd(N, seed=15) if bias else None
        calls.clear()
        got = ops.linear(x.cuda(), w.cuda(), b.cuda() if bias else None).cpu().to(F64)
        assert calls == want, (M, N, K)
        y, mag = product(x, w)
        y = y + b.to(F64) if bias else y
        assert ((got - y).abs() <= 2 ** -8 * y.abs() + K * 2.0 ** -24 * (mag + 1)).all()
    out = torch.empty(20, 20480, dtype=BF16, device="cuda")
    x, w = rnd(20, 64).cuda(), rnd(20480, 64).cuda()
    assert ops.linear(x, w, out=out) is out and torch.equal(out, ops.linear(x, w))


def layers(device, T_dec, prompts, monkeypatch, force=False, seed=3, **cut):
    """(rows, residual, cache) of both forms of the layers on one step."""
    cfg = get_config("llama3-8b@L2")
    for k, v in cut.items():
        setattr(cfg, k, v)
    m = LlamaModel(cfg, device, BF16, init="random", seed=seed)
    g = torch.Generator().manual_seed(seed)
    lens = [int(n) for n in torch.randint(1, 60, (T_dec,), generator=g)]
    seqs = T_dec + len(prompts)
    kv = torch.randn(2, 2, seqs * 8 + 1, cfg.num_kv_heads, 16, cfg.head_dim, generator=g).to(BF16).to(device)
    bt = (torch.arange(seqs * 8) + 1).view(seqs, 8).to(torch.int32)
    pos = [n - 1 for n in lens] + [t for p in prompts for t in range(p)]
    row = list(range(T_dec)) + [T_dec + j for j, p in enumerate(prompts) for _ in range(p)]
    slots = [int(bt[r, t // 16]) * 16 + t % 16 for r, t in zip(row, pos)]
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=device)  # noqa: E731
    meta = AttnMeta(positions=i32(pos), slot_mapping=i32(slots), num_decode=T_dec, dec_block_tables=bt[:T_dec].to(device),
                    dec_context_lens=i32(lens), dec_max_splits=1, dec_part_size=1 << 20, num_prefill_tokens=sum(prompts))
    if prompts:
        cu = [sum(prompts[:i]) for i in range(len(prompts) + 1)]
        meta.pre_block_tables, meta.pre_cu_seqlens, meta.pre_context_lens = bt[T_dec:].to(device), i32(cu), i32(prompts)
    h = (torch.randn(len(pos), cfg.hidden_size, generator=g)).to(BF16).to(device)
    trim = torch.tensor([0, len(pos) - 1], device=device) if prompts else None
    out = []
    for stream in (False, True):
        monkeypatch.setattr(LlamaModel, "_stream_ok", (lambda self, h: stream) if not stream or force else real_stream_ok)
        m.kv_cache = kv.clone()
        a, r = m.forward_layers(h.clone(), meta, trim_last=trim)
        out.append((a.float().cpu(), r.float().cpu(), m.kv_cache.float().cpu()))
    return out


real_stream_ok = LlamaModel._stream_ok


def close(a, b):
    # bf16 layers summed in other orders: roundings of 2^-9 that go through two layers
    for x, y in zip(a, b):
        assert ((x - y).norm() / y.norm()).item() < 0.01


def test_layers_compose_on_the_cpu(monkeypatch):
    plain, stream = layers("cpu", 5, [7, 1], monkeypatch, force=True, hidden_size=256, intermediate_size=320, num_heads=4, num_kv_heads=2,
                           head_dim=64)
    close(stream, plain)


@pytest.mark.gpu
@pytest.mark.parametrize("T,prompts", [(17, []), (64, []), (100, []), (9, [20, 1, 33]), (0, [70])])
def test_layers_on_the_gpu(monkeypatch, T, prompts):
    names, real = [], ops._call
    monkeypatch.setattr(ops, "_call", lambda name, *a: (names.append(name), real(name, *a))[1])
    plain, stream = layers("cuda", T, prompts, monkeypatch, hidden_size=2048, intermediate_size=4160, num_heads=16, num_kv_heads=4)
    close(stream, plain)
    # both forms ran, one after the other
    first = names.index("rope_cache_parts")
    assert "rope_cache" in names[:first] and "add_rmsnorm_parts" not in names[:first]
    assert names[first:].count("rope_cache_parts") == 2 and "rope_cache" not in names[first:] and names[first:].count("add_rmsnorm_parts") == 3


@pytest.mark.gpu
@pytest.mark.parametrize("T,K,stream", [(2, 4096, False), (3, 4096, True), (16, 4096, True), (8, 3072, False), (9, 3072, True), (16, 2048, False)])
def test_few_rows(monkeypatch, T, K, stream):
    """Rows and widths around the line between the fused layers and these."""
    names, real = [], ops._call
    monkeypatch.setattr(ops, "_call", lambda name, *a: (names.append(name), real(name, *a))[1])
    plain, got = layers("cuda", T, [], monkeypatch, hidden_size=K, intermediate_size=5632, num_heads=16, num_kv_heads=4)
    close(got, plain)
    assert names.count("fused_skinny") and names.count("rope_cache_parts") == (2 if stream else 0)


@pytest.mark.gpu
def test_a_step_takes_them_and_replays(monkeypatch):
    """17 rows of a 2048-wide model: the layers run on the streaming products, eagerly and as a graph that is replayed between other work."""
    from dgi.engine import EngineConfig, LLMEngine
    from dgi.sched.request import SamplingParams
    cfg = get_config("llama3-8b@L2")
    cfg.hidden_size, cfg.intermediate_size, cfg.num_heads, cfg.num_kv_heads, cfg.vocab_size = 2048, 4096, 16, 4, 4096
    m = LlamaModel(cfg, "cuda", BF16, init="random", seed=5)
    names = []
    real = ops._call
    monkeypatch.setattr(ops, "_call", lambda name, *a: (names.append(name), real(name, *a))[1])
    outs = []
    for graphs in (False, True):
        eng = LLMEngine(EngineConfig(model=cfg.name, device="cuda", num_blocks=256, max_num_seqs=24, max_model_len=256,
                                     max_num_batched_tokens=512, use_graphs=graphs, graph_buckets=(24,)), model_cfg=cfg, model=m)
        reqs = eng.generate([[(7 * i + j) % 4000 for j in range(5 + i)] for i in range(18)], SamplingParams(max_tokens=8, temperature=0.0,
                                                                                                         ignore_eos=True))
        outs.append([r.output for r in reqs])
    assert "add_rmsnorm_parts" in names and "rope_cache_parts" in names
    assert outs[0] == outs[1]


def test_weights_are_looked_at_once(monkeypatch):
    """The look at every weight of every layer is not repeated at each step, but is after a weight is replaced."""
    looks = []

    class Weight:
        dtype = BF16

        def __init__(self, *shape, at=0):
            self.shape, self.at = shape, at

        def is_contiguous(self):
            looks.append(self)
            return True

        def data_ptr(self):
            return self.at

    def layer():
        return LlamaLayerWeights(Weight(2048), Weight(3072, 2048), Weight(2048, 2048), Weight(2048), Weight(8192, 2048), Weight(2048, 4096))

    monkeypatch.setattr(ops, "stream_ok", lambda x, w: True)
    m = LlamaModel.__new__(LlamaModel)
    m.reduce, m.capture_layers, m.layers = None, (), [layer() for _ in range(3)]
    h = torch.zeros(20, 2048, dtype=BF16)
    assert m._stream_ok(h) and len(looks) == 18
    assert m._stream_ok(h) and not m._stream_ok(h.float()) and len(looks) == 18
    m.layers[1].down = Weight(2048, 4096, at=8)
    assert not m._stream_ok(h)
    m.layers[1].down = Weight(2048, 4096)
    assert m._stream_ok(h)
    m.layers[2].qkv_bias = Weight(3072)
    m.layers[2].qkv_bias.dtype = torch.float32
    assert not m._stream_ok(h)
    m.layers[2] = layer()
    assert m._stream_ok(h)


def test_sizes_that_stream():
    """Rounds of the chip that are mostly idle, wide rows many times over and parts of two large pieces stay with the vendor's product."""
    rows = lambda N, K: [M for M in (17, 64, 65, 96, 97, 128, 129) if ops._stream_sizes(M, N, K)]  # noqa: E731
    assert rows(37888, 3584) == rows(34816, 4096) == rows(45056, 5120) == []
    assert rows(65536, 5120) == rows(20480, 3584) == rows(128256, 8192) == rows(17408, 5120) == rows(16384, 3584) == [17, 64]
    assert rows(32000, 8192) == rows(128256, 4096) == rows(20480, 512) == [17, 64, 65, 96]
    assert rows(4096, 14336) == rows(16384, 4096) == rows(520, 98304) == [17, 64, 65, 96, 97, 128]
    assert rows(4096, 4096) == []
    glu = lambda I, K: [M for M in (1, 32, 33, 64, 65, 96, 97, 128) if ops.glu_streams(M, I, K)]  # noqa: E731
    assert glu(18944, 3584) == glu(17408, 5120) == []
    assert glu(14336, 4096) == glu(13824, 5120) == glu(8960, 1536) == [1, 32, 33, 64, 65, 96, 97, 128]
    assert glu(8192, 4096) == glu(28672, 8192) == glu(24576, 6144) == [1, 32, 33, 64]
    assert glu(4096, 2048) == [1, 32]
    over = lambda I, K: [M for M in (1, 2, 3, 8, 9, 16) if ops.stream_over_fused(M, I, K)]  # noqa: E731
    assert over(14336, 4096) == over(5632, 4096) == [3, 8, 9, 16] and over(8192, 3072) == [9, 16]
    assert over(17408, 4096) == over(8192, 2048) == []
