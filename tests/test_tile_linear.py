"""Products past 128 rows that run on the ping-pong kernel: the logits of large vocabularies (``ops.linear``) and products of long rows, around
the rows and sizes at which the rules change, against the product in fp32."""
import pytest
import torch

from dgi import ops


@pytest.mark.gpu
@pytest.mark.parametrize("M", [129, 255, 256, 257, 353, 512, 513, 1024, 1025])
@pytest.mark.parametrize("N,K", [(384 * 256, 128), (384 * 256 - 256, 128), (501 * 256, 192), (384 * 256 + 8, 64), (448 * 256, 64), (8192, 16384)])
def test_linear_past_the_streamed_rows(M, N, K):
    g = torch.Generator(device="cuda")
    g.manual_seed(M + N)
    x = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    w = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).bfloat16()
    y = ops.linear(x, w).float()
    ref = x.float() @ w.float().t()
    # one rounding to bf16; sums of K products in fp32, in another order
    assert (y - ref).abs().max() <= 2.0 ** -8 * ref.abs().max() + 1e-4
    assert ((y - ref).norm() / ref.norm()) <= 2.0 ** -8


def test_rows_of_the_rules():
    assert [ops.tile_gemm(m, 128256) for m in (128, 129, 256, 257, 512, 1024, 1025)] == [False, True, True, True, True, True, False]
    assert [ops.tile_gemm(200, n) for n in (32000, 384 * 256 - 256, 384 * 256, 448 * 256, 512 * 256, 594 * 256)] == [False, False, False, True, True, False]
    assert [ops.split_gemm(m, 8192, 28672) for m in (128, 129, 512, 513)] == [False, True, True, False]
    assert [ops.split_gemm(200, n, k) for n, k in [(4096, 14336), (8192, 16384), (8192, 16383), (4096, 16384)]] == [False, True, False, False]


@pytest.mark.gpu
@pytest.mark.parametrize("M", [129, 300, 512])
def test_split_product(M):
    g = torch.Generator(device="cuda")
    g.manual_seed(M)
    x = torch.randn(M, 16448, device="cuda", generator=g).bfloat16()
    w = (torch.randn(8192, 16448, device="cuda", generator=g) * 16448 ** -0.5).bfloat16()
    ref = x.float() @ w.float().t()
    assert ((ops.mfma_gemm(x, w).float() - ref).norm() / ref.norm()) <= 2.0 ** -8


@pytest.mark.gpu
@pytest.mark.parametrize("M", [64, 200])
def test_linear_keeps_its_derivatives(M):
    """Rows that want a gradient stay with the differentiable product, whatever its size."""
    g = torch.Generator(device="cuda")
    g.manual_seed(M)
    x = torch.randn(M, 64, device="cuda", generator=g).bfloat16().requires_grad_()
    w = torch.randn(501 * 256, 64, device="cuda", generator=g).bfloat16()
    up = torch.randn(M, 501 * 256, device="cuda", generator=g).bfloat16()
    ops.linear(x, w).backward(up)
    ref = up.float() @ w.float()
    assert ((x.grad.float() - ref).norm() / ref.norm()) <= 2.0 ** -7


def test_what_is_plain():
    """Operands of a transform, of a trace or with history are not for kernels that know values alone."""
    from torch._subclasses import FakeTensorMode
    from torch.autograd import forward_ad
    seen = []
    look = lambda t: (seen.append(ops.plain_values(t)), t * 2)[1]  # noqa: E731
    x, p = torch.randn(3, 4), torch.nn.Parameter(torch.randn(3, 4))
    torch.func.vmap(look)(x)
    torch.func.jvp(look, (x,), (x,))
    torch.func.grad(lambda t: look(t).sum())(x)
    with FakeTensorMode() as mode:
        look(torch.empty(3, 4))
    look(mode.from_tensor(x))
    with forward_ad.dual_level():
        look(forward_ad.make_dual(x, x))
        assert ops.plain_values(x)
    look(p)
    look(x * p)
    assert seen == [False] * 8
    with torch.no_grad():
        assert ops.plain_values(x, None, p)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(8, 4096, 1024), (64, 20480, 64), (128, 4096, 12288), (200, 501 * 256, 64)])
@pytest.mark.parametrize("of", ["x", "w", "bias"])
def test_linear_keeps_every_derivative(M, N, K, of):
    """Backward and forward derivatives of each operand alone, at the sizes of each kernel, and operands without data."""
    from torch._subclasses import FakeTensorMode
    from torch.autograd import forward_ad
    g = torch.Generator(device="cuda")
    g.manual_seed(M)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).bfloat16()  # noqa: E731
    a = {"x": rnd(M, K), "w": rnd(N, K) * K ** -0.5, "bias": rnd(N) if M <= 128 else None}
    if a[of] is None:
        pytest.skip("no bias at this size")
    up, tan = rnd(M, N), rnd(*a[of].shape)
    f = {k: None if v is None else v.float() for k, v in a.items()}
    want = {"x": up.float() @ f["w"], "w": up.float().t() @ f["x"], "bias": up.float().sum(0)}[of]
    leaf = a[of].clone().requires_grad_()
    ops.linear(**{**a, of: leaf}).backward(up)
    # sums in fp32, rounded to bf16 on both ways
    assert ((leaf.grad.float() - want).norm() / want.norm()) <= 2.0 ** -7
    want = {"x": lambda t: t @ f["w"].t(), "w": lambda t: f["x"] @ t.t(), "bias": lambda t: t.expand(M, N)}[of](tan.float())
    with forward_ad.dual_level():
        got = forward_ad.unpack_dual(ops.linear(**{**a, of: forward_ad.make_dual(a[of], tan)})).tangent
        assert ((got.float() - want).norm() / want.norm()) <= 2.0 ** -7
    with FakeTensorMode(allow_non_fake_inputs=True) as mode:
        assert ops.linear(**{**a, of: mode.from_tensor(a[of])}).shape == (M, N)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(64, 20480, 64), (20, 4096, 12288), (20, 20480, 20480), (200, 501 * 256, 64)])
def test_linear_takes_what_the_plain_product_takes(M, N, K):
    """Biases and results of other shapes, types and places, results over the operands, weights off their 16 bytes and of one row."""
    g = torch.Generator(device="cuda")
    g.manual_seed(M)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).bfloat16()  # noqa: E731
    x, flat = rnd(M, K), rnd(N * K + 1) * K ** -0.5
    w = flat[:-1].view(N, K)
    y = x.float() @ w.float().t()

    def check(got, want):
        # one rounding to bf16; sums of K products in fp32, in another order
        assert got.shape == want.shape and ((got.float() - want).norm() / want.norm()) <= 2.0 ** -8

    for bias in (rnd(1), rnd(M, N), rnd(1, N)):
        check(ops.linear(x, w, bias), y + bias.float())
    for out in (torch.empty(M, N, device="cuda"), torch.empty(M, N, dtype=torch.bfloat16), torch.empty(2, M, N, device="cuda"),
                torch.empty(N, M, device="cuda").bfloat16().t(), rnd(M, N + 4)[:, :N]):
        assert ops.linear(x, w, out=out) is out
        check(out.cuda(), y.expand_as(out))
    if N == K:
        both = x.clone()
        assert ops.linear(both, w, out=both) is both
        check(both, y)
        del both
        one = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
        check(ops.linear(x[:1].expand(M, K), w, out=one), y[:1].expand(M, N))
    off = flat[1:].view(N, K)
    check(ops.linear(x, off), x.float() @ off.float().t())
    check(ops.linear(x, w[0]), x.float() @ w[0].float())
    with pytest.raises(RuntimeError):
        ops.linear(x, w.new_zeros(N, K + 64))
    with pytest.raises(RuntimeError):
        ops.linear(x, w, out=torch.empty(M + 1, N, device="cuda").bfloat16())


def test_the_last_mlp_has_a_workspace_of_its_own(monkeypatch):
    """Models stepped from several threads or streams share a device: their split products must not share partial sums."""
    from types import SimpleNamespace
    from dgi.models.llama import LlamaModel
    seen = []
    monkeypatch.setattr(ops, "split_gemm", lambda *a: True)
    monkeypatch.setattr(ops, "mfma_gemm_ok", lambda *a: True)
    monkeypatch.setattr(ops, "mfma_gemm", lambda x, w, **k: (seen.append(k), x @ w.t())[1])
    layer = SimpleNamespace(gate_up=torch.randn(16, 8), down=torch.randn(8, 8))
    LlamaModel._last_mlp(torch.randn(3, 8), layer)
    assert seen == [{"own_space": True}]


@pytest.mark.gpu
def test_split_products_of_two_streams():
    """Two threads, each with a stream and operands of its own: every product has the bits that it has alone; and captured."""
    import threading
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    sets = []
    for i, M in enumerate((129, 300)):
        x = torch.randn(M, 16384, device="cuda", generator=g).bfloat16()
        w = (torch.randn(8192, 16384, device="cuda", generator=g) * 2 ** -7).bfloat16()
        v = torch.randn(448 * 256, 16384, device="cuda", generator=g).bfloat16() if i else None
        sets.append((x, w, v, ops.mfma_gemm(x, w, own_space=True)))
        assert torch.equal(ops.mfma_gemm(x, w), sets[-1][3])
        ref = x.float() @ w.float().t()
        assert ((sets[-1][3].float() - ref).norm() / ref.norm()) <= 2.0 ** -8
    torch.cuda.synchronize()
    wrong = [0, 0]

    def work(i):
        x, w, v, want = sets[i]
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(30):
                got = ops.mfma_gemm(x, w, own_space=True)
                if v is not None and _ % 8 == 0:
                    ops.linear(x, v)
                wrong[i] += int(not torch.equal(got, want))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert wrong == [0, 0]
    x, w, _, want = sets[0]
    with torch.inference_mode():                     # as engines capture: the generator's state is one of torch's inference tensors then
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            got = ops.mfma_gemm(x, w, own_space=True)
        for _ in range(3):
            got.zero_()
            graph.replay()
            assert torch.equal(got, want) and torch.equal(ops.mfma_gemm(x, w), want)


def test_rows_that_are_split():
    """Four pieces of 24 to 64 tiles; short sums of few rows stay with the vendor's product."""
    split = lambda N, K: [M for M in (129, 160, 161, 256, 257, 512) if ops.split_gemm(M, N, K)]  # noqa: E731
    assert split(8192, 28672) == split(6144, 24576) == [129, 160, 161, 256, 257, 512]
    assert split(8192, 16384) == [161, 256, 257, 512] and split(16384, 16384) == [161, 256] and split(16384, 53248) == [129, 160, 161, 256]
    assert split(4096, 32768) == [257, 512] and split(5120, 27648) == [257, 512]


@pytest.mark.gpu
def test_linear_leaves_outputs_in_whole_vendor_tiles(monkeypatch):
    """The ping-pong kernel only where it is the faster: outputs that are no multiple of 512, rows that fill a third of their last tile."""
    calls = []
    real = ops._call
    monkeypatch.setattr(ops, "_call", lambda name, *a: (calls.append(name), real(name, *a))[1])
    for M, N, want in [(129, 501 * 256, True), (353, 501 * 256, True), (352, 501 * 256, False), (257, 501 * 256, False), (512, 1001 * 256, True),
                       (200, 512 * 256, False), (512, 500 * 256, False), (129, 592 * 256, False)]:
        x, w = torch.randn(M, 64, device="cuda").bfloat16(), torch.randn(N, 64, device="cuda").bfloat16()
        calls.clear()
        ops.linear(x, w)
        assert calls == (["mfma_gemm"] if want else []), (M, N)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(8, 4096, 1024), (64, 20480, 64), (128, 4096, 12288), (200, 501 * 256, 64)])
def test_operands_of_another_device(monkeypatch, M, N, K):
    """Kernels are launched on the current device: operands of another one stay with torch's product, which goes to theirs."""
    calls = []
    monkeypatch.setattr(ops, "_call", lambda name, *a: calls.append(name))
    x, w = torch.randn(M, K, device="cuda").bfloat16(), torch.randn(N, K, device="cuda").bfloat16()
    ops.linear(x, w)
    assert calls
    calls.clear()
    monkeypatch.setattr(torch.cuda, "current_device", lambda: x.device.index + 1)
    y = ops.linear(x, w)
    ops.row_sumsq(x, torch.empty(M, 2, device="cuda"))
    assert not calls
    ref = x.float() @ w.float().t()
    assert ((y.float() - ref).norm() / ref.norm()) <= 2.0 ** -8
