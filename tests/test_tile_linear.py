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
