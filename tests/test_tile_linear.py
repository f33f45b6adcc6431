"""``ops.linear`` past 128 rows where it runs on the ping-pong kernel: the logits of large vocabularies and products of long rows, around the
rows and sizes at which the rule changes, against the product in fp32."""
import pytest
import torch

from dgi import ops


@pytest.mark.gpu
@pytest.mark.parametrize("M", [129, 255, 256, 257, 353, 512, 513, 1024, 1025])
@pytest.mark.parametrize("N,K", [(384 * 256, 128), (384 * 256 - 256, 128), (501 * 256, 192), (384 * 256 + 8, 64), (8192, 16384), (8192, 16448)])
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


def test_rows_of_the_rule():
    assert [ops.tile_gemm_rows(n, k) for n, k in [(128256, 4096), (128256, 8192), (384 * 256, 64), (384 * 256 - 8, 64), (32000, 4096),
                                                  (8192, 28672), (4096, 14336), (8192, 16384), (8192, 16383), (57344, 8192)]] == \
        [1024, 1024, 1024, 0, 0, 512, 0, 512, 0, 0]
