"""``ops.row_sumsq``: sums of squares of bf16 rows in fp32, the other columns zero, against 64 bits; rows with a stride of their own and sizes
that the kernel leaves to tensor operations."""
import pytest
import torch

from dgi import ops


@pytest.mark.gpu
@pytest.mark.parametrize("T,H,pad,cols", [(1, 8, 0, 1), (3, 2048, 8, 8), (129, 4096, 0, 16), (5, 8200, 24, 33), (7, 100, 0, 8), (4, 64, 4, 300)])
def test_row_sumsq(T, H, pad, cols):
    x = torch.randn(T, H + pad, generator=torch.Generator().manual_seed(H)).bfloat16().cuda()[:, :H]
    out = torch.full((T, cols + 3), 7.0, device="cuda")
    ops.row_sumsq(x, out[:, :cols])
    ref = x.cpu().double().pow(2).sum(1)
    # a tree over the row: well under 64 roundings of 2^-24
    assert ((out[:, 0].cpu().double() - ref).abs() <= 64 * 2.0 ** -24 * ref).all()
    assert (out[:, 1:cols] == 0).all() and (out[:, cols:] == 7.0).all()


@pytest.mark.gpu
def test_history_and_other_places():
    """Rows that want a gradient keep it; statistics may lie elsewhere."""
    x = torch.randn(5, 64, generator=torch.Generator().manual_seed(2)).bfloat16().cuda()
    leaf = x.clone().requires_grad_()
    ops.row_sumsq(leaf, torch.empty(5, 3, device="cuda"))[:, 0].sum().backward()
    assert torch.equal(leaf.grad, (2 * x.float()).bfloat16())
    out = ops.row_sumsq(x, torch.empty(5, 3))
    assert out.device.type == "cpu" and torch.allclose(out[:, 0], x.float().pow(2).sum(-1).cpu(), rtol=1e-5) and not out[:, 1:].any()
