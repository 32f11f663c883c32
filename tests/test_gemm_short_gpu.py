"""bf16 products with fp32 results through LDS rings: the bits of the form that takes any row, at the edges of tiles and of the ring."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [64, 128, 448, 1024])
@pytest.mark.parametrize("m,n", [(1, 4), (15, 60), (16, 64), (17, 68), (33, 1000), (64, 128), (65, 132), (130, 1028)])
def test_bits(m, n, k):
    from nanovllm import ops
    g = torch.Generator().manual_seed(m * n + k)
    x, w = torch.randn(m, k, generator=g).bfloat16().cuda(), (torch.randn(n, k, generator=g) * 0.1).bfloat16().cuda()
    wide = torch.empty(m, k + 1, dtype=torch.bfloat16, device="cuda")
    wide[:, :-1] = x
    got = ops.linear_any(x, w, out_f32=True)
    assert got.dtype is torch.float32 and torch.equal(got, ops.linear_any(wide[:, :-1], w, out_f32=True))
    want = x.double() @ w.double().t().contiguous()
    slack = (x.double().abs() @ w.double().abs().t().contiguous()) * k * 2.0 ** -24      # fp32 sums of exact products
    assert ((got.double() - want).abs() <= slack).all()
