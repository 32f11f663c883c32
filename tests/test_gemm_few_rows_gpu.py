"""Products over 33 .. 64 rows: narrow tiles, at the edges of their columns and of the ring, give the bits of the 128-column ones."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [64, 320, 384, 1024])
@pytest.mark.parametrize("n", [4, 16, 20, 1024, 4096, 4100, 4128, 8192, 8196])
@pytest.mark.parametrize("m", [33, 48, 63, 64])
def test_bits(m, n, k):
    from nanovllm import _hip, ops
    g = torch.Generator().manual_seed(m * n + k)
    x, w, b = ((torch.randn(s, generator=g) * 0.5).bfloat16().cuda() for s in ((m, k), (n, k), (n,)))
    got = ops.linear(x, w, b)
    with _hip.switch("NVH_GEMM_FORCE_TILE", 4):              # 64 x 128
        assert torch.equal(got, ops.linear(x, w, b))
    # fp32 sums of exact products, k roundings at most, and the result's own
    want = x.double() @ w.double().t().contiguous() + b.double()
    slack = (x.double().abs() @ w.double().abs().t().contiguous()) * k * 2.0 ** -24
    assert ((got.double() - want).abs() <= want.abs() * 2.0 ** -8 + slack).all()
