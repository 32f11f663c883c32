"""Products whose 128 x 64 tiles would take a second round over the CUs: 128 x 128 ones give the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [64, 320, 1024, 2112])
@pytest.mark.parametrize("m,n", [(257, 6148), (300, 5632), (520, 4100), (1000, 2112), (1025, 1860)])
def test_bits(m, n, k):
    from nanovllm import _hip, ops
    g = torch.Generator().manual_seed(m * n + k)
    x, w, b = ((torch.randn(s, generator=g) * 0.5).bfloat16().cuda() for s in ((m, k), (n, k), (n,)))
    for f in (lambda: ops.linear(x, w, b), lambda: ops.linear_swiglu(x, w)) if n % 32 == 0 else (lambda: ops.linear(x, w, b),):
        got = f()
        with _hip.switch("NVH_GEMM_FORCE_TILE", 5):          # 64 x 64
            assert torch.equal(got, f())
    want = x.double() @ w.double().t().contiguous() + b.double()
    slack = (x.double().abs() @ w.double().abs().t().contiguous()) * k * 2.0 ** -24
    assert ((ops.linear(x, w, b).double() - want).abs() <= want.abs() * 2.0 ** -8 + slack).all()
