"""Eight-wave tiles with three stages (128 x 128, 128 x 192, 256 x 128), one a CU: from fewer k-tiles than stages on, ragged edges, widths that end in a
narrower strip of tiles, K-slabs: the bits of 64 x 64 tiles."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def plan(m, n, k):
    import ctypes as C
    from nanovllm import _hip
    out = C.create_string_buffer(512)
    assert _hip.lib().nvh_gemm_plan(m, n, k, 1, 0, out, 512) == 0
    return out.value.decode()


def check(f, x, w, b):
    from nanovllm import _hip
    got = f()
    with _hip.switch("NVH_GEMM_FORCE_TILE", 5), _hip.switch("NVH_GEMM_NO_KGROUPS"):      # 64 x 64, one wave group
        assert torch.equal(got, f())
    want = x.double() @ w.double().t().contiguous() + (0 if b is None else b.double())
    slack = (x.double().abs() @ w.double().abs().t().contiguous()) * x.shape[1] * 2.0 ** -24
    assert ((got.double() - want).abs() <= want.abs() * 2.0 ** -8 + slack).all()


@pytest.mark.parametrize("k", [64, 128, 192, 256, 320, 1024])
@pytest.mark.parametrize("m,n,tile", [(1024, 4096, "128x128"), (897, 3972, "128x128"), (769, 4604, "128x128"), (1024, 6144, "128x192"), (1001, 5252, "128x192"), (513, 9604, "128x192")])
def test_bits(m, n, tile, k):
    from nanovllm import ops
    assert plan(m, n, k).startswith(f"tile {tile} waves 2x4 stages 3")
    g = torch.Generator().manual_seed(m + n + k)
    x, w, b = ((torch.randn(s, generator=g) * 0.5).bfloat16().cuda() for s in ((m, k), (n, k), (n,)))
    check(lambda: ops.linear(x, w, b), x, w, b)


@pytest.mark.parametrize("m,n,k", [(1024, 8192, 1024), (1016, 7172, 1088), (769, 8188, 1152)])
def test_tall_bits(m, n, k):
    from nanovllm import ops
    assert plan(m, n, k).startswith("tile 256x128 waves 2x4 stages 3")
    g = torch.Generator().manual_seed(m + n + k)
    x, w = ((torch.randn(s, generator=g) * 0.5).bfloat16().cuda() for s in ((m, k), (n, k)))
    check(lambda: ops.linear(x, w), x, w, None)


@pytest.mark.parametrize("m,n,k,s", [(256, 5120, 768, 3), (300, 2560, 832, 4), (128, 5120, 5184, 6)])
def test_slabs(m, n, k, s):
    """Slabs of 3 to 14 k-tiles, the last one shorter; each slab is a sum over its part of K alone."""
    from nanovllm import ops
    g = torch.Generator().manual_seed(m + n + k)
    x, w = ((torch.randn(sh, generator=g) * 0.5).bfloat16().cuda() for sh in ((m, k), (n, k)))
    got = ops.linear_splitk(x, w, s)
    per = -(-(k // 64) // s) * 64
    for p in range(s):
        a, c = x[:, p * per:(p + 1) * per].double(), w[:, p * per:(p + 1) * per].double()
        assert ((got[p].double() - a @ c.t().contiguous()).abs() <= a.abs() @ c.abs().t().contiguous() * per * 2.0 ** -24 + 1e-30).all()


@pytest.mark.parametrize("m,n,k", [(1024, 1024, 1024), (833, 1020, 1152), (1000, 964, 3072), (1000, 964, 3200)])
def test_two_groups(m, n, k):
    """64 x 64 tiles of two wave groups: stages requested behind the reads (K up to 3072) and ahead of them."""
    from nanovllm import ops
    assert plan(m, n, k).startswith("kgroups")
    g = torch.Generator().manual_seed(m + n + k)
    x, w, b = ((torch.randn(s, generator=g) * 0.5).bfloat16().cuda() for s in ((m, k), (n, k), (n,)))
    got = ops.linear(x, w, b).double()
    want = x.double() @ w.double().t().contiguous() + b.double()
    slack = (x.double().abs() @ w.double().abs().t().contiguous()) * k * 2.0 ** -24
    assert ((got - want).abs() <= want.abs() * 2.0 ** -8 + slack).all()
