"""Eight-wave tiles with three stages (128 x 128, 128 x 192, 256 x 128), one a CU: from fewer k-tiles than stages on, ragged edges with results stored 16 and 8
bytes at a time, weights read past the caches, widths that end in a narrower strip of tiles, K-slabs: the bits of 64 x 64 tiles.  And two-group tiles: the
bits of their two sums."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def plan(m, n, k, slabs=1):
    import ctypes as C
    from nanovllm import _hip
    out = C.create_string_buffer(512)
    assert _hip.lib().nvh_gemm_plan(m, n, k, slabs, 0, out, 512) == 0
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


@pytest.mark.parametrize("m,n,k,tile", [(1000, 1852, 192, "128x64 waves 2x2"), (1024, 1664, 192, "128x64 waves 2x2"), (1280, 12800, 192, "256x256 waves 2x4"),
                                        (1270, 13052, 192, "256x256 waves 2x4"), (700, 604, 192, "64x64 waves 2x2"), (1008, 64, 192, "64x64 waves 2x2")])
def test_grids_of_odd_and_twice_odd_widths(m, n, k, tile):
    """Tiles in strips of which the last is narrower (29, 50 and 51 tiles wide) and in the grid's own order (26, 10 and 1): each is computed, once."""
    from nanovllm import ops
    assert plan(m, n, k).startswith(f"tile {tile}")
    g = torch.Generator().manual_seed(m + n + k)
    x, w = ((torch.randn(s, generator=g) * 0.5).bfloat16().cuda() for s in ((m, k), (n, k)))
    check(lambda: ops.linear(x, w), x, w, None)


@pytest.mark.parametrize("m,n,k", [(1024, 8192, 1024), (1016, 7172, 1088), (769, 8188, 1152)])
def test_tall_bits(m, n, k):
    from nanovllm import ops
    assert plan(m, n, k).startswith("tile 256x128 waves 2x4 stages 3")
    g = torch.Generator().manual_seed(m + n + k)
    x, w = ((torch.randn(s, generator=g) * 0.5).bfloat16().cuda() for s in ((m, k), (n, k)))
    check(lambda: ops.linear(x, w), x, w, None)


@pytest.mark.parametrize("m,n,k,tile", [(1016, 7176, 1024, "256x128 waves 2x4 stages 3 grid"), (1001, 5256, 320, "128x192 waves 2x4 stages 3 grid"),
                                        (897, 3976, 192, "128x128 waves 2x4 stages 3 grid"), (100, 37984, 1024, "128x192 waves 2x4 stages 3 nt"),
                                        (128, 37980, 128, "128x192 waves 2x4 stages 3 nt"), (200, 28680, 1024, "256x128 waves 2x4 stages 3 nt"),
                                        (256, 28676, 1088, "256x128 waves 2x4 stages 3 nt")])
def test_ragged_and_streamed_bits(m, n, k, tile):
    """Rows past the last one in tiles whose results leave 16 bytes a lane (N a multiple of 8), and weights of one row of tiles, read non-temporally."""
    from nanovllm import ops
    assert plan(m, n, k).startswith(f"tile {tile}")
    g = torch.Generator().manual_seed(m + n + k)
    x, w = ((torch.randn(s, generator=g) * 0.5).bfloat16().cuda() for s in ((m, k), (n, k)))
    guard = torch.full((m + 8, n), 7.0, dtype=torch.bfloat16, device="cuda")                  # rows behind the result keep what they hold

    def f():
        from nanovllm import _hip
        _hip.call("nvh_gemm_bf16_nt", x.data_ptr(), k, w.data_ptr(), 0, guard.data_ptr(), n, m, n, k, 1, 0, torch.cuda.current_stream().cuda_stream)
        assert bool((guard[m:] == 7.0).all())
        return guard[:m].clone()

    check(f, x, w, None)


@pytest.mark.parametrize("m,n,k,s", [(256, 5120, 768, 3), (300, 2560, 832, 4), (128, 5120, 5184, 6), (128, 4096, 832, 8)])
def test_slabs(m, n, k, s):
    """Slabs of 1 to 14 k-tiles, the last one shorter or empty (13 k-tiles by two in 8 slabs); each slab is a sum over its part of K alone."""
    from nanovllm import ops
    assert plan(m, n, k, s).replace(" nt", "").startswith("tile 128x128 waves 2x4 stages 3 slabs")
    g = torch.Generator().manual_seed(m + n + k)
    x, w = ((torch.randn(sh, generator=g) * 0.5).bfloat16().cuda() for sh in ((m, k), (n, k)))
    got = ops.linear_splitk(x, w, s)
    per = -(-(k // 64) // s) * 64
    for p in range(s):
        a, c = x[:, p * per:(p + 1) * per].double(), w[:, p * per:(p + 1) * per].double()
        assert ((got[p].double() - a @ c.t().contiguous()).abs() <= a.abs() @ c.abs().t().contiguous() * per * 2.0 ** -24 + 1e-30).all()


@pytest.mark.parametrize("m,n,k", [(1024, 1024, 1024), (833, 1020, 1152), (1000, 964, 3072), (1000, 964, 3200), (832, 1216, 1024), (896, 1152, 1024), (896, 1152, 1536)])
def test_two_groups(m, n, k):
    """64 x 64 tiles of two wave groups: stages requested behind the reads (K up to 3072) and ahead of them."""
    from nanovllm import ops
    assert plan(m, n, k).startswith("kgroups")
    g = torch.Generator().manual_seed(m + n + k)
    x, w, b = ((torch.randn(s, generator=g) * 0.5).bfloat16().cuda() for s in ((m, k), (n, k), (n,)))
    got = ops.linear(x, w, b)
    # group 0 adds up the even k-tiles, group 1 the odd ones: two K-slabs of the same operands with the even k-tiles in front
    # (k-tiles of both groups are as many, K is a multiple of 128)
    even, odd = (torch.cat([torch.arange(c, c + 64) for c in range(first, k, 128)]) for first in (0, 64))
    order = torch.cat([even, odd]).cuda()
    parts = ops.linear_splitk(x[:, order].contiguous(), w[:, order].contiguous(), 2)
    assert torch.equal(got, (parts[0] + parts[1] + b.float()).bfloat16())
    want = x.double() @ w.double().t().contiguous() + b.double()
    slack = (x.double().abs() @ w.double().abs().t().contiguous()) * k * 2.0 ** -24
    assert ((got.double() - want).abs() <= want.abs() * 2.0 ** -8 + slack).all()
