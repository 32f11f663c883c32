"""fp32 products through the waves' LDS rings: the bits of the form that reads any row, at the edges of tiles and of a wave's chunks."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def odd_rows(t):
    wide = torch.empty(t.shape[0], t.shape[1] + 1, device=t.device)
    wide[:, :-1] = t
    return wide[:, :-1]


@pytest.mark.parametrize("k", [32, 96, 128, 160, 256, 416, 1024])
@pytest.mark.parametrize("m,n", [(1, 1), (16, 16), (17, 63), (32, 64), (33, 65), (64, 100), (65, 128), (130, 1030), (300, 2050)])
def test_plain(m, n, k):
    from nanovllm import ops
    g = torch.Generator().manual_seed(m * n + k)
    x, w, b = torch.randn(m, k, generator=g).cuda(), torch.randn(n, k, generator=g).cuda(), torch.randn(n, generator=g).cuda()
    want = ops.linear_any(odd_rows(x), w, b)
    assert torch.equal(ops.linear_any(x, w, b), want)
    for r in {0, m // 2, m - 1}:
        assert torch.equal(ops.linear_any(x[r:r + 1].contiguous(), w, b)[0], want[r])


@pytest.mark.parametrize("k", [32, 96, 160, 1024])
@pytest.mark.parametrize("m", [1, 4, 15, 16])
@pytest.mark.parametrize("n", [8192, 8193, 8210, 33000])
def test_few_rows_of_many_columns(m, n, k):
    """Around the width from which small tiles take more than a round: the general form's bits, and those of a call of one row."""
    from nanovllm import ops
    g = torch.Generator().manual_seed(m * n + k)
    x, w, b = torch.randn(m, k, generator=g).cuda(), torch.randn(n, k, generator=g).cuda(), torch.randn(n, generator=g).cuda()
    want = ops.linear_any(odd_rows(x), w, b)
    assert torch.equal(ops.linear_any(x, w, b), want)
    assert torch.equal(ops.linear_any(x[m - 1:].contiguous(), w, b)[0], want[m - 1])
    exact = x.double() @ w.double().t().contiguous() + b.double()
    size = x.double().abs() @ w.double().abs().t().contiguous() + b.double().abs()
    assert ((want.double() - exact).abs() <= size * (k + 4) * 2.0 ** -24).all()


@pytest.mark.parametrize("relu2", [False, True])
@pytest.mark.parametrize("n,k", [(16, 32), (33, 96), (100, 576), (576, 1024)])
def test_grouped(n, k, relu2):
    from nanovllm import ops
    sizes = [0, 1, 15, 16, 17, 31, 32, 33, 48, 49, 64, 65, 130]
    g = torch.Generator().manual_seed(n + k)
    ids = torch.repeat_interleave(torch.arange(len(sizes)), torch.tensor(sizes))[torch.randperm(sum(sizes), generator=g)].int()[:, None].cuda()
    x, w = torch.randn(ids.shape[0], k, generator=g).cuda(), torch.randn(len(sizes), n, k, generator=g).cuda()
    plan = ops.moe_align(ids, len(sizes))
    act = "relu2" if relu2 else None
    at = plan["pos_of_pair"].long()
    want = ops.linear_grouped(odd_rows(x), w, plan, True, act=act)[at]
    assert torch.equal(ops.linear_grouped(x, w, plan, True, act=act)[at], want)
    assert torch.equal(ops.linear_grouped(x[plan["src_token"].long()], w, plan, False, act=act)[at], want)


@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("sizes", [[0, 1, 16, 17, 32, 33, 48, 49, 64, 65, 130], [128], [33, 0, 64], [700, 20]])
@pytest.mark.parametrize("n,k", [(4, 32), (40, 96), (200, 1024), (1030, 64)])
def test_grouped_forms(sizes, n, k, many, monkeypatch):
    """Tiles by 64 columns, by 32, and by 32 with a tile's rows in two workgroups (small grids)."""
    from nanovllm import ops
    monkeypatch.setattr(ops, "GROUPED_MANY_ROWS_F32", 0 if many else 1 << 30)
    g = torch.Generator().manual_seed(n + k)
    ids = torch.repeat_interleave(torch.arange(len(sizes)), torch.tensor(sizes))[torch.randperm(sum(sizes), generator=g)].int()[:, None].cuda()
    x, w = torch.randn(ids.shape[0], k, generator=g).cuda(), torch.randn(len(sizes), n, k, generator=g).cuda()
    plan = ops.moe_align(ids, len(sizes))
    at = plan["pos_of_pair"].long()
    want = ops.linear_grouped(odd_rows(x), w, plan, True)[at]
    assert torch.equal(ops.linear_grouped(x, w, plan, True)[at], want)
    exact = torch.einsum("tk,tnk->tn", x.double().cpu(), w.double().cpu()[ids[:, 0].long().cpu()])
    size = torch.einsum("tk,tnk->tn", x.double().abs().cpu(), w.double().abs().cpu()[ids[:, 0].long().cpu()])
    assert ((want.double().cpu() - exact).abs() <= size * (k + 4) * 2.0 ** -24).all()
