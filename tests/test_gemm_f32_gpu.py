"""fp32 products on the matrix cores: every edge of a tile, a chunk and a vector load, one row alone against the same row among others."""
import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24                                             # half a unit of the last place: one rounding of a product or a sum


def bound(x, w, extra=4):
    """K products and K - 1 sums in any order: at most (K + extra) roundings of the sum of the magnitudes."""
    return (x.shape[-1] + extra) * EPS * (x.abs().double() @ w.abs().double().t()) + 1e-30


@pytest.mark.parametrize("k", [1, 3, 4, 15, 16, 17, 20, 63, 64, 65, 68, 512, 1000])
@pytest.mark.parametrize("m,n", [(1, 1), (15, 17), (16, 16), (17, 31), (31, 33), (33, 32), (70, 100)])
def test_products_and_rows(m, n, k):
    from nanovllm import ops
    g = torch.Generator().manual_seed(m * 1000 + n * 10 + k)
    x, w, b = torch.randn(m, k, generator=g), torch.randn(n, k, generator=g), torch.randn(n, generator=g)
    want = x.double() @ w.double().t()
    xg, wg = x.cuda(), w.cuda()
    got = ops.linear_any(xg, wg)
    assert ((got.cpu().double() - want).abs() <= bound(x, w)).all()
    assert ((ops.linear_any(xg, wg, b.cuda()).cpu().double() - want - b.double()).abs() <= bound(x, w) + 4 * EPS * (want + b).abs()).all()
    for r in {0, m // 2, m - 1}:                             # (a row alone takes the small tiles)
        assert torch.equal(ops.linear_any(xg[r:r + 1].contiguous(), wg)[0], got[r])
    wide = torch.randn(m, k + 3, generator=g).cuda()         # rows that no 16-byte load may be used on
    wide[:, :k] = xg
    assert torch.equal(ops.linear_any(wide[:, :k], wg), got)


@pytest.mark.parametrize("n,k", [(33, 20), (96, 64), (64, 1026)])
@pytest.mark.parametrize("relu2", [False, True])
def test_grouped_rows(n, k, relu2):
    """Blocks of 0, 1, 15, 16, 17, 32, 33, 64 and 65 rows (a tile of the list is 64: upper and lower half, few rows): each row as the plain product
    gives it."""
    from nanovllm import ops
    sizes = [0, 1, 15, 16, 17, 32, 33, 64, 65]
    g = torch.Generator().manual_seed(n + k)
    ids = torch.repeat_interleave(torch.arange(len(sizes)), torch.tensor(sizes))[torch.randperm(sum(sizes), generator=g)].int()
    x, w = torch.randn(len(ids), k, generator=g), torch.randn(len(sizes), n, k, generator=g)
    plan = ops.moe_align(ids.view(-1, 1).cuda(), len(sizes))
    got = ops.linear_grouped(x.cuda(), w.cuda(), plan, True, act="relu2" if relu2 else None)
    pos = plan["pos_of_pair"].view(-1).long()
    for e in range(len(sizes)):
        rows = (ids == e).nonzero().view(-1)
        if rows.numel():
            plain = ops.linear_any(x[rows].cuda(), w[e].cuda())
            assert torch.equal(got[pos[rows.cuda()]], plain.clamp(min=0) ** 2 if relu2 else plain), e
