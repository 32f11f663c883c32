"""nvh_glu_clamp_pairs over more elements than a grid has threads: the pairs on both sides of every cut, most pairs having no row."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pairs,inter", [((1 << 22) + 3, 1025), (3, 1 << 20), (1, 8200)])
def test_many_pairs(pairs, inter):
    from nanovllm import _hip, ops
    g = torch.Generator().manual_seed(pairs)
    most = max((1 << 31) // inter, 1)
    picked = sorted({p for p in (0, most - 1, most, 2 * most - 1, 2 * most, pairs - 1) if p < pairs})
    pos = torch.full((pairs,), -1, dtype=torch.int32, device="cuda")
    pos[picked] = torch.arange(len(picked), dtype=torch.int32, device="cuda")
    weights = torch.rand(pairs, device="cuda")
    rows = torch.randn(len(picked), 2 * inter, generator=g).bfloat16().cuda()
    y = torch.zeros(len(picked), inter, dtype=torch.bfloat16, device="cuda")
    _hip.call("nvh_glu_clamp_pairs", rows.data_ptr(), 2 * inter, pos.data_ptr(), weights.data_ptr(), y.data_ptr(), inter, pairs, inter, 1.5, 1.702, 0, ops._stream())
    w = weights[picked][:, None].double()
    gate, up = (rows[:, :inter].double() * w).clamp(max=1.5), (rows[:, inter:].double() * w).clamp(-1.5, 1.5)
    want = gate * torch.sigmoid(1.702 * gate) * (up + 1)
    # a bf16 rounding of the result; fp32 roundings of the products and the exponential stay below 2^-20 of values of a few units
    assert ((y.double() - want).abs() <= want.abs() * 2.0 ** -8 + 2.0 ** -20).all()
