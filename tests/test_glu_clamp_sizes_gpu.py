"""nvh_glu_clamp_pairs over more elements than a grid has threads: the pairs on both sides of every cut, most pairs having no row."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pairs,inter", [((1 << 22) + 3, 1025), ((1 << 22) + 3, 1024), ((1 << 22) + 3, 1032), (3, 1 << 20), (1, 8200)])
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


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("inter", [24, 768, 1001, 1024, 1032, 3072])
def test_forms_agree(inter, dtype):
    """Around the sizes where one form takes over from the next: the bits of rows that no 16-byte load may be used on, and of a call of a few pairs."""
    from nanovllm import ops
    g = torch.Generator().manual_seed(inter)
    for total in (1 << 19, 1 << 20, 1 << 21):
        for pairs in sorted({max(total // inter + d, 1) for d in (-1, 0, 1, 2)}):
            plan = ops.moe_align(torch.zeros(pairs, 1, dtype=torch.int32, device="cuda"), 1)
            rows = torch.empty(pairs, 2 * inter + 1, dtype=dtype, device="cuda").uniform_(-3, 3)
            weights = torch.rand(pairs, 1, generator=g).cuda()
            want = ops.glu_clamp_pairs(rows[:, :-1], plan, weights, 1.5)
            got = ops.glu_clamp_pairs(rows[:, :-1].contiguous(), plan, weights, 1.5)
            assert torch.equal(got, want)
            few = ops.moe_align(torch.zeros(7, 1, dtype=torch.int32, device="cuda"), 1)
            at = plan["pos_of_pair"][-7:].long()
            alone = ops.glu_clamp_pairs(rows[at, :-1].contiguous(), dict(few, pos_of_pair=torch.arange(7, dtype=torch.int32, device="cuda")), weights[-7:].contiguous(), 1.5)
            assert torch.equal(alone, want[at])
