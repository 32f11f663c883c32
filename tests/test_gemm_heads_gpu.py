"""Products per head through LDS rings: the bits of the form that takes any row, with and without a gate, at the edges of tiles and of the ring."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("k", [64, 192, 448])
@pytest.mark.parametrize("m", [1, 16, 17, 33, 64, 65, 130])
@pytest.mark.parametrize("heads,n", [(1, 4), (3, 60), (16, 192), (5, 68)])
def test_bits(heads, n, m, k, gated):
    from nanovllm import ops
    g = torch.Generator().manual_seed(m * n + k + heads)
    head_out = n + 8
    x = torch.randn(m, heads * k, generator=g).bfloat16().cuda()
    w = (torch.randn(heads, n, k, generator=g) * 0.1).bfloat16().cuda()
    gate = torch.randn(m, heads * n, generator=g).bfloat16().cuda() if gated else None
    wide = torch.empty(m, heads * k + 1, dtype=torch.bfloat16, device="cuda")         # (rows that 16-byte loads do not fit)
    wide[:, :-1] = x
    outs = []
    for src in (x, wide[:, :-1]):
        out = torch.full((m, heads * head_out), 7.0, dtype=torch.bfloat16, device="cuda")
        outs.append(ops.linear_heads(src, w, k, out=out, out_head_stride=head_out, gate=gate))
    assert torch.equal(outs[0], outs[1])
    got = outs[0].view(m, heads, head_out)
    assert (got[:, :, n:] == 7.0).all()                      # what lies between two heads stays
    want = torch.stack([x.view(m, heads, k)[:, h].double() @ w[h].double().t().contiguous() for h in range(heads)], 1)
    slack = torch.stack([x.view(m, heads, k)[:, h].double().abs() @ w[h].double().abs().t().contiguous() for h in range(heads)], 1) * k * 2.0 ** -24
    if gated:
        s = torch.sigmoid(gate.double()).view(m, heads, n)
        want, slack = want * s, slack * s + (want * s).abs() * 2.0 ** -21            # (the sigmoid's own fp32 roundings)
    assert ((got[:, :, :n].double() - want).abs() <= want.abs() * 2.0 ** -8 + slack).all()
