"""Activations and logits, eight elements a lane, against rows that allow one at a time: the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def odd_rows(t):
    wide = torch.empty(t.shape[0], t.shape[1] + 1, dtype=t.dtype, device=t.device)
    wide[:, :-1] = t
    return wide[:, :-1]


def rows(rows, cols, dtype):
    return (torch.randn(rows, cols, generator=torch.Generator().manual_seed(rows + cols)) * 3).to(dtype).cuda()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,inter", [(1, 8), (65, 1000), (1057, 1000), (512, 2048), (43700, 24)])
def test_activations(n, inter, dtype):
    from nanovllm import ops
    x = rows(n, 2 * inter, dtype)
    assert torch.equal(ops.gelu_tanh_mul(x), ops.gelu_tanh_mul(odd_rows(x)))
    for act in ("silu", "gelu_tanh", "relu2"):
        for gated in (True, False):
            assert torch.equal(ops.act_mul(x, act, gated), ops.act_mul(odd_rows(x), act, gated))
    g = torch.nn.functional.silu(x[:, :inter].double()) * x[:, inter:].double()
    assert ((ops.act_mul(x, "silu", True).double() - g).abs() <= g.abs() * (2.0 ** -8 if dtype is torch.bfloat16 else 2.0 ** -20)).all()
    ids = torch.arange(n).remainder(3).int()[:, None].cuda()
    plan = ops.moe_align(ids, 3)
    w = torch.rand(n, 1, generator=torch.Generator().manual_seed(n)).cuda()
    assert torch.equal(ops.glu_clamp_pairs(x, plan, w, 2.0), ops.glu_clamp_pairs(odd_rows(x), plan, w, 2.0))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,vocab", [(1, 8), (3, 1000), (33, 32768), (1100, 1000)])
def test_logits(n, vocab, dtype):
    from nanovllm import ops
    z = rows(n, vocab, dtype)
    assert torch.equal(ops.logit_softcap(z, 2.0), ops.logit_softcap(odd_rows(z), 2.0))
    for cap in (0.0, 3.0):
        assert torch.equal(ops.logits_scale(z, 0.7, cap), ops.logits_scale(odd_rows(z), 0.7, cap))
    want = 2.0 * torch.tanh(z.double() / 2.0)
    assert ((ops.logit_softcap(z, 2.0).double() - want).abs() <= 2.0 ** -20 * want.abs() + 2.0 ** -22).all()
