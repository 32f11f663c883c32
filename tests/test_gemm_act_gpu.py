"""Projections with their ungated activation in the product's epilogue (nvh_gemm_act_bf16_nt)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 15, 16, 17, 32, 33, 63, 64])
@pytest.mark.parametrize("n,k", [(4, 64), (36, 1024), (1024, 192), (4096, 1024), (4100, 1024), (8192, 128)])
@pytest.mark.parametrize("act", ["relu2", "xielu"])
def test_the_bits_of_two_launches(m, n, k, act):
    """Every tile it takes, rows and columns that end inside one, with and without a bias, from rows of a wider buffer: the bits of the product followed by the
    activation, and within bf16's rounding (twice 2^-9, of the product and of the result) of the formula in float64."""
    from nanovllm import _hip, ops
    g = torch.Generator().manual_seed(m * 10007 + n + k)
    x = torch.randn(m, k + 8, generator=g).bfloat16().cuda()[:, :k]
    w = (torch.randn(n, k, generator=g) * k ** -0.5 * 2).bfloat16().cuda()
    params = torch.tensor([0.4, -0.7]).bfloat16().cuda() if act == "xielu" else None
    for bias in (None, torch.randn(n, generator=g).bfloat16().cuda()):
        got = ops.linear_act(x, w, bias, act, params)
        assert (got is not None) == bool(_hip.lib().nvh_gemm_act_supported(m, n, k)) and got is not None
        mid = ops.linear_any(x, w, bias)
        want = ops.xielu(mid, params) if act == "xielu" else ops.act_mul(mid, "relu2", False)
        assert torch.equal(got, want)
        z = x.double() @ w.double().t() + (0 if bias is None else bias.double())
        if act == "relu2":
            ref, slope = z.clamp_min(0) ** 2, 2 * z.abs()
        else:
            p, q = torch.nn.functional.softplus(params.double())
            ref = torch.where(z > 0, p * z * z, (0.5 + q) * (torch.expm1(z.clamp_max(0)) - z)) + 0.5 * z
            slope = torch.where(z > 0, 2 * p * z + 0.5, torch.full_like(z, 1.6))
        assert ((got.double() - ref).abs() <= 2.0 ** -8 * (slope * z.abs() + ref.abs()) + 1e-4).all()


def test_what_it_leaves_to_two_launches():
    from nanovllm import ops
    w = torch.randn(256, 128).bfloat16().cuda()
    for x in (torch.randn(65, 128).bfloat16().cuda(), torch.randn(4, 128).cuda(), torch.randn(4, 132).bfloat16().cuda()[:, 4:], torch.randn(0, 128).bfloat16().cuda()):
        assert ops.linear_act(x, w if x.dtype == w.dtype else w.float(), None, "relu2") is None


def test_a_watched_activation_sees_the_product():
    """A hook on the projection or the activation, or another forward: both modules are called."""
    from nanovllm.layers.activation import Act
    from nanovllm.layers.linear import MergedLinear
    from nanovllm.layers.moe import project_act
    torch.set_default_dtype(torch.bfloat16)
    try:
        up, act = MergedLinear(128, [256]).cuda(), Act("relu2")
    finally:
        torch.set_default_dtype(torch.float32)
    up.weight.data.normal_()
    x, seen = torch.randn(8, 128).bfloat16().cuda(), []
    plain = project_act(up, act, x)
    handle = act.register_forward_hook(lambda mod, args, out: seen.append(args[0]))
    assert torch.equal(project_act(up, act, x), plain) and len(seen) == 1 and torch.equal(seen[0], up(x))
    handle.remove()
    act.forward = lambda z: z
    assert torch.equal(project_act(up, act, x), up(x))
