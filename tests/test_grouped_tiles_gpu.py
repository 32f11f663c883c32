"""Grouped bf16 products: every tile form gives a row the bits of the plain any-shape product."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("experts,top,k", [(1, 1, 8), (3, 2, 1000), (16, 4, 1024), (64, 64, 1536), (65, 7, 520), (300, 80, 2048)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_routing(experts, top, k, dtype):
    """Choices and weights against the logits that the same launch hands out: the largest, ties to the lower number, -inf and NaN never before others."""
    from nanovllm import ops
    g = torch.Generator().manual_seed(experts * top)
    T = 9
    x, w = torch.randn(T, k, generator=g).to(dtype).cuda(), (torch.randn(experts, k, generator=g) * 0.1).to(dtype).cuda()
    if experts > 2:
        w[2] = w[0]                                          # a tie
    ids, weights, logits = ops.moe_route_linear(x, w, None, top, want_logits=True)
    want = x.double().cpu() @ w.double().cpu().t()
    assert ((logits.double().cpu() - want).abs() <= (k + 8) * 2.0 ** -24 * (x.double().abs().cpu() @ w.double().abs().cpu().t())).all()
    order = torch.sort(logits.cpu(), dim=1, descending=True, stable=True).indices[:, :top]
    assert torch.equal(ids.cpu().long(), order)
    soft = torch.softmax(logits.cpu().double().gather(1, order), 1)
    assert torch.allclose(weights.cpu().double(), soft, rtol=1e-5, atol=1e-12)
    ids, weights = ops.moe_route_linear(x, w, None, top, sigmoid_scores=True)
    assert torch.equal(ids.cpu().long(), order) and torch.allclose(weights.cpu().double(), torch.sigmoid(logits.cpu().double().gather(1, order)), rtol=1e-5, atol=1e-12)
    ids, weights, _, scores = ops.moe_route_scored(x, w, top, want_scores=True, renorm=True)
    order = torch.sort(scores.cpu(), dim=1, descending=True, stable=True).indices[:, :top]
    assert torch.equal(ids.cpu().long(), order)
    picked = scores.cpu().double().gather(1, order)
    assert torch.allclose(weights.cpu().double(), picked / picked.sum(1, keepdim=True), rtol=1e-5)
    x[0] = float("nan")                                      # whatever is chosen then are different experts of the list
    ids = ops.moe_route_scored(x, w, top)[0]
    assert ids[0].min() >= 0 and ids[0].max() < experts and ids[0].unique().numel() == top
