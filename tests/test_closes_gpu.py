"""Closes of a sublayer: rows kept in registers against rows that no vector load may be used on, and a mixture's sum inside the close."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def odd_rows(t):
    wide = torch.empty(t.shape[0], t.shape[1] + 1, dtype=t.dtype, device=t.device)
    wide[:, :-1] = t
    return wide[:, :-1]


def close_to(a, b, dtype):
    """The same sums in fp32 in another order: 1e-5 of the rows' size and, in bf16, one rounding of the result."""
    a, b = a.double(), b.double()
    return ((a - b).abs() <= (1e-5 + (2.0 ** -7 if dtype is torch.bfloat16 else 0.0)) * b.abs() + 1e-5 * b.pow(2).mean().sqrt()).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,dim", [(1, 4), (3, 64), (5, 1020), (2, 1024), (3, 1028), (2, 2052), (2, 4100), (1, 8192)])
def test_registers_and_columns(rows, dim, dtype):
    from nanovllm import ops
    g = torch.Generator().manual_seed(rows * dim)
    def t(*shape):
        return torch.randn(*shape, generator=g).to(dtype).cuda()
    a, b, c, w1, w2, w3, w4 = t(rows, dim), t(rows, dim), t(rows, dim), t(dim), t(dim), t(dim), t(dim)
    c32, x = torch.randn(rows, dim, generator=g).cuda(), torch.randn(rows, dim, generator=g).cuda()
    forms = [(ops.residual_norm, dict(a=a, a_weight=w1, b=b, b_weight=w2, branch_scale=0.5, branch_eps=1e-6, c=c, c32=c32, norm="layer", weight=w3, bias=w4, eps=1e-5)),
             (ops.residual_norm, dict(c=c, norm="rms", weight=w3, eps=1e-5)), (ops.residual_norm, dict(a=a, b=b)),
             (ops.residual_postnorm, dict(weight=w1, eps=1e-6, y=a, y32=c32, layer_scale=w2, alpha=2.0, weight_offset=1.0)),
             (ops.residual_postnorm, dict(weight=w1, eps=1e-6, y=a, in_place=False)),
             (ops.residual_subnorm, dict(weight=w1[:1], eps=1e-6, mult=0.5, a=a, a_scale=0.6, b=b, b_scale=0.9, c32=c32)),
             (ops.residual_subnorm, dict(weight=w1, eps=1e-6, a=a))]
    for op, kw in forms:
        one, other = x.clone(), x.clone()
        h = op(one, **kw)
        k = op(other, **{n: odd_rows(v) if torch.is_tensor(v) and v.dim() == 2 else v for n, v in kw.items()})
        assert close_to(one, other, torch.float32) and (h is None or close_to(h, k, dtype))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("tokens,dim,top,experts", [(1, 8, 1, 1), (7, 1024, 2, 16), (5, 1028, 4, 6), (3, 2048, 5, 9), (4, 30, 3, 7)])
def test_a_mixture_inside_the_close(tokens, dim, top, experts, dtype):
    """Bit for bit what moe_combine and the close after it give; weights or none, a shared expert with a gate, without, or none; a pair without a row."""
    from nanovllm import ops
    g = torch.Generator().manual_seed(tokens * dim)
    ids = torch.stack([torch.randperm(experts, generator=g)[:top] for _ in range(tokens)]).int()
    if tokens > 2:
        ids[1, 0] = -1
    plan = ops.moe_align(ids.cuda(), experts)
    def t(*shape):
        return torch.randn(*shape, generator=g).to(dtype).cuda()
    y, shared, w, wn = t(tokens * top, dim), t(tokens, dim), torch.rand(tokens, top, generator=g).cuda(), t(dim)
    gate, x = torch.randn(tokens, 1, generator=g).cuda(), torch.randn(tokens, dim, generator=g).cuda()
    for weights, sh, gt in ((w, shared, gate), (w, shared, None), (None, None, None)):
        summed = ops.moe_combine(y, plan, weights, sh, gt, top=top)
        moe = dict(y=y, plan=plan, weights=weights, shared=sh, gate=gt, top=top)
        for op, kw, name in ((ops.residual_norm, dict(norm="rms", weight=wn, eps=1e-5), "c32"), (ops.residual_postnorm, dict(weight=wn, eps=1e-5, alpha=2.0), "y32"),
                             (ops.residual_subnorm, dict(weight=wn[:1], eps=1e-5), "c32")):
            one, other = x.clone(), x.clone()
            assert torch.equal(op(one, **kw, moe=moe), op(other, **kw, **{name: summed})) and torch.equal(one, other)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("dim", [4, 252, 256, 260, 1024, 2048, 4096, 4100, 5120, 5124, 6144, 6148, 8192])
def test_every_form_of_the_norm_close(dim, dtype):
    """Calls with a second branch, with one and further terms, with one alone and without any, at the edges of the columns a lane and a wave hold."""
    from nanovllm import ops
    rows = 3
    g = torch.Generator().manual_seed(dim)
    def t(*shape):
        return torch.randn(*shape, generator=g).to(dtype).cuda()
    a, b, c, w1, w2, w3, w4 = t(rows, dim), t(rows, dim), t(rows, dim), t(dim), t(dim), t(dim), t(dim)
    c32, x = torch.randn(rows, dim, generator=g).cuda(), torch.randn(rows, dim, generator=g).cuda()
    branch, second = dict(a=a, a_weight=w1, branch_scale=0.5, branch_eps=1e-6), dict(b=b, b_weight=w2)
    rms, layer = dict(norm="rms", weight=w3, eps=1e-5), dict(norm="layer", weight=w3, bias=w4, eps=1e-5)
    for kw in ({**branch, **second, **rms}, {**branch, **second, "c": c, **layer}, {**branch, **rms}, {"a": a, **rms}, branch, {**branch, **layer}, {"a": a, "c32": c32, **rms},
               {**branch, "c": c, "c32": c32, **layer}, rms, layer, {"c": c, **rms}, {"c32": c32, **layer}, {"c": c, "c32": c32}, second, {"b": b, "c32": c32, **rms}):
        one, other = x.clone(), x.clone()
        h = ops.residual_norm(one, **kw)
        k = ops.residual_norm(other, **{n: odd_rows(v) if torch.is_tensor(v) and v.dim() == 2 else v for n, v in kw.items()})
        assert close_to(one, other, torch.float32) and (h is None or close_to(h, k, dtype)), kw.keys()
