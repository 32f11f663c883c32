"""One-token steps of the recurrences: a form of their own, the bits of the form that walks portions."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _slots(B, g):
    slots = torch.randperm(B + 2, generator=g)[:B].int()
    ctx = torch.randint(2, 900, (B,), generator=g).int()
    if B > 2:
        slots[1], ctx[2] = -1, 1                             # a padded row; a sequence that starts here
    return slots.cuda(), ctx.cuda(), torch.arange(B + 1, dtype=torch.int32).cuda()


@pytest.mark.parametrize("read_first,scalar", [(False, False), (False, True), (True, False)])
@pytest.mark.parametrize("B,H,G,dk,dv", [(1, 1, 1, 64, 1), (3, 2, 1, 64, 24), (5, 4, 2, 128, 72), (3, 2, 2, 256, 40), (40, 16, 16, 64, 65), (33, 8, 8, 128, 128), (17, 16, 8, 256, 33)])
def test_gated_linear_scan(B, H, G, dk, dv, read_first, scalar):
    from nanovllm import ops
    g = torch.Generator().manual_seed(B + dk + dv)
    slots, ctx, cu = _slots(B, g)
    q, k = torch.randn(B, G * dk, generator=g).cuda(), torch.randn(B, G * dk, generator=g).cuda()
    v, w = torch.randn(B, H * dv, generator=g).cuda(), torch.rand(B, H if scalar else H * dk, generator=g).cuda()
    state = torch.randn(B + 2, H, dv, dk, generator=g).cuda()
    state[slots[2] if B > 2 else 0] = float("nan") if B > 2 else 1.0          # (what a fresh sequence's slot held must not be read)
    kw = dict(qk_groups=G, kscale=torch.rand(B, H, generator=g).cuda(), skip=torch.randn(H, generator=g).cuda(), read_first=read_first,
              bonus=torch.randn(H * dk, generator=g).cuda() if read_first else None)
    one, many = state.clone(), state.clone()
    a = ops.gated_linear_scan(q, k, w, v, one, slots, None, ctx, H, dk, dv, **kw)
    b = ops.gated_linear_scan(q, k, w, v, many, slots, cu, ctx, H, dk, dv, max_seqlen_q=1, **kw)
    real = slots >= 0
    assert torch.equal(a[real], b[real]) and torch.equal(one.view(torch.int32), many.view(torch.int32))
    wide = torch.randn(B, G * dk + 1, generator=g).cuda()    # rows that no 16-byte load may be used on
    wide[:, :G * dk] = q
    again = state.clone()
    assert torch.equal(ops.gated_linear_scan(wide[:, :G * dk], k, w, v, again, slots, None, ctx, H, dk, dv, **kw)[real], a[real])


@pytest.mark.parametrize("B,H,dk,dv", [(1, 1, 64, 4), (3, 2, 64, 36), (5, 3, 128, 72), (3, 2, 256, 64), (40, 16, 64, 64), (33, 16, 128, 128), (70, 8, 128, 100), (5, 3, 64, 30)])
def test_delta_rule(B, H, dk, dv):
    from nanovllm import ops
    g = torch.Generator().manual_seed(B + dk + dv)
    slots, ctx, cu = _slots(B, g)
    rows = torch.randn(B, H, 5 * dk + dv, generator=g).cuda() * 0.3
    state = torch.randn(B + 2, H, dk, dv, generator=g).cuda()
    if B > 2:
        state[slots[2]] = float("nan")
    one, many = state.clone(), state.clone()
    a = ops._delta_scan(rows, one, slots, None, ctx, H, dk, dv, 1)
    b = ops._delta_scan(rows, many, slots, cu, ctx, H, dk, dv, 1)
    real = slots >= 0
    assert torch.equal(a[real], b[real]) and torch.equal(one.view(torch.int32), many.view(torch.int32))
