"""The delta rule's chunked form against the recurrence in float64 and against the token-by-token form."""
import pytest
import torch

from nanovllm.ops import DELTA_CHUNK_MIN as MIN

pytestmark = pytest.mark.gpu


def recurrence(rows, dk, state):
    """rows [T, H, 5 dk + dv] = r | k | w | u | au | v, state [H, dk, dv], all float64."""
    r, k, w, u, au, v = rows.split([dk] * 5 + [rows.shape[2] - 5 * dk], 2)
    S, out = state.clone(), []
    for t in range(rows.shape[0]):
        uS = (u[t, :, :, None] * S).sum(1)
        S = w[t, :, :, None] * S - au[t, :, :, None] * uS[:, None, :] + k[t, :, :, None] * v[t, :, None, :]
        out.append((r[t, :, :, None] * S).sum(1))
    return torch.stack(out), S


def pack(T, H, dk, dv, g, decay):
    r, k, v = torch.randn(T, H, dk, generator=g), torch.randn(T, H, dk, generator=g), torch.randn(T, H, dv, generator=g)
    u = k / (k * k).sum(-1, keepdim=True).sqrt()
    a = torch.rand(T, H, dk, generator=g)
    w = {"mild": 0.55 + 0.45 * torch.rand(T, H, dk, generator=g), "one": torch.ones(T, H, dk),
         "steep": torch.rand(T, H, dk, generator=g) ** 40, "none": torch.zeros(T, H, dk)}[decay]
    return torch.cat([r, k, w, u, a * u * (1.0 if decay != "one" else 0.5), v], 2)


def scan(rows, state, slots, cu, ctx, H, dk, dv, longest):
    from nanovllm import ops
    st = state.cuda()
    out = ops._delta_scan(rows.cuda(), st, slots.cuda(), cu.cuda(), ctx.cuda(), H, dk, dv, longest)
    return out.cpu().view(-1, H, dv), st.cpu()


@pytest.mark.parametrize("decay", ["mild", "one", "steep", "none"])
@pytest.mark.parametrize("H,dk,dv", [(3, 64, 64), (2, 128, 128), (2, 16, 48), (1, 96, 16), (2, 48, 32), (1, 32, 144)])
def test_portions_of_every_kind(H, dk, dv, decay):
    """Portions below, at and above the threshold, with and without a partial last chunk, fresh and carried, padded rows between.  The bound is
    eight times what the token-by-token form is off (both sum in fp32, in another order), and 1e-6 of the largest value."""
    lens, carried = [MIN, 5, MIN + 15, 0, MIN + 16, MIN - 1, 1, MIN + 113], [0, 7, 3, 2, 0, 0, 9, 1]
    g = torch.Generator().manual_seed(dk + dv)
    T, B = sum(lens), len(lens)
    rows = pack(T, H, dk, dv, g, decay)
    state = torch.randn(B + 2, H, dk, dv, generator=g)
    slots = torch.randperm(B + 2, generator=g)[:B].int()
    slots[5] = -1
    cu = torch.tensor([0] + lens).cumsum(0).int()
    ctx = torch.tensor([n + c for n, c in zip(lens, carried)]).int()
    serial, serial_state = scan(rows, state, slots, cu, ctx, H, dk, dv, 0)
    got, got_state = scan(rows, state, slots, cu, ctx, H, dk, dv, max(lens))
    used = set(slots[slots >= 0].tolist())
    for b, n in enumerate(lens):
        at, s = int(cu[b]), int(slots[b])
        if not n or s < 0:
            continue
        start = state[s].double() if carried[b] else torch.zeros(H, dk, dv, dtype=torch.float64)
        want, end = recurrence(rows[at:at + n].double(), dk, start)
        for x, y, z in ((got[at:at + n], serial[at:at + n], want), (got_state[s], serial_state[s], end)):
            if n < MIN:
                assert torch.equal(x, y)
            assert (x.double() - z).abs().max() <= 8 * (y.double() - z).abs().max() + 1e-6 * z.abs().max(), (b, n)
    for s in range(B + 2):
        if s not in used or lens[slots.tolist().index(s)] == 0:
            assert torch.equal(got_state[s], state[s])


def test_error_against_64_bits():
    """1024 tokens at the served sizes, in the 2-norm: outputs and states are nearer to float64 than token by token."""
    for H, dk, dv in ((16, 64, 64), (8, 128, 128)):
        g = torch.Generator().manual_seed(3)
        rows = pack(1024, H, dk, dv, g, "mild")
        cu, ctx, slots = torch.tensor([0, 1024]).int(), torch.tensor([1024]).int(), torch.tensor([0]).int()
        state = torch.zeros(1, H, dk, dv)
        want, end = recurrence(rows.double().cuda(), dk, state[0].double().cuda())
        off = []
        for longest in (0, 1024):
            out, st = scan(rows, state, slots, cu, ctx, H, dk, dv, longest)
            off.append([(out.double() - want.cpu()).norm(), (st[0].double() - end.cpu()).norm()])
        (out_serial, state_serial), (out_chunks, state_chunks) = off
        assert out_chunks < out_serial and state_chunks < state_serial, (H, off)


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("at", [37, MIN + 9])
@pytest.mark.parametrize("field", range(6))
def test_values_that_are_not_finite(field, at, value):
    """One such value of r, k, w, u, au or v, with whole chunks before and behind it or in the partial last chunk of a portion that is chunked: the tokens
    before it, and other heads, stay as they are (of v: other columns as well), and what is not finite token by token is not finite in chunks."""
    H, dk, dv, T = 2, 64, 32, MIN + 12
    g = torch.Generator().manual_seed(11)
    rows = pack(T, H, dk, dv, g, "mild")
    cu, ctx, slots, state = torch.tensor([0, T]).int(), torch.tensor([T]).int(), torch.tensor([0]).int(), torch.zeros(1, H, dk, dv)
    want, want_state = scan(rows, state, slots, cu, ctx, H, dk, dv, T)
    plain, _ = scan(rows, state, slots, cu, ctx, H, dk, dv, 0)
    assert not torch.equal(want, plain)                      # (the two forms round differently: the chunked one ran)
    rows[at, 1, field * dk + 5] = value
    serial, serial_state = scan(rows, state, slots, cu, ctx, H, dk, dv, 0)
    got, got_state = scan(rows, state, slots, cu, ctx, H, dk, dv, T)
    close = dict(rtol=1e-5, atol=1e-5 * want.abs().max().item())
    torch.testing.assert_close(got[:at], want[:at], **close)
    torch.testing.assert_close(got[:, 0], want[:, 0], **close)
    torch.testing.assert_close(got_state[0, 0], want_state[0, 0], **close)
    assert not got[at, 1].isfinite().all()
    assert not (got.isfinite() & ~serial.isfinite()).any() and not (got_state.isfinite() & ~serial_state.isfinite()).any()
    if field == 0:                                           # a read-out alone
        torch.testing.assert_close(got[at + 1:], want[at + 1:], **close)
        torch.testing.assert_close(got_state, want_state, **close)
    if field == 5:
        keep = [c for c in range(dv) if c != 5]
        torch.testing.assert_close(got[:, 1][:, keep], want[:, 1][:, keep], **close)
        torch.testing.assert_close(got_state[0, 1][:, keep], want_state[0, 1][:, keep], **close)


def test_cuts_at_whole_chunks():
    """A portion cut at a multiple of 16 tokens into two that are chunked: the same bits."""
    H, dk, dv, T, cut = 2, 64, 64, 3 * MIN + 5, MIN + 16
    g = torch.Generator().manual_seed(5)
    rows, state = pack(T, H, dk, dv, g, "mild"), torch.randn(1, H, dk, dv, generator=g)
    slots, at = torch.tensor([0]).int(), lambda *n: torch.tensor(n).int()
    whole, whole_state = scan(rows, state, slots, at(0, T), at(T + 1), H, dk, dv, T)
    one, mid = scan(rows[:cut].contiguous(), state, slots, at(0, cut), at(cut + 1), H, dk, dv, cut)
    two, end = scan(rows[cut:].contiguous(), mid, slots, at(0, T - cut), at(T + 1), H, dk, dv, T - cut)
    assert torch.equal(torch.cat([one, two]), whole) and torch.equal(end, whole_state)
