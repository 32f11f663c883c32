"""The gated linear scan's chunked form against the recurrence in float64 and against the token-by-token form."""
import pytest
import torch

from nanovllm.ops import SCAN_CHUNK_MIN as MIN

pytestmark = pytest.mark.gpu


def recurrence(x, state, read_first):
    """Operands [T, H, ...] and state [H, dv, dk], all float64."""
    S, out = state.clone(), []
    for t in range(x["v"].shape[0]):
        kv = x["v"][t, :, :, None] * (x["c"][t, :, None] * x["k"][t])[:, None, :]
        new = x["w"][t, :, None, :] * S + kv
        seen = S + kv * x["bonus"][:, None, :] if read_first else new
        out.append((seen * x["q"][t, :, None, :]).sum(-1) + x["skip"][:, None] * x["v"][t])
        S = new
    return torch.stack(out), S


def operands(T, H, G, dk, dv, g, decay, scalar):
    r = lambda *s: torch.randn(*s, generator=g)
    u = torch.rand(T, H, 1 if scalar else dk, generator=g)
    w = {"mild": 0.55 + 0.45 * u, "slow": 1 - 0.02 * u, "steep": u ** 40, "none": 0 * u}[decay]
    return dict(q=r(T, G, dk), k=r(T, G, dk), w=w, v=r(T, H, dv), c=torch.rand(T, H, generator=g), skip=r(H), bonus=r(H, dk))


def scan(x, state, slots, cu, ctx, H, G, dk, dv, longest, read_first, plain=False):
    from nanovllm import ops
    st, T = state.cuda(), x["v"].shape[0]
    flat = lambda n: x[n].reshape(T, -1).cuda()
    out = ops.gated_linear_scan(flat("q"), flat("k"), flat("w"), flat("v"), st, slots.cuda(), cu.cuda(), ctx.cuda(), H, dk, dv, G,
                                None if plain else x["c"].cuda(), None if plain else x["skip"].cuda(), longest, read_first,
                                x["bonus"].cuda() if read_first and not plain else None)
    return out.cpu().view(T, H, dv), st.cpu()


def full(x, H, G, dk, plain=False):
    """The operands as the recurrence takes them, in float64."""
    T = x["v"].shape[0]
    y = {n: t.double() for n, t in x.items()}
    y["q"], y["k"], y["w"] = y["q"].repeat_interleave(H // G, 1), y["k"].repeat_interleave(H // G, 1), y["w"].expand(T, H, dk)
    if plain:
        y["c"], y["skip"], y["bonus"] = torch.ones(T, H).double(), torch.zeros(H).double(), torch.zeros(H, dk).double()
    return y


@pytest.mark.parametrize("read_first", [False, True])
@pytest.mark.parametrize("decay", ["mild", "slow", "steep", "none"])
@pytest.mark.parametrize("H,G,dk,dv,scalar", [(3, 3, 64, 64, False), (4, 2, 128, 256, True), (2, 1, 128, 64, False), (2, 2, 16, 48, True), (1, 1, 96, 16, False),
                                              (2, 2, 48, 32, False), (1, 1, 32, 144, False)])
def test_portions_of_every_kind(H, G, dk, dv, scalar, decay, read_first):
    """Portions below, at and above the threshold, with and without a partial last chunk, fresh and carried, padded rows between.  The bound is
    eight times what the token-by-token form is off (both sum in fp32, in another order), and 1e-6 of the largest value."""
    lens, carried = [MIN, 5, MIN + 15, 0, MIN + 16, MIN - 1, 1, MIN + 113], [0, 7, 3, 2, 0, 0, 9, 1]
    g = torch.Generator().manual_seed(dk + dv)
    T, B, plain = sum(lens), len(lens), dk == 48
    x = operands(T, H, G, dk, dv, g, decay, scalar)
    state = torch.randn(B + 2, H, dv, dk, generator=g)
    slots = torch.randperm(B + 2, generator=g)[:B].int()
    slots[5] = -1
    cu = torch.tensor([0] + lens).cumsum(0).int()
    ctx = torch.tensor([n + c for n, c in zip(lens, carried)]).int()
    serial, serial_state = scan(x, state, slots, cu, ctx, H, G, dk, dv, 0, read_first, plain)
    got, got_state = scan(x, state, slots, cu, ctx, H, G, dk, dv, max(lens), read_first, plain)
    y, used = full(x, H, G, dk, plain), set(slots[slots >= 0].tolist())
    for b, n in enumerate(lens):
        at, s = int(cu[b]), int(slots[b])
        if not n or s < 0:
            continue
        start = state[s].double() if carried[b] else torch.zeros(H, dv, dk, dtype=torch.float64)
        want, end = recurrence({m: t if m in ("skip", "bonus") else t[at:at + n] for m, t in y.items()}, start, read_first)
        for a, c, z in ((got[at:at + n], serial[at:at + n], want), (got_state[s], serial_state[s], end)):
            if n < MIN:
                assert torch.equal(a, c)
            assert (a.double() - z).abs().max() <= 8 * (c.double() - z).abs().max() + 1e-6 * z.abs().max(), (b, n)
    for s in range(B + 2):
        if s not in used or lens[slots.tolist().index(s)] == 0:
            assert torch.equal(got_state[s], state[s])


@pytest.mark.parametrize("decay", ["mild", "slow"])
def test_error_against_64_bits(decay):
    """1024 tokens at the served sizes, in the 2-norm: outputs and states are no further from float64 than token by token."""
    for H, G, dk, dv, read_first in ((16, 16, 64, 64, True), (4, 4, 128, 256, False)):
        g = torch.Generator().manual_seed(3)
        x = operands(1024, H, G, dk, dv, g, decay, False)
        cu, ctx, slots = torch.tensor([0, 1024]).int(), torch.tensor([1024]).int(), torch.tensor([0]).int()
        state = torch.zeros(1, H, dv, dk)
        want, end = recurrence({m: t.cuda() for m, t in full(x, H, G, dk).items()}, state[0].double().cuda(), read_first)
        off = []
        for longest in (0, 1024):
            out, st = scan(x, state, slots, cu, ctx, H, G, dk, dv, longest, read_first)
            off.append([((out.double() - want.cpu()).norm() / want.cpu().norm()).item(), ((st[0].double() - end.cpu()).norm() / end.cpu().norm()).item()])
        (out_serial, state_serial), (out_chunks, state_chunks) = off
        assert out_chunks <= out_serial and state_chunks <= state_serial, (H, off)


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("field", ["q", "k", "w", "v"])
def test_values_that_are_not_finite(field, value):
    """One such value at token 37 of 76 leaves the tokens before it, and other heads, as they are; a value of v leaves the other columns as well."""
    H, dk, dv, T, at = 2, 64, 32, MIN + 12, 37
    g = torch.Generator().manual_seed(11)
    x = operands(T, H, H, dk, dv, g, "mild", False)
    cu, ctx, slots, state = torch.tensor([0, T]).int(), torch.tensor([T]).int(), torch.tensor([0]).int(), torch.zeros(1, H, dv, dk)
    want, want_state = scan(x, state, slots, cu, ctx, H, H, dk, dv, T, False)
    x[field][at, 1, 5] = value
    got, got_state = scan(x, state, slots, cu, ctx, H, H, dk, dv, T, False)
    close = dict(rtol=1e-5, atol=1e-5 * want.abs().max().item())
    torch.testing.assert_close(got[:at], want[:at], **close)
    torch.testing.assert_close(got[:, 0], want[:, 0], **close)
    torch.testing.assert_close(got_state[0, 0], want_state[0, 0], **close)
    assert not got[at, 1].isfinite().all()
    if field == "v":
        keep = [c for c in range(dv) if c != 5]
        torch.testing.assert_close(got[:, 1][:, keep], want[:, 1][:, keep], **close)


@pytest.mark.parametrize("read_first", [False, True])
@pytest.mark.parametrize("H,G,dk,dv,scalar,lens", [(2, 2, 64, 24, False, [1, 555]), (2, 1, 128, 40, True, [513, 2]), (1, 1, 256, 64, False, [600, 3]),
                                                   (2, 2, 48, 40, False, [300, 70, 512]), (2, 1, 256, 32, True, [9, 300]),
                                                   (16, 16, 16, 16, False, [512, 256, 600, 9, 512, 512, 255, 512])])
def test_segments(H, G, dk, dv, scalar, lens, read_first):
    """Head sizes without a chunked form, and one with it whose heads fill the chip: portions of 256 tokens and more in four segments, in eight where the
    longest has 512, beside shorter ones; fresh and carried.  The bound is eight times what the token-by-token form is off, and 1e-6 of the largest
    value."""
    from nanovllm import _hip, ops
    assert _hip.lib().nvh_scan_segmentable(dk)
    crowded = 64 * sum(lens) * H > ops.SCAN_CHUNK_HEADS * dk * max(lens)
    assert crowded or not _hip.lib().nvh_scan_chunk_workspace_bytes(sum(lens), len(lens), H, dk, dv)
    assert max(lens) >= ops.SCAN_SEGMENT_MIN_TOKENS and len(lens) <= ops.SCAN_SEGMENT_MAX_BATCH
    g = torch.Generator().manual_seed(dk + dv)
    T, B, plain = sum(lens), len(lens), dk == 48
    x = operands(T, H, G, dk, dv, g, "slow", scalar)
    state = torch.randn(B + 1, H, dv, dk, generator=g)
    slots, cu, carried = torch.randperm(B + 1, generator=g)[:B].int(), torch.tensor([0] + lens).cumsum(0).int(), [4 * (b % 2 == 0) for b in range(B)]
    ctx = torch.tensor([n + c for n, c in zip(lens, carried)]).int()
    serial, serial_state = scan(x, state, slots, cu, ctx, H, G, dk, dv, 0, read_first, plain)
    got, got_state = scan(x, state, slots, cu, ctx, H, G, dk, dv, max(lens), read_first, plain)
    y = full(x, H, G, dk, plain)
    for b, n in enumerate(lens):
        at, s = int(cu[b]), int(slots[b])
        want, end = recurrence({m: t if m in ("skip", "bonus") else t[at:at + n] for m, t in y.items()},
                               state[s].double() if carried[b] else torch.zeros(H, dv, dk, dtype=torch.float64), read_first)
        for a, c, z in ((got[at:at + n], serial[at:at + n], want), (got_state[s], serial_state[s], end)):
            assert torch.equal(a, c) == (n < ops.SCAN_SEGMENT_MIN_TOKENS), (b, n)      # (long ones round differently: they were cut)
            assert (a.double() - z).abs().max() <= 8 * (c.double() - z).abs().max() + 1e-6 * z.abs().max(), (b, n)


@pytest.mark.parametrize("extra", [1, 9, 15])
def test_infinite_values_in_the_last_chunk(extra):
    """Infinite values at the last token of a portion that ends within a chunk: the state becomes infinite or not finite exactly where it does token by
    token, and with the same signs; everything else stays as it is."""
    H, dk, dv, T = 2, 64, 32, MIN + extra
    g = torch.Generator().manual_seed(extra)
    x = operands(T, H, H, dk, dv, g, "mild", False)
    cu, ctx, slots, state = torch.tensor([0, T]).int(), torch.tensor([T]).int(), torch.tensor([0]).int(), torch.zeros(1, H, dv, dk)
    x["v"][T - 1, 1, 5], x["v"][T - 1, 0, 7] = float("inf"), float("-inf")
    want, want_state = scan(x, state, slots, cu, ctx, H, H, dk, dv, 0, False)
    got, got_state = scan(x, state, slots, cu, ctx, H, H, dk, dv, T, False)
    assert want_state.isinf().sum() == 2 * dk and not want_state.isnan().any()
    torch.testing.assert_close(got_state, want_state, rtol=1e-5, atol=1e-5 * want_state[want_state.isfinite()].abs().max().item())
    assert torch.equal(got.isfinite(), want.isfinite())
    torch.testing.assert_close(got[want.isfinite()], want[want.isfinite()], rtol=1e-5, atol=1e-5 * want[want.isfinite()].abs().max().item())


def test_cuts_at_whole_chunks():
    """A portion cut at a multiple of 16 tokens into two that are chunked: the same bits."""
    H, dk, dv, T, cut = 2, 64, 64, 3 * MIN + 5, MIN + 16
    g = torch.Generator().manual_seed(5)
    x, state = operands(T, H, H, dk, dv, g, "mild", False), torch.randn(1, H, dv, dk, generator=g)
    part = lambda lo, hi: {m: t if m in ("skip", "bonus") else t[lo:hi] for m, t in x.items()}
    slots, at = torch.tensor([0]).int(), lambda *n: torch.tensor(n).int()
    whole, whole_state = scan(x, state, slots, at(0, T), at(T + 1), H, H, dk, dv, T, False)
    one, mid = scan(part(0, cut), state, slots, at(0, cut), at(cut + 1), H, H, dk, dv, cut, False)
    two, end = scan(part(cut, T), mid, slots, at(0, T - cut), at(T + 1), H, H, dk, dv, T - cut, False)
    assert torch.equal(torch.cat([one, two]), whole) and torch.equal(end, whole_state)
