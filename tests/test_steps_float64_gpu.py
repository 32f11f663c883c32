"""Rotary preparation, closes, one-token recurrences and the operands of the convolutions against their formulas in float64, in the forms for
aligned rows and in those for any: their tests against each other show that the forms agree, these that both are right."""
import pytest
import torch

import test_delta_chunk_gpu as D

pytestmark = pytest.mark.gpu
U = 2.0 ** -24                                               # half a unit of fp32


def rounding(dtype):
    return 2.0 ** -8 if dtype is torch.bfloat16 else 2 * U    # of a result on its way out


def odd_rows(t):
    wide = torch.empty(t.shape[0], t.shape[1] + 1, dtype=t.dtype, device=t.device)
    wide[:, :-1] = t
    return wide[:, :-1]


def turn(x, angle, inter, mag=1.0):
    """Pairs of x [T, heads, n] rotated by angle [T, n / 2], times mag: neighbours, or element i and i + n / 2."""
    n = x.shape[-1]
    a, b = (x[..., 0::2], x[..., 1::2]) if inter else (x[..., :n // 2], x[..., n // 2:])
    c, s = mag * angle.cos()[:, None], mag * angle.sin()[:, None]
    a, b = a * c - b * s, b * c + a * s
    return torch.stack([a, b], -1).flatten(-2) if inter else torch.cat([a, b], -1)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("norm", ["none", "row", "head"])
@pytest.mark.parametrize("H,G,dim,vdim,rot,inter,turns,v_inter", [(2, 1, 16, 16, 16, False, True, False), (16, 8, 128, 128, 64, True, False, False), (8, 8, 128, 64, 128, False, True, False),
                                                                  (4, 2, 40, 24, 32, False, True, True), (4, 4, 32, 16, 0, False, False, False)])
@pytest.mark.parametrize("T", [3, 150])
def test_rotary_prep(T, H, G, dim, vdim, rot, inter, turns, v_inter, norm, dtype):
    """q, k after norm and rotation, v turned, the gate.  Bound: half of n roundings and eight for a norm over n squares; eight of its pair's size for a
    rotation, whose sines and cosines are off by 2^-20 (fp32) or, from the hardware (bf16), 2^-12; and the result's own rounding."""
    from nanovllm import ops
    g = torch.Generator().manual_seed(T + H * dim)
    nq, nk, nv, page = H * dim, G * dim, G * vdim, 32
    row = torch.randn(T, -(-(nq + nk + nv + H) // 8) * 8, generator=g).to(dtype).cuda()
    slots = (torch.randperm(5 * page, generator=g)[:T] + page).int().cuda()
    positions = torch.randint(0, 900, (T,), generator=g).cuda()
    w = [None, None] if norm == "none" else [(torch.rand(n, generator=g) + 0.5).to(dtype).cuda() for n in ((nq, nk) if norm == "row" else (dim, dim))]
    freq = torch.rand(rot // 2, generator=g).cuda() if rot else None
    vfreq = torch.rand(vdim // 2, generator=g).cuda() if turns else None

    def part(lo, n, d):
        return row[:, lo:lo + n].double().view(T, -1, d)

    def angle(f):                                            # (position times frequency is an fp32 number)
        return (positions.float()[:, None] * f).double()
    want, sizes = [], []
    for x, wn in ((part(0, nq, dim), w[0]), (part(nq, nk, dim), w[1])):
        if norm != "none":
            ms = (x * x).mean((1, 2) if norm == "row" else 2, keepdim=True)
            x = x / (ms + 1e-5).sqrt() * (wn.double().view(1, -1, dim) if norm == "row" else wn.double())
        size = x.abs()
        if rot:
            size[..., :rot] = 2.2 * size[..., :rot].amax(-1, keepdim=True)
            x = torch.cat([turn(x[..., :rot], angle(freq), inter, 1.1), x[..., rot:]], -1)
        want.append(x)
        sizes.append(size)
    v = part(nq + nk, nv, vdim)
    vsize = v.abs().amax(-1, keepdim=True) * 2
    if turns:
        v = turn(v, angle(vfreq), v_inter)
    sine = 2.0 ** -20 if dtype is torch.float32 else 2.0 ** -12
    n = max(nq, dim) if norm == "row" else dim
    for src in (row, odd_rows(row)):
        kc, vc = torch.zeros(6, page, G, dim, dtype=dtype, device="cuda"), torch.zeros(6, G, vdim, page, dtype=dtype, device="cuda")
        q, gate = ops.attn_rotary_prep(src[:, :nq + nk + nv + H], w[0], w[1], 1e-5, positions, freq, 1.1, rot, vfreq, kc, vc, slots, H, G, dim, vdim, True, inter, v_inter,
                                       norm_per_head=norm == "head")
        at = slots.long()
        k, got_v = kc.view(-1, G, dim)[at], vc.permute(0, 3, 1, 2).reshape(-1, G, vdim)[at]
        for a, b, size in ((q.view(T, H, dim), want[0], sizes[0]), (k, want[1], sizes[1])):
            slack = (n / 2 + 8) * U * b.abs() + ((sine if rot else 0) + 8 * U) * size
            assert ((a.double() - b).abs() <= slack + rounding(dtype) * (b.abs() + slack)).all()
        slack = (sine + 8 * U if turns else 0) * vsize
        assert ((got_v.double() - v).abs() <= slack + rounding(dtype) * v.abs()).all()
        assert ((gate.double() - torch.sigmoid(row[:, nq + nk + nv:nq + nk + nv + H].double())).abs() <= 8 * U).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,dim", [(3, 64), (5, 1020), (64, 1024), (3, 1028), (2, 4100), (1, 8192)])
def test_closes(rows, dim, dtype):
    """The three closes.  A row's statistics are sums of `dim` terms; their relative error is below (dim / 2 + 8) roundings, as is that of what they scale."""
    from nanovllm import ops
    g = torch.Generator().manual_seed(rows * dim)

    def t(*shape):
        return torch.randn(*shape, generator=g).to(dtype).cuda()
    a, b, c, w1, w2, w3, w4 = t(rows, dim), t(rows, dim), t(rows, dim), t(dim), t(dim), t(dim), t(dim)
    c32, x = torch.randn(rows, dim, generator=g).cuda(), torch.randn(rows, dim, generator=g).cuda()
    A, B, C, W1, W2, W3, W4, C32, X = (v.double() for v in (a, b, c, w1, w2, w3, w4, c32, x))

    def unit(v, eps):
        return v / (v.pow(2).mean(1, keepdim=True) + eps).sqrt()
    summed = X + 0.5 * (unit(A, 1e-6) * W1 + unit(B, 1e-6) * W2) + C + C32
    centred = summed - summed.mean(1, keepdim=True)
    post = unit(2.0 * X + W2 * (A + C32), 1e-6) * (1.0 + W1)
    sub = X + 0.5 * W1[:1] * unit(0.6 * A + 0.9 * B + C32, 1e-6)
    cases = [(ops.residual_norm, dict(a=a, a_weight=w1, b=b, b_weight=w2, branch_scale=0.5, branch_eps=1e-6, c=c, c32=c32, norm="layer", weight=w3, bias=w4, eps=1e-5), summed,
              unit(centred, 1e-5) * W3 + W4),
             (ops.residual_norm, dict(c=c, norm="rms", weight=w3, eps=1e-5), X + C, unit(X + C, 1e-5) * W3),
             (ops.residual_postnorm, dict(weight=w1, eps=1e-6, y=a, y32=c32, layer_scale=w2, alpha=2.0, weight_offset=1.0), post, post),
             (ops.residual_subnorm, dict(weight=w1[:1], eps=1e-6, mult=0.5, a=a, a_scale=0.6, b=b, b_scale=0.9, c32=c32), sub, sub)]
    for odd in (False, True):
        for op, kw, want_x, want_h in cases:
            got = x.clone()
            h = op(got, **{n: odd_rows(v) if odd and torch.is_tensor(v) and v.dim() == 2 else v for n, v in kw.items()})
            for out, want, last in ((got, want_x, 2 * U), (h, want_h, rounding(dtype))):
                slack = (dim / 2 + 8) * U * (want.abs() + want.pow(2).mean(1, keepdim=True).sqrt() * 4)
                assert ((out.double() - want).abs() <= slack + last * want.abs()).all()


@pytest.mark.parametrize("read_first,scalar", [(False, False), (False, True), (True, False)])
@pytest.mark.parametrize("B,H,G,dk,dv", [(3, 2, 1, 64, 24), (5, 4, 2, 128, 72), (33, 8, 8, 128, 128), (3, 2, 2, 256, 40), (3, 2, 2, 48, 20)])
def test_one_token_of_the_gated_scan(B, H, G, dk, dv, read_first, scalar):
    from nanovllm import ops
    g = torch.Generator().manual_seed(B + dk + dv)
    slots, ctx = torch.randperm(B + 2, generator=g)[:B].int(), torch.randint(2, 900, (B,), generator=g).int()
    ctx[2] = 1                                               # (starts here)
    q, k, v = torch.randn(B, G * dk, generator=g), torch.randn(B, G * dk, generator=g), torch.randn(B, H * dv, generator=g)
    w, state = torch.rand(B, H if scalar else H * dk, generator=g), torch.randn(B + 2, H, dv, dk, generator=g)
    ks, skip, bonus = torch.rand(B, H, generator=g), torch.randn(H, generator=g), torch.randn(H * dk, generator=g)
    S = state[slots.long()].double()
    S[2] = 0
    Q, K = (x.double().view(B, G, 1, dk).repeat_interleave(H // G, 1) for x in (q, k))
    V, W = v.double().view(B, H, dv, 1), w.double().view(B, H, 1, 1 if scalar else dk)
    kv = K * (ks.double().view(B, H, 1, 1) * V)
    new = W * S + kv
    read = S + bonus.double().view(1, H, 1, dk) * kv if read_first else new
    want = (read * Q).sum(-1) + skip.double().view(1, H, 1) * V[..., 0]
    size = (((W * S).abs() + S.abs() + (1 + bonus.abs().max()) * kv.abs()) * Q.abs()).sum(-1) + (skip.double().view(1, H, 1) * V[..., 0]).abs()
    st = state.cuda()
    out = ops.gated_linear_scan(q.cuda(), k.cuda(), w.cuda(), v.cuda(), st, slots.cuda(), None, ctx.cuda(), H, dk, dv, qk_groups=G, kscale=ks.cuda(), skip=skip.cuda(),
                                read_first=read_first, bonus=bonus.cuda() if read_first else None)
    assert ((out.cpu().double().view(B, H, dv) - want).abs() <= (dk + 8) * U * size).all()       # (at most dk sums and eight roundings of a term)
    assert ((st.cpu()[slots.long()].double() - new).abs() <= 4 * U * ((W * S).abs() + kv.abs())).all()


@pytest.mark.parametrize("B,H,dk,dv", [(3, 2, 64, 36), (5, 3, 128, 72), (33, 16, 128, 128), (3, 2, 256, 64), (3, 2, 64, 30), (2, 3, 48, 16)])
def test_one_token_of_the_delta_rule(B, H, dk, dv):
    g = torch.Generator().manual_seed(B + dk + dv)
    rows, state = torch.randn(B, H, 5 * dk + dv, generator=g) * 0.3, torch.randn(B + 2, H, dk, dv, generator=g)
    slots, ctx = torch.randperm(B + 2, generator=g)[:B].int(), torch.randint(2, 900, (B,), generator=g).int()
    ctx[1] = 1
    from nanovllm import ops
    st = state.cuda()
    out = ops._delta_scan(rows.cuda(), st, slots.cuda(), None, ctx.cuda(), H, dk, dv, 1).cpu().double().view(B, H, dv)
    for b in range(B):
        S = state[slots[b]].double() * (0 if b == 1 else 1)
        want, new = D.recurrence(rows[b:b + 1].double(), dk, S)
        r, k, w, u, au, v = rows[b].double().split([dk] * 5 + [dv], 1)
        uS = (u[:, :, None] * S).abs().sum(1)
        size = (w[:, :, None] * S).abs() + au[:, :, None].abs() * uS[:, None] + (k[:, :, None] * v[:, None]).abs()
        assert ((st[slots[b]].cpu().double() - new).abs() <= (dk + 8) * U * size).all()          # (u^T S: dk sums)
        assert ((out[b] - want[0]).abs() <= (2 * dk + 8) * U * (r[:, :, None].abs() * size).sum(1)).all()


def conv(rows, state, w, carried):
    """Causal convolution of one sequence's rows [n, c] with w [c, taps], from state [taps - 1, c] or zeros; and the sizes of the terms."""
    taps, n = w.shape[1], rows.shape[0]
    seq = torch.cat([state if carried else torch.zeros_like(state), rows])
    return (sum(seq[k:k + n] * w[:, k] for k in range(taps)), sum((seq[k:k + n] * w[:, k]).abs() for k in range(taps)), seq[n:])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("taps,heads,inner,gn", [(4, 2, 64, 16), (2, 3, 48, 8), (3, 1, 20, 7), (5, 2, 32, 8)])
def test_ssd_step(taps, heads, inner, gn, dtype):
    """silu(z) of a sum of taps + 1 terms: its slope is at most 1.1; dt and decay are a few fp32 functions of numbers of some units."""
    from nanovllm import ops
    g = torch.Generator().manual_seed(taps * inner)
    B, c = 6, inner + 2 * gn

    def t(*shape):
        return torch.randn(*shape, generator=g).to(dtype)
    xbc, dt, w, bias, dtb, al = t(B, c), t(B, heads), t(c, taps), t(c), t(heads), t(heads)
    state = torch.randn(B + 1, taps - 1, c, generator=g)
    slots, ctx = torch.tensor([3, 0, 6, 5, 1, 2]).int(), torch.tensor([1, 4, 3, 1, 99, 3]).int()
    st = state.cuda()
    ox, ob, oc, odt, odecay = ops.ssd_conv_prep(*(v.cuda() for v in (xbc, dt, w, bias, dtb, al)), st, slots.cuda(), None, ctx.cuda(), heads, inner, gn)
    got = torch.cat([ox, ob, oc], 1).cpu().double()
    for b in range(B):
        z, size, new = conv(xbc[b:b + 1].double(), state[slots[b]].double(), w.double(), int(ctx[b]) > 1)
        z, size = z[0] + bias.double(), size[0] + bias.double().abs()
        assert ((got[b] - z * torch.sigmoid(z)).abs() <= 1.1 * (taps + 2) * U * size + 16 * U * z.abs()).all()
        assert torch.equal(st[slots[b]].cpu(), new.float())
    step = torch.nn.functional.softplus(dt.double() + dtb.double())
    assert ((odt.cpu().double() - step).abs() <= 16 * U * step.clamp(min=1)).all()
    rate = al.double().exp()
    assert ((odecay.cpu().double() - (-rate * step).exp()).abs() <= 16 * U * (1 + rate * step)).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("taps,heads,groups,dk,dv", [(4, 16, 8, 64, 32), (2, 16, 16, 20, 24), (3, 8, 2, 128, 128), (5, 16, 8, 16, 16)])
def test_delta_operands(taps, heads, groups, dk, dv, dtype):
    """q / |q| sqrt(dk), k / |k|, beta, decay and their products for runs of tokens.  A norm is off by at most what its terms are, relatively to their sizes."""
    from nanovllm import ops
    g = torch.Generator().manual_seed(taps * dk)
    lens, carried = [5, 1, 300, 2], [0, 4, 3, 0]
    T, c, nqk = sum(lens), 2 * groups * dk + heads * dv, groups * dk

    def t(*shape):
        return torch.randn(*shape, generator=g).to(dtype)
    qkv, b, a, w, dtb, al = t(T, c), t(T, heads), t(T, heads), t(c, taps), t(heads), t(heads)
    state, cu = torch.randn(len(lens), taps - 1, c, generator=g), torch.tensor([0] + lens).cumsum(0).int()
    slots, ctx = torch.tensor([2, 0, 3, 1]).int(), torch.tensor([n + p for n, p in zip(lens, carried)]).int()
    out = torch.empty(T, heads, 5 * dk + dv, device="cuda")
    dev = [v.cuda() for v in (qkv, b, a, w, dtb, al, state, slots, cu, ctx)]
    ops._hip.call("nvh_gated_delta_prep", dev[0].data_ptr(), c, dev[1].data_ptr(), heads, dev[2].data_ptr(), heads, *(v.data_ptr() for v in dev[3:]), out.data_ptr(),
                  len(lens), T, taps, heads, groups, dk, dv, int(dtype is torch.float32), ops._stream())
    parts = [conv(qkv[lo:lo + n].double(), state[s].double(), w.double(), p) for lo, n, s, p in zip(cu.tolist(), lens, slots.tolist(), carried)]
    z, size = torch.cat([p[0] for p in parts]), torch.cat([p[1] for p in parts])
    y, off = z * torch.sigmoid(z), 1.1 * (taps + 1) * U * size + 16 * U * z.abs()

    def heads_of(x, lo):
        return x[:, lo:lo + nqk].view(T, groups, dk).repeat_interleave(heads // groups, 1)
    beta = torch.sigmoid(b.double())[..., None]
    dec = (-al.double().exp() * torch.nn.functional.softplus(a.double() + dtb.double())).exp()[..., None]
    dec_off = 16 * U * (1 + (al.double().exp() * torch.nn.functional.softplus(a.double() + dtb.double())))[..., None]
    got = out.cpu().double().split([dk] * 5 + [dv], 2)
    units = []
    for lo, scale in ((0, dk ** -0.5), (nqk, 1.0)):
        x, d = heads_of(y, lo), heads_of(off, lo)
        length = (x.pow(2).sum(-1, keepdim=True) + 1e-6).sqrt()
        slack = d / length + x.abs() / length * (d.norm(dim=-1, keepdim=True) / length + (dk / 2 + 8) * U)
        units.append((x / length * scale, slack * scale))
    (q, dq), (k, dk_off) = units
    v, dv_off = y[:, 2 * nqk:].view(T, heads, dv), off[:, 2 * nqk:].view(T, heads, dv)
    for x, want, slack in ((got[0], q, dq), (got[1], beta * k, beta * dk_off + 16 * U * k.abs()), (got[2], dec.expand_as(k), dec_off), (got[3], k, dk_off),
                           (got[4], beta * dec * k, beta * dec * dk_off + (16 * U + dec_off) * k.abs()), (got[5], v, dv_off)):
        assert ((x - want).abs() <= slack).all()


@pytest.mark.parametrize("dk,dv", [(16, 16), (32, 32), (48, 16), (64, 32), (96, 48), (128, 16)])
def test_chunk_counts(dk, dv):
    """Sequences of 8 to 17 chunks in one call, so that every remainder of the records in flight and both parities of the shared places end a sequence: outputs
    and states as near to float64 as eight times the token-by-token form's distance."""
    H, lens = 3, [D.MIN + 16 * j + (5 if j % 3 == 1 else 0) for j in range(10)]
    g = torch.Generator().manual_seed(dk + dv)
    rows, state = D.pack(sum(lens), H, dk, dv, g, "mild"), torch.randn(len(lens), H, dk, dv, generator=g)
    slots, cu, ctx = torch.randperm(len(lens), generator=g).int(), torch.tensor([0] + lens).cumsum(0).int(), torch.tensor([n + 3 for n in lens]).int()
    serial = D.scan(rows, state, slots, cu, ctx, H, dk, dv, 0)
    got = D.scan(rows, state, slots, cu, ctx, H, dk, dv, max(lens))
    assert not torch.equal(got[0], serial[0])                # (another form did run)
    for b, n in enumerate(lens):
        lo, s = int(cu[b]), int(slots[b])
        want, end = D.recurrence(rows[lo:lo + n].double(), dk, state[s].double())
        for x, y, z in ((got[0][lo:lo + n], serial[0][lo:lo + n], want), (got[1][s], serial[1][s], end)):
            assert (x.double() - z).abs().max() <= 8 * (y.double() - z).abs().max() + 1e-6 * z.abs().max(), (b, n)
