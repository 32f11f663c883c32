"""bf16 paged attention of any head size: one-token steps whose sequences are dealt out by length."""
import pytest
import torch

pytestmark = pytest.mark.gpu
PAGE = 256


def caches(g, ctx, G, dim, vdim):
    pages = [-(-c // PAGE) for c in ctx]
    order, table, at = torch.randperm(sum(pages) + 1, generator=g).int(), torch.full((len(ctx), max(max(pages), 1)), -1, dtype=torch.int32), 0
    for b, n in enumerate(pages):
        table[b, :n] = order[at:at + n]
        at += n
    k, v = torch.randn(at + 1, PAGE, G, dim, generator=g).bfloat16(), torch.randn(at + 1, G, vdim, PAGE, generator=g).bfloat16()
    return k, v, table


def reference(q, k, v, table, ctx, past, H, G, dim, vdim, window, keep, chunk, sinks):
    """q [n, H dim] of one sequence behind `past` tokens, float64 on the CPU."""
    rows = table[:-(-ctx // PAGE)].long()
    K = k[rows].reshape(-1, G, dim)[:ctx].double()
    V = v[rows].permute(0, 3, 1, 2).reshape(-1, G, vdim)[:ctx].double()
    n = q.shape[0]
    i, j = torch.arange(past, past + n)[:, None], torch.arange(ctx)[None, :]
    seen = (j <= i)
    if window:
        seen &= (i - j < window) | (j < keep)
    if chunk:
        seen &= j >= i // chunk * chunk
    out = torch.empty(n, H, vdim, dtype=torch.float64)
    for h in range(H):
        s = (q.double().view(n, H, dim)[:, h] @ K[:, h // (H // G)].t().contiguous()) * dim ** -0.5
        s = s.masked_fill(~seen, -torch.inf)
        if sinks is not None:
            s = torch.cat([s, sinks[h].double().expand(n, 1)], 1)
        out[:, h] = torch.softmax(s, 1)[:, :ctx] @ V[:, h // (H // G)].contiguous()
    return out.view(n, H * vdim)


def close_to(got, want):
    """Weights enter with 16 bits, sums are fp32: 2^-14 of the largest value, and the result's own rounding to bf16."""
    want = want.to(got.device)
    return ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -13 * want.abs().max()).all()


@pytest.mark.parametrize("window,keep,chunk", [(0, 0, 0), (200, 5, 0), (0, 0, 128)])
@pytest.mark.parametrize("B", [33, 100, 256, 257])
def test_a_step_of_many_sequences(B, window, keep, chunk):
    """The sequences of a large batch, dealt out by length, give the bits that they give in small batches; equal lengths, one key, none."""
    from nanovllm import ops
    g = torch.Generator().manual_seed(B + window)
    H, G, dim, vdim = 16, 8, 64, 64
    ctx = torch.randint(1, 700, (B,), generator=g).tolist()
    ctx[3], ctx[7:12], ctx[20] = 0, [511] * 5, 1
    k, v, table = caches(g, ctx, G, dim, vdim)
    q = torch.randn(B, H * dim, generator=g).bfloat16().cuda()
    k, v, table, lens = k.cuda(), v.cuda(), table.cuda(), torch.tensor(ctx).int().cuda()
    kw = dict(window=window, keep_first=keep, chunk=chunk)
    got = ops.attn_paged_any(q, k, v, None, lens, table, dim ** -0.5, H, G, dim, vdim, **kw)
    n = 24                                                   # (too few to be dealt out, too many for key parts)
    for lo in range(0, B - n, n):
        assert torch.equal(ops.attn_paged_any(q[lo:lo + n].contiguous(), k, v, None, lens[lo:lo + n].contiguous(), table[lo:lo + n].contiguous(), dim ** -0.5, H, G, dim, vdim, **kw),
                           got[lo:lo + n])
    for b in (3, 20, B - 1):
        if ctx[b]:
            assert close_to(got[b:b + 1], reference(q[b:b + 1].cpu(), k.cpu(), v.cpu(), table[b].cpu(), ctx[b], ctx[b] - 1, H, G, dim, vdim, window, keep, chunk, None))
        else:
            assert (got[b] == 0).all()


@pytest.mark.parametrize("window,keep,chunk", [(0, 0, 0), (700, 5, 0), (0, 0, 640)])
@pytest.mark.parametrize("lens", ["longer", "at the line", "alike", "one long", "short"])
@pytest.mark.parametrize("B", [33, 64, 65, 128, 129])
def test_dealt_out_or_not(B, lens, window, keep, chunk):
    """Either side of the lines between which the sequences of a step are dealt out: their number, the longest one and how far they differ."""
    from nanovllm import ops
    g = torch.Generator().manual_seed(B + window + chunk)
    H, G, dim, vdim = 8, 8, 64, 64
    lo, hi = {"longer": (1, 1200), "at the line": (300, 512), "alike": (460, 600), "one long": (1, 40), "short": (1, 192)}[lens]
    ctx = torch.randint(lo, hi + 1, (B,), generator=g).tolist()
    ctx[5], ctx[B - 1] = {"longer": (0, 1281), "at the line": (513 if B & 1 else 512, 1), "alike": (600, 450 if B & 1 else 451), "one long": (0, 1100), "short": (193 if B & 1 else 192, 0)}[lens]
    k, v, table = caches(g, ctx, G, dim, vdim)
    q = torch.randn(B, H * dim, generator=g).bfloat16().cuda()
    k, v, table, dev = k.cuda(), v.cuda(), table.cuda(), torch.tensor(ctx).int().cuda()
    kw = dict(window=window, keep_first=keep, chunk=chunk)
    got = ops.attn_paged_any(q, k, v, None, dev, table, dim ** -0.5, H, G, dim, vdim, **kw)
    for at in range(0, B, 30):                               # (too few workgroups to be dealt out, too many for key parts)
        n = slice(min(at, B - 30), min(at, B - 30) + 30)
        assert torch.equal(ops.attn_paged_any(q[n].contiguous(), k, v, None, dev[n].contiguous(), table[n].contiguous(), dim ** -0.5, H, G, dim, vdim, **kw), got[n])
    for b in (0, 5, B - 1):
        if ctx[b]:
            assert close_to(got[b:b + 1], reference(q[b:b + 1].cpu(), k.cpu(), v.cpu(), table[b].cpu(), ctx[b], ctx[b] - 1, H, G, dim, vdim, window, keep, chunk, None))
        else:
            assert (got[b] == 0).all()


@pytest.mark.parametrize("H,G,dim,vdim", [(2, 1, 128, 128), (2, 2, 64, 128), (1, 1, 256, 192), (2, 2, 48, 80)])
@pytest.mark.parametrize("window,keep,chunk,sink", [(0, 0, 0, False), (100, 0, 0, True), (200, 70, 0, False), (0, 0, 192, True)])
def test_tiles_seen_whole(H, G, dim, vdim, window, keep, chunk, sink):
    """Prompts against float64; a portion behind cached tokens gives the bits of the whole prompt, whichever tiles its waves see whole."""
    from nanovllm import ops
    g = torch.Generator().manual_seed(dim + window + chunk)
    ctx = [1, 63, 64, 65, 130, 450]
    k, v, table = caches(g, ctx, G, dim, vdim)
    q = torch.randn(sum(ctx), H * dim, generator=g).bfloat16()
    sinks = torch.randn(H, generator=g) if sink else None
    kc, vc, tab = k.cuda(), v.cuda(), table.cuda()
    kw = dict(window=window, keep_first=keep, chunk=chunk, sinks=None if sinks is None else sinks.cuda())

    def run(rows, lens, ctx_lens, tables):
        cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
        return ops.attn_paged_any(rows.cuda(), kc, vc, cu, torch.tensor(ctx_lens).int().cuda(), tables.contiguous(), dim ** -0.5, H, G, dim, vdim, **kw)

    got = run(q, ctx, ctx, tab)
    lo = 0
    for b, n in enumerate(ctx):
        assert close_to(got[lo:lo + n], reference(q[lo:lo + n], k, v, table[b], n, 0, H, G, dim, vdim, window, keep, chunk, sinks)), b
        for cut in (1, 15, 16, 40, 64, 100, 127, 200, 333):
            if cut < n - 1:                                  # (one query left would be a step of another form)
                assert torch.equal(run(q[lo + cut:lo + n], [n - cut], [n], tab[b:b + 1]), got[lo + cut:lo + n]), (b, cut)
        lo += n


@pytest.mark.parametrize("H,G,dim,vdim", [(2, 1, 128, 128), (4, 2, 64, 64), (1, 1, 128, 256), (2, 1, 192, 128), (1, 1, 192, 192), (2, 1, 256, 192), (1, 1, 256, 256), (2, 1, 160, 128)])
def test_windows_that_reach_everything(H, G, dim, vdim):
    """A window, or a chunk, of more than the context leaves out nothing: the bits of the call without one, whichever form of the loop either takes."""
    from nanovllm import ops
    g = torch.Generator().manual_seed(dim + vdim)
    for lens, ctx in ([1, 63, 64, 65, 130, 450], [1, 63, 64, 65, 130, 450]), ([40, 1, 129], [333, 700, 257]), ([1] * 40, list(range(1, 800, 20))):
        k, v, table = caches(g, ctx, G, dim, vdim)
        q = torch.randn(sum(lens), H * dim, generator=g).bfloat16()
        cu = torch.tensor([0] + lens).cumsum(0).int()
        args = (k.cuda(), v.cuda(), None if max(lens) == 1 else cu.cuda(), torch.tensor(ctx).int().cuda(), table.cuda(), dim ** -0.5, H, G, dim, vdim)
        got = ops.attn_paged_any(q.cuda(), *args)
        for kw in dict(window=5000), dict(chunk=8192), dict(slopes=torch.zeros(H).cuda()):
            assert torch.equal(ops.attn_paged_any(q.cuda(), *args, **kw), got), kw
        for b in range(0, len(ctx), 3):
            lo, n = int(cu[b]), lens[b]
            assert close_to(got[lo:lo + n], reference(q[lo:lo + n], k, v, table[b], ctx[b], ctx[b] - n, H, G, dim, vdim, 0, 0, 0, None)), (lens, b)
