"""Paged attention on the matrix cores where scores lie far from zero or at the ends of fp32's range: a weight is as exact as its distance from the row's maximum."""
import pytest
import torch

pytestmark = pytest.mark.gpu

PAGE, FAR = 64, 2.0 ** 20
LOWEST = torch.finfo(torch.float32).min
SHAPES = [(4, 2, 128, 128), (4, 4, 32, 32), (4, 2, 48, 80), (2, 1, 192, 128), (2, 2, 256, 192)]
STEPS = {"prompts": ([1, 17, 64, 130, 40], [1, 17, 64, 130, 241]), "single": ([1] * 6, [1, 16, 64, 65, 193, 900])}


def caches(ctxs, heads, groups, dim, vdim, g):
    """Page tables, keys whose products with the query of `queries` are FAR + the key's second element, and values."""
    width = max(-(-c // PAGE) for c in ctxs)
    tables = torch.randperm(len(ctxs) * width, generator=g).int().view(len(ctxs), width)
    kc = torch.zeros(len(ctxs) * width, PAGE, groups, dim)
    kc[..., 0] = FAR ** 0.5
    kc[..., 1] = torch.randint(-32, 33, kc.shape[:3], generator=g) / 8    # (FAR + a multiple of 1/8 is an fp32 number: scores carry no rounding at all)
    vc = torch.randn(len(ctxs) * width, groups, vdim, PAGE, generator=g)
    return tables, kc.bfloat16(), vc.bfloat16()


def queries(tokens, heads, dim, far=True):
    q = torch.zeros(tokens, heads, dim)
    q[..., 0], q[..., 1] = FAR ** 0.5 if far else 0.0, 1.0
    return q.reshape(tokens, heads * dim).bfloat16()


def run(lens, ctxs, q, tables, kc, vc, heads, groups, dim, vdim, **opts):
    from nanovllm import ops
    cu = None if max(lens) == 1 else torch.tensor([0] + lens).cumsum(0).int().cuda()
    return ops.attn_paged_any(q.cuda(), kc.cuda(), vc.cuda(), cu, torch.tensor(ctxs, dtype=torch.int32).cuda(), tables.cuda(), 1.0, heads, groups, dim, vdim,
                              **{n: x.cuda() for n, x in opts.items()}).cpu().double().view(-1, heads, vdim)


def rows(lens, ctxs, tables, kc, vc, heads, groups):
    """Per sequence: its rows, the keys' own part of a score, values, distances and which keys a row sees."""
    at = 0
    for b, (n, c) in enumerate(zip(lens, ctxs)):
        t = tables[b].long()
        k = kc[t].flatten(0, 1)[:c, :, 1].double().repeat_interleave(heads // groups, 1)
        v = vc[t].permute(0, 3, 1, 2).flatten(0, 1)[:c].double().repeat_interleave(heads // groups, 1)
        dist = torch.arange(c - n, c)[:, None] - torch.arange(c)[None, :]
        yield slice(at, at + n), k.t()[:, None].expand(-1, n, -1), v, dist, dist >= 0
        at += n


def close(got, w, v):
    want, mass = torch.einsum("hts,shd->thd", w, v), torch.einsum("hts,shd->thd", w, v.abs())
    # the result's rounding to bf16, and weights of 16 bits (hi + lo)
    assert ((got - want).abs() <= want.abs() * 2.0 ** -8 + mass * 2.0 ** -15).all()


@pytest.mark.parametrize("form", ["plain", "slopes", "bias", "sinks"])
@pytest.mark.parametrize("step", sorted(STEPS))
@pytest.mark.parametrize("heads,groups,dim,vdim", SHAPES)
def test_far_from_zero(heads, groups, dim, vdim, step, form):
    lens, ctxs = STEPS[step]
    g = torch.Generator().manual_seed(dim + vdim)
    tables, kc, vc = caches(ctxs, heads, groups, dim, vdim, g)
    slopes, bias, sinks = torch.full((heads,), 0.125), torch.randint(-16, 17, (heads, 50), generator=g) / 8, FAR + torch.arange(heads) * 1.0
    opts = {"slopes": dict(slopes=slopes), "bias": dict(bias=bias), "sinks": dict(sinks=sinks)}.get(form, {})
    got = run(lens, ctxs, queries(sum(lens), heads, dim), tables, kc, vc, heads, groups, dim, vdim, **opts)
    for at, x, v, dist, seen in rows(lens, ctxs, tables, kc, vc, heads, groups):
        if form == "slopes":
            x = x - 0.125 * dist
        if form == "bias":
            x = x + bias.double()[:, dist.clamp(0, 49)]
        x = x.masked_fill(~seen, -torch.inf)
        if form == "sinks":
            x = torch.cat([x, (sinks.double() - FAR)[:, None, None].expand(-1, x.shape[1], 1)], -1)
        close(got[at], torch.softmax(x, -1)[..., :v.shape[0]], v)


@pytest.mark.parametrize("step", sorted(STEPS))
@pytest.mark.parametrize("heads,groups,dim,vdim", SHAPES)
def test_ends_of_the_range(heads, groups, dim, vdim, step):
    """A bias of fp32's lowest value takes a score in (its sum is the lowest value again) and is still a number: keys that all have it weigh the same, and nothing
    beside one that has not.  A sink of the lowest value is none, one of the highest leaves nothing."""
    lens, ctxs = STEPS[step]
    g = torch.Generator().manual_seed(dim + vdim + 1)
    tables, kc, vc = caches(ctxs, heads, groups, dim, vdim, g)
    q = queries(sum(lens), heads, dim, far=False)
    near = torch.full((heads, 50), LOWEST)
    near[:, :3] = 0.0
    for opts in (dict(bias=torch.full((heads, 50), LOWEST)), dict(bias=near), dict(sinks=torch.full((heads,), LOWEST)), dict(sinks=torch.full((heads,), -LOWEST))):
        got = run(lens, ctxs, q, tables, kc, vc, heads, groups, dim, vdim, **opts)
        for at, x, v, dist, seen in rows(lens, ctxs, tables, kc, vc, heads, groups):
            if "bias" in opts:
                b = opts["bias"][:, dist.clamp(0, 49)]
                x = x.float() + b
            x = x.masked_fill(~seen, -torch.inf)
            if "sinks" in opts:
                x = torch.cat([x, opts["sinks"].double()[:, None, None].expand(-1, x.shape[1], 1)], -1)
            close(got[at], torch.softmax(x.double(), -1)[..., :v.shape[0]], v)
