"""Decode attention with 1 .. 8 query heads a kv head: trips that the new token opens, ends or lies inside, ranges, pages that hold no numbers behind a
context's end; against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CTX = [1, 2, 15, 16, 17, 63, 64, 65, 66, 127, 128, 129, 192, 193, 255, 256, 257, 320, 321, 700]


def rope_head(x, w, cs, eps):
    """The q/k epilogue at its rounding points: norm -> bf16, times weight -> bf16, rotated halves -> bf16."""
    n = (x.float() / torch.sqrt((x.float() ** 2).mean(-1, keepdim=True) + eps)).bfloat16().float()
    n = (n * w.float()).bfloat16().float()
    cos, sin = cs[..., :64], cs[..., 64:]
    a, b = n[..., :64], n[..., 64:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1).bfloat16()


@pytest.mark.parametrize("splits", [1, 5])
@pytest.mark.parametrize("group", [1, 2, 4, 5, 8])
def test_new_token_and_edges(group, splits):
    from nanovllm import ops
    hkv, hq, eps = 2, 2 * group, 1e-6
    g = torch.Generator().manual_seed(group * 10 + splits)
    b, width = len(CTX), 3
    tables = torch.randperm(b * width, generator=g).int().view(b, width)
    kc, vc = (torch.randn(b * width, 256, hkv, 128, generator=g).bfloat16() for _ in range(2))
    for i, n in enumerate(CTX):                              # what a page held before is no number at all, from the new token's own place on
        for page in range(width):
            first = max(0, n - 1 - 256 * page)
            kc[tables[i, page].long(), first:] = vc[tables[i, page].long(), first:] = float("nan")
    qkv = torch.randn(b, (hq + 2 * hkv) * 128, generator=g).bfloat16()
    qw, kw = (torch.rand(128, generator=g).bfloat16() + 0.5 for _ in range(2))
    cs = torch.randn(1024, 128, generator=g)
    pos = torch.tensor(CTX) - 1
    kg, vg = kc.cuda(), vc.cuda()
    got = ops.attn_decode_fused_qkv(qkv.cuda(), hq, hkv, qw.cuda(), kw.cuda(), eps, pos.cuda(), cs.cuda(), kg, vg, torch.tensor(CTX, dtype=torch.int32).cuda(), tables.cuda(),
                                    128 ** -0.5, splits).cpu().double()
    heads = qkv.view(b, hq + 2 * hkv, 128)
    q, k_new = rope_head(heads[:, :hq], qw, cs[pos][:, None], eps), rope_head(heads[:, hq:hq + hkv], kw, cs[pos][:, None], eps)
    for i, n in enumerate(CTX):
        t = tables[i].long()
        k, v = kc[t].reshape(-1, hkv, 128)[:n].clone(), vc[t].reshape(-1, hkv, 128)[:n].clone()
        k[n - 1], v[n - 1] = k_new[i], heads[i, hq + hkv:]
        for cache, new in ((kg, k[n - 1]), (vg, v[n - 1])):
            # (a rounding of the norm apart at most: one unit of bf16)
            assert ((cache[t[(n - 1) // 256], (n - 1) % 256].cpu().double() - new.double()).abs() <= new.double().abs() * 2.0 ** -7 + 1e-6).all()
        k, v = (x.double().repeat_interleave(group, 1) for x in (k, v))
        w = torch.softmax((k * q[i].double()).sum(-1) * 128 ** -0.5, 0)
        want = (w[:, :, None] * v).sum(0)
        scale = (w[:, :, None] * v.abs()).sum(0)
        # the result's own rounding, and scores of fp32 sums over bf16 products with inputs up to a rounding apart
        assert ((got[i] - want).abs() <= want.abs() * 2.0 ** -8 + scale * 0.03).all(), n
        assert ((got[i] - want).norm() / want.norm()) < 0.01, n
    plain = ops.attn_decode(q.cuda(), kg, vg, torch.tensor(CTX, dtype=torch.int32).cuda(), tables.cuda(), 128 ** -0.5, splits).cpu().double()
    assert ((plain - got).norm() / got.norm()) < 0.01


@pytest.mark.parametrize("splits", [1, 5])
@pytest.mark.parametrize("group", [1, 2, 4, 5, 8])
def test_weights_in_fp32(group, splits):
    """Two keys of a context carry its weights and their values nearly cancel, so that the result shows the weights to more than 16 bits."""
    from nanovllm import ops
    hkv, hq, scale = 2, 2 * group, 128 ** -0.5
    g = torch.Generator().manual_seed(100 + group * 10 + splits)
    ctxs = [2, 17, 64, 65, 130, 257, 700]
    b, width = len(ctxs), 3
    tables = torch.randperm(b * width, generator=g).int().view(b, width)
    u = (torch.randn(b, hkv, 128, generator=g) * 1.2).bfloat16()
    q = u[:, :, None].expand(b, hkv, group, 128).reshape(b, hq, 128).contiguous()
    kc = torch.zeros(b * width, 256, hkv, 128, dtype=torch.bfloat16)
    vc = torch.randn(b * width, 256, hkv, 128, generator=g).bfloat16()
    wants, seen = [], [0, 0]
    for i, n in enumerate(ctxs):
        t = tables[i].long()
        k, v = (-2.0 * u[i].float()).bfloat16()[None].repeat(n, 1, 1), vc[t].reshape(-1, hkv, 128)[:n].clone()      # (weights of e^-40 and less)
        one, two = (int(x) for x in torch.randperm(n, generator=g)[:2])
        k[one] = (u[i].float() * (0.9 + 0.1 * torch.rand(hkv, 1, generator=g))).bfloat16()
        k[two] = (u[i].float() * (0.9 + 0.1 * torch.rand(hkv, 1, generator=g))).bfloat16()
        s = (k.double() * u[i].double()).sum(-1) * scale
        w = torch.softmax(s, 0)
        v[two] = (-v[one].double() * (w[one] / w[two])[:, None]).bfloat16()
        for p in range(width):
            part = slice(256 * p, min(n, 256 * (p + 1)))
            kc[t[p], :max(0, part.stop - part.start)], vc[t[p], :max(0, part.stop - part.start)] = k[part], v[part]
        want, mass = (w[:, :, None] * v.double()).sum(0), (w[:, :, None] * v.double().abs()).sum(0)
        # the result's rounding, and two weights from scores that carry 130 roundings of fp32
        bound = want.abs() * 2.0 ** -8 + mass * 2 * ((w * s.abs()).sum(0)[:, None] + 4) * 130 * 2.0 ** -24
        wants.append((want, bound))
        for kind, coarse in enumerate((w.bfloat16().double(), torch.softmax(s.bfloat16().double(), 0))):     # what the bound is to see: weights, scores of 16 bits
            coarse = coarse / coarse.sum(0)
            seen[kind] += bool((((coarse[:, :, None] * v.double()).sum(0) - want).abs() > bound).any())
    assert min(seen) >= 4, seen
    got = ops.attn_decode(q.cuda(), kc.cuda(), vc.cuda(), torch.tensor(ctxs, dtype=torch.int32).cuda(), tables.cuda(), scale, splits).cpu().double()
    for i, (want, bound) in enumerate(wants):
        err = (got[i].view(hkv, group, 128) - want[:, None]).abs()
        assert (err <= bound[:, None]).all(), (ctxs[i], (err / bound[:, None]).max().item())


def ulp(x):
    return torch.exp2(torch.floor(torch.log2(x.abs())) - 23)


@pytest.mark.parametrize("group", [1, 2, 4, 5, 8])
def test_scores_are_summed_in_pairs(group):
    """A score's 128 products add up by halves: over many pairs of keys the weights' 2-norm error is what the roundings of such a sum and of the scaled score leave.
    (A running sum in four steps, each rounded at up to its full size, has 1.5 times that.)"""
    from nanovllm import ops
    hkv, hq, scale, b = 2, 2 * group, 128 ** -0.5, 600
    g = torch.Generator().manual_seed(group)
    u = (torch.randn(b, hkv, 128, generator=g) * 1.2).bfloat16()
    k = (u.float()[:, None] * (0.9 + 0.1 * torch.rand(b, 2, hkv, 1, generator=g))).bfloat16()
    d = (k.double() * u.double()[:, None]).sum(-1)           # [b, 2, hkv], some 175
    w = torch.softmax(d * scale, 1)
    v = torch.randn(b, 2, hkv, 128, generator=g).bfloat16()
    v[:, 1] = (-v[:, 0].double() * (w[:, 0] / w[:, 1])[..., None]).bfloat16()          # the values nearly cancel: what is left shows the weights
    kc = torch.zeros(b, 256, hkv, 128, dtype=torch.bfloat16, device="cuda")
    vc = torch.zeros_like(kc)
    kc[:, :2], vc[:, :2] = k.cuda(), v.cuda()
    q = u[:, :, None].expand(b, hkv, group, 128).reshape(b, hq, 128).contiguous()
    got = ops.attn_decode(q.cuda(), kc, vc, torch.full((b,), 2, dtype=torch.int32).cuda(), torch.arange(b).int().view(b, 1).cuda(), scale, 1).cpu().double().view(b, hkv, group, 128)
    want, mass = (w[..., None] * v.double()).sum(1), (w[..., None] * v.double().abs()).sum(1)
    # (where the result itself is rounded at below 2^-23 of the mass)
    err = ((got - want[:, :, None]) / mass[:, :, None])[(want.abs() < mass * 2.0 ** -14)[:, :, None].expand(-1, -1, group, -1)]
    # variances in units of log2: the product with the scale, then 1, 2, 4 and 8 sums of halves, quarters ..; the result moves by half of the scores' difference
    log2e = 1.4426950408889634
    var = ulp(d * scale * log2e) ** 2 + sum(2.0 ** j * (ulp(d / 2 ** j) * scale * log2e) ** 2 for j in range(4))
    bound = ((var / 12).sum(1).mean() ** 0.5 / log2e / 2).item()
    assert err.numel() > 3000 and (err ** 2).mean().item() ** 0.5 < 1.2 * bound, ((err ** 2).mean().item() ** 0.5, bound)
