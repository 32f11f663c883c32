"""fp32 paged attention on the matrix cores against float64: the edges of a block of 16 keys, of a tile of four and of a query tile, every option,
and head sizes beside the ones that it is built for."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

OPTIONS = {
    "plain": {}, "window": dict(window=37, keep_first=3), "chunk": dict(chunk=50), "slopes": dict(slopes=True), "bias": dict(bias=29), "masking bias": dict(bias=29, masked=20),
    "sinks": dict(sinks=True), "softcap": dict(softcap=2.0, q_temp=(0.1, 16)), "pool": dict(window=40, pool=16), "gates": dict(gate=True, gate_elems=True),
    "all": dict(window=70, keep_first=20, slopes=True, bias=100, sinks=True, softcap=5.0, gate=True),
}


def draw(H, G, d, dv, ends, takes, page, opt, seed):
    g = torch.Generator().manual_seed(seed)
    T, B, pages = sum(takes), len(ends), sum(-(-e // page) for e in ends) + 2
    x = dict(q=torch.randn(T, H * d, generator=g), k=torch.randn(pages, page, G, d, generator=g), v=torch.randn(pages, G, dv, page, generator=g))
    order, at = torch.randperm(pages, generator=g).int(), 0
    x["tables"] = torch.zeros(B, max(1, max(-(-e // page) for e in ends)), dtype=torch.int32)
    for b, e in enumerate(ends):
        n = -(-e // page)
        x["tables"][b, :n] = order[at:at + n]
        at += n
        if e % page:                                         # what a page holds past the last key is nobody's
            x["k"][x["tables"][b, n - 1], e % page:] = float("nan")
            x["v"][x["tables"][b, n - 1], :, :, e % page:] = float("nan")
    kw = {n: opt[n] for n in ("window", "keep_first", "chunk", "softcap", "q_temp", "pool") if n in opt}
    if opt.get("slopes"):
        kw["slopes"] = torch.rand(H, generator=g) * 0.1
    if opt.get("bias"):
        kw["bias"] = torch.randn(H, opt["bias"], generator=g)
        kw["bias"][:, opt.get("masked", opt["bias"]):] = -math.inf
    if opt.get("sinks"):
        kw["sinks"] = torch.randn(H, generator=g)
    if opt.get("gate"):
        kw["gate"] = torch.rand(T, H, generator=g)
    if opt.get("gate_elems"):
        kw["gate_elems"] = torch.randn(T, H * dv, generator=g)
    if opt.get("pool"):
        rows = -(-page // opt["pool"])
        kw["pooled"] = (torch.randn(pages, rows, G, d, generator=g), torch.randn(pages, rows, G, dv, generator=g))
    return x, kw


def run(x, kw, H, G, d, dv, ends, takes, scale):
    from nanovllm import ops
    cuda = lambda t: t.cuda() if isinstance(t, torch.Tensor) else tuple(map(cuda, t)) if isinstance(t, tuple) and isinstance(t[0], torch.Tensor) else t
    cu = None if all(n == 1 for n in takes) else torch.tensor([0] + takes).cumsum(0).int().cuda()
    return ops.attn_paged_any(x["q"].cuda(), x["k"].cuda(), x["v"].cuda(), cu, torch.tensor(ends).int().cuda(), x["tables"].cuda(), scale, H, G, d, dv,
                              **{n: cuda(t) for n, t in kw.items()}).cpu()


def oracle(x, kw, H, G, d, dv, ends, takes, scale):
    """(output, bound): the bound is 64 roundings of the scores' and of the outputs' magnitudes (scores |q| |k|, through the exponential)."""
    page, T = x["k"].shape[1], sum(takes)
    out, tol, at = torch.zeros(T, H, dv, dtype=torch.float64), torch.zeros(T, H, dv, dtype=torch.float64), 0
    window, keep, chunk, cap, pool = kw.get("window", 0), kw.get("keep_first", 0), kw.get("chunk", 0), kw.get("softcap", 0.0), kw.get("pool", 0)
    for b, (e, n) in enumerate(zip(ends, takes)):
        if not e:
            at += n
            continue
        tab, keys = x["tables"][b].long(), torch.arange(e)
        K, V = x["k"].double()[tab[keys // page], keys % page], x["v"].double()[tab[keys // page], :, :, keys % page]          # [e, G, d], [e, G, dv]
        for r in range(n):
            p = e - n + r
            see = (keys <= p) & ((p - keys < window) | (keys < keep) if window else keys >= 0) & ((keys >= p // chunk * chunk) if chunk else keys >= 0)
            kk, vv, dist = K[see], V[see], p - keys[see]
            if pool and p >= window:
                blocks = torch.arange((p - window + 1) // pool)
                pi = (blocks * pool + pool - 1) // page
                row = blocks - pi * page // pool
                kk = torch.cat([kw["pooled"][0].double()[tab[pi], row], kk])
                vv = torch.cat([kw["pooled"][1].double()[tab[pi], row], vv])
            kk, vv = kk.repeat_interleave(H // G, 1), vv.repeat_interleave(H // G, 1)
            q = x["q"][at + r].double().view(H, d) * scale
            if "q_temp" in kw:
                q = q * (1 + kw["q_temp"][0] * math.log((p + 1) // kw["q_temp"][1] + 1))
            s, size = torch.einsum("hd,khd->hk", q, kk), torch.einsum("hd,khd->hk", q.abs(), kk.abs()).max().item()
            if cap:
                s = cap * torch.tanh(s / cap)
            if "slopes" in kw:
                s = s - kw["slopes"].double()[:, None] * dist
                size += kw["slopes"].max().item() * p
            if "bias" in kw:
                s = s + kw["bias"].double()[:, dist.clamp(max=kw["bias"].shape[1] - 1)]
            z = torch.cat([s, kw["sinks"].double()[:, None]], 1) if "sinks" in kw else s
            w = torch.softmax(z, 1)[:, :s.shape[1]]
            o, a = torch.einsum("hk,khv->hv", w, vv), torch.einsum("hk,khv->hv", w, vv.abs())
            if "gate" in kw:
                o, a = o * kw["gate"][at + r].double()[:, None], a * kw["gate"][at + r].double()[:, None]
            if "gate_elems" in kw:
                o = o * torch.sigmoid(kw["gate_elems"][at + r].double().view(H, dv))
            out[at + r], tol[at + r] = o, a * 64 * 2.0 ** -24 * (1 + size) + 1e-7
        at += n
    return out.view(T, -1), tol.view(T, -1)


@pytest.mark.parametrize("option", OPTIONS)
@pytest.mark.parametrize("H,G,d,dv,page", [(4, 2, 128, 128, 256), (2, 2, 64, 128, 48), (3, 1, 16, 16, 16), (2, 1, 128, 64, 64), (2, 1, 256, 192, 64), (2, 2, 80, 80, 48)])
def test_prompts(H, G, d, dv, page, option):
    ends, takes = [1, 16, 17, 63, 65, 150, 0, 129], [1, 16, 17, 40, 1, 33, 0, 129]
    x, kw = draw(H, G, d, dv, ends, takes, page, OPTIONS[option], d + len(option))
    scale = d ** -0.5
    got = run(x, kw, H, G, d, dv, ends, takes, scale)
    want, tol = oracle(x, kw, H, G, d, dv, ends, takes, scale)
    assert ((got.double() - want).abs() <= tol).all(), (got.double() - want).abs().max()


@pytest.mark.parametrize("option", OPTIONS)
@pytest.mark.parametrize("H,G,d,dv", [(4, 2, 128, 128), (40, 2, 64, 64), (16, 1, 256, 192), (3, 3, 32, 32)])
def test_one_query(H, G, d, dv, option):
    """Heads of a group as the rows, a sequence without keys among the others; and the bits of the same queries as part of longer portions."""
    ends = [1, 300, 0, 64, 65]
    takes = [1] * len(ends)
    x, kw = draw(H, G, d, dv, ends, takes, 64, OPTIONS[option], d + H)
    scale = d ** -0.5
    got = run(x, kw, H, G, d, dv, ends, takes, scale)
    want, tol = oracle(x, kw, H, G, d, dv, ends, takes, scale)
    keep = [0, 1, 3, 4]
    assert ((got.double() - want).abs() <= tol)[keep].all(), (got.double() - want).abs()[keep].max()
    assert (got[2] == 0).all()
    more = [1, 20, 0, 1, 3]                                  # (the last query of a portion is the same token)
    last = torch.tensor(more).cumsum(0) - 1
    y, wide = dict(x), {}
    y["q"] = torch.randn(sum(more), H * d)
    y["q"][last[keep]] = x["q"][keep]
    for n, t in kw.items():
        wide[n] = t
        if n in ("gate", "gate_elems"):
            wide[n] = torch.rand(sum(more), t.shape[1])
            wide[n][last[keep]] = t[keep]
    again = run(y, wide, H, G, d, dv, ends, more, scale)
    assert torch.equal(again[last[keep]], got[keep])
