"""Paged attention on the matrix cores, prompts and single queries, heads up to 256 wide: windows, chunks, slopes, caps, biases and sinks at the edges of tiles of 16
queries and 64 keys, scores far from zero; against float64."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

FORMS = {"plain": {}, "window": dict(window=70, keep_first=3), "chunk": dict(chunk=96), "slopes": dict(slopes=True), "cap": dict(softcap=20.0), "bias": dict(bias=True), "sinks": dict(sinks=True)}


def reference(q, k, v, past, scale, window=0, keep_first=0, chunk=0, slopes=None, softcap=0.0, bias=None, sinks=None):
    """[T, H, dim], [S, H, dim], [S, H, vdim] in float64 -> result and what its weights would give the values' magnitudes."""
    t, s = q.shape[0], k.shape[0]
    i, j = torch.arange(past, past + t)[:, None], torch.arange(s)[None, :]
    seen = j <= i
    if window:
        seen = seen & ((i - j < window) | (j < keep_first))
    if chunk:
        seen = seen & (i // chunk == j // chunk)
    x = torch.einsum("thd,shd->hts", q, k) * scale
    if bias is not None:
        x = x + bias[:, (i - j).clamp(0, bias.shape[1] - 1)]
    if softcap:
        x = softcap * torch.tanh(x / softcap)
    if slopes is not None:
        x = x - slopes[:, None, None] * (i - j)
    x = x.masked_fill(~seen, -math.inf)
    top = x.amax(-1, keepdim=True)
    if sinks is not None:
        top = torch.maximum(top, sinks[:, None, None])
    e = torch.exp(x - top)
    den = e.sum(-1, keepdim=True) + (0 if sinks is None else torch.exp(sinks[:, None, None] - top))
    return torch.einsum("hts,shd->thd", e / den, v), torch.einsum("hts,shd->thd", e / den, v.abs()), x[:, seen].abs().max().item()


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("heads,groups,dim,vdim", [(4, 2, 128, 128), (4, 4, 32, 32), (2, 1, 192, 128), (2, 2, 256, 192), (4, 2, 48, 80)])
def test_forms(heads, groups, dim, vdim, form):
    from nanovllm import ops
    page = 64
    g = torch.Generator().manual_seed(dim + vdim + len(form))
    steps = ([1, 15, 16, 17, 63, 64, 65, 130, 1, 40], [1, 15, 16, 17, 63, 64, 65, 130, 200, 241]), ([1] * 6, [1, 16, 64, 65, 193, 300])
    for lens, ctxs in steps:
        width = max(-(-c // page) for c in ctxs)
        tables = torch.randperm(len(lens) * width, generator=g).int().view(len(lens), width)
        kc = torch.randn(len(lens) * width, page, groups, dim, generator=g).bfloat16()
        vc = torch.randn(len(lens) * width, groups, vdim, page, generator=g).bfloat16()
        q = (2.0 * torch.randn(sum(lens), heads * dim, generator=g)).bfloat16()
        opts = dict(FORMS[form])
        if "slopes" in opts:
            opts["slopes"] = torch.rand(heads, generator=g) * 0.05
        if "bias" in opts:
            opts["bias"] = torch.randn(heads, 50, generator=g)
        if "sinks" in opts:
            opts["sinks"] = torch.randn(heads, generator=g) * 3
        cu = None if max(lens) == 1 else torch.tensor([0] + lens).cumsum(0).int().cuda()
        scale = 1.5 * dim ** -0.5
        got = ops.attn_paged_any(q.cuda(), kc.cuda(), vc.cuda(), cu, torch.tensor(ctxs, dtype=torch.int32).cuda(), tables.cuda(), scale, heads, groups, dim, vdim,
                                 **{n: x.cuda() if torch.is_tensor(x) else x for n, x in opts.items()}).cpu().double().view(-1, heads, vdim)
        at = 0
        for b, (n, c) in enumerate(zip(lens, ctxs)):
            t = tables[b].long()
            k = kc[t].reshape(-1, groups, dim)[:c].double().repeat_interleave(heads // groups, 1)
            v = vc[t].permute(0, 3, 1, 2).reshape(-1, groups, vdim)[:c].double().repeat_interleave(heads // groups, 1)
            want, mass, big = reference(q[at:at + n].double().view(n, heads, dim), k, v, c - n, scale, **{n_: x.double() if torch.is_tensor(x) else x for n_, x in opts.items()})
            # the result's rounding to bf16; weights of 16 bits (hi + lo) and exponents of scores that carry dim + 4 roundings of fp32
            bound = want.abs() * 2.0 ** -8 + mass * (2.0 ** -15 + 2 * (big + 4) * (dim + 4) * 2.0 ** -24) + 1e-30
            assert ((got[at:at + n] - want).abs() <= bound).all(), (form, b, n, c)
            at += n
