"""Queries, keys and values from the projection row: pieces of eight elements and value tiles against the form that takes any row."""
import pytest
import torch

pytestmark = pytest.mark.gpu
PAGE = 64


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("norm", ["none", "row", "head"])
@pytest.mark.parametrize("H,G,dim,vdim,rot,inter,turn,v_inter", [
    (1, 1, 8, 8, 8, True, True, True), (2, 1, 16, 16, 16, False, True, False), (16, 8, 128, 128, 64, True, False, False), (8, 8, 128, 64, 128, False, True, False),
    (4, 2, 40, 24, 32, False, True, True), (16, 8, 128, 128, 0, False, True, False), (32, 16, 128, 72, 96, True, False, False)])
@pytest.mark.parametrize("T", [1, 5, 127, 128, 200])
def test_forms_agree(T, H, G, dim, vdim, rot, inter, turn, v_inter, norm, dtype):
    """Equal but for the order in which a norm adds its squares: 1e-5 of the value (of a rotated pair's larger one) and a rounding of the result; values
    are the same bits."""
    from nanovllm import ops
    if T > 128 and H * dim > 2048:
        T = 130
    g = torch.Generator().manual_seed(T + H * dim)
    nq, nk, nv = H * dim, G * dim, G * vdim
    width = nq + nk + nv + H
    row = torch.randn(T, (width + 8) // 8 * 8, generator=g).to(dtype).cuda()
    odd = torch.empty(T, row.shape[1] + 1, dtype=dtype, device="cuda")
    odd[:, :-1] = row
    pages = -(-T // PAGE) + 1
    slots = torch.randperm((pages - 1) * PAGE, generator=g)[:T].int() + PAGE     # (the first page is left to the run below)
    if T > 4:
        slots[3] = -1
        slots[64:64 + PAGE] = torch.arange(len(slots[64:64 + PAGE])).int()    # tokens that lie side by side in a page
    positions = torch.randint(0, 5000, (T,), generator=g).cuda()
    w = [None, None] if norm == "none" else [(torch.rand(n, generator=g) + 0.5).to(dtype).cuda() for n in ((nq, nk) if norm == "row" else (dim, dim))]
    freq = torch.rand(rot // 2, generator=g).cuda() if rot else None
    vfreq = torch.rand(vdim // 2, generator=g).cuda() if turn else None
    outs = []
    for src in (row, odd):
        kc, vc = torch.zeros(pages, PAGE, G, dim, dtype=dtype, device="cuda"), torch.zeros(pages, G, vdim, PAGE, dtype=dtype, device="cuda")
        q, gate = ops.attn_rotary_prep(src[:, :width], w[0], w[1], 1e-5, positions, freq, 1.1, rot, vfreq, kc, vc, slots.cuda(), H, G, dim, vdim, True, inter, v_inter,
                                       norm_per_head=norm == "head")
        outs.append((q, gate, kc, vc))
    (q, gate, kc, vc), (q2, gate2, kc2, vc2) = outs
    assert torch.equal(gate, gate2) and torch.equal(vc, vc2)
    for a, b in ((q, q2), (kc, kc2)):
        a, b = a.double(), b.double()
        top = b.abs().amax() if rot else b.abs()
        assert ((a - b).abs() <= 1e-5 * top + (2.0 ** -7 * b.abs() if dtype is torch.bfloat16 else 0)).all()


@pytest.mark.parametrize("per_head", [False, True])
@pytest.mark.parametrize("H,G,dim", [(16, 8, 128), (4, 2, 64), (4, 2, 256), (8, 2, 40), (1, 1, 8), (20, 4, 128), (32, 16, 128)])
def test_norms_are_no_less_precise(H, G, dim, per_head):
    """Both forms' root mean square distance of 1 / rms (read off an element of 1 with weights of 1) from float64, over about 100 000 norms, of which it is
    known to 0.3 %.  The other form's sums were the only ones once."""
    from nanovllm import ops
    nq, nk = H * dim, G * dim
    norms = H + G if per_head else 2
    T = 4096
    g = torch.Generator(device="cuda").manual_seed(dim)
    at, pages = torch.arange(T, device="cuda"), T // PAGE
    w = [torch.ones(n, device="cuda") for n in ((dim, dim) if per_head else (nq, nk))]
    off = [[], []]
    for _ in range(-(-100_000 // (T * norms))):
        row = torch.randn(T, -(-(nq + 2 * nk) // 4) * 4, generator=g, device="cuda")
        parts = [(0, nq), (nq, nk)]
        for lo, n in parts:
            row[:, lo:lo + n:dim if per_head else n] = 1
        odd = torch.empty(T, row.shape[1] + 1, device="cuda")
        odd[:, :-1] = row
        for i, src in enumerate((row, odd)):
            kc, vc = torch.zeros(pages, PAGE, G, dim, device="cuda"), torch.zeros(pages, G, dim, PAGE, device="cuda")
            q, _ = ops.attn_rotary_prep(src[:, :nq + 2 * nk], w[0], w[1], 1e-5, at, None, 1.0, 0, None, kc, vc, at.int(), H, G, dim, dim, False, norm_per_head=per_head)
            for (lo, n), got in zip(parts, (q, kc.view(T, nk))):
                d = dim if per_head else n
                want = 1 / (row[:, lo:lo + n].double().view(T, -1, d).pow(2).mean(-1) + 1e-5).sqrt()
                off[i].append(((got[:, ::d].double() - want) / want).flatten())
    vec, other = (float(torch.cat(o).pow(2).mean().sqrt()) for o in off)
    assert vec <= 1.015 * other, (vec, other)
