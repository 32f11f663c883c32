"""The delta rule's operands of many tokens at once against the same tokens a few at a time: the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,H,dk,rank", [(513, 16, 64, 64), (2049, 3, 80, 8), (1027, 5, 16, 24), (514, 16, 64, 20)])
def test_tokens_together(T, H, dk, rank, dtype):
    from nanovllm import _hip
    g = torch.Generator().manual_seed(T)
    n = H * dk
    rows = torch.randn(T, 4 * n + rank + 8, generator=g).to(dtype).cuda()
    r, k, v, a, low = rows[:, :n], rows[:, n:2 * n], rows[:, 2 * n:3 * n], rows[:, 3 * n:4 * n], rows[:, 4 * n:4 * n + rank]
    w2, w0, bias = (torch.randn(n, rank, generator=g) * 0.3).to(dtype).cuda(), torch.randn(n, generator=g).to(dtype).cuda(), torch.randn(n, generator=g).to(dtype).cuda()
    ld = rows.stride(0)

    def prep(lo, hi):
        out = torch.full((hi - lo, H, 6 * dk), float("nan"), device="cuda")
        at = lambda x: x[lo:hi].data_ptr()
        _hip.call("nvh_delta_prep", at(r), ld, at(k), ld, at(v), ld, at(a), ld, at(low), ld, w2.data_ptr(), w0.data_ptr(), bias.data_ptr(), out.data_ptr(),
                  hi - lo, H, dk, rank, 0.6, int(dtype == torch.float32), torch.cuda.current_stream().cuda_stream)
        return out.cpu()

    whole = prep(0, T)
    parts = torch.cat([prep(i, min(i + 100, T)) for i in range(0, T, 100)])
    assert whole.isfinite().all() and torch.equal(whole, parts)
    z = w0.double() + torch.tanh(low.double()) @ w2.double().t()
    want = torch.exp(-0.6 * torch.sigmoid(z)).view(T, H, dk).cpu()
    assert (whole[:, :, 2 * dk:3 * dk].double() - want).abs().max() <= (rank + 8) * 2.0 ** -24 * (1 + z.abs().max().item())
