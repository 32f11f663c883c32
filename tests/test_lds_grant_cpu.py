"""fp32 ring tiles of more than 64 KB of LDS ask for it before they launch; a refusal (here: there is no device) is reported as one and launches nothing."""
import pytest
import torch

from nanovllm import _hip

pytestmark = pytest.mark.skipif(torch.cuda.is_available(), reason="the calls are made to be refused, and hold no addresses of a GPU's memory")
ENOSYS = -38


def last():
    return _hip.lib().nvh_last_error().decode()


def test_refused():
    lib, p = _hip.lib(), 4096
    assert lib.nvh_gemm_any_nt(p, 64, p, None, p, 8192, 300, 8192, 64, 1, 1, None) == ENOSYS and "LDS" in last()
    for name in ("nvh_gemm_grouped_any_nt", "nvh_gemm_grouped_many_nt"):
        assert getattr(lib, name)(p, 64, None, p, p, 64, p, p, p, 4, 64, 64, 0, 1, 1, None) == ENOSYS and "LDS" in last()
