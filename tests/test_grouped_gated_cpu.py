"""nvh_gemm_grouped_gated_nt refuses what the two launches it stands for refuse (argument checks alone: a list of no tiles launches nothing)."""
import pytest

from nanovllm import _hip


def gated(act, limit):
    # (16-byte aligned addresses that nothing reads)
    return _hip.lib().nvh_gemm_grouped_gated_nt(4096, 64, 4096, 4096, 4096, 32, 4096, 4096, 4096, 0, 32, 64, act, 4096, None, 1, limit, 1.702, 0, None)


@pytest.mark.parametrize("limit", [0.0, -1.0, float("nan")])
def test_capped_unit_needs_a_limit(limit):
    pair = _hip.lib().nvh_glu_clamp_pairs(4096, 64, 4096, None, 4096, 32, 0, 32, limit, 1.702, 0, None)
    assert pair != 0 and gated(3, limit) == pair
    assert gated(3, 1.5) == 0 and gated(0, limit) == 0       # (no other activation reads it)
