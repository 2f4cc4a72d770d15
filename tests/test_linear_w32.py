"""Which linear layers with fp32 parameters are served (host side only)."""
import pytest
import torch


@pytest.fixture(scope="module")
def codes():
    from metalhlo_amd import kernels
    return kernels.DTYPE_CODE[torch.bfloat16], kernels.DTYPE_CODE[torch.float16]


def test_both_operands_stay_below_the_out_of_range_offset(lib, codes):
    """Loads past the edge use a byte offset of 2^31, so x [M, K] and w [N, K] each have to end below it."""
    for dt in codes:
        edge = 2 ** 31 // (192 * 2) // 8 * 8                      # K from which x of 192 rows spans 2^31 bytes
        assert lib.mhip_linear_w32_ok(192, 8, edge - 8, dt)
        for K in (edge + 8, 2 ** 31 // (72 * 4) // 8 * 8 - 72):   # (w of 8 columns alone ends below 2^31)
            assert (8 + 64) * (K + 64) * 4 < 2 ** 31 <= 192 * K * 2
            assert not lib.mhip_linear_w32_ok(192, 8, K, dt)
        assert lib.mhip_linear_w32_ok(128, 8, edge + 8, dt)       # (fewer rows of the same length are served)
