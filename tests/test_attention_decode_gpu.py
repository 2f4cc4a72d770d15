"""GPU parity of the decode-step attention kernel (attention_decode.hip): 1 to 16 query rows, key counts
around the 32-key blocks, the four waves' 128 keys and the parts of a split range, masks, views.  Bars as for
the other attention kernels (tests/test_attention_gpu.py)."""
import numpy as np
import pytest
import torch

from oracle import oracle
from tests.util import NAME, TOL, as_f64, assert_close, to_dev

pytestmark = pytest.mark.gpu


def _qkv(B, H, Sq, Skv, D, dtype, seed):
    rng = np.random.default_rng(seed)
    return (to_dev(rng.standard_normal((B, H, n, D)), dtype) for n in (Sq, Skv, Skv))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,H,Sq,Skv", [(1, 1, 1, 1), (2, 3, 1, 31), (1, 2, 2, 33), (1, 5, 4, 127), (3, 2, 16, 129), (1, 1, 15, 511), (1, 2, 1, 513), (2, 4, 8, 2100),
                                        (1, 1, 1, 8192), (70, 8, 1, 300)], ids=lambda v: str(v))
def test_decode(B, H, Sq, Skv, D, dtype):
    from metalhlo_amd import kernels
    q, k, v = _qkv(B, H, Sq, Skv, D, dtype, 3)
    got = kernels.flash_attention(q, k, v, scale=-0.2 if Skv == 127 else None)
    exp = oracle.attention(as_f64(q), as_f64(k), as_f64(v), scale=-0.2 if Skv == 127 else None)
    assert_close(got, exp, TOL[dtype], f"decode {(B, H, Sq, Skv, D)}")


@pytest.mark.parametrize("Skv", [40, 1000])
def test_decode_mask_and_views(Skv):
    """An additive mask (one row fully masked: zeros) and operands that are views of a cache [B, S, H, D]."""
    from metalhlo_amd import kernels
    B, H, Sq, D = 2, 3, 4, 64
    rng = np.random.default_rng(5)
    cache = to_dev(rng.standard_normal((2, B, Skv + 8, H, D)), torch.bfloat16)
    k, v = (cache[i, :, :Skv].permute(0, 2, 1, 3) for i in range(2))
    q = to_dev(rng.standard_normal((B, Sq, H, D)), torch.bfloat16).permute(0, 2, 1, 3)
    m = rng.standard_normal((B, 1, Sq, Skv))
    m[..., Skv // 2:] = -np.inf
    m[1, 0, 2] = -np.inf
    md = to_dev(m, torch.bfloat16)
    got = kernels.flash_attention(q, k, v, mask=md)
    exp = oracle.attention(as_f64(q), as_f64(k), as_f64(v), mask=as_f64(md))
    assert_close(got, exp, TOL[torch.bfloat16], "decode mask + views")
    assert torch.count_nonzero(got[1, :, 2]) == 0
