"""GPU parity of attention over few keys (attention_short.hip): queries and keys around its groups of 32 rows and 32 keys, more queries than keys and fewer, views, a negative scale.  Bars as for the other attention kernels (tests/test_attention_gpu.py)."""
import numpy as np
import pytest
import torch

from oracle import oracle
from tests.util import NAME, TOL, as_f64, assert_close, to_dev

pytestmark = pytest.mark.gpu


def _check(B, H, Sq, Skv, D, causal, dtype, scale=None):
    from metalhlo_amd import kernels
    rng = np.random.default_rng(Sq * 131 + Skv)
    q, k, v = (to_dev(rng.standard_normal((B, H, n, D)), dtype) for n in (Sq, Skv, Skv))
    got = kernels.flash_attention(q, k, v, is_causal=causal, scale=scale)
    exp = oracle.attention(as_f64(q), as_f64(k), as_f64(v), scale=scale, is_causal=causal)
    assert_close(got, exp, TOL[dtype], f"short {(B, H, Sq, Skv, D, causal)}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,H,Sq,Skv", [(1, 1, 17, 1), (2, 3, 31, 31), (1, 2, 64, 64), (1, 2, 65, 63), (3, 1, 20, 64), (1, 2, 33, 17), (5, 4, 16, 16), (40, 8, 64, 64)], ids=str)
def test_few_keys(B, H, Sq, Skv, D, dtype):
    _check(B, H, Sq, Skv, D, True, dtype, scale=-0.2 if Skv == 17 else None)


def test_same_bits_in_any_batch():
    from metalhlo_amd import kernels
    q, k, v = (to_dev(np.random.default_rng(i).standard_normal((40, 16, 50, 64)), torch.bfloat16) for i in range(3))
    lots = kernels.flash_attention(q, k, v, is_causal=True)
    few = kernels.flash_attention(*(t[:1, :3].contiguous() for t in (q, k, v)), is_causal=True)
    assert torch.equal(few, lots[:1, :3])


def test_projection_in_place():
    from metalhlo_amd import kernels
    B, H, S, D = 3, 4, 21, 64
    qkv = to_dev(np.random.default_rng(2).standard_normal((B * S, 3 * H * D)), torch.bfloat16)
    q, k, v = (as_f64(t) for t in qkv.view(B, S, 3, H, D).permute(2, 0, 3, 1, 4).unbind(0))
    got = kernels.causal_attention(qkv, B, H).view(B, S, H, D).permute(0, 2, 1, 3)
    assert_close(got, oracle.attention(q, k, v, is_causal=True), TOL[torch.bfloat16], "short, in place")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("S", [1, 17, 32, 33, 37, 64])
def test_a_row_keeps_its_bits_when_its_sequence_goes_on(S, D, dtype):
    """What stands behind a row is hidden from it: the kernels for longer sequences form the same products and sums in the same order."""
    from metalhlo_amd import kernels
    q, k, v = (to_dev(np.random.default_rng(i + S).standard_normal((2, 3, 300, D)) * 2, dtype) for i in range(3))
    scale = -0.2 if S == 33 else None
    short = kernels.flash_attention(*(t[:, :, :S].contiguous() for t in (q, k, v)), is_causal=True, scale=scale)
    for n in (65, 129, 300):
        longer = kernels.flash_attention(*(t[:, :, :n].contiguous() for t in (q, k, v)), is_causal=True, scale=scale)
        assert torch.equal(short, longer[:, :, :S]), n
