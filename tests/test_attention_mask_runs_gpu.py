"""GPU parity of additive masks that attention reads four keys at a time, and of masks whose rows, batch strides or
address do not allow that: the same bars as tests/test_attention_gpu.py."""
import numpy as np
import pytest
import torch

from oracle import oracle
from tests.util import NAME, TOL, as_f64, assert_close, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("D", [64, 128, 96])
@pytest.mark.parametrize("Sq,Skv,causal,odd", [(40, 4, False, False), (130, 68, True, False), (33, 200, False, False), (33, 200, False, True), (70, 130, True, False), (200, 127, False, False)],
                         ids=lambda v: str(v))
def test_mask(Sq, Skv, causal, odd, D, dtype):
    from metalhlo_amd import kernels
    B, H = 2, 3
    rng = np.random.default_rng(Skv)
    q, k, v = (to_dev(rng.standard_normal((B, H, n, D)), dtype) for n in (Sq, Skv, Skv))
    m = rng.standard_normal((B, H, Sq, Skv))
    m[1, :, :, -3:] = -np.inf                      # padding
    m[0, 1, 7] = -np.inf                           # a row without keys: zeros
    m[0, 2, 5] = float(torch.finfo(dtype).min)     # the type's lowest value everywhere
    md = to_dev(np.concatenate([np.zeros(1), m.reshape(-1)]), dtype)[1:].view(m.shape) if odd else to_dev(m, dtype)
    got = kernels.flash_attention(q, k, v, is_causal=causal, mask=md)
    exp = oracle.attention(as_f64(q), as_f64(k), as_f64(v), is_causal=causal, mask=as_f64(md))
    assert np.count_nonzero(as_f64(got)[0, 1, 7]) == 0
    assert_close(got, exp, TOL[dtype], "masked")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("B,H,Sq,Skv,D,causal", [(2, 3, 4, 40, 64, False), (2, 3, 4, 1000, 64, False), (1, 2, 16, 2100, 128, False), (16, 17, 33, 70, 128, False),
                                                 (2, 2, 140, 140, 32, True), (2, 2, 140, 139, 80, True)], ids=lambda v: str(v))
def test_lowest_number_as_mask(B, H, Sq, Skv, D, causal, dtype):
    """Keys hidden with the type's lowest number: every key of a row (they share it alike, hidden or not), the first or the
    last half, and beside keys hidden with -inf; a query of NaN gives NaN whatever its mask.  Decode steps with and without a split key range, both fp32 kernels,
    head sizes of every 16-bit kernel."""
    from metalhlo_amd import kernels
    rng = np.random.default_rng(D)
    q, k, v = (to_dev(rng.standard_normal((B, H, n, D)), dtype) for n in (Sq, Skv, Skv))
    q[0, 0, 2] = float("nan")
    q[-1, -1, 3] = float("nan")
    low = float(torch.finfo(dtype).min)
    m = rng.standard_normal((B, 1, Sq, Skv))
    m[:, 0, 0] = low
    m[:, 0, 1, :Skv // 2] = low
    m[:, 0, 2, Skv // 2:] = low
    m[:, 0, 3] = low
    m[:, 0, 3, ::2] = -np.inf
    md = to_dev(m, dtype)
    got = kernels.flash_attention(q, k, v, is_causal=causal, mask=md)
    assert_close(got, oracle.attention(as_f64(q), as_f64(k), as_f64(v), is_causal=causal, mask=as_f64(md)), TOL[dtype], "lowest number")
