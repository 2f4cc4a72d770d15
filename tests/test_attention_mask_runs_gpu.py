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
    keep = np.ones((B, H, Sq), bool)
    keep[0, 2, 5] = False                          # (in 32 bits the scores vanish against the mask: any weights, finite)
    g = as_f64(got)
    assert np.isfinite(g).all() and np.count_nonzero(g[0, 1, 7]) == 0
    assert_close(got[torch.from_numpy(keep).cuda()], exp[keep], TOL[dtype], "masked")
