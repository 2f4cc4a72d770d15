"""GPU parity of fp32 attention with the keys dealt over the waves (attention_f32.hip): query and key counts around
its 32-row tiles, 32-key blocks and four waves, causal, masks; and of the tile rule's other side.  fp32 bar of
tests/test_attention_gpu.py."""
import numpy as np
import pytest
import torch

from oracle import oracle
from tests.util import TOL, as_f64, assert_close, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [32, 64, 96, 128])
@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
@pytest.mark.parametrize("B,H,Sq,Skv", [(1, 1, 1, 1), (2, 3, 31, 33), (1, 8, 33, 31), (1, 2, 96, 127), (1, 5, 129, 129), (2, 4, 64, 300), (1, 1, 257, 40), (9, 32, 40, 70)],
                         ids=lambda v: str(v))
def test_split(B, H, Sq, Skv, causal, D):
    from metalhlo_amd import kernels
    rng = np.random.default_rng(D)
    q, k, v = (to_dev(rng.standard_normal((B, H, n, D)), torch.float32) for n in (Sq, Skv, Skv))
    guard = torch.full((B * H * Sq * D + 64,), float("nan"), device="cuda")
    got = kernels.flash_attention(q, k, v, is_causal=causal, out=guard[:-64].view(B, H, Sq, D))
    assert_close(got, oracle.attention(as_f64(q), as_f64(k), as_f64(v), is_causal=causal), TOL[torch.float32], f"split {(B, H, Sq, Skv, D)}")
    assert torch.isnan(guard[-64:]).all()


@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
def test_split_mask(causal):
    """Masks per batch entry, one row fully hidden (zeros), one hiding whole blocks; negative scale."""
    from metalhlo_amd import kernels
    B, H, Sq, Skv, D = 2, 3, 70, 200, 64
    rng = np.random.default_rng(2)
    q, k, v = (to_dev(rng.standard_normal((B, H, n, D)), torch.float32) for n in (Sq, Skv, Skv))
    m = rng.standard_normal((B, 1, Sq, Skv))
    m[1, 0, :, :64] = -np.inf
    m[0, 0, 5] = -np.inf
    md = to_dev(m, torch.float32)
    got = kernels.flash_attention(q, k, v, scale=-0.2, is_causal=causal, mask=md)
    exp = oracle.attention(as_f64(q), as_f64(k), as_f64(v), scale=-0.2, is_causal=causal, mask=as_f64(md))
    assert_close(got, exp, TOL[torch.float32], "split mask")
    assert torch.count_nonzero(got[0, :, 5]) == 0
