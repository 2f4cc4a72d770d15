"""GPU parity of decode attention on workgroups of eight waves and of four (attention_decode.hip): numbers of heads at the edges of the
rule, key counts at the edges of what eight waves take at once, with and without a workspace and a mask.  Bars as in test_attention_gpu.py."""
import pytest
import torch

from tests.util import NAME, TOL, as_f64, assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("heads,Sq,Skv,D", [(1, 1, 128, 64), (1, 16, 129, 128), (5, 3, 255, 64), (1, 16, 16384, 64), (8, 16, 2049, 64), (64, 2, 1025, 128), (65, 1, 640, 64),
                                            (86, 4, 2000, 128), (192, 1, 257, 64), (191, 5, 513, 64), (256, 8, 320, 128), (257, 1, 300, 64)], ids=str)
def test_waves(lib, heads, Sq, Skv, D, dtype):
    from metalhlo_amd import kernels
    g = torch.Generator(device="cuda").manual_seed(heads * 7 + Skv)
    q, k, v = (torch.randn(1, heads, n, D, generator=g, device="cuda").to(dtype) for n in (Sq, Skv, Skv))
    mask = torch.randn(1, 1, Sq, Skv, generator=g, device="cuda").to(dtype)
    mask[..., Skv * 2 // 3:] = float("-inf")
    for m in (None, mask):
        s = q.double() @ k.double().transpose(-1, -2).contiguous() * D ** -0.5
        exp = as_f64(torch.softmax(s if m is None else s + m.double(), -1) @ v.double())
        assert_close(kernels.flash_attention(q, k, v, mask=m), exp, TOL[dtype], f"waves {(heads, Sq, Skv, D)}")
        alone = torch.full_like(q, float("nan"))                     # without a workspace: a head's keys in one workgroup
        assert lib.mhip_flash_attention(torch.cuda.current_stream().cuda_stream, q.data_ptr(), k.data_ptr(), v.data_ptr(), None if m is None else m.data_ptr(),
                                        alone.data_ptr(), 1, heads, Sq, Skv, D, D ** -0.5, 0, 0, 0, kernels.DTYPE_CODE[dtype]) == 0
        assert_close(alone, exp, TOL[dtype], f"waves, no workspace {(heads, Sq, Skv, D)}")
