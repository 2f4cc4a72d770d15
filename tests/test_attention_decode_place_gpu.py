"""GPU test that the bits of decode attention (attention_decode.hip) do not say where in the launch a head is: equal heads have equal results, and heads in another order the same
results in that order, whole and in parts of the keys, with and without a mask."""
import pytest
import torch

from tests.util import NAME

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("B,H,Sq,Skv,D", [(8, 32, 1, 4096, 128), (8, 32, 1, 1024, 64), (4, 12, 3, 3000, 128), (2, 4, 1, 16384, 128), (2, 8, 16, 2047, 64), (32, 12, 4, 1111, 128),
                                          (64, 5, 1, 900, 128)], ids=str)
def test_a_head_has_the_same_bits_wherever_it_is(B, H, Sq, Skv, D, dtype):
    from metalhlo_amd import kernels
    g = torch.Generator(device="cuda").manual_seed(B * 1000 + Skv)
    q, k, v = (torch.randn(B, H, n, D, generator=g, device="cuda").to(dtype) for n in (Sq, Skv, Skv))
    mask = torch.randn(1, 1, Sq, Skv, generator=g, device="cuda").to(dtype)
    mask[..., Skv * 2 // 3:] = float("-inf")
    order = torch.randperm(B * H, generator=g, device="cuda")

    def moved(t):
        return t.reshape(B * H, -1)[order].reshape(t.shape)
    for m in (None, mask):
        out = kernels.flash_attention(q, k, v, mask=m)
        assert torch.equal(kernels.flash_attention(moved(q), moved(k), moved(v), mask=m), moved(out))
        first = [t[:1, :1].expand_as(t).contiguous() for t in (q, k, v)]
        alike = kernels.flash_attention(*first, mask=m)
        assert torch.equal(alike, alike[:1, :1].expand_as(alike)) and torch.equal(alike[0, 0], out[0, 0])
