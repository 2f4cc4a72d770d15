"""Attention over few tiles (attention_flow.hip) forms every sum in the order of the kernel for many: a sequence's bits do not
depend on the batch it is in.  Sizes around its tiles (128 queries, 32 a wave, 64 keys), q, k, v as views of one projection."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (31, 31, 1), (32, 33, 1), (64, 64, 1), (65, 200, 1), (127, 127, 1), (128, 128, 0), (129, 129, 1), (200, 63, 1),
         (40, 320, 0), (257, 257, 1), (130, 449, 0), (190, 500, 1), (129, 192, 0), (321, 321, 1)]


def _views(B, H, S, D, x):
    return x.view(B, S, 1, H, D).permute(2, 0, 3, 1, 4)[0]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Sq,Skv,causal", SIZES)
def test_same_bits_in_any_batch(dtype, D, Sq, Skv, causal):
    from metalhlo_amd import kernels
    H = 2
    many = 512 // H + 1                                     # more tiles than two workgroups a compute unit
    g = torch.Generator(device="cuda").manual_seed(Sq * 1000 + Skv)
    q, k, v = (torch.randn(3, s * H * D, generator=g, device="cuda").to(dtype) for s in (Sq, Skv, Skv))
    q[1] *= 40                                              # scores whose maximum moves the reference from block to block
    k[2, -D:] = float("inf")                                # scores that are not finite
    for scale in (None, -0.3):
        few = kernels.flash_attention(_views(3, H, Sq, D, q), _views(3, H, Skv, D, k), _views(3, H, Skv, D, v), scale, bool(causal))
        Q, K, V = (t.repeat(many, 1) for t in (q, k, v))
        lots = kernels.flash_attention(_views(3 * many, H, Sq, D, Q), _views(3 * many, H, Skv, D, K), _views(3 * many, H, Skv, D, V), scale,
                                       bool(causal))
        if not causal and Sq <= 16:
            continue
        assert torch.equal(few.view(torch.int16), lots[:3].view(torch.int16))
        assert torch.equal(few.view(torch.int16), lots[-3:].view(torch.int16))
    exp = torch.softmax(torch.where(
        torch.ones(Sq, Skv, dtype=torch.bool, device="cuda").tril() if causal else torch.ones(Sq, Skv, dtype=torch.bool, device="cuda"),
        _views(3, H, Sq, D, q).double()[:1] @ _views(3, H, Skv, D, k).double()[:1].transpose(-1, -2).contiguous() * -0.3, float("-inf")),
        -1) @ _views(3, H, Skv, D, v).double()[:1].contiguous()
    err = (few[:1].double() - exp).norm() / exp.norm()
    assert err <= (8e-3 if dtype == torch.bfloat16 else 1e-3), float(err)      # two roundings: weights and result
