"""GPU parity of attention and its projection in one launch (attend_project and attend_project_layer of linear_w32.hip): one and two groups of 32 queries, rows around its groups of 16, heads in one
part and in several, columns around its strips of 32 and the eighths that an XCD takes.

The attention in front is causal_attention's, bit for bit (one code), so the sums differ from its result times the rounded weights in 64 bits by fp32 additions of K products
alone: at most K 2^-23 of the sum of their magnitudes, a product of 16-bit numbers being exact."""
import numpy as np
import pytest
import torch

from tests.util import NAME, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("B,S,H,N", [(1, 1, 4, 8), (1, 31, 12, 768), (1, 32, 4, 264), (1, 33, 12, 40), (1, 64, 8, 1032), (2, 16, 4, 72), (2, 20, 12, 768), (2, 32, 8, 256), (4, 1, 1, 32), (3, 5, 2, 1000)], ids=str)
def test_sums(B, S, H, N, dtype):
    from metalhlo_amd import kernels
    assert kernels.attend_project_served(B, S, H, 64, N, dtype)
    rng = np.random.default_rng(B * 1000 + S + N)
    qkv = to_dev(rng.standard_normal((B * S, 3 * H * 64)), dtype)
    w = to_dev(rng.standard_normal((H * 64, N)), torch.float32)
    sums = kernels.attend_project(qkv, w, B, H, ahead=(to_dev(rng.standard_normal((64, 128)), torch.float32),))
    assert sums.dtype == torch.float32 and sums.shape[1:] == (B * S, N)
    x, r = kernels.causal_attention(qkv, B, H).double(), w.to(dtype).double()
    error = (sums.double().sum(0) - x @ r).abs()
    assert bool((error <= H * 64 * 2.0 ** -23 * (x.abs() @ r.abs())).all()), float(error.max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("B,S,H,N", [(1, 1, 1, 8), (1, 8, 12, 768), (1, 16, 12, 136), (1, 17, 16, 1032), (1, 32, 12, 768), (2, 16, 8, 24), (2, 8, 12, 768), (2, 8, 16, 40), (7, 2, 3, 136), (4, 8, 4, 264), (3, 5, 5, 128), (16, 2, 1, 72), (5, 3, 3, 8)], ids=str)
def test_layer(B, S, H, N, dtype):
    """One rounding to the type behind the sum and one behind the residual, of a sum off by K 2^-23 of its products."""
    from metalhlo_amd import kernels
    assert kernels.attend_project_layer_served(B, S, H, 64, N, dtype)
    rng = np.random.default_rng(B * 1000 + S + N)
    qkv, res = (to_dev(rng.standard_normal(n), dtype) for n in ((B * S, 3 * H * 64), (B * S, N)))
    w, bias = (to_dev(rng.standard_normal(n), torch.float32) for n in ((H * 64, N), (N,)))
    ahead = (to_dev(rng.standard_normal((64, 128)), torch.float32),)
    x, r = kernels.causal_attention(qkv, B, H).double(), w.to(dtype).double()
    sum_, off = x @ r + bias.to(dtype).double(), (H * 64 + 1) * 2.0 ** -23 * (x.abs() @ r.abs() + bias.abs().double())
    unit = torch.finfo(dtype).eps / 2
    got = kernels.attend_project_layer(qkv, w, bias, res, B, H, ahead=ahead).double()
    one = sum_.abs() * unit + off * (1 + unit)
    error = (got - sum_ - res.double()).abs()
    assert bool((error <= one + (got.abs() + one) * unit * (1 + unit)).all()), float(error.max())
    bare = kernels.attend_project_layer(qkv, w, None, None, B, H).double()
    error = (bare - x @ r).abs()
    assert bool((error <= (x @ r).abs() * unit + off * (1 + unit)).all()), float(error.max())
    # in a batch of its own and in one with others a sequence has the same bits
    if B > 1:
        assert torch.equal(kernels.attend_project_layer(qkv[:S], w, bias, res[:S], 1, H).double(), got[:S])


def test_a_part_that_sees_nothing_behind_its_rows():
    """Infinities and NaN behind the last row, of qkv and of W, reach no sum."""
    from metalhlo_amd import kernels
    rng = np.random.default_rng(5)
    room = torch.full((64, 3 * 256), float("nan"), dtype=torch.bfloat16, device="cuda")
    room[:37] = to_dev(rng.standard_normal((37, 768)), torch.bfloat16)
    w = to_dev(rng.standard_normal((256, 72)), torch.float32)
    wide = torch.full((320, 72), float("inf"), device="cuda")
    wide[:256] = w
    assert torch.equal(kernels.attend_project(room[:37], wide[:256], 1, 4), kernels.attend_project(room[:37].clone(), w, 1, 4))


@pytest.mark.parametrize("B,S,H,D,N,dtype", [(1, 65, 4, 64, 64, torch.bfloat16), (3, 22, 4, 64, 64, torch.bfloat16), (1, 8, 4, 128, 64, torch.bfloat16), (1, 8, 4, 64, 60, torch.bfloat16),
                                             (1, 8, 4, 64, 64, torch.float32), (0, 8, 4, 64, 64, torch.bfloat16), (1, 8, 4, 64, 0, torch.bfloat16)], ids=str)
def test_what_is_not_served(B, S, H, D, N, dtype):
    from metalhlo_amd import kernels
    assert not kernels.attend_project_served(B, S, H, D, N, dtype)


@pytest.mark.parametrize("B,S,H,D,N,dtype", [(1, 33, 12, 64, 64, torch.bfloat16), (2, 9, 12, 64, 64, torch.bfloat16), (3, 5, 12, 64, 64, torch.bfloat16), (4, 9, 4, 64, 64, torch.bfloat16), (1, 8, 17, 64, 64, torch.bfloat16),
                                             (1, 8, 4, 128, 64, torch.bfloat16), (1, 8, 4, 64, 60, torch.bfloat16), (1, 8, 4, 64, 64, torch.float32), (1, 0, 4, 64, 64, torch.bfloat16)], ids=str)
def test_what_no_layer_serves(B, S, H, D, N, dtype):
    from metalhlo_amd import kernels
    assert not kernels.attend_project_layer_served(B, S, H, D, N, dtype)
    assert not kernels.attend_project_layer_served(2 ** 32 + B, S, H, D, N, dtype)
