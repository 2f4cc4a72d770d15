"""Which (head, tile of queries) a workgroup takes: heads that eight divides go to an XCD each, the up to seven left over are dealt out by
tiles.  Every tile is computed, and once: a row of each 32 is compared with float64, so that a tile not written shows (the result
starts as NaN)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# two roundings of 16 bits (weights and result), four times what a sum in another order shows in fp32
BOUND = {torch.bfloat16: 8e-3, torch.float16: 1e-3, torch.float32: 1e-5}


@pytest.mark.parametrize("heads,S,D,dtype", [
    (1, 65, 64, torch.bfloat16), (3, 129, 64, torch.float16), (7, 300, 64, torch.bfloat16), (9, 257, 128, torch.bfloat16),
    (12, 1000, 64, torch.bfloat16), (15, 640, 128, torch.float16), (17, 129, 96, torch.bfloat16), (70, 1000, 64, torch.bfloat16),
    (5, 700, 64, torch.float32), (12, 128, 64, torch.float32), (77, 1000, 64, torch.float32), (17, 4096, 128, torch.bfloat16),
    (36, 4096, 128, torch.bfloat16), (3, 32768, 128, torch.bfloat16)])
@pytest.mark.parametrize("causal", [True, False])
def test_every_tile_is_computed(heads, S, D, dtype, causal):
    from metalhlo_amd import kernels
    g = torch.Generator(device="cuda").manual_seed(heads * 100000 + S)
    q, k, v = (torch.randn(1, heads, S, D, generator=g, device="cuda").to(dtype) for _ in range(3))
    out = torch.full_like(q, float("nan"))
    kernels.flash_attention(q, k, v, is_causal=causal, out=out)
    assert bool(torch.isfinite(out).all())
    rows = torch.arange(31 if S > 31 else 0, S, 32, device="cuda")
    for h in range(heads):
        scores = q[0, h, rows].double() @ k[0, h].double().T / D ** 0.5
        if causal:
            scores.masked_fill_(torch.arange(S, device="cuda") > rows[:, None], float("-inf"))
        exp = torch.softmax(scores, -1) @ v[0, h].double()
        err = (out[0, h, rows].double() - exp).norm(dim=-1) / exp.norm(dim=-1)
        assert float(err.max()) <= 2 * BOUND[dtype], (h, float(err.max()))
