"""GPU test that a query's bits in decode attention (attention_decode.hip) do not follow from how many queries are beside it, for numbers of heads and keys at the edges of what chooses a
workgroup's waves and over up to sixteen parts of the keys (more of them are added up by as many threads as the number of queries leaves)."""
import pytest
import torch

from tests.util import NAME

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("heads,Skv,D", [(1, 130, 64), (12, 256, 128), (256, 250, 128), (192, 129, 64), (128, 512, 128), (128, 256, 64), (16, 2048, 64), (64, 1000, 128), (257, 300, 64), (256, 128, 128)], ids=str)
def test_queries_beside_it(heads, Skv, D, dtype):
    from metalhlo_amd import kernels
    g = torch.Generator(device="cuda").manual_seed(heads * 1000 + Skv)
    q, k, v = (torch.randn(1, heads, n, D, generator=g, device="cuda").to(dtype) for n in (16, Skv, Skv))
    all_ = kernels.flash_attention(q, k, v)
    for n in (1, 4, 8, 9):
        assert torch.equal(kernels.flash_attention(q[:, :, :n].contiguous(), k, v), all_[:, :, :n])
