"""GPU test of the order in which finish_norm adds parts up: four are asked for at a time, and the sum is the one of fp32 additions from the first part on, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [8, 768, 1024, 1032])
@pytest.mark.parametrize("parts", [1, 2, 3, 4, 5, 7, 8, 9, 13])
def test_parts_in_order(parts, N):
    from metalhlo_amd import kernels
    g = torch.Generator(device="cuda").manual_seed(parts * 10000 + N)
    sums = torch.randn(parts, 33, N, generator=g, device="cuda") * 10.0 ** torch.randint(-3, 4, (parts, 33, N), generator=g, device="cuda")
    sums[-1, 5] = float("inf")
    sums[0, 6], sums[-1, 6] = -0.0, -0.0
    total = torch.zeros(33, N, device="cuda")
    for p in sums:
        total = total + p
    c, h = kernels.finish_norm(sums, None, torch.zeros(33, N, dtype=torch.bfloat16, device="cuda"), (torch.ones(N, device="cuda"), None, 1e-5))
    assert torch.equal(c, total.to(torch.bfloat16))
    assert bool(h[:5].isfinite().all()) and not bool(h[5].isfinite().any())
