"""GPU test that finish_norm adds the parts of a sum up from the first one on, with parts whose order decides the result by whole units: two of them are 2^26 and -2^26, beside
which the others, whole numbers of up to three, are lost, so that what is left is the sum of those behind the second.  It is a whole number that bf16 holds."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _parts(parts, rows, N):
    g = torch.Generator().manual_seed(parts * 10000 + N)
    small = torch.randint(1, 4, (parts, rows, N), generator=g) * (2 * torch.randint(0, 2, (parts, rows, N), generator=g) - 1)
    place = torch.rand(parts, rows, N, generator=g).argsort(0)
    return torch.where(place == 0, 2 ** 26, torch.where(place == 1, -2 ** 26, small)).float()


def _added(parts):
    total = torch.zeros_like(parts[0])
    for p in parts:
        total = total + p
    return total


def _grouped(parts, size):
    return _added([_added(parts[i:i + size]) for i in range(0, len(parts), size)])


@pytest.mark.parametrize("N", [8, 768, 1024, 1032, 4096])
@pytest.mark.parametrize("parts", [3, 4, 5, 6, 7, 8, 9, 13])
def test_parts_are_added_from_the_first_on(parts, N):
    from metalhlo_amd import kernels
    sums = _parts(parts, 33, N)
    total = _added(sums)
    # other orders show in these numbers, in bf16 too: the last part first, pairs first where there are two, fours first where there are two of several parts
    others = [_added(sums.flip(0))] + ([_grouped(sums, 2)] if parts >= 4 else []) + ([_grouped(sums, 4)] if parts >= 6 else [])
    assert all(bool((other.bfloat16() != total.bfloat16()).float().mean() > 0.05) for other in others)
    c, h = kernels.finish_norm(sums.cuda(), None, torch.zeros(33, N, dtype=torch.bfloat16, device="cuda"), (torch.ones(N, device="cuda"), None, 1e-5))
    assert torch.equal(c.cpu(), total.bfloat16())
    assert bool(h.isfinite().all())
