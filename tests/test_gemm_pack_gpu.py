"""16-bit products whose operands are copied to rows on 16-byte boundaries, against the kernel that reads them as they are (the
same bits below K 4096) and float64: one or both operands off, k padded to whole stages, rows and columns ragged."""
import pytest
import torch

from metalhlo_amd import _lib, kernels

pytestmark = pytest.mark.gpu

EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _inside_nan(shape, dtype, g, scale=1.0):
    """A dense matrix with NaN in front of it and behind it: what lies outside must not be multiplied."""
    n = shape[0] * shape[1]
    buf = torch.full((n + 96,), float("nan"), dtype=dtype, device="cuda")
    x = buf[16:16 + n].view(*shape)
    x.copy_(torch.randn(*shape, generator=g, device="cuda") * scale)
    return x


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(201, 203, 3001), (769, 515, 2001), (264, 257, 3008), (257, 264, 3016), (2049, 2051, 2041), (193, 9, 4999), (300, 1, 3002)])
def test_copies(dtype, ta, tb, M, N, K):
    lib, code = _lib.load(), kernels.DTYPE_CODE[dtype]
    g = torch.Generator(device="cuda").manual_seed(K)
    a, b = _inside_nan((K, M) if ta else (M, K), dtype, g), _inside_nan((N, K) if tb else (K, N), dtype, g, K ** -0.5)
    bias, res = torch.randn(N, generator=g, device="cuda").to(dtype), torch.randn(M, N, generator=g, device="cuda").to(dtype)

    def product(bytes_):
        out = torch.full((M * N + 64,), 7.0, dtype=dtype, device="cuda")
        work = torch.full((max(bytes_, 1),), 255, dtype=torch.uint8, device="cuda")
        assert lib.mhip_gemm_ws(torch.cuda.current_stream().cuda_stream, a.data_ptr(), b.data_ptr(), bias.data_ptr(), res.data_ptr(), out.data_ptr(), M, N, K, 1, 0, 0, 0,
                                ta, tb, 1, code, work.data_ptr() if bytes_ else None, bytes_) == 0
        assert (out[M * N:] == 7.0).all()
        return out[:M * N].view(M, N)

    need = lib.mhip_gemm_workspace(M, N, K, 1, ta, tb, code)
    if (ta and M % 8 != 0) or (not ta and K % 8 != 0) or (tb and K % 8 != 0) or (not tb and N % 8 != 0):
        assert need >= 2 * min(M, N) * K
    got = product(need)
    exp = torch.relu((a.double().T if ta else a.double()).contiguous() @ (b.double().T if tb else b.double()).contiguous() + bias.double())
    assert ((got.double() - exp - res.double()).abs() <= 2 * EPS[dtype] * (exp.abs() + res.double().abs()).clamp(min=1.0)).all()
    if K < 4096:
        assert torch.equal(got, product(0))
    assert torch.isfinite(product(need // 2)).all()              # less than the copies take: as they are


def test_copies_from_a_graph():
    g = torch.Generator(device="cuda").manual_seed(1)
    a, b = torch.randn(301, 3001, generator=g, device="cuda").bfloat16(), torch.randn(3001, 501, generator=g, device="cuda").bfloat16()
    kernels.matmul(a, b)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = kernels.matmul(a, b)
    for i in range(3):
        a.normal_(generator=g)
        want = kernels.matmul(a, b)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tile", [2560, 2561, 2564, 2566, 2567, 2568, 2569, 2570])
@pytest.mark.parametrize("ta", [0, 1])
def test_the_last_row_of_k_ends_in_an_odd_column(monkeypatch, dtype, tile, ta):
    """The descriptors of the ring kernels reach the last element of a copied row whose length is odd: only the last k is not zero."""
    lib, code = _lib.load(), kernels.DTYPE_CODE[dtype]
    M, N, K = 3841 if ta else 3848, 6273, 3008               # 192 tiles of 256x384; K is whole stages, so nothing is padded behind it
    g = torch.Generator(device="cuda").manual_seed(tile)
    a, b = torch.zeros((K, M) if ta else (M, K), dtype=dtype, device="cuda"), torch.zeros(K, N, dtype=dtype, device="cuda")
    u, v = torch.randn(M, generator=g, device="cuda").to(dtype), torch.randn(N, generator=g, device="cuda").to(dtype)
    a[K - 1 if ta else slice(None), slice(None) if ta else K - 1] = u
    b[K - 1] = v
    need = lib.mhip_gemm_workspace(M, N, K, 1, ta, 0, code)
    work, out = torch.full((need,), 255, dtype=torch.uint8, device="cuda"), torch.empty(M, N, dtype=dtype, device="cuda")
    monkeypatch.setenv("MHIP_GEMM_TILE", str(tile))
    assert lib.mhip_gemm_ws(torch.cuda.current_stream().cuda_stream, a.data_ptr(), b.data_ptr(), None, None, out.data_ptr(), M, N, K, 1, 0, 0, 0, ta, 0, 0, code,
                            work.data_ptr(), need) == 0
    assert lib.mhip_gemm_last_variant() == tile
    assert torch.equal(out, (u.float()[:, None] * v.float()[None, :]).to(dtype))


@pytest.mark.parametrize("K", [4065, 4090, 4095])
@pytest.mark.parametrize("N,M", [(300, (200, 1001, 2001)), (1001, (264, 1001))])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_padding_k_to_4096_leaves_the_order_of_a_sum(ta, tb, N, M, K):
    """From 193 rows on a row has the same bits for any number of rows while the caller's K is below 4096, also where the copies
    have 4096 columns."""
    lib, code = _lib.load(), kernels.DTYPE_CODE[torch.bfloat16]
    g = torch.Generator(device="cuda").manual_seed(K)
    a, b = torch.randn(max(M), K, generator=g, device="cuda").bfloat16(), torch.randn(K, N, generator=g, device="cuda").bfloat16()
    rhs, rows = b.T.contiguous() if tb else b, {}
    for m in M:
        lhs, need = a[:m].T.contiguous() if ta else a[:m], lib.mhip_gemm_workspace(m, N, K, 1, ta, tb, code)
        assert need >= 2 * (m + N) * K                            # both are copied
        for bytes_ in (need, 0):
            out, work = torch.empty(m, N, dtype=torch.bfloat16, device="cuda"), torch.empty(need, dtype=torch.uint8, device="cuda")
            assert lib.mhip_gemm_ws(torch.cuda.current_stream().cuda_stream, lhs.data_ptr(), rhs.data_ptr(), None, None, out.data_ptr(), m, N, K, 1, 0, 0, 0, ta, tb, 0,
                                    code, work.data_ptr() if bytes_ else None, bytes_) == 0
            rows[m, bytes_ > 0] = out[:min(M)]
    assert all(torch.equal(v, rows[M[0], False]) for v in rows.values())
