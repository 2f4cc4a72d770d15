"""GPU parity of the GEMM kernels for problems with few rows or few tiles (gemm_skinny.hip,
gemm_mid.hip): edges of their tiles, remainders, operands without vector alignment, split K.

Bound: a product of K terms summed in fp32 is off by at most K 2^-24 of sum |a||b|; the result is then
rounded once to its type (unit roundoff 2^-8 for bf16's 8-bit significand, 2^-11 for f16's 11), twice with a
residual."""
import numpy as np
import pytest
import torch

from tests.util import NAME, as_f64, to_dev

pytestmark = pytest.mark.gpu
ROUNDOFF = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}


def _check(M, N, K, dtype, ta, tb, residual, seed=7, batch=()):
    from metalhlo_amd import kernels
    rng = np.random.default_rng(seed)
    a = to_dev(rng.standard_normal(batch + ((K, M) if ta else (M, K))), dtype)
    b = to_dev(rng.standard_normal(batch + ((N, K) if tb else (K, N))), dtype)
    bias = None if batch else to_dev(rng.standard_normal(N), dtype)
    r = to_dev(rng.standard_normal(batch + (M, N)), dtype) if residual else None
    guard = torch.full((int(np.prod(batch + (M,))) * N + 64,), float("nan"), dtype=dtype, device="cuda")
    out = guard[:-64].view(batch + (M, N))
    kernels.matmul(a, b, bias=bias, activation="relu", trans_a=ta, trans_b=tb, residual=r, out=out)
    A, B = as_f64(a), as_f64(b)
    A, B = (np.swapaxes(A, -1, -2) if ta else A), (np.swapaxes(B, -1, -2) if tb else B)
    e = A @ B + (0 if bias is None else as_f64(bias))
    fp32 = (K + 2) * 2.0 ** -24 * (np.abs(A) @ np.abs(B) + (0 if bias is None else np.abs(as_f64(bias))))
    e = np.maximum(e, 0)
    bound = fp32 + ROUNDOFF[dtype] * (np.abs(e) + fp32)
    if residual:
        e = e + as_f64(r)
        bound = bound + ROUNDOFF[dtype] * (np.abs(e) + bound)
    assert np.all(np.abs(as_f64(out) - e) <= bound + 1e-30), (M, N, K, dtype, ta, tb)
    assert torch.isnan(guard[-64:]).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=lambda d: NAME[d])
@pytest.mark.parametrize("tb", [False, True], ids=["nn", "nt"])
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (1, 64, 8), (15, 31, 33), (16, 40, 264), (17, 4104, 2056), (32, 520, 6400), (33, 50, 100), (64, 129, 1027),
                                   (4, 4096, 4096), (16, 8200, 72)], ids=lambda v: str(v))
def test_few_rows(M, N, K, tb, dtype):
    _check(M, N, K, dtype, False, tb, residual=M % 2 == 1)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("layout", [(False, False), (False, True), (True, False), (True, True)], ids=["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("M,N,K", [(40, 8, 8), (72, 64, 136), (136, 136, 1000), (192, 264, 3000), (200, 392, 264), (264, 520, 4104), (768, 1536, 4096), (1000, 1000, 72)],
                         ids=lambda v: str(v))
def test_few_tiles(M, N, K, layout, dtype):
    _check(M, N, K, dtype, *layout, residual=N % 16 == 8)


def test_few_tiles_batched():
    _check(72, 200, 136, torch.bfloat16, False, False, True, batch=(5,))
    _check(20, 77, 45, torch.float32, False, True, True, batch=(3,))


def test_splitting_needs_its_workspace(lib):
    """Without the workspace the same problem runs unsplit; a misaligned one is refused."""
    M, N, K = 768, 1536, 8192
    need = lib.mhip_gemm_workspace(M, N, K, 1, 1, 0, 3)
    assert need > 0 and lib.mhip_gemm_workspace(4096, 4096, 4096, 1, 0, 0, 3) == 0
    a, b = (torch.randn(K, n, device="cuda").bfloat16() for n in (M, N))
    c = [torch.empty(M, N, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    args = lambda out: (torch.cuda.current_stream().cuda_stream, a.data_ptr(), b.data_ptr(), None, None, out.data_ptr(), M, N, K, 1, 0, 0, M * N, 1, 0, 0, 3)
    assert lib.mhip_gemm_ws(*args(c[0]), ws.data_ptr(), need) == 0
    assert lib.mhip_gemm_ws(*args(c[1]), None, 0) == 0
    assert lib.mhip_gemm_ws(*args(c[1]), ws.data_ptr() + 8, need - 8) == 1
    e = a.double().t().cpu() @ b.double().cpu()
    for out in c:        # K 2^-24 sum |a||b| is below 2^-8 sqrt(K) here; one rounding to bf16
        assert ((out.double().cpu() - e).abs() <= 2.0 ** -8 * (e.abs() + K ** 0.5)).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=lambda d: NAME[d])
@pytest.mark.parametrize("M,N,K", [(16, 1, 4096), (13, 1, 4100), (33, 1, 4099), (16, 2, 4096), (16, 3, 4096), (40, 3, 4099), (7, 5, 4096)], ids=lambda v: str(v))
def test_split_sums_of_few_columns(M, N, K, dtype):
    """A split K whose result has fewer columns than the four elements a thread of gemm_finish_kernel makes: the bias
    of each element is that of its own column.  What lies behind the bias in memory is NaN."""
    from metalhlo_amd import _lib, kernels
    code = {torch.bfloat16: 3, torch.float32: 1}[dtype]
    assert _lib.load().mhip_gemm_workspace(M, N, K, 1, 0, 1, code) > 0           # (the problem is split)
    rng = np.random.default_rng(M)
    a, b = to_dev(rng.standard_normal((M, K)), dtype), to_dev(rng.standard_normal((N, K)), dtype)
    bias = to_dev(np.concatenate([rng.standard_normal(N) * 100, np.full(16, np.nan)]), dtype)[:N]
    got = as_f64(kernels.matmul(a, b, bias=bias, trans_b=True))
    A, B, c = as_f64(a), as_f64(b).T, as_f64(bias)
    e = A @ B + c
    fp32 = (K + 2) * 2.0 ** -24 * (np.abs(A) @ np.abs(B) + np.abs(c))
    assert np.all(np.abs(got - e) <= fp32 + ROUNDOFF[dtype] * (np.abs(e) + fp32))


@pytest.mark.parametrize("M,line,tb,dtype", [(4, 2560, False, torch.bfloat16), (16, 3584, True, torch.bfloat16), (17, 2560, True, torch.bfloat16), (12, 2560, True, torch.float32),
                                             (40, 3072, False, torch.float32)], ids=str)
def test_both_sides_of_the_split_lines(M, line, tb, dtype):
    """From K = line on a few-row product is split; eight k before it is not."""
    from metalhlo_amd import _lib
    code = {torch.bfloat16: 3, torch.float32: 1}[dtype]
    assert _lib.load().mhip_gemm_workspace(M, 264, line, 1, 0, int(tb), code) > 0
    assert _lib.load().mhip_gemm_workspace(M, 264, line - 8, 1, 0, int(tb), code) == 0
    for K in (line - 8, line):
        _check(M, 264, K, dtype, False, tb, residual=True)


@pytest.mark.parametrize("N,K,dtype", [(768, 768, torch.bfloat16), (2304, 768, torch.float16), (768, 3072, torch.bfloat16), (768, 4088, torch.bfloat16), (770, 771, torch.bfloat16),
                                       (768, 3072, torch.float32), (2304, 770, torch.float32)], ids=str)
@pytest.mark.parametrize("tb", [False, True], ids=["nn", "nt"])
def test_rows_of_a_batch_keep_their_bits(N, K, tb, dtype):
    """From 193 rows on, and K below 4096, the kernels add a row's products in one order: more rows beside it change nothing."""
    from metalhlo_amd import kernels
    rng = np.random.default_rng(K)
    a, b = to_dev(rng.standard_normal((3000, K)), dtype), to_dev(rng.standard_normal((N, K) if tb else (K, N)), dtype)
    want = kernels.matmul(a[:193].contiguous(), b, trans_b=tb)
    for M in (256, 1000, 3000):
        assert torch.equal(kernels.matmul(a[:M].contiguous(), b, trans_b=tb)[:193], want), M


def test_workspaces_under_capture_and_on_a_side_stream():
    """Split products and a split decode step whose workspaces are allocated per call: recorded into one graph and replayed
    with new inputs, with eager calls of the same kernels between the replays, and run on another stream behind a long
    product there; every result is the eager one bit for bit."""
    from metalhlo_amd import kernels
    rng = np.random.default_rng(4)
    t = lambda *shape: to_dev(rng.standard_normal(shape), torch.bfloat16)  # noqa: E731
    w, x, dy, k, v = t(4096, 512), t(4, 4096), t(4096, 512), t(2, 4, 2100, 64), t(2, 4, 2100, 64)

    def step(a, q):
        return (kernels.matmul(a, w), kernels.flash_attention(q, k, v), kernels.matmul(dy, w, trans_a=True, activation="relu"), kernels.matmul(a * 2, dy))
    a, q = x.clone(), t(2, 4, 1, 64)
    step(a, q)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step(a, q)
    for i in range(4):
        na, nq = t(4, 4096), t(2, 4, 1, 64)
        a.copy_(na)
        q.copy_(nq)
        graph.replay()
        want = step(na, nq)
        step(nq.new_ones(4, 4096), nq)
        assert all(torch.equal(o, e) for o, e in zip(out, want)), i
    big, side = t(8192, 4096), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        late = kernels.matmul(big, t(4096, 4096))[:4].contiguous()
        got = step(late, nq)
    torch.cuda.current_stream().wait_stream(side)
    assert all(torch.equal(o, e) for o, e in zip(got, step(late, nq)))


@pytest.mark.parametrize("M,N,K", [(8, 256, 4096), (1, 64, 3584)], ids=lambda v: str(v))
def test_few_rows_off_16_bytes_are_split(lib, M, N, K):
    """Sizes whose strips hold all of K on 16 bytes: other addresses are served in parts, which lie in the workspace afterwards."""
    need = lib.mhip_gemm_workspace(M, N, K, 1, 0, 1, 3)
    assert need > 0
    a, b = torch.randn(M, K, device="cuda").bfloat16(), torch.randn(N * K + 1, device="cuda").bfloat16()
    for off in (0, 1):
        w = b[off:off + N * K].view(N, K)
        out, ws = torch.empty(M, N, dtype=torch.bfloat16, device="cuda"), torch.full((need,), 170, dtype=torch.uint8, device="cuda")
        assert lib.mhip_gemm_ws(torch.cuda.current_stream().cuda_stream, a.data_ptr(), w.data_ptr(), None, None, out.data_ptr(), M, N, K, 1, 0, 0, 0, 0, 1, 0, 3,
                                ws.data_ptr(), need) == 0
        e, fp32 = a.double() @ w.double().t(), K * 2.0 ** -24 * (a.double().abs() @ w.double().abs().t())
        assert ((out.double() - e).abs() <= fp32 + ROUNDOFF[torch.bfloat16] * (e.abs() + fp32)).all()
        assert bool((ws[:2 * M * N * 4] != 170).any()) == bool(off)
