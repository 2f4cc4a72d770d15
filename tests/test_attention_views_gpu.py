"""Attention on views beyond the 16-bit types with D 64 / 128 (mhip_flash_attention_views), and the programs whose head split and
merge become such views: the same bits as the packed tensors give, on both fp32 kernels (128 rows, keys over the waves)
and in the padded head sizes; what the packed form refuses stays refused."""
import ctypes as C

import numpy as np
import pytest
import torch

from metalhlo_amd import _lib, capi, kernels
from metalhlo_amd import programs as P

pytestmark = pytest.mark.gpu
CODE = kernels.DTYPE_CODE


@pytest.mark.parametrize("dtype,D", [(torch.float32, 32), (torch.float32, 64), (torch.float32, 96), (torch.float32, 128),
                                     (torch.bfloat16, 32), (torch.float16, 72)])
@pytest.mark.parametrize("B,H,S", [(1, 2, 1), (2, 3, 33), (2, 12, 200), (24, 12, 129)])
def test_views_give_the_bits_of_packed_tensors(dtype, D, B, H, S):
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(S + D)
    x = torch.randn(B, S, 3, H, D, generator=g, device="cuda").to(dtype)
    q, k, v = x.permute(2, 0, 3, 1, 4).unbind(0)
    mask = torch.zeros(B, 1, S, S, dtype=dtype, device="cuda")
    mask[:, :, :, (S + 1) // 2:] = float("-inf")
    for causal, m in ((True, None), (False, None), (False, mask)):
        want = kernels.flash_attention(q.contiguous(), k.contiguous(), v.contiguous(), is_causal=causal, mask=m)
        out = torch.full((B, S, H, D), float("nan"), dtype=dtype, device="cuda")
        W = 3 * H * D
        st = (C.c_int64 * 12)(*([S * W, D, W] * 3 + [S * H * D, D, H * D]))
        assert lib.mhip_flash_attention_views(torch.cuda.current_stream().cuda_stream, q.data_ptr(), k.data_ptr(), v.data_ptr(), m.data_ptr() if m is not None else None,
                                              out.data_ptr(), B, H, S, S, D, D ** -0.5, int(causal), S * S, 0, CODE[dtype], C.addressof(st)) == 0
        # (up to 16 queries without the causal rule take another kernel where they are packed)
        if dtype != torch.float32 and S <= 16 and not causal:
            continue
        assert torch.equal(out.permute(0, 2, 1, 3), want)


@pytest.mark.parametrize("dtype,D", [(torch.float32, 32), (torch.float32, 64), (torch.float32, 128), (torch.bfloat16, 32), (torch.float16, 72)])
@pytest.mark.parametrize("B,H", [(2, 3), (24, 12)])
@pytest.mark.parametrize("S", [1, 5, 27, 28, 33, 40])
def test_nothing_behind_the_last_key_counts(dtype, D, B, H, S):
    """Rows of NaN behind the last key of every sequence, the other sequences' rows among them: a view reads what it spans."""
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(S + D)
    rows, W = S + 96, 3 * H * D
    x = torch.full((B, rows, 3, H, D), float("nan"), dtype=dtype, device="cuda")
    x[:, :S] = torch.randn(B, S, 3, H, D, generator=g, device="cuda").to(dtype)
    q, k, v = x[:, :S].permute(2, 0, 3, 1, 4).unbind(0)
    st = (C.c_int64 * 12)(*([rows * W, D, W] * 3 + [S * H * D, D, H * D]))
    for causal in (False, True):
        want = kernels.flash_attention(q.contiguous(), k.contiguous(), v.contiguous(), is_causal=causal)
        out = torch.full((B, S, H, D), float("nan"), dtype=dtype, device="cuda")
        assert lib.mhip_flash_attention_views(torch.cuda.current_stream().cuda_stream, q.data_ptr(), k.data_ptr(), v.data_ptr(), None, out.data_ptr(),
                                              B, H, S, S, D, D ** -0.5, int(causal), 0, 0, CODE[dtype], C.addressof(st)) == 0
        got = out.permute(0, 2, 1, 3)
        assert torch.isfinite(got).all()
        assert torch.equal(got, want)


def test_refused_views():
    lib = _lib.load()
    x = torch.zeros(4096, dtype=torch.float32, device="cuda")
    p = x.data_ptr()
    for strides, D in (([2048, 1024, 130] * 4, 64), ([2048, 1024, 40] * 4, 40)):      # no 16-byte pieces; no such head size
        st = (C.c_int64 * 12)(*strides)
        assert lib.mhip_flash_attention_views(None, p, p, p, None, p, 1, 1, 8, 8, D, 1.0, 0, 0, 0, CODE[torch.float32], C.addressof(st)) == 2


@pytest.fixture(scope="module")
def sess():
    s = capi.Session()
    yield s
    s.close()


def _args(B, S, H, D, F, dtype):
    rng, d = np.random.default_rng(3), H * D
    n = lambda *s, m=0.05: (m * rng.standard_normal(s)).astype(np.float32)      # noqa: E731
    a = [n(B, S, d, m=1), 1 + n(d), n(d), n(d, 3 * d), n(3 * d), n(d, d), n(d), 1 + n(d), n(d), n(d, F), n(F), n(F, d), n(d)]
    return [(x, "f32") for x in a] if dtype == "f32" else [(torch.from_numpy(x).bfloat16().view(torch.int16).numpy().view(np.uint16), "bf16") for x in a]


@pytest.mark.parametrize("dtype,H,D", [("f32", 12, 64), ("f32", 4, 32), ("bf16", 4, 32)])
@pytest.mark.parametrize("B,S", [(1, 37), (2, 130)])
def test_a_block_gives_the_bits_of_its_copies(sess, dtype, H, D, B, S):
    """Level 1 runs the same kernels with the split and the merge copied; a split value that the program also returns is
    still produced."""
    text, args = P.transformer_block(B, S, H, D, 256, dtype), _args(B, S, H, D, 256, dtype)
    hs = "tensor<%dx%dx%dx%dx%s>" % (B, H, S, D, dtype)
    x3 = "tensor<%dx%dx%dx%s>" % (B, S, H * D, dtype)
    shared = text.replace(") -> %s {" % x3, ") -> (%s, %s) {" % (x3, hs)).replace("return %%res2 : %s" % x3, "return %%res2, %%kh : %s, %s" % (x3, hs))
    for t in (text, shared):
        got = []
        for level in (1, 2, 3):
            exe = sess.compile(t, level)
            runs = [sess.run(exe, args) for _ in range(3)]
            got.append(runs)
            sess.lib.mhlo_executable_destroy(exe)
        for runs in got:
            for r in runs:
                assert all(np.array_equal(x, y) for x, y in zip(r, got[0][0])) and len(r) == len(got[0][0])
