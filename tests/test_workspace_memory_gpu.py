"""A workspace only makes a product faster: where the device has no room for one the call takes its form without, with the same
bits from 193 rows on below K 4096."""
import ctypes as C

import numpy as np
import pytest
import torch

from metalhlo_amd import _lib, capi, kernels

pytestmark = pytest.mark.gpu

M, N, K = 301, 16001, 4001                     # both operands are copied: 131 MB


def _need():
    return _lib.load().mhip_gemm_workspace(M, N, K, 1, 0, 0, kernels.DTYPE_CODE[torch.bfloat16])


def _operands():
    g = torch.Generator(device="cuda").manual_seed(1)
    return torch.randn(M, K, generator=g, device="cuda").bfloat16(), torch.randn(K, N, generator=g, device="cuda").bfloat16()


def test_matmul():
    a, b = _operands()
    torch.cuda.empty_cache()                   # (blocks of their own for what stays)
    out, want = (torch.empty(M, N, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    kernels.matmul(a, b, out=want)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    assert _need() > 96 << 20
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (64 << 20)) / torch.cuda.mem_get_info()[1])
        with pytest.raises(torch.OutOfMemoryError):
            torch.empty(_need(), dtype=torch.uint8, device="cuda")
        kernels.matmul(a, b, out=out)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(out, want)


@pytest.fixture(scope="module")
def sess():
    s = capi.Session()
    yield s
    s.close()


@pytest.mark.parametrize("arena", ["1", "0"])
def test_compiled_program(sess, arena, monkeypatch):
    x, w, y = f"tensor<{M}x{K}xbf16>", f"tensor<{K}x{N}xbf16>", f"tensor<{M}x{N}xbf16>"
    text = (f"func.func @main(%x: {x}, %w: {w}) -> {y} {{\n    %y = stablehlo.dot_general %x, %w, contracting_dims = [1] x [0] : ({x}, {w}) -> {y}\n"
            f"    return %y : {y}\n}}")
    ins = [sess.buffer(t.view(torch.int16).cpu().numpy().view(np.uint16), "bf16") for t in _operands()]

    def execute(exe):
        args, outs, n = (C.c_void_p * 2)(*ins), (C.c_void_p * 1)(), C.c_int32()
        rc = sess.lib.mhlo_execute(exe, args, 2, outs, C.byref(n))
        assert rc == 0, sess.lib.mhlo_get_last_error()
        r = sess.to_numpy(outs[0])
        sess.lib.mhlo_buffer_destroy(outs[0])
        return r

    monkeypatch.setenv("METALHLO_ARENA", "1")       # (its memory goes back with the executable)
    exe = sess.compile(text)
    want = execute(exe)
    sess.lib.mhlo_executable_destroy(exe)
    monkeypatch.setenv("METALHLO_ARENA", arena)
    exe, held = sess.compile(text), []
    torch.cuda.empty_cache()
    for size in (8 << 30, 1 << 30, 128 << 20, 32 << 20):
        while torch.cuda.mem_get_info()[0] - size > 64 << 20:
            try:
                held.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
            except torch.OutOfMemoryError:
                break
    try:
        assert torch.cuda.mem_get_info()[0] < _need()
        got = execute(exe)
    finally:
        held.clear()
        torch.cuda.empty_cache()
    assert np.array_equal(got, want)
    sess.lib.mhlo_executable_destroy(exe)
    for b in ins:
        sess.lib.mhlo_buffer_destroy(b)
