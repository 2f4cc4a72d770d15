"""Host-side launch helpers over the kernel C-ABI.

torch is used only as plumbing here: it owns device memory and the current HIP
stream.  Every function validates shapes, allocates the output and calls one
``mhip_*`` entry point through ctypes; none has a fallback implementation.

The names follow the reference's kernel registry
(Sources/MetalHLOCore/Metal/Kernels/KernelRegistry.swift:17): softmax,
layer_norm, rms_norm, gelu, flash_attention, plus matmul.
"""
from __future__ import annotations

import ctypes as C
import math
from typing import Optional

import torch

from . import _lib

# MHLOElementType numbering (Sources/CMetalHLO/include/metalhlo.h:62-76)
DTYPE_CODE = {
    torch.float16: 0, torch.float32: 1, torch.float64: 2, torch.bfloat16: 3, torch.bool: 4,
    torch.int8: 5, torch.int16: 6, torch.int32: 7, torch.int64: 8, torch.uint8: 9,
}
ACTIVATION_CODE = {"none": 0, "relu": 1, "gelu": 2, "silu": 3, "tanh": 4, "sigmoid": 5, "gelu_exact": 6}


_native = None


def _host():
    """The compiled host path (csrc/python/native.cpp): checks, result tensor, stream and launch."""
    global _native
    if _native is None:
        _lib.load()                                   # (names the build command when the library is missing)
        _native = _lib.load_native()
    return _native


def _code(t: torch.Tensor) -> int:
    try:
        return DTYPE_CODE[t.dtype]
    except KeyError:
        raise TypeError(f"unsupported dtype {t.dtype}") from None


def _dev(*ts):
    for t in ts:
        if t is None:
            continue
        if not t.is_cuda:
            raise RuntimeError("metalhlo_amd kernels need device tensors (no CPU path exists)")
        if not t.is_contiguous():
            raise ValueError("tensors must be dense row-major (contiguous)")


def _stream() -> int:
    return torch.cuda.current_stream().cuda_stream


def _ptr(t: Optional[torch.Tensor]):
    return None if t is None else t.data_ptr()


def softmax(x: torch.Tensor, axis: int = -1) -> torch.Tensor:
    return (_native or _host()).softmax(x, axis)


def layer_norm(x, gamma=None, beta=None, eps: float = 1e-5):
    return (_native or _host()).layer_norm(x, gamma, beta, eps)


def rms_norm(x, gamma=None, eps: float = 1e-5):
    return (_native or _host()).rms_norm(x, gamma, eps)


def bias_gelu(x, bias=None, exact: bool = False):
    """gelu(x + bias): the tanh approximation, or with `exact` 0.5 v (1 + erf(v / sqrt 2))."""
    return (_native or _host()).bias_gelu(x, bias, exact)


def gelu(x, exact: bool = False):
    return bias_gelu(x, None, exact)


def matmul(a, b, bias=None, activation: str = "none", trans_a: bool = False,
           trans_b: bool = False, out: Optional[torch.Tensor] = None,
           residual: Optional[torch.Tensor] = None):
    """act(op(a) @ op(b) + bias) (+ residual, which has the result's shape and may be `out`);
    leading dims of `a` are batch dims when `b` is batched too, otherwise they fold into M.  Up to 192 rows,
    and from K 4096 on, the last bits of a row may depend on how many rows there are."""
    return (_native or _host()).matmul(a, b, bias, ACTIVATION_CODE[activation], trans_a, trans_b, out, residual)


def flash_attention(q, k, v, scale: Optional[float] = None, is_causal: bool = False,
                    mask: Optional[torch.Tensor] = None, out: Optional[torch.Tensor] = None):
    """softmax(scale * q k^T + mask, causal) v for [B,H,S,D] tensors.
    Default scale 1/sqrt(D) (FlashAttentionKernel.swift:55).  q, k, v (and `out`, when given)
    may be views with arbitrary batch / head / row strides as long as the last axis is
    contiguous, e.g. slices of a fused QKV projection; packed tensors take the plain entry.  The last bits of a
    row may depend on B * H for fp32 and for up to 16 queries without the causal rule, as mhip.h says."""
    return (_native or _host()).flash_attention(q, k, v, scale, is_causal, mask, out)


def linear(x, weight, bias=None, activation: str = "none", trans_b: bool = False, residual=None, parts: int = 0, ahead=()):
    """act(x @ op(weight) + bias) (+ residual) in x's 16-bit type with parameters held in fp32, each rounded to that type at
    use: what convert and matmul compute, in one launch; `linear_served` says for which sizes.  `parts` > 0 gives
    the fp32 sums of so many shares of K ([parts, M, N], for finish_norm; `linear_parts` says how many).  `ahead`: up to two
    weight matrices [K, N] that the next calls read (a hint, see mhip_linear_w32)."""
    return (_native or _host()).linear(x, weight, bias, residual, ACTIVATION_CODE[activation], trans_b, parts, ahead)


def linear_served(M: int, N: int, K: int, dtype) -> bool:
    return bool(_lib.load().mhip_linear_w32_ok(M, N, K, DTYPE_CODE[dtype]))


def linear_parts(M: int, N: int, K: int) -> int:
    return _lib.load().mhip_linear_w32_parts(M, N, K)


def linear_layer(x, weight, bias=None, activation: str = "none", residual=None, norm=None, ahead=()):
    """`linear` with weight [K, N], of LayerNorm(x) where `norm` is (gamma, beta, eps) in fp32; a long K without it is split over the device and
    added up in the same launch.  `linear_norm_served` says which rows are normalised."""
    return (_native or _host()).linear_layer(x, norm, weight, bias, residual, ACTIVATION_CODE[activation], ahead)


def linear_norm_served(M: int, N: int, K: int, dtype) -> bool:
    return bool(_lib.load().mhip_linear_w32_norm_ok(M, N, K, DTYPE_CODE[dtype]))


def tied_head(x, weight):
    """x [M, K] @ weight [N, K].T in x's 16-bit type, the fp32 weight rounded to it at use; `tied_head_served` says for which sizes."""
    return (_native or _host()).tied_head(x, weight)


def tied_head_served(M: int, N: int, K: int, dtype) -> bool:
    return bool(_lib.load().mhip_tied_head_ok(M, N, K, DTYPE_CODE[dtype]))


def matmul_sums(a, b, parts: int):
    """The fp32 sums of so many shares of K of a [M, K] @ b [K, N] in a 16-bit type: [parts, M, N], for finish_norm."""
    return (_native or _host()).matmul_sums(a, b, parts)


def matmul_sums_parts(M: int, N: int, K: int, dtype) -> int:
    """A good number of parts for these sizes, 0 where matmul_sums does not serve them."""
    return _lib.load().mhip_gemm_sums_parts(M, N, K, DTYPE_CODE[dtype])


def finish_norm(sums, bias, residual, norm):
    """(c, LayerNorm(c)) with c = round(sums.sum(0) + bias) + residual, or c = residual where sums is None; fp32 parameters."""
    return (_native or _host()).finish_norm(sums, bias, residual, *norm)


def causal_attention(qkv, batch: int, n_head: int):
    """flash_attention(is_causal=True) over a fused projection [B * S, 3 H D], read in place -> [B * S, H D]."""
    return (_native or _host()).causal_attention(qkv, batch, n_head)


def attend_project(qkv, weight, batch: int, n_head: int, ahead=()):
    """matmul of causal_attention(qkv) and the fp32 weight [H D, N], rounded at use, in one launch: fp32 sums [parts, B * S, N] for finish_norm.
    `attend_project_served` says for which sizes; `ahead` as in `linear`."""
    return (_native or _host()).attend_project(qkv, weight, batch, n_head, ahead)


def attend_project_served(batch: int, length: int, n_head: int, head_size: int, N: int, dtype) -> bool:
    return bool(_lib.load().mhip_attend_project_parts(batch, length, n_head, head_size, N, DTYPE_CODE[dtype]))


def attend_project_layer(qkv, weight, bias, residual, batch: int, n_head: int, ahead=()):
    """linear_layer(causal_attention(qkv), weight, bias, residual=residual) in one launch; `attend_project_layer_served` says for which sizes."""
    return (_native or _host()).attend_project_layer(qkv, weight, bias, residual, batch, n_head, ahead)


def attend_project_layer_served(batch: int, length: int, n_head: int, head_size: int, N: int, dtype) -> bool:
    return bool(_lib.load().mhip_attend_project_layer_ok(batch, length, n_head, head_size, N, DTYPE_CODE[dtype]))


# ---- glue -------------------------------------------------------------------
def gather_rows(table, indices):
    _dev(table, indices)
    lib = _lib.load()
    row = math.prod(table.shape[1:])
    out = torch.empty(tuple(indices.shape) + tuple(table.shape[1:]), dtype=table.dtype,
                      device=table.device)
    _lib.check(lib.mhip_gather_rows(_stream(), table.data_ptr(), indices.data_ptr(), out.data_ptr(),
                                    indices.numel(), table.shape[0], row, _code(table),
                                    _code(indices)))
    return out


def embed_tokens(ids, wte, wpe, out_dtype):
    _dev(ids, wte, wpe)
    lib = _lib.load()
    if ids.dtype != torch.int32 or ids.dim() != 2:
        raise TypeError("ids must be int32 [B,S]")
    B, S = ids.shape
    if S > wpe.shape[0]:
        raise ValueError("sequence longer than the position table")
    out = torch.empty(B, S, wte.shape[1], dtype=out_dtype, device=ids.device)
    _lib.check(lib.mhip_embed_tokens(_stream(), ids.data_ptr(), wte.data_ptr(), wpe.data_ptr(),
                                     out.data_ptr(), B, S, wte.shape[1], wte.shape[0], _code(wte),
                                     DTYPE_CODE[out_dtype]))
    return out


def add(a, b):
    _dev(a, b)
    lib = _lib.load()
    if a.shape != b.shape or a.dtype != b.dtype:
        raise ValueError("add needs equal shapes and dtypes")
    y = torch.empty_like(a)
    _lib.check(lib.mhip_add(_stream(), a.data_ptr(), b.data_ptr(), y.data_ptr(), a.numel(), _code(a)))
    return y


def rope(x, freqs):
    """Rotary position embedding: x [.., S, D]; freqs [S, D] (cos | sin halves) or [S, D / 2] (angles)."""
    _dev(x, freqs)
    lib = _lib.load()
    if x.dim() < 2 or x.shape[-1] % 2 or freqs.dtype != x.dtype:
        raise ValueError("rope needs x [.., S, D] with even D and freqs of x's element type")
    S, D = x.shape[-2], x.shape[-1]
    fd = freqs.shape[-1] if freqs.dim() else 0
    if fd not in (D, D // 2) or freqs.numel() != S * fd:
        raise ValueError("rope: freqs must be [S, D] or [S, D / 2]")
    y = torch.empty_like(x)
    _lib.check(lib.mhip_rope(_stream(), x.data_ptr(), freqs.data_ptr(), y.data_ptr(), x.numel() // D if D else 0, S, D,
                             1 if fd == D // 2 else 0, _code(x)))
    return y


def batch_norm(x, gamma, beta, mean, variance, eps=1e-5):
    """y = (x - mean) / sqrt(variance + eps) * gamma + beta, the four vectors along x's last axis."""
    _dev(x, gamma, beta, mean, variance)
    lib = _lib.load()
    C_ = x.shape[-1] if x.dim() else 1
    for t in (gamma, beta, mean, variance):
        if t.numel() != C_ or t.dtype != x.dtype:
            raise ValueError("batch_norm: gamma, beta, mean and variance must be [channels] of x's element type")
    y = torch.empty_like(x)
    _lib.check(lib.mhip_batch_norm(_stream(), x.data_ptr(), gamma.data_ptr(), beta.data_ptr(), mean.data_ptr(), variance.data_ptr(),
                                   y.data_ptr(), x.numel() // C_ if C_ else 0, C_, float(eps), _code(x)))
    return y


def depth_attention(q, k, v, scale=1.0):
    """softmax(q k^T scale) v for one query row per leading index: q [.., 1, H] or [.., H], k and v
    [.., depth, H] with depth <= 64; the result has q's shape."""
    _dev(q, k, v)
    lib = _lib.load()
    if k.dim() < 2 or k.shape != v.shape or not (q.dtype == k.dtype == v.dtype):
        raise ValueError("depth_attention: k and v must be [.., depth, H] of q's element type")
    depth, H = k.shape[-2], k.shape[-1]
    lead = tuple(k.shape[:-2])
    if tuple(q.shape) not in (lead + (1, H), lead + (H,)):
        raise ValueError("depth_attention: q must be [.., 1, H] or [.., H] over k's leading axes")
    out = torch.empty_like(q)
    rows = q.numel() // H if H else 0
    _lib.check(lib.mhip_depth_attention(_stream(), q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), rows, depth, H,
                                        float(scale), _code(q)))
    return out


CHAIN_UNARY_CODE = {"exponential": 0, "tanh": 1, "rsqrt": 2, "sqrt": 3, "negate": 4, "logistic": 5, "abs": 6, "log": 7,
                    "sine": 9, "cosine": 10, "floor": 11, "ceil": 12}
CHAIN_BINARY_CODE = {"add": 100, "subtract": 101, "multiply": 102, "divide": 103, "maximum": 104, "minimum": 105}


def elementwise_chain(inputs, ops):
    """One launch for a chain of elementwise operations: the running value starts as inputs[0], a
    binary operation takes the next input as its right operand, a unary one transforms the running
    value.  Inputs have the result's shape (that of inputs[0]) or one element."""
    import ctypes as C
    _dev(*inputs)
    lib = _lib.load()
    codes = []
    for name in ops:
        if name in CHAIN_BINARY_CODE:
            codes.append(CHAIN_BINARY_CODE[name])
        elif name in CHAIN_UNARY_CODE:
            codes.append(CHAIN_UNARY_CODE[name])
        else:
            raise ValueError(f"Unsupported operation in fused chain: {name}")
    need = 1 + sum(c >= 100 for c in codes)
    if len(inputs) < need:
        raise ValueError("Not enough inputs for the operations of the chain")
    inputs = list(inputs[:need])
    if any(t.dtype != inputs[0].dtype for t in inputs):
        raise ValueError("every input must have one element type")
    shape = max((t.shape for t in inputs), key=lambda sh: int(torch.Size(sh).numel()))
    y = torch.empty(shape, dtype=inputs[0].dtype, device=inputs[0].device)
    ptrs = (C.c_void_p * need)(*[t.data_ptr() for t in inputs])
    counts = (C.c_int64 * need)(*[t.numel() for t in inputs])
    arr = (C.c_int32 * len(codes))(*codes)
    _lib.check(lib.mhip_elementwise_chain(_stream(), need, ptrs, counts, len(codes), arr, y.data_ptr(), y.numel(), _code(y)))
    return y


def convert(x, dtype):
    _dev(x)
    lib = _lib.load()
    y = torch.empty(x.shape, dtype=dtype, device=x.device)
    _lib.check(lib.mhip_convert(_stream(), x.data_ptr(), y.data_ptr(), x.numel(), _code(x),
                                DTYPE_CODE[dtype]))
    return y


def transpose_0213(x):
    _dev(x)
    lib = _lib.load()
    d0, d1, d2, d3 = x.shape
    y = torch.empty(d0, d2, d1, d3, dtype=x.dtype, device=x.device)
    _lib.check(lib.mhip_transpose_0213(_stream(), x.data_ptr(), y.data_ptr(), d0, d1, d2, d3,
                                       _code(x)))
    return y


def split_qkv_heads(qkv, n_head: int):
    _dev(qkv)
    lib = _lib.load()
    B, S, three_d = qkv.shape
    D = three_d // (3 * n_head)
    q, k, v = (torch.empty(B, n_head, S, D, dtype=qkv.dtype, device=qkv.device) for _ in range(3))
    _lib.check(lib.mhip_split_qkv_heads(_stream(), qkv.data_ptr(), q.data_ptr(), k.data_ptr(),
                                        v.data_ptr(), B, S, n_head, D, _code(qkv)))
    return q, k, v


def iota(shape, dim: int, dtype, device="cuda"):
    lib = _lib.load()
    y = torch.empty(shape, dtype=dtype, device=device)
    _lib.check(lib.mhip_iota(_stream(), y.data_ptr(), math.prod(shape[:dim]), shape[dim],
                             math.prod(shape[dim + 1:]), DTYPE_CODE[dtype]))
    return y


def argmax(x, index_dtype=torch.int32, return_values: bool = False):
    if index_dtype not in (torch.int32, torch.int64):
        raise _lib.MhipError(2, f"mhip_argmax: index dtype {index_dtype} (need i32 or i64)")
    return (_native or _host()).argmax(x, index_dtype == torch.int64, return_values)


def autotune_matmul(a, b, bias=None, activation: str = "none", trans_a: bool = False,
                    trans_b: bool = False, iters: int = 10):
    """Times the GEMM kernel variants for this 2-D problem and stores the fastest in the
    library's tuning table (used by every later matmul of the same shape, layout and
    type).  Returns (variant code 128 | 256 | 2560 | 2561, microseconds per launch)."""
    _dev(a, b, bias)
    lib = _lib.load()
    if a.dim() != 2 or b.dim() != 2 or a.dtype != b.dtype:
        raise ValueError("autotune_matmul takes two 2-D operands of one dtype")
    M, K = (a.shape[1], a.shape[0]) if trans_a else (a.shape[0], a.shape[1])
    N = b.shape[0] if trans_b else b.shape[1]
    out = torch.empty((M, N), dtype=a.dtype, device=a.device)
    variant, us = C.c_int(0), C.c_float(0.0)
    _lib.check(lib.mhip_gemm_autotune(_stream(), a.data_ptr(), b.data_ptr(), _ptr(bias), out.data_ptr(), M, N, K, 1,
                                      0, 0, M * N, int(trans_a), int(trans_b), ACTIVATION_CODE[activation], _code(a),
                                      int(iters), C.byref(variant), C.byref(us)))
    return variant.value, us.value


def autotune_row(op: str, x, gamma=None, beta=None, eps: float = 1e-5, iters: int = 10):
    """Times the launch forms of a row operator ("softmax", "layer_norm", "rms_norm") for x
    [rows, cols] and stores the fastest in the tuning table.  Returns ((kind, rows per wave
    group, ordered, workgroups per CU), microseconds per launch)."""
    _dev(x, gamma, beta)
    lib = _lib.load()
    code = {"softmax": 0, "layer_norm": 1, "rms_norm": 2}[op]
    cols = x.shape[-1]
    out = torch.empty_like(x)
    choice, us = (C.c_int * 4)(), C.c_float(0.0)
    _lib.check(lib.mhip_row_autotune(_stream(), code, x.data_ptr(), _ptr(gamma), _ptr(beta), out.data_ptr(),
                                     x.numel() // cols, cols, float(eps), _code(x), int(iters), choice, C.byref(us)))
    return tuple(choice), us.value


def autotune_attention(q, k, v, scale=None, is_causal: bool = False, iters: int = 5):
    """Times the attention kernels that can serve packed q [B,H,Sq,D], k, v [B,H,Skv,D] and stores
    the fastest in the tuning table.  Returns (variant 1 | 2 | 3, microseconds per launch)."""
    _dev(q, k, v)
    lib = _lib.load()
    B, H, Sq, D = q.shape
    out = torch.empty_like(q)
    variant, us = C.c_int(0), C.c_float(0.0)
    _lib.check(lib.mhip_attention_autotune(_stream(), q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), B, H, Sq,
                                           k.shape[2], D, float(D ** -0.5 if scale is None else scale), int(is_causal),
                                           _code(q), int(iters), C.byref(variant), C.byref(us)))
    return variant.value, us.value


def tuning_device() -> str:
    """The current device's key in the tuning table (architecture name / compute units)."""
    return _lib.load().mhip_tuning_device().decode()


def tuning_save(path: str) -> None:
    _lib.check(_lib.load().mhip_tuning_save(str(path).encode()))


def tuning_load(path: str) -> None:
    _lib.check(_lib.load().mhip_tuning_load(str(path).encode()))


def shipped_tuning_table() -> str:
    """Path of the table that ships for the current device (it may not exist); the kernel library
    loads it by itself at first use unless the table was cleared before."""
    import os
    return os.path.join(os.path.dirname(os.path.abspath(__file__)), "tuning", tuning_device().replace("/", "_") + ".txt")


def tuning_clear() -> None:
    _lib.load().mhip_tuning_clear()


def tuning_count() -> int:
    return _lib.load().mhip_tuning_count()
