"""The work a user has this framework do, as cases that can be timed: single operators through
`metalhlo_amd.kernels`, a GPT-2 forward through `metalhlo_amd.gpt2`, and a compiled StableHLO program
through the C API (`metalhlo_amd.capi`).

Sizes are those of the benchmark, the tests and the GPT-2 configuration, or generic ones; `draw`
spreads over the ranges between them.  Every case is a dict with a "kind":

  gemm    one dot_general with its fused epilogue
  attn    one attention forward
  rows    one row operator
  gpt2    a GPT-2 forward: launched call by call, or replayed from a captured graph
  block   a transformer block in StableHLO text: upload of x, mhlo_execute, download of the result
"""
import ctypes
import math

import numpy as np
import torch

from metalhlo_amd import capi, kernels, programs
from metalhlo_amd.gpt2 import GPT2, GPT2Config

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
SIZE = {"bf16": 2, "f16": 2, "f32": 4}


def _gemm(M, N, K, dtype="bf16", batch=1, ta=False, tb=False, bias=False, act="none", residual=False, **kw):
    return dict(kind="gemm", M=M, N=N, K=K, dtype=dtype, batch=batch, ta=ta, tb=tb, bias=bias, act=act, residual=residual, **kw)


def _attn(B, H, Sq, Skv, D, dtype="bf16", causal=True, mask=False, **kw):
    return dict(kind="attn", B=B, H=H, Sq=Sq, Skv=Skv, D=D, dtype=dtype, causal=causal, mask=mask, **kw)


def _rows(op, rows, cols, dtype="bf16", **kw):
    return dict(kind="rows", op=op, rows=rows, cols=cols, dtype=dtype, **kw)


def _gpt2(B, S, graph, dtype="bf16", **kw):
    return dict(kind="gpt2", B=B, S=S, graph=graph, dtype=dtype, **kw)


def _block(B, S, H, D, F, dtype="f32", opt=2, **kw):
    return dict(kind="block", B=B, S=S, H=H, D=D, F=F, dtype=dtype, opt=opt, **kw)


def listed():
    return [
        # a linear layer of a decode step: a handful of tokens against a whole weight matrix
        _gemm(4, 4096, 4096, bias=True, name="gemm_decode"),
        # an ordinary layer on a ragged batch of tokens, bias and activation fused
        _gemm(1000, 3000, 1000, bias=True, act="gelu", name="gemm_ragged"),
        # the weight gradient of a 768 -> 3072 layer over 8192 tokens: x^T dy, a long contraction
        _gemm(768, 3072, 8192, ta=True, name="gemm_grad"),
        # the matrix product of the benchmark
        _gemm(4096, 4096, 4096, name="gemm_large"),
        # prefill of a long prompt (the benchmark's attention)
        _attn(4, 32, 4096, 4096, 128, name="attn_prefill"),
        # one decode step of eight sequences against their caches
        _attn(8, 32, 1, 4096, 128, causal=False, name="attn_decode"),
        # prefill of a few prompts of uneven length with GPT-2's head size
        _attn(3, 12, 1000, 1000, 64, name="attn_ragged"),
        # normalisation of a large batch of tokens (the benchmark's rows)
        _rows("layer_norm", 32768, 4096, name="rows_large"),
        # next-token distributions over GPT-2's vocabulary, whose rows start at odd addresses
        _rows("softmax", 128, 50257, name="rows_vocab"),
        # GPT-2-small over a short prompt of whatever length a user typed, launched call by call
        _gpt2(1, 37, False, name="gpt2_prompt"),
        # GPT-2-small over the benchmark's full batch, replayed from a captured graph
        _gpt2(8, 1024, True, name="gpt2_batch"),
        # one transformer block in plain fp32 StableHLO, batch 1, 128 tokens, 12 heads, through the C API
        _block(1, 128, 12, 64, 3072, name="block_capi"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A size between lo and hi: mostly a multiple of 64 or 8 as layers have them, sometimes any number."""
    n, u = _log(rng, lo, hi), rng.random()
    step = 64 if u < 0.5 else 8 if u < 0.8 else 1
    return max(lo, min(hi, -(-n // step) * step))


def draw(rng):
    kind = rng.choice(("decode_gemm", "gemm", "grad", "large_gemm", "prefill", "decode", "rows", "rows", "prompt", "batch", "block"))
    half = rng.choice(("bf16", "bf16", "f16"))
    act = rng.choice(("none", "none", "gelu", "relu", "silu"))
    if kind == "decode_gemm":        # few tokens; the weights stored [K, N] or [N, K]
        return _gemm(_log(rng, 1, 64), _size(rng, 512, 16384), _size(rng, 512, 8192), rng.choice((half, half, "f32")),
                     tb=rng.random() < 0.5, bias=rng.random() < 0.5, act=act)
    if kind == "gemm":
        batch = rng.choice((1, 1, 1, _log(rng, 2, 16)))
        top = 2048 if batch == 1 else 768
        return _gemm(_size(rng, 64, top), _size(rng, 64, top), _size(rng, 64, top), rng.choice((half, half, "f32")), batch,
                     tb=rng.random() < 0.5, bias=batch == 1 and rng.random() < 0.5, act=act, residual=rng.random() < 0.3)
    if kind == "grad":               # dW = x^T dy (long contraction) or dx = dy W^T
        tokens = _size(rng, 1024, 16384)
        n_in, n_out = (_size(rng, 512, 3072) for _ in range(2))
        dtype = rng.choice((half, half, "f32"))
        return _gemm(n_in, n_out, tokens, dtype, ta=True) if rng.random() < 0.6 else _gemm(tokens, n_in, n_out, dtype, tb=True)
    if kind == "large_gemm":
        return _gemm(64 * _log(rng, 32, 128) - rng.choice((0, 0, 3)), 64 * _log(rng, 12, 80), 64 * _log(rng, 12, 64), half,
                     tb=rng.random() < 0.5, bias=rng.random() < 0.5, act=act)
    if kind == "prefill":
        dtype = rng.choice((half, half, half, "f32"))
        D = rng.choice((64, 128, 64, 128, 96, 32))
        S = _size(rng, 64, 4096)
        budget = 5.5e11 if dtype != "f32" and D in (64, 128) else 2e10      # FLOP of the whole case
        heads = max(1, min(128, int(budget / (4.0 * S * S * D)), _log(rng, 4, 128)))
        H = max(h for h in (1, 2, 4, 8, 12, 16, 32) if h <= heads)
        return _attn(max(1, heads // H), H, S, S if rng.random() < 0.8 else _size(rng, 64, min(4096, 2 * S)), D, dtype,
                     rng.random() < 0.7, rng.random() < 0.15 and S <= 1024)
    if kind == "decode":
        D, H = rng.choice((64, 128)), rng.choice((8, 12, 16, 32))
        Skv = _size(rng, 128, 16384)
        B = max(1, min(_log(rng, 1, 64), int(2e9 / (4 * H * Skv * D))))
        return _attn(B, H, rng.choice((1, 1, 1, 4, 8)), Skv, D, half, False)
    if kind == "rows":
        op = rng.choice(("softmax", "layer_norm", "rms_norm", "bias_gelu", "argmax"))
        cols = rng.choice((768, 3072, 4096, 50257, _size(rng, 64, 16384), _size(rng, 64, 16384)))
        return _rows(op, _log(rng, 1, min(32768, 134217728 // cols)), cols, rng.choice((half, half, "f32")))
    if kind == "prompt":
        return _gpt2(_log(rng, 1, 4), _log(rng, 4, 256), False, half)
    if kind == "batch":
        B = _log(rng, 1, 8)
        return _gpt2(B, _size(rng, 64, 1024), True, half)
    H, D = rng.choice(((12, 64), (8, 64), (16, 64), (4, 32), (8, 128)))
    return _block(_log(rng, 1, 8), _size(rng, 16, 512), H, D, 4 * H * D, rng.choice(("f32", "f32", "bf16")), rng.choice((2, 2, 3)))


def _draws(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def normal(shape, dtype=torch.float32, scale=1.0, shift=0.0):
        return torch.randn(shape, generator=g, device="cuda").mul_(scale).add_(shift).to(dtype)
    return g, normal


class _Program:
    """A compiled program and its resident parameters, released with the object."""
    session = None

    def __init__(self, text, opt, params, x, element_type):
        if _Program.session is None:
            _Program.session = capi.Session()         # a process has one client
        self.s, self.x, self.type = _Program.session, x, element_type
        self.exe = self.s.compile(text, opt)
        self.params = [self.s.buffer(p, element_type) for p in params]
        self.args = (ctypes.c_void_p * (1 + len(params)))(None, *self.params)
        self.outs, self.got = (ctypes.c_void_p * 1)(), ctypes.c_int32()

    def __call__(self):
        lib = self.s.lib
        x = self.s.buffer(self.x, self.type)
        self.args[0] = x
        rc = lib.mhlo_execute(self.exe, self.args, len(self.args), self.outs, ctypes.byref(self.got))
        if rc:
            raise capi.MHLOError(rc, (lib.mhlo_get_last_error() or b"").decode())
        y = self.s.to_numpy(self.outs[0])
        lib.mhlo_buffer_destroy(self.outs[0])
        lib.mhlo_buffer_destroy(x)
        return torch.from_numpy(y) if self.type == "f32" else torch.from_numpy(y.view(np.int16)).view(DTYPES[self.type])

    def __del__(self):
        for b in self.params:
            self.s.lib.mhlo_buffer_destroy(b)
        self.s.lib.mhlo_executable_destroy(self.exe)


def _host(t, dtype):
    """The host array the C API takes: fp32, or the bit patterns of a 16-bit type."""
    return t.cpu().numpy() if dtype == "f32" else t.view(torch.int16).cpu().numpy().view(np.uint16)


def prepare(case, seed):
    g, normal = _draws(seed)
    kind, c = case["kind"], case
    dt = DTYPES[c["dtype"]]
    if kind == "gemm":
        lead = (c["batch"],) if c["batch"] > 1 else ()
        a = normal(lead + ((c["K"], c["M"]) if c["ta"] else (c["M"], c["K"])), dt)
        b = normal(lead + ((c["N"], c["K"]) if c["tb"] else (c["K"], c["N"])), dt, c["K"] ** -0.5)
        return dict(case=c, a=a, b=b, bias=normal((c["N"],), dt, 0.1) if c["bias"] else None,
                    residual=normal(lead + (c["M"], c["N"]), dt) if c["residual"] else None)
    if kind == "attn":
        q = normal((c["B"], c["H"], c["Sq"], c["D"]), dt)
        k, v = (normal((c["B"], c["H"], c["Skv"], c["D"]), dt) for _ in range(2))
        mask = None
        if c["mask"]:                # padding: every sequence hides the tail of its keys
            keep = torch.randint(c["Skv"] // 2, c["Skv"] + 1, (c["B"], 1, 1, 1), generator=g, device="cuda")
            hide = torch.arange(c["Skv"], device="cuda") >= keep
            mask = torch.zeros(c["B"], 1, c["Sq"], c["Skv"], dtype=dt, device="cuda").masked_fill_(hide, float("-inf"))
        return dict(case=c, q=q, k=k, v=v, mask=mask)
    if kind == "rows":
        x = torch.empty((c["rows"], c["cols"]), dtype=dt, device="cuda").normal_(0.0, 2.0, generator=g)
        return dict(case=c, x=x, gamma=normal((c["cols"],), dt, 0.1, 1.0), beta=normal((c["cols"],), dt, 0.1))
    if kind == "gpt2":
        cfg = GPT2Config()
        d, f = cfg.d_model, cfg.d_ff

        def w(*shape):
            return normal(shape, scale=0.02).cpu().numpy()

        def one(*shape):
            return normal(shape, scale=0.05, shift=1.0).cpu().numpy()
        layers = [dict(ln1_g=one(d), ln1_b=w(d), w_qkv=w(d, 3 * d), b_qkv=w(3 * d), w_o=w(d, d), b_o=w(d), ln2_g=one(d), ln2_b=w(d),
                       w_fc=w(d, f), b_fc=w(f), w_proj=w(f, d), b_proj=w(d)) for _ in range(cfg.n_layer)]
        model = GPT2(cfg, dict(wte=w(cfg.vocab, d), wpe=w(cfg.n_pos, d), layers=layers, lnf_g=one(d), lnf_b=w(d)), compute_dtype=dt)
        ids = torch.randint(0, cfg.vocab, (c["B"], c["S"]), generator=g, device="cuda", dtype=torch.int32)
        return dict(case=c, step=model.capture(ids) if c["graph"] else model.forward, ids=ids)
    d, F = c["H"] * c["D"], c["F"]
    host = lambda shape, scale=0.02, shift=0.0: _host(normal(shape, dt, scale, shift), c["dtype"])  # noqa: E731
    params = [host((d,), 0.05, 1.0), host((d,)), host((d, 3 * d)), host((3 * d,)), host((d, d)), host((d,)),
              host((d,), 0.05, 1.0), host((d,)), host((d, F)), host((F,)), host((F, d)), host((d,))]
    text = programs.transformer_block(c["B"], c["S"], c["H"], c["D"], F, c["dtype"])
    return dict(case=c, program=_Program(text, c["opt"], params, host((c["B"], c["S"], d), 1.0), c["dtype"]))


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "gemm":
        return kernels.matmul(state["a"], state["b"], bias=state["bias"], activation=c["act"], trans_a=c["ta"], trans_b=c["tb"],
                              residual=state["residual"])
    if kind == "attn":
        return kernels.flash_attention(state["q"], state["k"], state["v"], is_causal=c["causal"], mask=state["mask"])
    if kind == "rows":
        op, x = c["op"], state["x"]
        if op == "softmax":
            return kernels.softmax(x)
        if op == "layer_norm":
            return kernels.layer_norm(x, state["gamma"], state["beta"])
        if op == "rms_norm":
            return kernels.rms_norm(x, state["gamma"])
        if op == "bias_gelu":
            return kernels.bias_gelu(x, state["beta"])
        return kernels.argmax(x)
    if kind == "gpt2":
        return state["step"](state["ids"])
    return state["program"]()


def work(case):
    c, kind, e = case, case["kind"], SIZE[case["dtype"]]
    if kind == "gemm":
        M, N, K, b = c["M"], c["N"], c["K"], c["batch"]
        return dict(bytes=e * (b * (M * K + K * N + M * N * (2 if c["residual"] else 1)) + (N if c["bias"] else 0)), flops=2.0 * b * M * N * K)
    if kind == "attn":
        B, H, Sq, Skv, D = c["B"], c["H"], c["Sq"], c["Skv"], c["D"]
        if c["causal"]:              # pairs with key <= query
            n = min(Sq, Skv)
            pairs = n * (n + 1) / 2 + (Sq - n) * Skv
        else:
            pairs = Sq * Skv
        return dict(bytes=e * (2 * B * H * (Sq + Skv) * D + (B * Sq * Skv if c["mask"] else 0)), flops=4.0 * B * H * pairs * D)
    if kind == "rows":
        n = c["rows"] * c["cols"]
        if c["op"] == "argmax":
            return dict(bytes=e * n + 4 * c["rows"], flops=n)
        return dict(bytes=2 * e * n + 2 * e * c["cols"], flops=8.0 * n)
    if kind == "gpt2":
        cfg = GPT2Config()
        d, f = cfg.d_model, cfg.d_ff
        params = cfg.n_layer * (3 * d * d + d * d + 2 * d * f + 9 * d + f) + (cfg.vocab + cfg.n_pos) * d
        return dict(bytes=4.0 * params + e * c["B"] * c["S"] * cfg.vocab, flops=GPT2.flops(cfg, c["B"], c["S"]))
    d, T = c["H"] * c["D"], c["B"] * c["S"]
    params = 4 * d * d + 2 * d * c["F"] + 9 * d + c["F"]
    return dict(bytes=e * (params + 2.0 * T * d), flops=2.0 * T * (4 * d * d + 2 * d * c["F"]) + 2.0 * T * c["S"] * d)


def tolerance(case):
    """Relative differences two correct implementations show: sums of fp32 products in another order
    (fp32 results), and beyond that one rounding of the result, of the probabilities inside attention
    or, in a whole network, of every intermediate tensor (16-bit results)."""
    c = case
    if c["kind"] == "rows" and c["op"] == "argmax":
        return "exact"
    if c["dtype"] == "f32":
        return dict(rel=1e-5)
    eps = 5e-3 if c["dtype"] == "bf16" else 1e-3
    return dict(rel=eps * {"gpt2": 4, "block": 2, "attn": 2}.get(c["kind"], 1))
