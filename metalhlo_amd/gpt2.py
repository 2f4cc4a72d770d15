"""GPT-2 forward through the fused kernels (the GPT-2-small benchmark configuration: B8 S1024).

The op sequence is the one the reference's fusion passes produce for a pre-LN
GPT-2 block — fused_layer_norm, fused_matmul_bias_activation (bias only, and
bias + tanh-GELU), fused_scaled_dot_product_attention with is_causal, residual
adds, token + position gather, tied output head — issued in order on one HIP
stream like the reference's integrated executor does
(Sources/MetalHLOCore/Runtime/IntegratedExecutor.swift:208-232), but with no
host synchronisation between launches.  Architecture constants:
Sources/GPT2EndToEnd/main.swift:35-40.

Parameters are held in fp32; every forward converts them to the compute type at
use (the `convert` ops of the fp32-params / bf16-compute graph), computes each
fused op with fp32 accumulation and rounds once at its output.
"""
from __future__ import annotations

from dataclasses import dataclass
from typing import Dict, List

import numpy as np
import torch

from . import kernels


@dataclass
class GPT2Config:
    n_layer: int = 12
    d_model: int = 768
    n_head: int = 12
    d_ff: int = 3072
    vocab: int = 50257
    n_pos: int = 1024


def init_params(cfg: GPT2Config, seed: int = 5) -> Dict:
    """Random-init N(0, 0.02) weights, zero biases, LN gamma 1 / beta 0 (numpy fp32)."""
    rng = np.random.default_rng(seed)
    d, f = cfg.d_model, cfg.d_ff
    w = lambda *s: rng.normal(0.0, 0.02, s).astype(np.float32)
    z = lambda *s: np.zeros(s, np.float32)
    o = lambda *s: np.ones(s, np.float32)
    layers = [dict(ln1_g=o(d), ln1_b=z(d), w_qkv=w(d, 3 * d), b_qkv=z(3 * d), w_o=w(d, d), b_o=z(d),
                   ln2_g=o(d), ln2_b=z(d), w_fc=w(d, f), b_fc=z(f), w_proj=w(f, d), b_proj=z(d))
              for _ in range(cfg.n_layer)]
    return dict(wte=w(cfg.vocab, d), wpe=w(cfg.n_pos, d), layers=layers, lnf_g=o(d), lnf_b=z(d))


class GPT2:
    def __init__(self, cfg: GPT2Config, params: Dict, compute_dtype=torch.bfloat16, device="cuda"):
        self.cfg, self.dtype = cfg, compute_dtype
        # All parameters live in ONE fp32 device buffer (each tensor starts on a
        # 16-byte boundary), so the per-step fp32 -> compute-type conversion is a
        # single streaming launch; the named entries are views into the buffers.
        flat, self._slots = [], []

        def put(path, a):
            a = np.ascontiguousarray(a, dtype=np.float32)
            off = sum(x.size for x in flat)
            pad = (-a.size) % 8
            flat.append(np.concatenate([a.reshape(-1), np.zeros(pad, np.float32)]))
            self._slots.append((path, off, tuple(a.shape)))

        # the tied output head multiplies by wte^T: rows padded with zeros to a multiple of 64
        # keep that GEMM on the aligned kernels; "wte" is the view of the real rows
        wte = np.asarray(params["wte"], dtype=np.float32)
        self.vocab_pad = -(-wte.shape[0] // 64) * 64
        put(("wte_pad",), np.concatenate([wte, np.zeros((self.vocab_pad - wte.shape[0], wte.shape[1]), np.float32)]))
        self._slots.append((("wte",), self._slots[-1][1], wte.shape))
        for name in ("wpe", "lnf_g", "lnf_b"):
            put((name,), params[name])
        self._layers_at = sum(x.size for x in flat)
        for i, l in enumerate(params["layers"]):
            for k, v in l.items():
                put(("layers", i, k), v)
        self.flat32 = torch.from_numpy(np.concatenate(flat)).to(device)
        self.p32 = self._views(self.flat32)

    def _views(self, flat: torch.Tensor, start: int = 0) -> Dict:
        """The parameters from element `start` of the buffer on, which `flat` holds."""
        out: Dict = {"layers": [dict() for _ in range(self.cfg.n_layer)]}
        for path, off, shape in self._slots:
            if off < start:
                continue
            v = torch.as_strided(flat, shape, (shape[1], 1) if len(shape) == 2 else (1,), off - start)
            if path[0] == "layers":
                out["layers"][path[1]][path[2]] = v
            else:
                out[path[0]] = v
        return out

    def forward(self, ids: torch.Tensor) -> torch.Tensor:
        """ids int32 [B,S] on the device -> logits [B,S,vocab] in the compute type.  With more than 768 tokens in all a
        sequence has the same bits in any batch (d_model and d_ff below 4096, where products keep the order of a sum); up to that
        fp32 sums are split by the number of tokens."""
        cfg = self.cfg
        B, S = ids.shape
        d, H = cfg.d_model, cfg.n_head
        if self._few_tokens(B * S):
            return self._forward_few(ids)
        o_parts, p_parts = self._sum_parts(B * S)
        # the graph's `convert` ops: fp32 parameters -> compute type, every step
        # (a short prompt's output head reads its fp32 rows where they are)
        fp32_head = o_parts and kernels.tied_head_served(B * S, self.vocab_pad, d, self.dtype)
        start = self._layers_at if fp32_head else 0
        p = self.p32 if self.dtype == torch.float32 else self._views(kernels.convert(self.flat32[start:], self.dtype), start)
        x = kernels.embed_tokens(ids, self.p32["wte"], self.p32["wpe"], self.dtype).reshape(B * S, d)
        # the strided attention entry covers 16-bit types and head sizes 64 / 128
        in_place = self.dtype in (torch.bfloat16, torch.float16) and d // H in (64, 128)
        if o_parts:
            # K of the layers in front of a residual over the whole device; the launch that adds the parts up forms the next LayerNorm
            layers = self.p32["layers"]
            norms = [(l["ln1_g"], l["ln1_b"], 1e-5) for l in layers] + [(self.p32["lnf_g"], self.p32["lnf_b"], 1e-5)]
            x, h = kernels.finish_norm(None, None, x, norms[0])
            for l, l32, norm in zip(p["layers"], layers, norms[1:]):
                a = kernels.causal_attention(kernels.matmul(h, l["w_qkv"], bias=l["b_qkv"]), B, H)
                x, h = kernels.finish_norm(kernels.matmul_sums(a, l["w_o"], o_parts), l32["b_o"], x, (l32["ln2_g"], l32["ln2_b"], 1e-5))
                u = kernels.matmul(h, l["w_fc"], bias=l["b_fc"], activation="gelu")
                x, h = kernels.finish_norm(kernels.matmul_sums(u, l["w_proj"], p_parts), l32["b_proj"], x, norm)
            logits = kernels.tied_head(h, self.p32["wte_pad"]) if fp32_head else kernels.matmul(h, p["wte_pad"], trans_b=True)
            return logits.reshape(B, S, self.vocab_pad)[..., :cfg.vocab]
        for l in p["layers"]:
            h = kernels.layer_norm(x, l["ln1_g"], l["ln1_b"], eps=1e-5)
            qkv = kernels.matmul(h, l["w_qkv"], bias=l["b_qkv"])
            if in_place:
                # attention reads Q, K, V in place ([B,S,3,H,D] views of the projection) and
                # writes [B,S,H,D]: no head split / merge passes over memory
                q, k, v = qkv.view(B, S, 3, H, d // H).permute(2, 0, 3, 1, 4).unbind(0)
                a = torch.empty(B, S, H, d // H, dtype=qkv.dtype, device=qkv.device)
                kernels.flash_attention(q, k, v, is_causal=True, out=a.permute(0, 2, 1, 3))
                a = a.view(B * S, d)
            else:
                q, k, v = kernels.split_qkv_heads(qkv.reshape(B, S, 3 * d), H)
                a = kernels.flash_attention(q, k, v, is_causal=True)
                a = kernels.transpose_0213(a).reshape(B * S, d)
            x = kernels.matmul(a, l["w_o"], bias=l["b_o"], residual=x)          # x + proj(a), one kernel
            h = kernels.layer_norm(x, l["ln2_g"], l["ln2_b"], eps=1e-5)
            u = kernels.matmul(h, l["w_fc"], bias=l["b_fc"], activation="gelu")
            x = kernels.matmul(u, l["w_proj"], bias=l["b_proj"], residual=x)
        x = kernels.layer_norm(x, p["lnf_g"], p["lnf_b"], eps=1e-5)
        logits = kernels.matmul(x, p["wte_pad"], trans_b=True)   # tied head: x . wte^T (padded columns are 0)
        return logits.reshape(B, S, self.vocab_pad)[..., :cfg.vocab]

    def _few_tokens(self, tokens: int) -> bool:
        """Whether every layer of this many tokens reads its parameters as they are held (kernels.linear)."""
        d, f, dt = self.cfg.d_model, self.cfg.d_ff, self.dtype
        if dt not in (torch.bfloat16, torch.float16) or d // self.cfg.n_head not in (64, 128) or d % self.cfg.n_head:
            return False
        # (each 64 rows read a matrix again, which from memory costs as much as converting it: us as they are held and converted,
        # replayed, 65 tokens 559 and 571, 80 567 and 585, 96 581 and 595, 97, which are blocks of 64 rows instead of 48, 616 and 595,
        # 128 643 and 615; a matrix of up to 4 MB stays in an L2)
        if tokens > 96 and 4 * d * f > 4 << 20:
            return False
        return d <= 4096 and all(kernels.linear_served(tokens, n, k, dt) for n, k in ((3 * d, d), (d, d), (f, d), (d, f), (self.vocab_pad, d)))

    # 64x64 tiles of the layers in front of a residual from which on they fill the device whole
    # (us whole and in parts, replayed: 193 tokens 810 and 642, 300 841 and 692, 576 949 and 844, 768 (144 tiles) 1098 and 1008;
    # 1024 (192 tiles) 1206 and 1202, which leaves a sequence of full length its bits in any batch)
    _full_tiles = 144
    # (narrower layers have so few tiles for more tokens, but a sequence keeps its bits from here on whatever the width)
    _most_tokens = 768

    def _sum_parts(self, tokens: int):
        """Shares of K for the two layers in front of a residual, (0, 0) where their tiles fill the device without."""
        d, f = self.cfg.d_model, self.cfg.d_ff
        if d // self.cfg.n_head not in (64, 128) or d % self.cfg.n_head or d > 4096 or tokens > self._most_tokens or -(-tokens // 64) * -(-d // 64) > self._full_tiles:
            return 0, 0
        if self.dtype not in (torch.bfloat16, torch.float16):
            return 0, 0
        parts = tuple(kernels.matmul_sums_parts(tokens, d, k, self.dtype) for k in (d, f))
        return parts if all(parts) else (0, 0)

    def _forward_few(self, ids: torch.Tensor) -> torch.Tensor:
        """The same operators for a short prompt: the parameters are rounded to the compute type where they are read
        (converting all of them first took 117 of 705 us of kernels), and the launch that adds up a residual layer's
        sums forms the next LayerNorm."""
        cfg, p = self.cfg, self.p32
        B, S = ids.shape
        linear, layers, T = kernels.linear, p["layers"], B * S
        o_parts, p_parts = (kernels.linear_parts(T, cfg.d_model, k) for k in (cfg.d_model, cfg.d_ff))
        norms = [(l["ln1_g"], l["ln1_b"], 1e-5) for l in layers] + [(p["lnf_g"], p["lnf_b"], 1e-5)]
        x = kernels.embed_tokens(ids, p["wte"], p["wpe"], self.dtype).reshape(T, cfg.d_model)
        if kernels.linear_norm_served(T, cfg.d_model, cfg.d_model, self.dtype):
            layer = kernels.linear_layer
            merged = kernels.attend_project_layer_served(B, S, cfg.n_head, cfg.d_model // cfg.n_head, cfg.d_model, self.dtype)
            for i, l in enumerate(layers):
                qkv = layer(x, l["w_qkv"], l["b_qkv"], norm=norms[i], ahead=(l["w_o"], l["w_fc"]))
                if merged:
                    x = kernels.attend_project_layer(qkv, l["w_o"], l["b_o"], x, B, cfg.n_head, ahead=(l["w_proj"],))
                else:
                    x = layer(kernels.causal_attention(qkv, B, cfg.n_head), l["w_o"], l["b_o"], residual=x, ahead=(l["w_proj"],))
                u = layer(x, l["w_fc"], l["b_fc"], "gelu", norm=(l["ln2_g"], l["ln2_b"], 1e-5))
                x = layer(u, l["w_proj"], l["b_proj"], residual=x, ahead=(layers[i + 1]["w_qkv"],) if i + 1 < len(layers) else ())
            return self._head(kernels.finish_norm(None, None, x, norms[-1])[1], B, S)
        x, h = kernels.finish_norm(None, None, x, norms[0])
        merged = kernels.attend_project_served(B, S, cfg.n_head, cfg.d_model // cfg.n_head, cfg.d_model, self.dtype)
        for i, l in enumerate(layers):
            qkv = linear(h, l["w_qkv"], l["b_qkv"], ahead=(l["w_o"], l["w_fc"]))
            if merged:
                sums = kernels.attend_project(qkv, l["w_o"], B, cfg.n_head, ahead=(l["w_proj"],))
            else:
                sums = linear(kernels.causal_attention(qkv, B, cfg.n_head), l["w_o"], parts=o_parts, ahead=(l["w_proj"],))
            x, h = kernels.finish_norm(sums, l["b_o"], x, (l["ln2_g"], l["ln2_b"], 1e-5))
            u = linear(h, l["w_fc"], l["b_fc"], "gelu")
            sums = linear(u, l["w_proj"], parts=p_parts, ahead=(layers[i + 1]["w_qkv"],) if i + 1 < len(layers) else ())
            x, h = kernels.finish_norm(sums, l["b_proj"], x, norms[i + 1])
        return self._head(h, B, S)

    def _head(self, h: torch.Tensor, B: int, S: int) -> torch.Tensor:
        """Logits of a short prompt from the fp32 table."""
        cfg, p, T = self.cfg, self.p32, B * S
        # (us, strips that walk the device against x that stays: 64 tokens 36.9 and 38.5, 65 48.5 and 39.2, 128 53.5 and 45.1)
        if T > 64 and kernels.tied_head_served(T, self.vocab_pad, cfg.d_model, self.dtype):
            logits = kernels.tied_head(h, p["wte_pad"])
        else:
            logits = kernels.linear(h, p["wte_pad"], trans_b=True)
        return logits.reshape(B, S, self.vocab_pad)[..., :cfg.vocab]

    def capture(self, ids: torch.Tensor) -> "GraphedForward":
        """Records one forward pass for ids of this shape into a HIP graph.  Every launch
        of the pass goes to the stream handed to the kernel library, so the whole
        pipeline (about 100 launches) replays with one submission instead of one host
        call per kernel."""
        static_ids = ids.clone()
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):           # first calls set kernel attributes; keep them out of the capture
            for _ in range(2):
                self.forward(static_ids)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            logits = self.forward(static_ids)
        return GraphedForward(graph, static_ids, logits)

    @staticmethod
    def flops(cfg: GPT2Config, B: int, S: int) -> float:
        d, f = cfg.d_model, cfg.d_ff
        per_tok = cfg.n_layer * (d * 3 * d + d * d + 2 * d * f) + d * cfg.vocab
        attn = cfg.n_layer * 2 * B * cfg.n_head * S * S * (d // cfg.n_head)   # causal: half of 4BHS^2D
        return 2.0 * per_tok * B * S + attn


class GraphedForward:
    """A captured forward pass: copy new token ids in, replay, read `logits` (a buffer
    owned by the graph, overwritten by the next replay)."""

    def __init__(self, graph, ids: torch.Tensor, logits: torch.Tensor):
        self.graph, self.ids, self.logits = graph, ids, logits

    def __call__(self, ids: torch.Tensor) -> torch.Tensor:
        if ids.shape != self.ids.shape or ids.dtype != self.ids.dtype:
            raise ValueError("captured for ids of shape %s" % (tuple(self.ids.shape),))
        self.ids.copy_(ids)
        self.graph.replay()
        return self.logits
