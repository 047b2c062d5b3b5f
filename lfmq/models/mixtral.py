"""Mixtral 8x7B MoE.

Same attention/backbone as Llama (GQA, RoPE θ=1e6, RMSNorm) with the MLP
replaced by a top-2 router over 8 experts.  Experts use the fused
w13 (gate|up) + w2 (down) projections like the Llama MLP, so GPTQ/AWQ/RTN
quantize each expert Linear exactly like any other layer.

GPU path, decode and prompts: tokens are routed and sorted by expert on the
device (csrc/moe_route.hip) and run through the grouped packed products
(csrc/dq_rows.hip, csrc/dq_tile.hip) — one launch for all experts' w13 (with
the silu·mul epilogue fused) and one for w2 — instead of launches per expert.
With expert parallelism (lfmq/dist/ep.py) tokens go through the all-to-all
dispatch/combine pair instead.
"""
from __future__ import annotations

import threading
from dataclasses import dataclass, asdict
from typing import Optional

import torch
import torch.nn as nn

from ..ops import functional as F
from .kvcache import KVCache
from .linear import Linear, hooked
from .llama import LlamaAttention, LlamaConfig, RMSNorm, attention_norm
from .qlinear import QLinear, gathers


@dataclass
class MixtralConfig:
    vocab_size: int = 32000
    hidden_size: int = 4096
    intermediate_size: int = 14336
    n_layers: int = 32
    n_heads: int = 32
    n_kv_heads: int = 8
    head_dim: int = 128
    n_experts: int = 8
    top_k: int = 2
    rms_eps: float = 1e-5
    rope_theta: float = 1000000.0
    max_seq: int = 8192
    arch: str = "mixtral"

    @classmethod
    def mixtral_8x7b(cls, **kw):
        return cls(**kw)

    @classmethod
    def tiny(cls, **kw):
        return cls(**{**dict(vocab_size=512, hidden_size=128,
                             intermediate_size=256, n_layers=2, n_heads=4,
                             n_kv_heads=2, head_dim=32, n_experts=4, top_k=2,
                             max_seq=256), **kw})

    def to_dict(self) -> dict:
        return asdict(self)

    @classmethod
    def from_dict(cls, d: dict) -> "MixtralConfig":
        return cls(**{k: v for k, v in d.items() if k in cls.__dataclass_fields__})


class MixtralExpert(nn.Module):
    def __init__(self, cfg: MixtralConfig, dtype):
        super().__init__()
        self.w13 = nn.Linear(cfg.hidden_size, 2 * cfg.intermediate_size,
                             bias=False, dtype=dtype)  # [gate | up]
        self.w2 = nn.Linear(cfg.intermediate_size, cfg.hidden_size,
                            bias=False, dtype=dtype)
        self.inter = cfg.intermediate_size

    def forward(self, x):
        gu = self.w13(x)
        return self.w2(F.silu_mul_gateup(gu, self.inter))


# the grouped kernels address 4 GiB of 16-bit rows
_ROWS_ELEMENTS = (1 << 31) - 1
_PACKED = ("qweight", "scales", "qzeros")
_STACKING = threading.Lock()


class MixtralMoE(nn.Module):
    """Top-k router + experts.  Forward modes:
      - loop (CPU; experts that are more than their packed matrices):
        per-expert forward of the tokens that chose it
      - grouped (GPU, stacked buffers): one launch pair of packed products
        for all experts
      - EP (world > 1): token all-to-all to the rank owning the expert
        (installed by lfmq.dist.ep.apply_expert_parallel)
    """

    def __init__(self, cfg: MixtralConfig, dtype):
        super().__init__()
        self.cfg = cfg
        self.n_experts = cfg.n_experts
        self.top_k = cfg.top_k
        self.gate = Linear(cfg.hidden_size, cfg.n_experts, dtype)  # router stays dense bf16
        self.experts = nn.ModuleList(MixtralExpert(cfg, dtype)
                                     for _ in range(cfg.n_experts))
        self._grouped = None  # set by consolidate()

    def route(self, x2):
        logits = self.gate(x2).float()
        weights, ids = torch.topk(logits, self.top_k, dim=-1)
        weights = torch.softmax(weights, dim=-1)
        return weights, ids

    def _layers(self):
        """The experts' layers [w13, w2, w13, ..], or None if one of them is
        not packed.  (Asked for in every forward: no module attributes.)"""
        ms = [e._modules.get(name) for e in self.experts._modules.values()
              for name in ("w13", "w2")]
        for m in ms:
            if not isinstance(m, QLinear):
                return None
        return ms

    def consolidate(self):
        """Stack the quantized experts' packed buffers for the grouped
        kernels: qweight [E, n, kw], scales [E, n, G], qzeros [E, n, zw].
        The experts' buffers become the stacks' parts: the weights are there
        once, and what is written to an expert is what the kernels read."""
        ms = self._layers()
        return None if ms is None else self._stacks(ms)

    def _stacks(self, ms=None) -> dict:
        """The stacks of the experts' buffers as they are now: replaced or
        moved ones are stacked again."""
        ms = ms or self._layers()
        g = self._current(ms)
        if g is None:
            with _STACKING:
                g = self._current(ms) or self._stack(ms)
        return g

    def _current(self, ms):
        g = self._grouped
        if g is None:
            return None
        for key, stacked in zip(_PACKED, g["at"]):
            if [m._buffers[key].data_ptr() for m in ms] != stacked or \
                    g["w13"][key].data_ptr() != stacked[0] or \
                    g["w2"][key].data_ptr() != stacked[1]:
                return None
        return g

    def _stack(self, ms) -> dict:
        g = {}
        # (ordinary tensors, which may be written to, in any mode)
        with torch.inference_mode(False), torch.no_grad():
            for name, mods in (("w13", ms[::2]), ("w2", ms[1::2])):
                g[name] = {key: torch.stack([getattr(m, key) for m in mods])
                           for key in _PACKED}
                g[name].update(bits=mods[0].bits, g=mods[0].group_size,
                               n=mods[0].out_features, k=mods[0].in_features)
        device = g["w2"]["qweight"].device
        if device.type == "cuda":
            if torch.cuda.is_current_stream_capturing():
                return g         # the graph's: filled whenever it runs
            # before another stream reads the stacks
            torch.cuda.current_stream(device).synchronize()
        for name, mods in (("w13", ms[::2]), ("w2", ms[1::2])):
            for key in _PACKED:
                for m, part in zip(mods, g[name][key]):
                    setattr(m, key, part)
        # where the layers' buffers are while they are parts of the stacks
        g["at"] = [[m._buffers[key].data_ptr() for m in ms] for key in _PACKED]
        self._grouped = g
        return g

    def forward(self, x):
        b, s, h = x.shape
        x2 = x.reshape(-1, h)
        t = x2.shape[0]
        # up to 64 rows go through the grouped kernels whoever watches the
        # experts; more do where the experts are nothing but their matrices
        ms = self._layers() if x.is_cuda else None
        if ms is not None and not any(map(gathers, ms)) and (
                t * self.top_k <= 64 or self._plain()):
            y2 = self._forward_grouped(x2, self._stacks(ms))
        else:
            weights, ids = self.route(x2)
            y2 = self._forward_loop(x2, weights, ids)
        return y2.reshape(b, s, h)

    def _plain(self) -> bool:
        """Routing and experts are what the grouped kernels do: no hook, class
        or forward of their own, and shapes that the kernels take."""
        cls = type(self)
        return (self.n_experts <= 64 and self.top_k <= 4
                and cls.route is MixtralMoE.route
                and cls._forward_loop is MixtralMoE._forward_loop
                and not {"route", "_forward_loop"} & self.__dict__.keys()
                and all(type(e) is MixtralExpert
                        and not hooked(e, e.w13, e.w2) for e in self.experts)
                and all(type(m) is QLinear and m.group_size % 32 == 0
                        for e in self.experts for m in (e.w13, e.w2)))

    def _forward_loop(self, x2, weights, ids):
        y = torch.zeros_like(x2)
        if x2.is_cuda and torch.cuda.is_current_stream_capturing():
            # every token through every expert: the host may not wait for
            # the routing
            for e, expert in enumerate(self.experts):
                w = (weights * (ids == e)).sum(dim=-1, keepdim=True)
                y += expert(x2) * w.to(y.dtype)
            return y
        for e in range(self.n_experts):
            mask = (ids == e)
            tok_mask = mask.any(dim=-1)
            if not bool(tok_mask.any()):
                continue
            xe = x2[tok_mask]
            ye = self.experts[e](xe)
            w = (weights * mask.float()).sum(dim=-1)[tok_mask]
            y[tok_mask] += ye * w.unsqueeze(-1).to(ye.dtype)
        return y

    def _forward_grouped(self, x2, g):
        """On the device from logits to sum, any number of tokens: routing
        and row tiles in one kernel, grouped products with silu·mul in the
        first one's epilogue, weighted sum of a token's rows."""
        from ..ops import hip_ext
        ext = hip_ext()
        a, b = g["w13"], g["w2"]
        logits16 = self.gate(x2).contiguous()  # dense bf16 router GEMV

        def part(x, logits):
            bm = ext.moe_tile(x.shape[0] * self.top_k, self.n_experts, a["k"],
                              a["g"], b["k"], b["g"])
            src, pos, w, tiles = ext.moe_plan(logits, self.top_k, bm)
            h = ext.moe_linear(x, src, tiles, a["qweight"], a["scales"],
                               a["qzeros"], a["bits"], a["g"], True, bm)
            rows = ext.moe_linear(h, None, tiles, b["qweight"], b["scales"],
                                  b["qzeros"], b["bits"], b["g"], False, bm)
            return ext.moe_sum(rows, pos, w)

        t = x2.shape[0]
        most = _ROWS_ELEMENTS // max(a["k"], self.top_k * b["k"])
        if t <= most:
            return part(x2, logits16)
        n = -(-t // most)
        return torch.cat([part(x, z) for x, z in zip(
            x2.tensor_split(n), logits16.tensor_split(n))])


class MixtralDecoderLayer(nn.Module):
    def __init__(self, cfg: MixtralConfig, dtype):
        super().__init__()
        lcfg = LlamaConfig(hidden_size=cfg.hidden_size, n_heads=cfg.n_heads,
                           n_kv_heads=cfg.n_kv_heads, head_dim=cfg.head_dim,
                           rope_theta=cfg.rope_theta, rms_eps=cfg.rms_eps)
        self.input_layernorm = RMSNorm(cfg.hidden_size, cfg.rms_eps, dtype)
        self.self_attn = LlamaAttention(lcfg, dtype)
        self.post_attention_layernorm = RMSNorm(cfg.hidden_size, cfg.rms_eps, dtype)
        self.moe = MixtralMoE(cfg, dtype)

    def forward(self, x, cache_k, cache_v, positions, seq_len_after,
                residual=None):
        if residual is None:
            residual = x
            h = self.input_layernorm(x)
        else:
            h, residual = F.rmsnorm_residual(x, residual,
                                             self.input_layernorm.weight,
                                             self.input_layernorm.eps)
        h, residual = attention_norm(
            self.self_attn, h, cache_k, cache_v, positions, seq_len_after,
            residual, self.post_attention_layernorm)
        h = self.moe(h)
        return h, residual

    def forward_decode_step(self, x, cache_k, cache_v, state, max_seq,
                            residual=None, tickets=None):
        if residual is None:
            residual = x
            h = self.input_layernorm(x)
        else:
            h, residual = F.rmsnorm_residual(x, residual,
                                             self.input_layernorm.weight,
                                             self.input_layernorm.eps)
        h = self.self_attn.forward_decode_graph(h, cache_k, cache_v, state,
                                                max_seq, tickets)
        h, residual = F.rmsnorm_residual(h, residual,
                                         self.post_attention_layernorm.weight,
                                         self.post_attention_layernorm.eps)
        h = self.moe(h)
        return h, residual


class MixtralForCausalLM(nn.Module):
    def __init__(self, cfg: MixtralConfig, dtype=torch.bfloat16):
        super().__init__()
        self.cfg = cfg
        self.dtype = dtype
        self.embed_tokens = nn.Embedding(cfg.vocab_size, cfg.hidden_size, dtype=dtype)
        self.layers = nn.ModuleList(MixtralDecoderLayer(cfg, dtype)
                                    for _ in range(cfg.n_layers))
        self.norm = RMSNorm(cfg.hidden_size, cfg.rms_eps, dtype)
        self.lm_head = Linear(cfg.hidden_size, cfg.vocab_size, dtype)

    @torch.no_grad()
    def init_random(self, seed: int = 0):
        g = torch.Generator().manual_seed(seed)
        for p in self.parameters():
            p.data.copy_(torch.randn(p.shape, generator=g, dtype=torch.float32)
                         .mul_(0.02).to(p.dtype))
        return self

    @torch.no_grad()
    def consolidate_moe(self):
        for layer in self.layers:
            layer.moe.consolidate()
        return self

    def make_cache(self, batch: int, max_seq: Optional[int] = None, device=None):
        dev = device or next(self.parameters()).device
        att = self.layers[0].self_attn
        return KVCache(self.cfg.n_layers, batch, att.n_kv_heads,
                       max_seq or self.cfg.max_seq, self.cfg.head_dim, dev,
                       dtype=self.dtype, n_heads=att.n_heads)

    def forward(self, input_ids, cache: KVCache, positions=None):
        b, s = input_ids.shape
        pos0 = cache.seq_len
        if positions is None:
            positions = torch.arange(
                pos0, pos0 + s, device=input_ids.device,
                dtype=torch.int32 if input_ids.is_cuda else None)
        if positions.is_cuda:
            positions = positions.to(torch.int32)    # once, not in every layer
        x = self.embed_tokens(input_ids)
        residual = None
        for i, layer in enumerate(self.layers):
            x, residual = layer(x, cache.k[i], cache.v[i], positions,
                                pos0 + s, residual)
        x = self.norm(x, residual=residual)
        logits = self.lm_head(x)
        cache.advance(s)
        return logits

    def forward_decode_step(self, input_ids, cache, state, max_seq):
        x = self.embed_tokens(input_ids)
        residual, tickets = None, getattr(cache, "tickets", None)
        for i, layer in enumerate(self.layers):
            x, residual = layer.forward_decode_step(
                x, cache.k[i], cache.v[i], state, max_seq, residual, tickets)
        x = self.norm(x, residual=residual)
        return self.lm_head(x)

    @torch.no_grad()
    def generate(self, input_ids, max_new_tokens: int = 16, cache=None,
                 gen_cfg=None, generator=None):
        from .generation import autoregressive_generate
        return autoregressive_generate(self, input_ids, max_new_tokens,
                                       cache, gen_cfg, generator)
