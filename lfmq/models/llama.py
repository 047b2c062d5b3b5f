"""Llama-3 family architecture, built natively for the MI355X decode path.

Random-init from a local config (no network => no pretrained weights).
MI355X-first choices:
  - fused qkv_proj and gate_up_proj Linears (one GEMV launch each at
    decode instead of 3/2 — launch overhead is the TP=8 risk)
  - static KV cache + pure-tensor decode step, hipGraph-capturable
  - attention decode / rmsnorm / rope / silu·mul via the gfx950 HIP
    kernels (lfmq.ops.functional)

TP sharding (applied by lfmq.dist.tp): qkv/gate_up/lm_head column-split,
o_proj/down_proj row-split with all-reduce.
"""
from __future__ import annotations

import math
from dataclasses import dataclass, field, asdict
from typing import Optional

import torch
import torch.nn as nn

from ..ops import functional as F
from .kvcache import KVCache
from .linear import Linear, hooked
from .qlinear import FEW_ROWS, QLinear, rows_fused


@dataclass
class LlamaConfig:
    vocab_size: int = 128256
    hidden_size: int = 4096
    intermediate_size: int = 14336
    n_layers: int = 32
    n_heads: int = 32
    n_kv_heads: int = 8
    head_dim: int = 128
    rms_eps: float = 1e-5
    rope_theta: float = 500000.0
    max_seq: int = 8192
    tie_embeddings: bool = False
    arch: str = "llama"

    @classmethod
    def llama3_8b(cls, **kw):
        return cls(**{**dict(vocab_size=128256, hidden_size=4096,
                             intermediate_size=14336, n_layers=32, n_heads=32,
                             n_kv_heads=8), **kw})

    @classmethod
    def llama3_70b(cls, **kw):
        return cls(**{**dict(vocab_size=128256, hidden_size=8192,
                             intermediate_size=28672, n_layers=80, n_heads=64,
                             n_kv_heads=8), **kw})

    @classmethod
    def tiny(cls, **kw):
        """2-layer 8B-shaped-per-layer test model."""
        return cls(**{**dict(vocab_size=512, hidden_size=256,
                             intermediate_size=512, n_layers=2, n_heads=4,
                             n_kv_heads=2, head_dim=64, max_seq=512), **kw})

    def to_dict(self) -> dict:
        return asdict(self)

    @classmethod
    def from_dict(cls, d: dict) -> "LlamaConfig":
        d = {k: v for k, v in d.items() if k in cls.__dataclass_fields__}
        return cls(**d)


class RMSNorm(nn.Module):
    def __init__(self, dim: int, eps: float, dtype=torch.bfloat16):
        super().__init__()
        self.eps = eps
        self.weight = nn.Parameter(torch.ones(dim, dtype=dtype))

    def forward(self, x, residual: Optional[torch.Tensor] = None):
        return F.rmsnorm(x, self.weight, self.eps, residual)


def linear_norm(p: nn.Module, x, residual, norm: RMSNorm):
    """F.rmsnorm_residual(p(x), residual) of the norm, and what it norms: in the
    product's own launches where p is a packed layer as it is.  (us, 77 rows of
    2048: the sum of parts 3.9 and the norm 3.2, both in one 4.0)"""
    if x.is_cuda and type(p) is QLinear and not hasattr(p, "perm") and \
            not hooked(p):
        return F.dq_linear_norm(x, p, residual, norm.weight, norm.eps)
    return F.rmsnorm_residual(p(x), residual, norm.weight, norm.eps)


def takes_factors(p: QLinear) -> bool:
    """Whether a norm in front of p is worth a launch of its own for 17 to 48
    rows: where a product without it may be `dq_mid`'s or `dq_short`'s.  A step of
    four layers of 2048, 4 bits: 17 rows 217 us with it, 219 without (groups of 64
    230 and 238), 32 rows 216 and 230, 48 rows 249 and 261; 8 bits 228 and 231 at 17.
    In a graph, that is: one by one the launches cost the host 4 us a layer (20 rows
    347 and 330)."""
    return p.bits == 8 or p.in_features >= 2048


def shares_k(p: nn.Module) -> bool:
    """Whether p's forward_resid is a packed layer's product and nothing else."""
    return type(p) is QLinear and not hasattr(p, "perm") \
        and unchanged(p, QLinear, "forward", "forward_resid") and not hooked(p)


def resid_product(p: QLinear, x, resid, tickets):
    """p.forward_resid(x, resid), by the kernel that shares k among workgroups where
    that gains: nowhere outside these sizes, and a look at p and the kernel's own
    rule take 5 us a layer of the host (a step of 8 without a graph, four layers of
    2048, 286 us with them, 262 without)."""
    k = x.shape[-1]
    if x.is_cuda and 2 < x.shape[0] <= 16 and k >= 8192 \
            and k * resid.shape[-1] >= 32 << 20 and shares_k(p):
        y = F.dq_linear_parts(x, p, resid, tickets)
        if y is not None:
            return y
    return p.forward_resid(x, resid)


class LlamaAttention(nn.Module):
    def __init__(self, cfg: LlamaConfig, dtype):
        super().__init__()
        self.cfg = cfg
        self.n_heads = cfg.n_heads
        self.n_kv_heads = cfg.n_kv_heads
        self.head_dim = cfg.head_dim
        qkv_out = (cfg.n_heads + 2 * cfg.n_kv_heads) * cfg.head_dim
        self.qkv_proj = nn.Linear(cfg.hidden_size, qkv_out, bias=False, dtype=dtype)
        self.o_proj = nn.Linear(cfg.n_heads * cfg.head_dim, cfg.hidden_size,
                                bias=False, dtype=dtype)
        self.scale = 1.0 / math.sqrt(cfg.head_dim)

    def forward(self, x: torch.Tensor, cache_k: torch.Tensor,
                cache_v: torch.Tensor, positions: torch.Tensor,
                seq_len_after: int) -> torch.Tensor:
        return self.o_proj(self.attend(x, cache_k, cache_v, positions,
                                       seq_len_after))

    def attend(self, x, cache_k, cache_v, positions, seq_len_after):
        """What o_proj projects."""
        b, s, _ = x.shape
        hq, hkv, d = self.n_heads, self.n_kv_heads, self.head_dim
        qkv = self.qkv_proj(x)
        pos0 = seq_len_after - s
        if x.is_cuda:
            # fused rope + KV append straight off the qkv buffer (one launch)
            q = F.qkv_rope_append(qkv, cache_k, cache_v, positions, pos0, hq,
                                  self.cfg.rope_theta)
            if s == 1:
                o = F.attn_decode(q.view(b, hq, 1, d), cache_k, cache_v,
                                  seq_len_after, self.scale)
                o = o.view(b, s, hq * d)
            elif F.USE_FLASH_PREFILL and d == 128:
                # one-kernel MFMA flash prefill; handles pos0 > 0 too
                # (LFMQ_FLASH_PREFILL=0 restores the matmul-chain path)
                o = F.attn_prefill_fused(q, cache_k, cache_v, pos0,
                                         self.scale).reshape(b, s, hq * d)
            else:
                qh = q.transpose(1, 2)
                kc = cache_k[:, :, pos0:seq_len_after]
                vc = cache_v[:, :, pos0:seq_len_after]
                if pos0 == 0:
                    o = F.attn_prefill(qh, kc, vc, causal=True, scale=self.scale)
                else:
                    o = self._chunk_attn(qh, cache_k, cache_v, pos0, seq_len_after)
                o = o.transpose(1, 2).reshape(b, s, hq * d)
            return o
        q, k, v = qkv.split([hq * d, hkv * d, hkv * d], dim=-1)
        q = q.reshape(b, s, hq, d)
        k = k.reshape(b, s, hkv, d)
        v = v.reshape(b, s, hkv, d)
        q, k = F.apply_rope(q, k, positions, self.cfg.rope_theta)
        F.kv_append(cache_k, cache_v, k, v, pos0)
        qh = q.transpose(1, 2)  # [b, hq, s, d]
        if s == 1:
            o = F.attn_decode(qh, cache_k, cache_v, seq_len_after, self.scale)
        elif pos0 == 0:
            o = F.attn_prefill(qh, k.transpose(1, 2), v.transpose(1, 2),
                               causal=True, scale=self.scale)
        else:  # chunked continuation: attend to full cache, causal inside chunk
            o = self._chunk_attn(qh, cache_k, cache_v, pos0, seq_len_after)
        return o.transpose(1, 2).reshape(b, s, hq * d)

    def forward_decode_graph(self, x, cache_k, cache_v, state, max_seq,
                             tickets=None):
        """hipGraph-capturable decode step (s == 1, GPU only)."""
        b, s, _ = x.shape
        o = self.decode_qkv_attn(x, cache_k, cache_v, state, max_seq,
                                 tickets=tickets)
        return self.o_proj(o)

    def decode_qkv_attn(self, x, cache_k, cache_v, state, max_seq,
                        rms_eps: float = -1.0, tickets=None, row_scale=None):
        """qkv GEMV -> ONE fused rope+KV-append+attention launch; returns
        [b, s, hq*d] (pre o_proj).  rms_eps >= 0 additionally fuses the
        input RMSNorm into the qkv GEMV (norm weight pre-folded); row_scale:
        as factors of x's rows, known already."""
        b, s, _ = x.shape
        if row_scale is not None:
            qkv = F.dq_linear_scaled(x, row_scale, self.qkv_proj)
        elif rms_eps >= 0:
            qkv = self.qkv_proj.forward_rms(x, rms_eps)
        else:
            qkv = self.qkv_proj(x)
        o = F.attn_decode_fused(qkv.view(b, -1), cache_k, cache_v, state,
                                max_seq, self.scale, self.n_heads,
                                self.cfg.rope_theta, tickets)
        return o.view(b, s, self.n_heads * self.head_dim)

    def _chunk_attn(self, q, cache_k, cache_v, pos0, seq_len_after):
        b, hq, s, d = q.shape
        hkv = cache_k.shape[1]
        rep = hq // hkv
        kc = cache_k[:, :, :seq_len_after].float().repeat_interleave(rep, dim=1)
        vc = cache_v[:, :, :seq_len_after].float().repeat_interleave(rep, dim=1)
        sc = torch.einsum("bhqd,bhtd->bhqt", q.float(), kc) * self.scale
        t_idx = torch.arange(seq_len_after, device=q.device)
        q_idx = pos0 + torch.arange(s, device=q.device)
        mask = t_idx[None, :] > q_idx[:, None]
        sc = sc.masked_fill(mask, float("-inf"))
        p = torch.softmax(sc, dim=-1)
        return torch.einsum("bhqt,bhtd->bhqd", p, vc).to(q.dtype)


class LlamaMLP(nn.Module):
    def __init__(self, cfg: LlamaConfig, dtype):
        super().__init__()
        self.gate_up_proj = nn.Linear(cfg.hidden_size, 2 * cfg.intermediate_size,
                                      bias=False, dtype=dtype)
        self.down_proj = nn.Linear(cfg.intermediate_size, cfg.hidden_size,
                                   bias=False, dtype=dtype)
        self.inter = cfg.intermediate_size

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return self.down_proj(self.gated(x))

    def gated(self, x: torch.Tensor) -> torch.Tensor:
        """What down_proj projects."""
        gp = self.gate_up_proj
        m = x.numel() // x.shape[-1]
        if (x.is_cuda and isinstance(gp, QLinear)
                and type(gp).forward is QLinear.forward
                and not hasattr(gp, "perm")
                and (m <= 4 or (gp.bias is None and rows_fused(gp)))):
            # fused gate_up product + silu·mul epilogue (no separate pass)
            return F.dq_gemv_gateup(x, gp.qweight, gp.scales, gp.qzeros,
                                    gp.bits, gp.group_size)
        return F.silu_mul_gateup(gp(x), self.inter)


def unchanged(m, cls: type, *names: str) -> bool:
    """Whether these calls of m are what cls does, and not a caller's: of a module
    or a method put in their place only the call is known."""
    return all(getattr(type(m), n, None) is getattr(cls, n)
               and n not in getattr(m, "__dict__", ()) for n in names)


def attention_norm(att: nn.Module, x, cache_k, cache_v, positions,
                   seq_len_after, residual, norm: RMSNorm):
    """F.rmsnorm_residual of att's result, and what it norms."""
    if unchanged(att, LlamaAttention, "forward") and not hooked(att):
        return linear_norm(att.o_proj, att.attend(
            x, cache_k, cache_v, positions, seq_len_after), residual, norm)
    return F.rmsnorm_residual(
        att(x, cache_k, cache_v, positions, seq_len_after), residual,
        norm.weight, norm.eps)


def mlp_norm(mlp: nn.Module, x, residual, norm: RMSNorm):
    """The same of the feed-forward's."""
    if unchanged(mlp, LlamaMLP, "forward") and not hooked(mlp):
        return linear_norm(mlp.down_proj, mlp.gated(x), residual, norm)
    return F.rmsnorm_residual(mlp(x), residual, norm.weight, norm.eps)


class LlamaDecoderLayer(nn.Module):
    def __init__(self, cfg: LlamaConfig, dtype):
        super().__init__()
        self.input_layernorm = RMSNorm(cfg.hidden_size, cfg.rms_eps, dtype)
        self.self_attn = LlamaAttention(cfg, dtype)
        self.post_attention_layernorm = RMSNorm(cfg.hidden_size, cfg.rms_eps, dtype)
        self.mlp = LlamaMLP(cfg, dtype)

    def forward(self, x, cache_k, cache_v, positions, seq_len_after,
                residual=None):
        """Fused-residual form: returns (mlp_out, residual_after_attn) so
        the NEXT norm folds the pending add (one rmsnorm_residual kernel
        instead of add + rmsnorm).  residual=None => x is the raw input."""
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
        h = self.mlp(h)
        return h, residual

    def forward_normed(self, h, residual, cache_k, cache_v, positions,
                       seq_len_after, norm):
        """forward between norms: of the layer's normed input and what that
        was to the same of the next layer, whose norm it is."""
        att, mlp, post = self.self_attn, self.mlp, self.post_attention_layernorm
        if h.shape[1] > 1 and unchanged(att, LlamaAttention, "forward") \
                and unchanged(mlp, LlamaMLP, "forward"):
            products = (att.qkv_proj, att.o_proj, mlp.gate_up_proj,
                        mlp.down_proj)
            if cache_k.shape[0] == h.shape[0] and self._in_one_call(products):
                return F.prompt_layer(h, residual, cache_k, cache_v, positions,
                                      seq_len_after - h.shape[1], att.n_heads,
                                      att.cfg.rope_theta, att.scale, products,
                                      post, norm)
        h, residual = attention_norm(att, h, cache_k, cache_v, positions,
                                     seq_len_after, residual, post)
        return mlp_norm(mlp, h, residual, norm)

    def _in_one_call(self, products) -> bool:
        att, mlp = self.self_attn, self.mlp
        return (F.USE_FLASH_PREFILL and att.head_dim == 128
                and not F._NANCHECK
                and all(type(p) is QLinear and "perm" not in p._buffers
                        and "perm" not in p.__dict__ for p in products)
                and products[2].bias is None and rows_fused(products[2])
                and not hooked(att, mlp, *products))

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
        h = self.mlp(h)
        return h, residual

    def forward_decode_fused(self, x, cache_k, cache_v, state, max_seq,
                             tickets=None):
        """Folded-norm decode step: both RMSNorms ride inside the GEMVs
        and both residual adds ride in the o/down epilogues — 6 kernels
        per layer, no separate norm/add launches.  Requires
        _in_norm_folded and _post_norm_folded (lfmq.quant.fold)."""
        eps = self.input_layernorm.eps
        o = self.self_attn.decode_qkv_attn(x, cache_k, cache_v, state,
                                           max_seq, eps, tickets)
        x = self.self_attn.o_proj.forward_resid(o, x)
        mlp, gp = self.mlp, self.mlp.gate_up_proj
        h, eps = x, self.post_attention_layernorm.eps
        if x.shape[0] > 32 and gp.in_features >= 4096 and \
                gp.in_features * gp.out_features >= 24 << 20:
            # (several ranks, steps of a caller's own; others by
            # forward_decode_rows)
            # the product for prompts, which takes normed rows, is faster
            # (28672 x 4096 at 48 rows: 41 us with its norm, 50)
            h, eps = self.post_attention_layernorm(x), -1.0
        h = F.dq_gemv_gateup(h, gp.qweight, gp.scales, gp.qzeros, gp.bits,
                             gp.group_size, rms_eps=eps)
        return resid_product(mlp.down_proj, h, x, tickets)

    def forward_decode_rows(self, x, scale, cache_k, cache_v, state, max_seq,
                            following: Optional["LlamaDecoderLayer"],
                            tickets=None):
        """forward_decode_fused for 17 to 48 rows: an RMSNorm is a factor of
        each row, which the product before it leaves beside its result
        (x, scale, or None -> the same of the following layer, if there is
        one).  The products, which do not
        have to see whole rows any more, may split k.  us a step of four
        layers, norms in the products and this way: hidden 4096, 4 bits 410 /
        372 at 17 rows, 452 / 378 at 32, 459 / 425 at 48; 8 bits 551 / 473 at
        32; hidden 2048 268 / 260 at 48.  Up to 16 rows the product that walks over
        columns has the norm for nothing (with a gate 18 us at 16 rows of
        28672 x 4096, 26 for this way's at 17)."""
        att, mlp = self.self_attn, self.mlp
        gp, eps = mlp.gate_up_proj, self.post_attention_layernorm.eps
        o = att.decode_qkv_attn(x, cache_k, cache_v, state, max_seq,
                                self.input_layernorm.eps, tickets, scale)
        if takes_factors(gp):
            x, scale = F.dq_linear_scaled(o, None, att.o_proj, x, eps)
            h = F.dq_gateup_scaled(x, scale, gp)
        else:
            x = att.o_proj.forward_resid(o, x)
            h = F.dq_gemv_gateup(x, gp.qweight, gp.scales, gp.qzeros, gp.bits,
                                 gp.group_size, rms_eps=eps)
        if following is None:              # nobody reads the last one's
            return mlp.down_proj.forward_resid(h, x), None
        return F.dq_linear_scaled(
            h, None, mlp.down_proj, x, following.input_layernorm.eps,
            takes_factors(following.self_attn.qkv_proj))


class LlamaForCausalLM(nn.Module):
    def __init__(self, cfg: LlamaConfig, dtype=torch.bfloat16):
        super().__init__()
        self.cfg = cfg
        self.dtype = dtype
        self.embed_tokens = nn.Embedding(cfg.vocab_size, cfg.hidden_size, dtype=dtype)
        self.layers = nn.ModuleList(LlamaDecoderLayer(cfg, dtype)
                                    for _ in range(cfg.n_layers))
        self.norm = RMSNorm(cfg.hidden_size, cfg.rms_eps, dtype)
        self.lm_head = Linear(cfg.hidden_size, cfg.vocab_size, dtype)
        if cfg.tie_embeddings:
            self.lm_head.weight = self.embed_tokens.weight

    @torch.no_grad()
    def init_random(self, seed: int = 0):
        g = torch.Generator().manual_seed(seed)
        for p in self.parameters():
            p.data.copy_(torch.randn(p.shape, generator=g, dtype=torch.float32)
                         .mul_(0.02).to(p.dtype))
        return self

    def make_cache(self, batch: int, max_seq: Optional[int] = None,
                   device=None) -> KVCache:
        dev = device or next(self.parameters()).device
        # TP: layers may hold a KV-head shard; size the cache from the module
        att = self.layers[0].self_attn
        return KVCache(self.cfg.n_layers, batch, att.n_kv_heads,
                       max_seq or self.cfg.max_seq, self.cfg.head_dim, dev,
                       dtype=self.dtype, n_heads=att.n_heads)

    def forward(self, input_ids: torch.Tensor, cache: KVCache,
                positions: Optional[torch.Tensor] = None) -> torch.Tensor:
        """input_ids [b, s] -> logits [b, s, vocab].  Advances the cache."""
        b, s = input_ids.shape
        pos0 = cache.seq_len
        if positions is None:
            positions = torch.arange(
                pos0, pos0 + s, device=input_ids.device,
                dtype=torch.int32 if input_ids.is_cuda else None)
        if positions.is_cuda:
            positions = positions.to(torch.int32)    # once, not in every layer
        seq_after = pos0 + s
        x = self.embed_tokens(input_ids)
        if self._norms_ride(x):
            norms = [l.input_layernorm for l in self.layers] + [self.norm]
            x, residual = norms[0](x), x
            for i, layer in enumerate(self.layers):
                x, residual = layer.forward_normed(
                    x, residual, cache.k[i], cache.v[i], positions, seq_after,
                    norms[i + 1])
        else:
            residual = None
            for i, layer in enumerate(self.layers):
                x, residual = layer(x, cache.k[i], cache.v[i], positions,
                                    seq_after, residual)
            x = self.norm(x, residual=residual)
        logits = self.lm_head(x)
        cache.advance(s)
        return logits

    def _norms_ride(self, x) -> bool:
        """Whether a layer's last product may take the next norm with it."""
        return x.is_cuda and len(self.layers) > 0 and all(
            type(l).forward is LlamaDecoderLayer.forward for l in self.layers
        ) and type(self.norm).forward is RMSNorm.forward and not hooked(
            self.norm, *self.layers)

    def _engine_for(self, cache, batch: int) -> bool:
        """Build/bind the persistent decode engine for this cache (lazy;
        one stream build per cache).  False => launched-kernel path.
        The env opt-in is re-read every step so LFMQ_ENGINE can be
        toggled within one process; only STRUCTURAL unsupport (arch /
        shape) latches."""
        import os
        if os.environ.get("LFMQ_ENGINE", "0") != "1":
            return False
        eng = getattr(self, "_engine", None)
        if eng is not None and eng.cache is cache:
            return True
        if getattr(self, "_engine_unsupported", False):
            return False
        from .engine import DecodeEngine, engine_supported
        if not engine_supported(self, batch):
            self._engine_unsupported = True
            return False
        self._engine = DecodeEngine(self, cache, cache.max_seq)
        return True

    def _decode_fused_ready(self) -> bool:
        for layer in self.layers:
            if not (getattr(layer, "_in_norm_folded", False)
                    and getattr(layer, "_post_norm_folded", False)):
                return False
            if not isinstance(layer.self_attn.qkv_proj, QLinear):
                return False
            for proj in (layer.self_attn.qkv_proj, layer.self_attn.o_proj,
                         layer.mlp.gate_up_proj, layer.mlp.down_proj):
                if hasattr(proj, "perm"):
                    # act-order: inputs need the perm gather — QLinear
                    # .forward handles it; the fused 6-kernel chain bypasses
                    # QLinear.forward, so fall back to the step path
                    return False
        return True

    def _rows_fused(self) -> bool:
        """Whether the products of a larger batch may take norm, gate and
        residual with them."""
        for layer in self.layers:
            mlp, att = layer.mlp, layer.self_attn
            ins, outs = (att.qkv_proj, mlp.gate_up_proj), \
                        (att.o_proj, mlp.down_proj)
            if not all(rows_fused(p) for p in ins) or \
                    mlp.gate_up_proj.bias is not None:
                return False
            if not all(isinstance(p, QLinear) and p.group_size % 64 == 0
                       and not hooked(p) for p in outs):
                return False
            if type(mlp).forward is not LlamaMLP.forward or hooked(
                    layer.input_layernorm, layer.post_attention_layernorm,
                    mlp):
                return False
        return True

    def _rows_scaled(self) -> bool:
        """Whether norms may also be left to the product before them."""
        return all(
            unchanged(layer, LlamaDecoderLayer, "forward_decode_fused")
            and unchanged(layer.self_attn, LlamaAttention, "decode_qkv_attn")
            and unchanged(layer.self_attn.qkv_proj, QLinear, "forward_rms")
            and all(unchanged(p, QLinear, "forward", "forward_resid")
                    for p in (layer.self_attn.o_proj, layer.mlp.down_proj))
            for layer in self.layers)

    def forward_decode_step(self, input_ids, cache, state, max_seq):
        """One hipGraph-capturable decode step: [b,1] ids -> [b,1,vocab]."""
        # persistent weight-streaming engine: the whole layer stack in ONE
        # kernel launch (csrc/engine.hip); lm_head stays a separate launch.
        if input_ids.is_cuda and self._engine_for(cache, input_ids.shape[0]):
            x = self._engine.step(input_ids, state)
            return self.lm_head(x)
        x = self.embed_tokens(input_ids)
        if getattr(self, "_fused_decode", None) is None:
            self._fused_decode = self._decode_fused_ready()
        b, tickets = input_ids.shape[0], getattr(cache, "tickets", None)
        if self._fused_decode and (b <= 4 or (b <= FEW_ROWS
                                              and self._rows_fused())):
            if b > 16 and self._rows_scaled():
                first, scale = self.layers[0], None
                if takes_factors(first.self_attn.qkv_proj):
                    scale = F.row_scale(x, first.input_layernorm.eps)
                for i, (layer, following) in enumerate(
                        zip(self.layers, [*self.layers[1:], None])):
                    x, scale = layer.forward_decode_rows(
                        x, scale, cache.k[i], cache.v[i], state, max_seq,
                        following, tickets)
            else:
                for i, layer in enumerate(self.layers):
                    x = layer.forward_decode_fused(x, cache.k[i], cache.v[i],
                                                   state, max_seq, tickets)
            x = self.norm(x)
        else:
            residual = None
            for i, layer in enumerate(self.layers):
                x, residual = layer.forward_decode_step(
                    x, cache.k[i], cache.v[i], state, max_seq, residual,
                    tickets)
            x = self.norm(x, residual=residual)
        return self.lm_head(x)

    @torch.no_grad()
    def generate(self, input_ids: torch.Tensor, max_new_tokens: int = 32,
                 cache: Optional[KVCache] = None, gen_cfg=None,
                 generator=None) -> torch.Tensor:
        from .generation import autoregressive_generate
        return autoregressive_generate(self, input_ids, max_new_tokens,
                                       cache, gen_cfg, generator)
