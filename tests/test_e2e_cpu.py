"""End-to-end CPU configs.

Config #1: OPT-125m-shaped per-tensor int8 RTN quantize +
CPU matmul decode — quantize -> save -> load -> greedy decode equivalence
vs fp32 within tolerance.  Plus tiny-Llama GPTQ/AWQ end-to-end fidelity.
"""
import types

import pytest
import torch

from lfmq import QuantConfig, build_model, load, quantize, save
from lfmq.models.kvcache import KVCache
from lfmq.models.llama import LlamaConfig, LlamaForCausalLM
from lfmq.models.mixtral import MixtralConfig
from lfmq.models.opt import OPTConfig
from lfmq.quant.calib import CalibStream


def test_config1_opt_int8_cpu_decode(tmp_path):
    cfg = OPTConfig.tiny()
    fp = build_model(cfg, seed=11)
    ids = torch.randint(0, cfg.vocab_size, (2, 12))
    ref_out = fp.generate(ids, max_new_tokens=8)
    ref_logits = fp(ids, fp.make_cache(2, 64))

    qcfg = QuantConfig(scheme="rtn", bits=8, per_tensor=True, group_size=0)
    qm = quantize(build_model(cfg, seed=11), qcfg)
    p = str(tmp_path / "opt")
    save(qm, p, qcfg)
    qm2 = load(p)

    q_logits = qm2(ids, qm2.make_cache(2, 64))
    # logits close in relative terms
    rel = (q_logits - ref_logits).abs().mean() / ref_logits.abs().mean()
    assert rel < 0.05
    q_out = qm2.generate(ids, max_new_tokens=8)
    agree = (q_out == ref_out).float().mean()
    assert agree > 0.85  # greedy tokens nearly identical


def test_tiny_llama_gptq_e2e(tmp_path):
    cfg = LlamaConfig.tiny()
    fp = build_model(cfg, seed=3)
    qcfg = QuantConfig(scheme="gptq", bits=4, group_size=64,
                       calib_n_seqs=4, calib_seq_len=64)
    calib = CalibStream(cfg.vocab_size, 64, 4, qcfg.calib_seed)
    qm = quantize(build_model(cfg, seed=3), qcfg, calib=calib)
    p = str(tmp_path / "llama_gptq")
    save(qm, p, qcfg)
    qm2 = load(p)

    ids = torch.randint(0, cfg.vocab_size, (1, 16))
    lf = fp(ids, fp.make_cache(1, 32)).float()
    lq = qm2(ids, qm2.make_cache(1, 32)).float()
    # logit KL under threshold (random-init tiny model: loose bound)
    pf = torch.log_softmax(lf, -1)
    pq = torch.log_softmax(lq, -1)
    kl = (pf.exp() * (pf - pq)).sum(-1).mean()
    assert kl < 0.5, f"KL={kl}"


def test_tiny_llama_awq_e2e(tmp_path):
    cfg = LlamaConfig.tiny()
    fp = build_model(cfg, seed=5)
    qcfg = QuantConfig(scheme="awq", bits=4, group_size=64,
                       calib_n_seqs=2, calib_seq_len=64, awq_grid=8)
    calib = CalibStream(cfg.vocab_size, 64, 2, qcfg.calib_seed)
    qm = quantize(build_model(cfg, seed=5), qcfg, calib=calib)
    p = str(tmp_path / "llama_awq")
    save(qm, p, qcfg)
    qm2 = load(p)
    ids = torch.randint(0, cfg.vocab_size, (1, 16))
    lf = fp(ids, fp.make_cache(1, 32)).float()
    lq = qm2(ids, qm2.make_cache(1, 32)).float()
    pf = torch.log_softmax(lf, -1)
    pq = torch.log_softmax(lq, -1)
    kl = (pf.exp() * (pf - pq)).sum(-1).mean()
    assert kl < 0.5, f"KL={kl}"


def test_quantized_decode_prefill_consistency():
    """Decode one-token-at-a-time must equal prefill logits (cache math)."""
    cfg = LlamaConfig.tiny()
    qcfg = QuantConfig(scheme="rtn", bits=4, group_size=64)
    qm = quantize(build_model(cfg, seed=9), qcfg)
    ids = torch.randint(0, cfg.vocab_size, (1, 8))
    lp = qm(ids, qm.make_cache(1, 32)).float()
    cache = qm.make_cache(1, 32)
    outs = []
    for t in range(8):
        outs.append(qm(ids[:, t:t + 1], cache).float())
    ld = torch.cat(outs, dim=1)
    assert torch.allclose(lp, ld, atol=2e-2, rtol=1e-2)


def test_opt_awq_e2e(tmp_path):
    """AWQ on the OPT arch (LayerNorm/v_proj/fc1 scale plan)."""
    from lfmq.quant.calib import CalibStream
    cfg = OPTConfig.tiny()
    fp = build_model(cfg, seed=14)
    qcfg = QuantConfig(scheme="awq", bits=4, group_size=32, awq_grid=6,
                       calib_n_seqs=2, calib_seq_len=32)
    calib = CalibStream(cfg.vocab_size, 32, 2, qcfg.calib_seed)
    qm = quantize(build_model(cfg, seed=14), qcfg, calib=calib)
    ids = torch.randint(0, cfg.vocab_size, (1, 10))
    lf = fp(ids, fp.make_cache(1, 24)).float()
    lq = qm(ids, qm.make_cache(1, 24)).float()
    pf = torch.log_softmax(lf, -1); pq = torch.log_softmax(lq, -1)
    kl = (pf.exp() * (pf - pq)).sum(-1).mean()
    assert kl < 0.5, float(kl)


def test_sym_quant_e2e_round_trip(tmp_path):
    """sym=True end-to-end: quantize -> save -> load -> decode; the
    packed layout stores the constant sym zero like any other zero."""
    import torch

    import lfmq
    from lfmq.models.llama import LlamaConfig
    cfg = LlamaConfig.tiny()
    qcfg = lfmq.QuantConfig(scheme="rtn", bits=4, group_size=32, sym=True)
    qm = lfmq.quantize(lfmq.build_model(cfg, seed=47), qcfg)
    p = str(tmp_path / "sym")
    lfmq.save(qm, p, qcfg)
    back = lfmq.load(p)
    ids = torch.arange(8).remainder(cfg.vocab_size).reshape(1, 8)
    a = qm(ids, qm.make_cache(1, 16))
    b = back(ids, back.make_cache(1, 16))
    assert torch.equal(a, b)
    out = back.generate(ids[:, :4], max_new_tokens=4)
    assert out.shape == (1, 8)


def test_per_channel_quant_e2e(tmp_path):
    """group_size=-1 (per-channel: one group = the whole row) through
    quantize -> save -> load -> forward."""
    import torch

    import lfmq
    from lfmq.models.llama import LlamaConfig
    cfg = LlamaConfig.tiny()
    qcfg = lfmq.QuantConfig(scheme="rtn", bits=4, group_size=-1)
    qm = lfmq.quantize(lfmq.build_model(cfg, seed=49), qcfg)
    p = str(tmp_path / "pc")
    lfmq.save(qm, p, qcfg)
    back = lfmq.load(p)
    ids = torch.arange(8).remainder(cfg.vocab_size).reshape(1, 8)
    assert torch.equal(qm(ids, qm.make_cache(1, 16)),
                       back(ids, back.make_cache(1, 16)))


def test_caches_own_their_arrival_counters():
    """Steps on two caches may overlap: nothing of theirs is shared, and there
    is a counter for every query head."""
    from lfmq.models.mixtral import MixtralConfig
    for cfg in (LlamaConfig.tiny(), MixtralConfig.tiny()):
        m = build_model(cfg, seed=0)
        a, b = m.make_cache(3, 16), m.make_cache(3, 16)
        assert a.tickets.data_ptr() != b.tickets.data_ptr()
        assert a.tickets.tolist() == [0] * 3 * cfg.n_heads


class Standin(torch.nn.Module):
    """A caller's module in the place of a layer's: a call, and nothing else."""

    def __init__(self, of):
        super().__init__()
        self.of = of

    def forward(self, *args):
        return self.of(*args)


@pytest.mark.parametrize("arch", ["llama", "mixtral"])
@pytest.mark.parametrize("names", [("self_attn",), ("mlp",), ("self_attn", "mlp")])
@pytest.mark.parametrize("norms_ride", [False, True])
def test_replaced_modules_are_called(arch, names, norms_ride, monkeypatch):
    """Attention and feed-forward that a caller has replaced take prompts and
    tokens, also where a layer's last product takes the next norm along (on the
    GPU)."""
    cfg = (LlamaConfig if arch == "llama" else MixtralConfig).tiny()
    m = build_model(cfg, seed=3)
    if norms_ride:
        monkeypatch.setattr(LlamaForCausalLM, "_norms_ride", lambda *a: True)
    ids = torch.randint(0, cfg.vocab_size, (2, 9))

    def logits():
        cache = m.make_cache(2, 16)
        return m(ids, cache), m(ids[:, :1], cache)

    want = logits()
    m.make_cache = lambda b, n: KVCache(
        cfg.n_layers, b, cfg.n_kv_heads, n, cfg.head_dim, "cpu", dtype=m.dtype)
    for layer in m.layers:
        for name in names:
            name = "moe" if arch == "mixtral" and name == "mlp" else name
            setattr(layer, name, Standin(getattr(layer, name)))
    for a, b in zip(logits(), want):
        assert torch.equal(a, b)


def out(x, n):
    return torch.zeros(*x.shape[:-1], n, dtype=x.dtype)


def shapes_alone(m, monkeypatch):
    """A captured step's products and attention (GPU only) as their shapes."""
    from lfmq.ops import functional as F
    d = m.cfg.head_dim
    monkeypatch.setattr(F, "dq_gemv_gateup", lambda x, q, *a, **kw: out(
        x, q.shape[0] // 2))
    monkeypatch.setattr(F, "dq_linear", lambda x, q, *a, **kw: out(x, q.shape[0]))
    monkeypatch.setattr(F, "attn_decode_fused", lambda qkv, k, v, st, n, sc, hq,
                        *a: torch.zeros(len(qkv), hq * d, dtype=qkv.dtype))
    monkeypatch.setattr(F, "row_scale", lambda x, eps: "embedding")
    monkeypatch.setattr(F, "dq_linear_scaled", lambda x, scale, p, resid=None,
                        eps=-1.0, apart=True: out(x, p.out_features)
                        if eps < 0 else (out(x, p.out_features), "product"))
    monkeypatch.setattr(F, "dq_gateup_scaled", lambda x, scale, p: out(
        x, p.out_features // 2))


def step(m, b):
    m.forward_decode_step(torch.zeros(b, 1, dtype=torch.long), m.make_cache(b, 8),
                          torch.zeros(3, dtype=torch.int32), 8)


@pytest.mark.parametrize("bits,parts", [(4, True), (4, False), (8, False)])
def test_factors_of_rows_that_somebody_reads(bits, parts, monkeypatch):
    """A step of 17 rows asks for the factors of a norm's rows only where a
    product reads them, and for a launch of their own only where the next product
    is worth one; what a product in parts leaves is taken anyhow."""
    from lfmq.ops import functional as F
    cfg = LlamaConfig.tiny()
    m = quantize(build_model(cfg, seed=3), QuantConfig(
        scheme="rtn", bits=bits, group_size=64, fold_rms=True))
    asked, given, read = [], [], []
    names = {id(p): f"{i}.{n}" for i, l in enumerate(m.layers) for n, p in
             (("qkv", l.self_attn.qkv_proj), ("o", l.self_attn.o_proj),
              ("gate_up", l.mlp.gate_up_proj), ("down", l.mlp.down_proj))}

    def factors(name):
        given.append(name)
        return name

    def linear_scaled(x, scale, p, resid=None, eps=-1.0, apart=True):
        y, name = out(x, p.out_features), names[id(p)]
        if scale is not None:
            read.append(scale)
        if eps < 0:
            return y
        asked.append((name, apart))
        return y, factors(name) if parts or apart else None

    shapes_alone(m, monkeypatch)
    monkeypatch.setattr(F, "row_scale", lambda x, eps: factors("embedding"))
    monkeypatch.setattr(F, "dq_linear_scaled", linear_scaled)
    monkeypatch.setattr(F, "dq_gateup_scaled", lambda x, scale, p: (
        read.append(scale), out(x, p.out_features // 2))[1])
    step(m, 17)
    assert m._fused_decode and m._rows_fused() and m._rows_scaled()
    last = len(m.layers) - 1
    assert last > 0
    assert given == read
    assert ("embedding" in given) == (bits == 8)
    assert asked == [(f"{i}.{n}", bits == 8) for i in range(last + 1)
                     for n in ("o", "down")
                     if (n == "o" and bits == 8) or (n == "down" and i < last)]


def test_products_that_share_k_are_a_packed_layers_own():
    """A caller's forward_resid or forward, hooks and gathers keep the call."""
    from lfmq.models.llama import shares_k
    from lfmq.models.qlinear import QLinear

    def layer():
        return QLinear(64, 8, 4, 64)
    assert shares_k(layer())
    own = type("Own", (QLinear,), {"forward_resid": lambda self, x, r: r})
    assert not shares_k(own(64, 8, 4, 64))
    for name in ("forward", "forward_resid"):
        p = layer()
        setattr(p, name, types.MethodType(lambda self, *a: a[-1], p))
        assert not shares_k(p)
    p = layer()
    p.register_forward_hook(lambda *a: None)
    assert not shares_k(p)
    p = layer()
    p.register_buffer("perm", torch.arange(64))
    assert not shares_k(p)


@pytest.mark.parametrize("where", ["class", "instance"])
@pytest.mark.parametrize("b", [3, 17])
@pytest.mark.parametrize("name", ["forward_decode_fused", "decode_qkv_attn"])
def test_a_callers_own_step_is_called(name, b, where, monkeypatch):
    """A layer's step, or its attention's, that a caller has overridden takes
    batches of every size, by the call that it knows."""
    cfg = LlamaConfig.tiny()
    m = quantize(build_model(cfg, seed=3), QuantConfig(
        scheme="rtn", bits=8, group_size=64, fold_rms=True))
    shapes_alone(m, monkeypatch)
    layer, calls = m.layers[1], []
    on = layer if name == "forward_decode_fused" else layer.self_attn
    old = getattr(type(on), name)

    def own(self, x, cache_k, cache_v, state, max_seq, *more):
        assert len(more) <= 2
        calls.append(x.shape[0])
        return old(self, x, cache_k, cache_v, state, max_seq, *more)

    if where == "class":
        on.__class__ = type("Own", (type(on),), {name: own})
    else:
        setattr(on, name, types.MethodType(own, on))
    step(m, b)
    assert m._fused_decode and calls == [b]
