"""The edges of what the GPU calls take: nothing at all, more than a counter
or an address holds, infinities, numbers below the normal range, tensors that
stand for more than their values, streams and graphs."""
import math

import pytest
import torch

from lfmq.ops import ref

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
BF = torch.bfloat16


def ext():
    from lfmq.ops import hip_ext
    return hip_ext()


def packed(n, k, g, bits=4, seed=0):
    """(dequantized weights, [qweight, scales, qzeros] on the GPU)"""
    gen = torch.Generator().manual_seed(seed)
    c, s, z = ref.quant_groupwise(torch.randn(n, k, generator=gen), bits, g,
                                  False)
    s = s.to(BF)
    return (ref.dequant_groupwise(c, s.float(), z, g),
            [ref.pack_codes(c, bits).to(DEV), s.to(DEV),
             ref.pack_zeros(z, bits).to(DEV)])


# ------------------------------------------------------------- attention
@pytest.mark.parametrize("scale", [0.0, -0.125])
@pytest.mark.parametrize("s,pos0", [(70, 0), (130, 33)])
def test_prompt_attention_takes_any_scale(scale, s, pos0):
    """A scale of 0 weighs all visible keys alike, a negative one prefers
    the least scores.  Weights are rounded to 8 bits, as the result is."""
    torch.manual_seed(s)
    hq, hkv, d, T = 4, 2, 128, pos0 + s
    q = torch.randn(1, s, hq, d).to(BF)
    kc, vc = (torch.randn(1, hkv, T + 9, d).to(BF) for _ in range(2))
    got = ext().attn_prefill(q.view(1, s, -1).to(DEV), kc.to(DEV), vc.to(DEV),
                             hq, pos0, scale)
    k, v = (t[0, :, :T].double().repeat_interleave(hq // hkv, 0)
            for t in (kc, vc))
    sc = q[0].double().transpose(0, 1) @ k.transpose(1, 2) * scale
    seen = torch.arange(T) <= pos0 + torch.arange(s).unsqueeze(1)
    w = torch.softmax(sc.masked_fill(~seen, -math.inf), -1)
    want = (w @ v).transpose(0, 1).reshape(s, hq * d)
    got = got.double().cpu().view(s, hq * d)
    assert bool(got.isfinite().all())
    assert float((got - want).abs().max() / want.abs().max()) < 2 ** -7


@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("b,s", [(1, 7), (2, 3), (5, 9), (17, 2), (1, 130)])
def test_prompt_attention_of_narrow_heads(d, b, s):
    """Head sizes that the kernel does not take: products of the library,
    whose operands are laid out for it.  Weights and result are rounded to 8
    bits."""
    from lfmq.ops import functional as F
    torch.manual_seed(s)
    hq, hkv = 8, 2
    q = torch.randn(b, s, hq, d).to(BF).to(DEV).transpose(1, 2)
    kc, vc = (torch.randn(b, hkv, s + 16, d).to(BF) for _ in range(2))
    got = F.attn_prefill(q, kc.to(DEV)[:, :, :s], vc.to(DEV)[:, :, :s])
    want = ref.attn_prefill(q.cpu().float(), kc[:, :, :s].float(),
                            vc[:, :, :s].float())
    assert float((got.float().cpu() - want).abs().max()
                 / want.abs().max()) < 2 ** -6


@pytest.mark.parametrize("T", [1, 33, 70, 300])
@pytest.mark.parametrize("fused", [False, True])
def test_decode_attention_of_an_infinite_value(T, fused):
    """An infinite value in the last row of the cache is weighed once."""
    torch.manual_seed(T)
    hq, hkv, d = 4, 2, 128
    kc, vc = (torch.randn(1, hkv, T + 5, d).to(BF).to(DEV) for _ in range(2))
    qkv = torch.randn(1, (hq + 2 * hkv) * d).to(BF).to(DEV)
    if fused:
        qkv.view(1, hq + 2 * hkv, d)[:, hq + hkv:, 7] = math.inf
        o = ext().attn_decode_fused(qkv, kc, vc, T, d ** -0.5,
                                    torch.ones(d // 2, device=DEV), hq, None,
                                    None)
    else:
        vc[:, :, T - 1, 7] = math.inf
        o = ext().attn_decode(qkv[:, :hq * d].view(1, hq, 1, d), kc, vc, T,
                              d ** -0.5, None)
    o = o.float().view(hq, d)
    assert bool((o[:, 7] == math.inf).all())
    assert bool(o[:, :7].isfinite().all() and o[:, 8:].isfinite().all())


@pytest.mark.parametrize("s,pos0", [(1, 0), (70, 0), (130, 33)])
def test_prompt_attention_of_an_infinite_value(s, pos0):
    """The same for a prompt's last query."""
    from lfmq.ops import functional as F
    torch.manual_seed(s)
    hq, hkv, d, T = 4, 2, 128, pos0 + s
    q = torch.randn(1, s, hq, d).to(BF).to(DEV)
    kc, vc = (torch.randn(1, hkv, T + 9, d).to(BF).to(DEV) for _ in range(2))
    vc[:, :, T - 1, 7] = math.inf
    o = F.attn_prefill_fused(q, kc, vc, pos0, d ** -0.5)
    o = o.float().view(s, hq, d)[-1]
    assert bool((o[:, 7] == math.inf).all())
    assert bool(o[:, :7].isfinite().all() and o[:, 8:].isfinite().all())


def test_decode_attention_of_no_sequences():
    """Refused, as a launch of nothing is."""
    kc = torch.zeros(0, 8, 64, 128, dtype=BF, device=DEV)
    with pytest.raises(RuntimeError, match="invalid configuration"):
        ext().attn_decode(torch.zeros(0, 32, 1, 128, dtype=BF, device=DEV),
                          kc, kc, 33, 0.1, None)
    with pytest.raises(RuntimeError, match="invalid configuration"):
        ext().attn_decode_fused(
            torch.zeros(0, 48 * 128, dtype=BF, device=DEV), kc, kc, 33, 0.1,
            torch.ones(64, device=DEV), 32, None, None)


def test_decode_attention_of_no_keys():
    """Refused: there is nothing to take a mean of."""
    kc = torch.zeros(1, 8, 64, 128, dtype=BF, device=DEV)
    for T in (0, -3):
        with pytest.raises(RuntimeError):
            ext().attn_decode(torch.zeros(1, 32, 1, 128, dtype=BF, device=DEV),
                              kc, kc, T, 0.1, None)
        with pytest.raises(RuntimeError):
            ext().attn_decode_fused(
                torch.zeros(1, 48 * 128, dtype=BF, device=DEV), kc, kc, T, 0.1,
                torch.ones(64, device=DEV), 32, None, None)


@torch.no_grad()
def test_decode_steps_that_overlap_on_two_streams():
    """Two captured steps of one model and one shape, each with a cache of
    its own and many key ranges a head, replayed at the same time."""
    import lfmq
    from lfmq.models.llama import LlamaConfig
    T = 2500
    cfg = LlamaConfig(vocab_size=512, hidden_size=512, intermediate_size=512,
                      n_layers=4, n_heads=8, n_kv_heads=2, head_dim=64)
    m = lfmq.quantize(lfmq.build_model(cfg, seed=0), lfmq.QuantConfig(
        scheme="rtn", bits=4, group_size=64)).to(DEV)
    runs = []
    for seed in range(2):
        torch.manual_seed(seed)
        cache = m.make_cache(1, max_seq=T + 8)
        for t in (cache.k_all, cache.v_all):
            t.normal_()
        tok = torch.randint(0, 512, (1, 1), device=DEV)
        state = torch.tensor([T - 1, T, 0], dtype=torch.int32, device=DEV)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            want = m.forward_decode_step(tok, cache, state, T + 8).clone()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            got = m.forward_decode_step(tok, cache, state, T + 8)
        runs.append((graph, side, got, want, (cache, tok, state)))
    a, b = (r[4][0].tickets for r in runs)
    assert a.data_ptr() != b.data_ptr() and not a.any() and not b.any()
    for _ in range(30):
        for graph, side, *_ in runs:
            with torch.cuda.stream(side):
                for _ in range(4):
                    graph.replay()
        torch.cuda.synchronize()
        for *_, got, want, _ in runs:
            assert torch.equal(got, want)
            got.zero_()
        torch.cuda.synchronize()
    assert not a.any() and not b.any()


# ------------------------------------------------------- packed products
def test_packed_product_of_nothing():
    """No rows: no rows, however large the matrix; no columns: refused, as a
    launch of nothing is."""
    n, k, g = 6144, 4096, 128
    p = [torch.zeros(n, k // 8, dtype=torch.int32, device=DEV),
         torch.ones(n, k // g, dtype=BF, device=DEV),
         torch.zeros(n, k // g // 8, dtype=torch.int32, device=DEV)]
    x, r = (torch.zeros(0, c, dtype=BF, device=DEV) for c in (k, n))
    for resid, eps in ((None, -1.0), (r, -1.0), (None, 1e-5)):
        y = ext().dq_linear(x, *p, 4, g, None, resid, eps, 0)
        assert y.shape == (0, n)
    assert ext().dq_gemv_gateup(x, *p, 4, g, -1.0, 0).shape == (0, n // 2)
    empty = [t[:0] for t in p]
    for m in (1, 8, 64):
        with pytest.raises(RuntimeError, match="invalid configuration"):
            ext().dq_linear(torch.zeros(m, k, dtype=BF, device=DEV), *empty, 4,
                            g, None, None, -1.0, 0)


@pytest.mark.parametrize("m", [1, 2, 4])
@pytest.mark.parametrize("k,g", [(12416, 32), (28672, 64)])
def test_norm_and_gate_of_more_groups_than_kernels_hold(m, k, g):
    """388 and 448 groups a row.  The norm's result is rounded to 8 bits (each
    of k terms by 2^-9: of their sum's size, 2^-9 in the root mean square),
    then sums, gate and result."""
    torch.manual_seed(m)
    n = 64
    codes = torch.randint(0, 16, (n, k), dtype=torch.int32)
    zeros = torch.randint(0, 16, (n, k // g), dtype=torch.int32)
    s16 = (torch.rand(n, k // g) * 0.02 + 0.01).to(BF)
    p = (ref.pack_codes(codes, 4).to(DEV), s16.to(DEV),
         ref.pack_zeros(zeros, 4).to(DEV), 4, g)
    w = ref.dequant_groupwise(codes, s16.float(), zeros, g).double()
    x = torch.randn(m, k).to(BF)
    xn = x.double() * torch.rsqrt(x.double().square().mean(1, True) + 1e-5)
    for v, eps in ((x.double(), -1.0), (xn, 1e-5)):
        want = v @ w.t()
        a, u = want.chunk(2, 1)
        for y, z in ((ext().dq_linear(x.to(DEV), *p, None, None, eps, 0),
                      want),
                     (ext().dq_gemv_gateup(x.to(DEV), *p, eps, 0),
                      torch.nn.functional.silu(a) * u)):
            err = (y.double().cpu() - z).square().mean().sqrt()
            assert float(err / z.square().mean().sqrt()) < 2 ** -7
    for hint in (1, 2, 4, 5):                  # the GEMV by name: refused
        with pytest.raises(RuntimeError):
            ext().dq_linear(x.to(DEV), *p, None, None, -1.0, hint)


def test_packed_product_of_no_group():
    """Groups of nothing are refused by name (a division by their size would
    end the process)."""
    x = torch.zeros(2, 128, dtype=BF, device=DEV)
    p = [t[None] for t in packed(8, 128, 64)[1]]
    tiles = torch.zeros(1, 3, dtype=torch.int32, device=DEV)
    for call in (
            lambda: ext().dq_linear(x, *(t[0] for t in p), 4, 0, None, None,
                                    -1.0, 0),
            lambda: ext().dq_gemv_gateup(x, *(t[0] for t in p), 4, 0, -1.0, 0),
            lambda: ext().moe_linear(x, None, tiles, *p, 4, 0, False, 16),
            lambda: ext().moe_tile(64, 2, 128, 0, 128, 0),
            lambda: ext().moe_plan(x[:, :8].contiguous(), 2, 0)):
        with pytest.raises(RuntimeError, match="at least one"):
            call()


def test_packed_product_with_a_matrix_past_four_gibibytes():
    """More rows than the kernel that addresses any matrix takes otherwise."""
    n, k, g, m = 131072 + 64, 65536, 128, 99
    gen = torch.Generator(DEV).manual_seed(0)
    p = [torch.randint(-2 ** 31, 2 ** 31 - 1, (n, k // 8), dtype=torch.int32,
                       generator=gen, device=DEV),
         torch.rand(n, k // g, generator=gen, device=DEV).to(BF),
         torch.randint(-2 ** 31, 2 ** 31 - 1, (n, k // g // 8),
                       dtype=torch.int32, generator=gen, device=DEV)]
    x = torch.randn(m, k, generator=gen, device=DEV).to(BF)
    at = torch.tensor([0, 1, n // 2 - 1, n // 2, 65600, 131071, 131072, n - 1],
                      device=DEV)

    def columns(i):
        w = ref.dequant_weight(*(t[i].cpu() for t in p), 4, g, k)
        return x.double() @ w.double().t().to(DEV)

    want = columns(at)
    y = ext().dq_linear(x, *p, 4, g, None, None, -1.0, 0)
    assert float((y[:, at].double() - want).abs().max()
                 / want.abs().max()) < 2 ** -8
    at = at[:3]
    want = torch.nn.functional.silu(columns(at)) * columns(at + n // 2)
    y = ext().dq_gemv_gateup(x, *p, 4, g, -1.0, 0)
    assert float((y[:, at].double() - want).abs().max()
                 / want.abs().max()) < 2 ** -6


def test_gate_of_rows_past_four_gibibytes():
    m, n, k, g = 524288 + 70, 128, 4096, 128
    w, p = packed(n, k, g)
    x = torch.randn(m, k, device=DEV, dtype=BF)
    y = ext().dq_gemv_gateup(x, *p, 4, g, -1.0, 0)
    assert y.shape == (m, n // 2)
    at = torch.tensor([0, 63, 64, 262143, 262144, 524287, 524288, m - 1],
                      device=DEV)
    a, u = (x[at].double() @ w.double().t().to(DEV)).chunk(2, 1)
    want = torch.nn.functional.silu(a) * u
    assert float((y[at].double() - want).abs().max()
                 / want.abs().max()) < 2 ** -6


@pytest.mark.parametrize("hint", [0, 1, 2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("m", [1, 3])
def test_gemv_takes_any_number_of_columns_for_a_hint(hint, m):
    """Numbers that it has no body for are another one's, whole."""
    n, k, g = 130, 4096, 128
    w, p = packed(n, k, g)
    x = torch.randn(m, k).to(BF)
    want = x.double() @ w.double().t()
    a, u = want.chunk(2, 1)
    for y, z in ((ext().dq_linear(x.to(DEV), *p, 4, g, None, None, -1.0, hint),
                  want),
                 (ext().dq_gemv_gateup(x.to(DEV), *p, 4, g, -1.0, hint),
                  torch.nn.functional.silu(a) * u)):
        assert float((y.double().cpu() - z).abs().max()
                     / z.abs().max()) < 2 ** -7


@pytest.mark.parametrize("m", [1, 40])
def test_guard_names_the_gate(m, monkeypatch):
    """LFMQ_NANCHECK finds the operation that made a value infinite."""
    from lfmq.ops import functional as F
    monkeypatch.setattr(F, "_NANCHECK", True)
    _, p = packed(64, 128, 64)
    x = torch.ones(m, 128, device=DEV, dtype=BF)
    F.dq_gemv_gateup(x, *p, 4, 64)
    x[0, 3] = math.inf
    with pytest.raises(FloatingPointError, match="dq_gemv_gateup"):
        F.dq_gemv_gateup(x, *p, 4, 64)


# ------------------------------------------------------------------ gptq
@pytest.mark.parametrize("tiny", [1e-40, 3e-38, 2e-36, 1e-33])
def test_gptq_block_of_numbers_below_the_normal_range(tiny):
    """Groups whose scale has no finite reciprocal, and remainders that leave
    the normal range: still the tensor loop's quotients."""
    from lfmq import QuantConfig
    from lfmq.quant import gptq

    from gptq_util import gpu_block
    torch.manual_seed(5)
    n, k, g = 40, 128, 64
    w = torch.randn(n, k, device=DEV)
    w[0] = 0
    w[0, 3] = tiny
    w[1, :g] *= tiny
    w[2] *= tiny
    w[3] = 0
    w[4, g:] = tiny
    u = torch.randn(k, k, device=DEV).triu_() * 0.05
    u.diagonal().copy_(torch.rand(k, device=DEV) + 0.5)
    cfg = QuantConfig(scheme="gptq", bits=4, group_size=g)

    def solve(f):
        out = (torch.zeros(n, k, dtype=torch.int32, device=DEV),
               torch.zeros(n, k // g, device=DEV),
               torch.zeros(n, k // g, dtype=torch.int32, device=DEV))
        return (*out, f(w, u, *out, 0, cfg, g))

    for got, want in zip(solve(gpu_block), solve(gptq._block)):
        assert torch.equal(got, want)


# --------------------------------------------------------------- routing
@pytest.mark.parametrize("t", [1, 2, 63, 64])
def test_route_to_as_many_experts_as_lanes(t):
    """64 experts have 65 bounds, one more than the threads that route up to
    64 tokens."""
    torch.manual_seed(t)
    E, top = 64, 4
    logits = torch.stack([torch.randperm(E) for _ in range(t)]).to(BF)
    # memory of the size that the bounds will take is not clean
    torch.full((E + 1,), -7, dtype=torch.int32, device=DEV)
    src, w, offsets, active = ext().moe_route(logits.to(DEV), top)
    top_l, ids = torch.topk(logits.float(), top, -1)
    count = torch.bincount(ids.flatten(), minlength=E)
    want = torch.zeros(E + 1, dtype=torch.int64)
    want[1:] = count.cumsum(0)
    assert offsets.tolist() == want.tolist()
    used = count.nonzero().flatten().tolist()
    assert active.tolist() == used + [-1] * (E - len(used))
    for e in used:
        at = slice(int(want[e]), int(want[e + 1]))
        assert sorted(src[at].tolist()) == \
            (ids == e).any(1).nonzero().flatten().tolist()


# ---------------------------------------------------------- grouped calls
def grouped_case(t, E, n, k, g, seed):
    torch.manual_seed(seed)
    w, p = packed(E * n, k, g)
    ids = torch.randint(0, E, (t,)).sort().values
    off = torch.zeros(E + 1, dtype=torch.int32)
    off[1:] = torch.bincount(ids, minlength=E).cumsum(0)
    x = torch.randn(t, k).to(BF)
    rows = torch.stack([x[i].double() @ w.view(E, n, k)[ids[i]].double().t()
                        for i in range(t)])
    return (x.to(DEV), off.to(DEV), [a.view(E, n, -1) for a in p], rows)


@pytest.mark.parametrize("n", [1, 37, 66])
def test_grouped_linear_of_any_width(n):
    x, off, p, rows = grouped_case(23, 5, n, 128, 32, n)
    got = ext().grouped_dq_linear(x, off, *p, 4, 32).double().cpu()
    assert float((got - rows).abs().max() / rows.abs().max()) < 2 ** -8
    x, off, p, rows = grouped_case(130, 3, n, 128, 64, n)
    tiles = torch.tensor([[e, int(a), int(b - a)] for e, (a, b) in enumerate(
        zip(off[:-1], off[1:]))], dtype=torch.int32, device=DEV)
    got = ext().moe_linear(x, None, tiles, *p, 4, 64, False, 128)
    assert float((got.cpu() - rows).abs().max() / rows.abs().max()) < 1e-5


@pytest.mark.parametrize("n", [37, 64])
def test_grouped_linear_scatter(n):
    """Adds a slot's row, weighted, to its token's."""
    x, off, p, rows = grouped_case(24, 5, n, 128, 64, n)
    off[-1] = rest = max(int(off[-2]), 20)     # the slots after it: nobody's
    dst = torch.randperm(24).to(torch.int32) % 12
    wt = torch.rand(24)
    y = torch.randn(12, n)
    want = y.double().index_add(0, dst[:rest].long(),
                                (rows * wt.double()[:, None])[:rest])
    y = y.to(DEV)
    ext().grouped_dq_linear_scatter(x, off, dst.to(DEV), wt.to(DEV), y, *p, 4,
                                    64, None)
    assert float((y.double().cpu() - want).abs().max()
                 / want.abs().max()) < 1e-5


# --------------------------------------------------------------- mixtral
def quantized_moe(hidden, inter, group=64, seed=3, **kw):
    from lfmq import QuantConfig
    from lfmq.models.mixtral import MixtralConfig, MixtralMoE
    from lfmq.models.qlinear import QLinear
    torch.manual_seed(seed)
    cfg = MixtralConfig.tiny(hidden_size=hidden, intermediate_size=inter, **kw)
    moe = MixtralMoE(cfg, BF).to(DEV)
    qc = QuantConfig(scheme="rtn", bits=4, group_size=group)
    for e in moe.experts:
        e.w13, e.w2 = QLinear.from_rtn(e.w13, qc), QLinear.from_rtn(e.w2, qc)
    return moe


def by_loop(moe, x):
    x2 = x.reshape(-1, x.shape[-1])
    return moe._forward_loop(x2, *moe.route(x2)).reshape(x.shape)


def close(a, b):
    a, b = a.double(), b.double()
    return float((a - b).abs().max() / b.abs().max()) < 2 ** -6


@pytest.mark.parametrize("t", [2, 70])
def test_mixtral_made_in_inference_mode(t):
    with torch.inference_mode():
        moe = quantized_moe(256, 256)
        x = torch.randn(1, t, 256, device=DEV).to(BF)
        assert close(moe(x), by_loop(moe, x))
    with torch.no_grad():
        moe.consolidate()
        assert close(moe(x.clone()), by_loop(moe, x.clone()))


@pytest.mark.parametrize("t", [1, 4, 70])
def test_mixtral_uses_the_weights_that_are_there(t):
    """Written in place, written past the version counters, replaced (the
    new ones at the old addresses, too), loaded, moved."""
    moe, other = quantized_moe(256, 256), quantized_moe(256, 256, seed=9)
    x = torch.randn(1, t, 256, device=DEV).to(BF)
    with torch.no_grad():
        moe(x)
        before = moe.experts[0].w2.scales
        for e in moe.experts:
            e.w2.scales.mul_(2)
        assert close(moe(x), by_loop(moe, x))
        for e in moe.experts:
            e.w2.scales.data.mul_(2)
        assert close(moe(x), by_loop(moe, x))
        assert before.data_ptr() == moe.experts[0].w2.scales.data_ptr()
        for e in moe.experts:
            new = e.w2.scales.flip(0).cpu()
            e.w2.scales = None
            e.w2.scales = new.to(DEV)
        assert close(moe(x), by_loop(moe, x))
        moe.load_state_dict(other.state_dict())
        assert close(moe(x), by_loop(moe, x))
        assert close(moe(x), other(x))
        moe = moe.cpu().to(DEV)
        assert close(moe(x), by_loop(moe, x))


def test_mixtral_weights_replaced_and_then_captured():
    """A graph that has to lay the experts out itself does so whenever it
    runs, and leaves nothing of its memory to later calls."""
    moe, other = quantized_moe(256, 256), quantized_moe(256, 256, seed=9)
    x = torch.randn(1, 2, 256, device=DEV).to(BF)
    with torch.no_grad():
        moe(x)
        moe.load_state_dict(other.state_dict(), assign=True)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            got = moe(x)
        want = by_loop(other, x)
        assert close(moe(x), want)
        for _ in range(3):
            got.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert close(got, want)
            assert close(moe(x), want)


@pytest.mark.parametrize("t", [1, 5, 70])
def test_mixtral_experts_with_a_gather(t):
    """Act-order experts take their columns in an order of their own, in a
    captured step too."""
    moe = quantized_moe(256, 256)
    x = torch.randn(1, t, 256, device=DEV).to(BF)
    with torch.no_grad():
        plain = moe(x)
        for i, e in enumerate(moe.experts):
            for m in (e.w13, e.w2):
                m.register_buffer("perm", torch.randperm(256).to(DEV))
        want = by_loop(moe, x)
        assert not close(plain, want)
        assert close(moe(x), want)
        if t > 5:
            return
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            got = moe(x)
        for _ in range(3):
            got.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert close(got, want)
            assert close(moe(x), want)


def test_mixtral_prompt_calls_what_was_put_in_its_way():
    """Hooks on all modules, an expert's own forward or class, routing of a
    subclass."""
    from lfmq.models import mixtral
    moe = quantized_moe(256, 256)
    x = torch.randn(1, 70, 256, device=DEV).to(BF)
    seen = []
    with torch.no_grad():
        want = moe(x)
        h = torch.nn.modules.module.register_module_forward_hook(
            lambda m, i, o: seen.append(m))
        try:
            got = moe(x)
        finally:
            h.remove()
        assert close(got, want)
        assert {id(e) for e in moe.experts} <= {id(m) for m in seen}

        e = moe.experts[0]
        e.forward = lambda v: torch.zeros_like(v)
        assert close(moe(x), by_loop(moe, x)) and not close(moe(x), want)
        del e.forward
        e.w2.forward = lambda v: torch.zeros(v.shape[0], 256, device=DEV,
                                             dtype=BF)
        assert close(moe(x), by_loop(moe, x)) and not close(moe(x), want)
        del e.w2.forward
        assert close(moe(x), want)

        class Twice(mixtral.MixtralExpert):
            def forward(self, v):
                return 2 * super().forward(v)

        e.__class__ = Twice
        assert close(moe(x), by_loop(moe, x)) and not close(moe(x), want)
        e.__class__ = mixtral.MixtralExpert

        class Last(mixtral.MixtralMoE):
            def route(self, x2):
                w, ids = super().route(x2)
                return w, torch.zeros_like(ids) + torch.arange(
                    2, device=DEV)

        moe.__class__ = Last
        assert close(moe(x), by_loop(moe, x)) and not close(moe(x), want)


def test_mixtral_prompt_past_four_gibibytes():
    """75000 tokens' activations in the experts are more than 4 GiB."""
    moe = quantized_moe(64, 14336)
    x = torch.randn(1, 75000, 64, device=DEV).to(BF)
    at = torch.tensor([0, 1, 37499, 37500, 65535, 65536, 74999], device=DEV)
    with torch.no_grad():
        y = moe(x)
        assert y.shape == x.shape
        assert close(y[:, at], by_loop(moe, x[:, at]))


def test_mixtral_prompt_of_more_tokens_than_a_grid_has_rows():
    moe = quantized_moe(64, 64)
    x = torch.randn(1, 70000, 64, device=DEV).to(BF)
    at = torch.tensor([0, 1, 65534, 65535, 65536, 69999], device=DEV)
    with torch.no_grad():
        assert close(moe(x)[:, at], by_loop(moe, x[:, at]))


# ---------------------------------------------------------------- linear
def test_linear_of_more_than_values():
    """Forward-mode tangents, vmap, tracing, a weight of another class, modes
    that watch calls: what the library's product gives."""
    import torch.autograd.forward_ad as fwAD
    from lfmq.models.linear import Linear
    torch.manual_seed(2)
    m = Linear(256, 64, BF).to(DEV).requires_grad_(False)
    x, dx = (torch.randn(3, 256, device=DEV).to(BF) for _ in range(2))
    want = torch.nn.functional.linear
    with fwAD.dual_level():
        t = fwAD.unpack_dual(m(fwAD.make_dual(x, dx))).tangent
        assert torch.equal(t, want(dx, m.weight))
        m2 = Linear(256, 64, BF).to(DEV).requires_grad_(False)
        del m2.weight
        m2.weight = fwAD.make_dual(m.weight.detach(), m.weight.detach())
        t = fwAD.unpack_dual(m2(x)).tangent
        assert torch.equal(t, want(x, m.weight))
    traced = torch.jit.trace(m, (x,), check_trace=False)
    assert torch.equal(traced(dx), want(dx, m.weight))

    class Scaled(torch.Tensor):
        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            r = super().__torch_function__(func, types, args, kwargs or {})
            return r * 2 if func is want else r

    m.weight = torch.nn.Parameter(m.weight.detach().as_subclass(Scaled),
                                  requires_grad=False)
    w = m.weight.detach().as_subclass(torch.Tensor)
    assert torch.equal(m(x).as_subclass(torch.Tensor), 2 * want(x, w))
    m.weight = torch.nn.Parameter(w, requires_grad=False)

    from torch.utils.flop_counter import FlopCounterMode
    with FlopCounterMode(display=False) as count:
        m(x)
    assert count.get_total_flops() == 2 * 3 * 256 * 64


def test_linear_under_transforms():
    from lfmq.models.linear import Linear
    torch.manual_seed(2)
    m = Linear(256, 64, BF).to(DEV).requires_grad_(False)
    x = torch.randn(3, 256, device=DEV).to(BF)
    want = torch.nn.functional.linear(x, m.weight).float()
    got = torch.func.vmap(m)(x)
    assert float((got.float() - want).abs().max()) < 2 ** -6
    _, t = torch.func.jvp(m, (x,), (x,))
    assert float((t.float() - want).abs().max()) < 2 ** -6
    with torch.device(DEV):                    # still the kernel
        from lfmq.ops import seq_ext
        assert torch.equal(m(x), seq_ext().linear_rows(x, m.weight, False))


def test_dense_layer_calls_an_instance_s_own_forward():
    from lfmq.models.mixers import DenseMLP
    torch.manual_seed(2)
    mlp = DenseMLP(256, 128, BF).to(DEV).requires_grad_(False)
    x = torch.randn(3, 256, device=DEV).to(BF)
    want = mlp(x)
    mlp.gate_up_proj.forward = lambda v: torch.zeros(3, 256, device=DEV,
                                                     dtype=BF)
    assert float(mlp(x).abs().max()) == 0
    del mlp.gate_up_proj.forward
    assert torch.equal(mlp(x), want)


# -------------------------------------------------------------- seqcache
def busy(n=20):
    """Work that is queued for a while."""
    x = torch.randn(4096, 4096, device=DEV)
    for _ in range(n):
        x = (x @ x).clamp_(-1, 1)


def tiny_packed():
    import lfmq
    from lfmq.models.rapivik import RapivikConfig
    return lfmq.build_model(RapivikConfig.tiny(n_layers=2), seed=1).to(DEV)


@torch.no_grad()
def test_batch_is_kept_for_a_step_on_another_stream():
    """A batch is dropped while the step that reads its numbers is queued on
    another stream; batches of the same sizes are made meanwhile."""
    m = tiny_packed()
    tok = torch.randint(0, 512, (80,), device=DEV)

    def step(cache, slots, counts):
        return m.forward_tokens(tok, cache.batch(slots, counts), cache)

    want = step(m.make_cache(4, 96), [1, 3], [70, 10])
    cache, side = m.make_cache(4, 96), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        busy(40)
    batch = cache.batch([1, 3], [70, 10])
    with torch.cuda.stream(side):
        got = m.forward_tokens(tok, batch, cache)
    del batch
    other = m.make_cache(4, 96)
    for _ in range(8):
        other.batch([2, 0], [10, 70])
    torch.cuda.synchronize()
    assert torch.equal(got, want)


@torch.no_grad()
def test_step_waits_for_numbers_that_another_stream_asked_for():
    """The layouts that a batch makes when they are asked for are queued on
    that step's stream."""
    m = tiny_packed()
    tok = torch.randint(0, 512, (80,), device=DEV)
    cache, side = m.make_cache(2, 96), torch.cuda.Stream()
    want = m.forward_tokens(tok, cache.batch([0, 1], [70, 10]), cache)
    cache, again = m.make_cache(2, 96), m.make_cache(2, 96)
    batch = cache.batch([0, 1], [70, 10])
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        busy()
        m.forward_tokens(tok, batch, cache)
    assert torch.equal(m.forward_tokens(tok, batch, again), want)
    assert {s for _, s in batch._queued} == {torch.cuda.current_stream(), side}


@torch.no_grad()
def test_step_of_a_batch_made_before_its_capture():
    m = tiny_packed()
    tok = torch.randint(0, 512, (80,), device=DEV)
    cache = m.make_cache(2, 96)
    fresh = cache.snapshot()
    batch = cache.batch([0, 1], [70, 10])
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        want = m.forward_tokens(tok, batch, cache)
    torch.cuda.synchronize()
    cache.restore(fresh)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = m.forward_tokens(tok, batch, cache)
    for _ in range(3):
        cache.restore(fresh)
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)


@pytest.mark.parametrize("m", [17, 49, 97, 100, 128, 129])
def test_packed_product_of_no_columns(m):
    """Refused with any number of rows, as a launch of nothing is."""
    k, g = 4096, 128
    p = [torch.zeros(0, k // 8, dtype=torch.int32, device=DEV),
         torch.ones(0, k // g, dtype=BF, device=DEV),
         torch.zeros(0, k // g // 8, dtype=torch.int32, device=DEV)]
    x = torch.zeros(m, k, dtype=BF, device=DEV)
    for call in (lambda: ext().dq_linear(x, *p, 4, g, None, None, -1.0, 0),
                 lambda: ext().dq_gemv_gateup(x, *p, 4, g, -1.0, 0)):
        with pytest.raises(RuntimeError, match="invalid configuration"):
            call()


@pytest.mark.parametrize("glu", [True, False])
@pytest.mark.parametrize("bm", [16, 128])
def test_grouped_product_of_no_experts(bm, glu):
    """Without experts there are no tiles, and nothing is computed."""
    k, n, g = 1024, 512, 128
    p = [torch.zeros(0, n, k // 8, dtype=torch.int32, device=DEV),
         torch.ones(0, n, k // g, dtype=BF, device=DEV),
         torch.zeros(0, n, k // g // 8, dtype=torch.int32, device=DEV)]
    x = torch.zeros(5, k, dtype=BF, device=DEV)
    tiles = torch.zeros(0, 3, dtype=torch.int32, device=DEV)
    y = ext().moe_linear(x, None, tiles, *p, 4, g, glu, bm)
    assert y.shape == (5, n // 2 if glu else n)


@pytest.mark.parametrize("glu", [True, False])
@pytest.mark.parametrize("bm", [16, 128])
def test_grouped_product_of_no_groups(bm, glu):
    """Rows of nothing have no chunk of k to begin with: refused."""
    n, g = 512, 128
    p = [torch.zeros(2, n, 0, dtype=torch.int32, device=DEV),
         torch.ones(2, n, 0, dtype=BF, device=DEV),
         torch.zeros(2, n, 0, dtype=torch.int32, device=DEV)]
    x = torch.zeros(5, 0, dtype=BF, device=DEV)
    tiles = torch.tensor([[0, 0, 5]], dtype=torch.int32, device=DEV)
    with pytest.raises(RuntimeError, match="invalid argument"):
        ext().moe_linear(x, None, tiles, *p, 4, g, glu, bm)
