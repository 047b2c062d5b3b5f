"""Packed products of a decode step against 64 bits: one row (dq_row) and up
to sixteen (dq_wide), where their waves, groups and tiles end.

Products of bf16 and codes are exact and summed in fp32, so a result is off
by its own rounding, 2^-9 of a value, and by the sums' error where it is small
beside its row."""
import re

import pytest
import torch
from torch.profiler import ProfilerActivity, profile

import lfmq
from lfmq.models.llama import LlamaConfig
from lfmq.ops import functional as F
from lfmq.ops import hip_ext as ext
from lfmq.ops import ref

pytestmark = pytest.mark.gpu
DEV, BF = "cuda", torch.bfloat16


def matrix(bits, n, k, g, experts=()):
    """Packed weights on the device, and what they stand for."""
    codes = torch.randint(0, 1 << bits, (*experts, n, k), dtype=torch.int32)
    zeros = torch.randint(0, 1 << bits, (*experts, n, k // g),
                          dtype=torch.int32)
    s = (torch.rand(*experts, n, k // g) * 0.02 + 0.01).to(BF)
    flat = [t.flatten(0, -2) for t in (codes, zeros, s)]
    w = ((flat[0].to(DEV).view(-1, k // g, g) - flat[1].to(DEV).unsqueeze(-1))
         .double() * flat[2].to(DEV).double().unsqueeze(-1)).flatten(1)
    packed = [ref.pack_codes(flat[0], bits), flat[2],
              ref.pack_zeros(flat[1], bits)]
    return [t.view(*experts, n, -1).to(DEV).contiguous() for t in packed], \
        w.view(*experts, n, k)


def close(y, want, rel=5e-3):
    err = (y.double() - want).abs()
    floor = 1e-3 * want.abs().amax(-1, keepdim=True) + 1e-30
    assert y.shape == want.shape
    assert float((err / (want.abs() + floor)).max()) < rel


def launched(call):
    """Names of the kernels that it launches."""
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        call()
        torch.cuda.synchronize()
    names = (re.search(r"(\w+)[<(]", e.key.replace("(anonymous namespace)", ""))
             for e in p.key_averages())
    return {n.group(1) for n in names if n}


def normed(x, eps):
    x = x.double()
    return x * torch.rsqrt((x ** 2).mean(-1, keepdim=True) + eps)


def gated(h):
    a, u = h.chunk(2, -1)
    return torch.nn.functional.silu(a) * u


def check(bits, m, n, k, g):
    p, w = matrix(bits, n, k, g)
    x = torch.randn(m, k, device=DEV).to(BF)
    if m > 1:
        x[0] = 0
    bias = torch.randn(n, device=DEV).to(BF)
    resid = torch.randn(m, n, device=DEV).to(BF)
    plain, rms = x.double() @ w.t(), normed(x, 1e-5) @ w.t()
    close(ext().dq_linear(x, *p, bits, g, bias, None, 1e-5, 0),
          rms + bias.double())
    close(ext().dq_linear(x, *p, bits, g, None, resid, -1.0, 0),
          plain + resid.double())
    if n % 2 == 0:
        # the gate turns its sum's error into at most its slope, 1.1, of it
        close(ext().dq_gemv_gateup(x, *p, bits, g, 1e-5, 0), gated(rms), 1e-2)
        close(ext().dq_gemv_gateup(x, *p, bits, g, -1.0, 0), gated(plain),
              1e-2)


# k in two to five parts, also of unequal length; columns that end inside a tile, and
# workgroups with a tile less than others; without a residual, and with a bias.
@pytest.mark.parametrize("bits,m,n,k,g", [
    (4, 3, 6148, 8192, 128), (4, 16, 4099, 8704, 64), (4, 8, 4096, 14336, 128),
    (8, 5, 5001, 12288, 128), (8, 16, 2050, 20352, 64), (4, 9, 4200, 17408, 128),
    (8, 4, 6160, 8704, 64), (4, 12, 4112, 11904, 64)])
def test_k_in_parts_that_one_launch_adds_up(bits, m, n, k, g):
    torch.manual_seed(m + n)
    p, w = matrix(bits, n, k, g)
    tickets = torch.zeros(256, dtype=torch.int32, device=DEV)
    bias = torch.randn(n, device=DEV).to(BF)
    resid = torch.randn(m, n, device=DEV).to(BF)
    x = torch.randn(m, k, device=DEV).to(BF)
    x[0] = 0
    for _ in range(3):                       # the counters are as they were
        y = ext().dq_linear_parts(x, *p, bits, g, bias, resid, tickets)
        close(y, x.double() @ w.t() + bias.double() + resid.double())
        y = ext().dq_linear_parts(x, *p, bits, g, None, None, tickets)
        close(y, x.double() @ w.t())
        assert not bool(tickets.any())
        x = torch.randn(m, k, device=DEV).to(BF)
    assert ext().dq_linear_parts(x, *p, bits, g, None, None, tickets[:8]) is None


@pytest.mark.parametrize("n,k,rounds", [(8176, 8960, 1), (10912, 9984, 2)])
def test_k_in_parts_is_one_round_of_workgroups(n, k, rounds):
    """Three parts of 511 column tiles, six of which a workgroup would leave 258 of
    them (seven do not), and of 682, which eight a workgroup would."""
    torch.manual_seed(n)
    p, w = matrix(4, n, k, 128)
    x = torch.randn(5, k, device=DEV).to(BF)
    tickets = torch.zeros(256, dtype=torch.int32, device=DEV)
    y = ext().dq_linear_parts(x, *p, 4, 128, None, None, tickets)
    assert (y is None) == (rounds > 1)
    if y is not None:
        close(y, x.double() @ w.t())


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("n,k,g", [
    (8198, 2048, 128), (8193, 2048, 64), (7946, 2112, 32), (4097, 4096, 128),
    (28674, 4096, 128), (4106, 5120, 128), (2731, 6400, 64), (1542, 8192, 128),
    (1030, 14336, 128), (774, 16384, 32)])
def test_one_row(bits, n, k, g):
    """One to eight waves along k, the last one short; rows that end inside a
    group of four, gates inside a pair; several groups a wave."""
    torch.manual_seed(n)
    check(bits, 1, n, k, g)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("n,k,g", [
    (2050, 2048, 32), (1366, 3072, 128), (1027, 4096, 64), (514, 8192, 128),
    (259, 16384, 64)])
def test_one_row_of_few_weights(bits, n, k, g):
    """The least that is not the GEMV's: fewer groups than waves, waves without
    any, a short last wave."""
    torch.manual_seed(n + bits)
    check(bits, 1, n, k, g)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m,n,k,g", [
    (2, 2049, 2048, 128), (3, 3074, 2304, 64), (4, 4098, 4096, 128),
    (5, 2050, 2048, 64), (8, 28674, 4096, 128), (9, 8198, 4352, 128),
    (12, 33000, 2048, 128), (16, 5126, 8192, 64), (16, 4110, 4096, 64),
    (6, 8210, 6144, 64)])
def test_few_rows_many_columns(bits, m, n, k, g):
    """Eight and sixteen waves along k, one and more steps of it; tiles that
    end inside a workgroup's last one; 4, 8 and 16 rows of sums."""
    torch.manual_seed(n)
    check(bits, m, n, k, g)


@pytest.mark.parametrize("bits,n,k,g", [(4, 2062, 2048, 128),
                                        (8, 2048, 4352, 64),
                                        (4, 2048, 6144, 64),
                                        (4, 4100, 4096, 128)])
@pytest.mark.parametrize("counts", [(1, 0, 2), (16, 3, 0), (0, 21, 9)])
def test_rows_by_expert(bits, n, k, g, counts):
    """One to sixteen rows a tile, experts without any, tiles that are none."""
    torch.manual_seed(n)
    p, w = matrix(bits, n, k, g, (len(counts),))
    ids = torch.tensor([e for e, c in enumerate(counts) for _ in range(c)],
                       device=DEV)
    src = torch.randperm(len(ids)).to(DEV)
    x = torch.randn(len(ids), k, device=DEV).to(BF)
    tiles, at = [], 0
    for e, c in enumerate(counts):
        tiles += [(e, at + i, min(16, c - i)) for i in range(0, c, 16)]
        at += c
    tiles.insert(1, (-1, 0, 0))
    tiles = torch.tensor(tiles + [(-1, 0, 0)], dtype=torch.int32, device=DEV)
    want = (x.double()[src].unsqueeze(1) @ w[ids].transpose(1, 2)).squeeze(1)
    s32 = src.to(torch.int32)
    close(ext().moe_linear(x, s32, tiles, *p, bits, g, True, 16), gated(want),
          1e-2)
    close(ext().moe_linear(x[src], None, tiles, *p, bits, g, False, 16), want)


# just below and above the number of groups whose scales dq_wide's LDS holds
@pytest.mark.parametrize("bits,k", [(4, 232960), (4, 240000), (4, 262144),
                                    (8, 194560), (8, 196608)])
@pytest.mark.parametrize("m", [2, 16])
def test_few_rows_of_more_groups_than_a_tile_holds(bits, k, m):
    n, g, gen = 8192, 64, torch.Generator(DEV).manual_seed(k)
    i32 = dict(dtype=torch.int32, device=DEV, generator=gen)
    q = torch.randint(-2 ** 31, 2 ** 31, (n, k * bits // 32), **i32)
    z = torch.randint(-2 ** 31, 2 ** 31, (n, -(-k // g * bits // 32)), **i32)
    s = (torch.rand(n, k // g, device=DEV, generator=gen) * 0.02 + 0.01).to(BF)
    x = torch.randn(m, k, device=DEV, generator=gen).to(BF)
    y = ext().dq_linear(x, q, s, z, bits, g, None, None, -1.0, 0)
    # the columns in parts, some of each
    for c in range(0, n, 1024):
        at = slice(c, c + 40)
        w = ref.dequant_groupwise(
            ref.unpack_codes(q[at], bits, k), s[at].float(),
            ref.unpack_zeros(z[at], bits, k // g), g).double()
        close(y[:, at], x.double() @ w.t())


@pytest.mark.parametrize("m", [1, 8])
def test_scales_that_start_on_an_odd_number(m):
    """dq_row and dq_wide read them in pairs: such a matrix is another kernel's."""
    bits, n, k, g = 4, 8194, 2048, 128
    (q, s, z), w = matrix(bits, n, k, g)
    odd = torch.zeros(s.numel() + 1, dtype=BF, device=DEV)[1:].view_as(s)
    odd.copy_(s)
    assert odd.data_ptr() % 4 == 2
    x = torch.randn(m, k, device=DEV).to(BF)
    want = x.double() @ w.t()
    close(ext().dq_linear(x, q, odd, z, bits, g, None, None, -1.0, 0), want)
    close(ext().dq_gemv_gateup(x, q, odd, z, bits, g, -1.0, 0), gated(want),
          1e-2)
    tiles = torch.tensor([[0, 0, m]], dtype=torch.int32, device=DEV)
    close(ext().moe_linear(x, None, tiles, q.unsqueeze(0), odd.unsqueeze(0),
                           z.unsqueeze(0), bits, g, False, 16), want)


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_one_row_of_values_that_are_not_finite(value):
    """Every column takes part in every value: no result is finite."""
    p, _ = matrix(4, 8198, 2048, 128)
    x = torch.randn(1, 2048, device=DEV).to(BF)
    x[0, 1000] = value
    for eps in (-1.0, 1e-5):
        y = ext().dq_linear(x, *p, 4, 128, None, None, eps, 0)
        assert not bool(torch.isfinite(y).any())


# matrices past 4 GiB (k 16384, 8 bits: 262144 rows are), whose last rows a
# 32-bit offset would not reach
@pytest.mark.parametrize("m", [1, 4])
def test_few_rows_past_4_gib(m):
    bits, n, k, g = 8, 263168, 16384, 128
    q = torch.zeros(n, k // 4, dtype=torch.int32, device=DEV)
    s = torch.zeros(n, k // g, dtype=BF, device=DEV)
    z = torch.zeros(n, k // g // 4, dtype=torch.int32, device=DEV)
    part, w = matrix(bits, 1024, k, g)
    for t, u in zip((q, s, z), part):
        t[-1024:] = u
    x = torch.randn(m, k, device=DEV).to(BF)
    y = ext().dq_linear(x, q, s, z, bits, g, None, None, -1.0, 0)
    close(y[:, -1024:], x.double() @ w.t())
    assert not bool(y[:, :-1024].any())


@pytest.mark.parametrize("bits,m,n,k,g", [
    (4, 2, 8191, 2048, 128), (4, 16, 8194, 2048, 128), (4, 9, 7290, 2304, 128),
    (4, 5, 4110, 4096, 128), (8, 3, 4095, 2048, 128), (8, 12, 4098, 2048, 64),
    (8, 16, 3650, 2304, 128), (8, 7, 2050, 4096, 64), (8, 4, 3300, 2688, 64)])
def test_few_rows_by_whole_lines(bits, m, n, k, g):
    """From 8 MiB of weights on, and just below: both pieces of a line, columns
    that end inside an eight, waves with a part of their chunks."""
    torch.manual_seed(n)
    check(bits, m, n, k, g)


@pytest.mark.parametrize("m,n,k,g,bits", [
    (17, 2048, 4096, 64, 4), (48, 4096, 14336, 128, 4), (33, 4104, 2048, 64, 8),
    (20, 8192, 4096, 128, 8), (48, 16384, 2048, 128, 4), (48, 512, 512, 64, 4),
    (31, 1028, 1024, 128, 8), (47, 1030, 2048, 64, 4), (18, 24576, 2048, 64, 4)])
def test_rows_times_their_factors(m, n, k, g, bits):
    """A norm as factors of x's rows, and the result's own factors from the sum
    of parts (rows of up to 2048, 4096, 8192 and 16384 columns, few and many
    parts), from whole products and from rows that no workgroup holds."""
    p, w = matrix(bits, n, k, g)
    x = torch.randn(m, k, device=DEV).to(BF)
    x[0] = 0
    bias = torch.randn(n, device=DEV).to(BF)
    resid = torch.randn(m, n, device=DEV).to(BF)
    scale = ext().row_scale(x, 1e-5)
    rms = normed(x, 1e-5) @ w.t()
    # a sum of k squares in fp32 and a reciprocal root
    own = torch.rsqrt((x.double() ** 2).mean(-1) + 1e-5)
    assert float((scale.double() / own - 1).abs().max()) < 1e-5
    y, = ext().dq_linear_scaled(x, scale, *p, bits, g, bias, None, -1.0)
    close(y, rms + bias.double())
    for s, want in ((None, x.double() @ w.t()), (scale, rms)):
        y, out = ext().dq_linear_scaled(x, s, *p, bits, g, None, resid, 1e-6)
        close(y, want + resid.double())
        own = torch.rsqrt((y.double() ** 2).mean(-1) + 1e-6)
        assert float((out.double() / own - 1).abs().max()) < 1e-5
    if n % 2 == 0:
        close(ext().dq_gateup_scaled(x, scale, *p, bits, g), gated(rms), 1e-2)


@pytest.mark.parametrize("m,n,k,g,bits,parts", [
    (17, 2048, 2048, 64, 4, False), (32, 2048, 4096, 128, 4, False),
    (48, 4096, 14336, 128, 4, True), (33, 4104, 2048, 64, 8, None),
    (47, 1030, 2048, 64, 4, None), (18, 24576, 2048, 64, 4, None)])
def test_factors_without_a_launch_of_their_own(m, n, k, g, bits, parts):
    """Where the product's parts are summed the same factors, elsewhere none."""
    p, _ = matrix(bits, n, k, g)
    x = torch.randn(m, k, device=DEV).to(BF)
    resid = torch.randn(m, n, device=DEV).to(BF)
    y, want = ext().dq_linear_scaled(x, None, *p, bits, g, None, resid, 1e-6)
    z, *own = ext().dq_linear_scaled(x, None, *p, bits, g, None, resid, 1e-6,
                                     False)
    assert torch.equal(y, z) and all(torch.equal(t, want) for t in own)
    assert parts is None or bool(own) == parts


@pytest.mark.parametrize("m,n,k,g,bits", [
    (77, 2048, 8192, 64, 8), (40, 4096, 14336, 128, 4), (64, 4104, 4096, 64, 4),
    (50, 8192, 4096, 128, 8), (33, 16384, 2048, 128, 4), (100, 1032, 4096, 128, 4),
    (20, 2044, 8192, 64, 4), (60, 2046, 2048, 64, 8), (3, 2048, 2048, 128, 4),
    (300, 2048, 2048, 64, 4)])
@pytest.mark.parametrize("shift", [0, 2])
def test_norm_after_a_product(m, n, k, g, bits, shift):
    """The sum of parts with residual and norm (rows of up to 2048, 4096, 8192 and
    16384 columns), a product in one piece, and rows that no workgroup holds or
    that lie off 8 bytes: as the product and the norm apart."""
    torch.manual_seed(n + m)
    p, w = matrix(bits, n, k, g)
    x = torch.randn(m, k, device=DEV).to(BF)
    bias = torch.randn(n, device=DEV).to(BF)
    to = torch.randn(m * n + shift, device=DEV).to(BF)[shift:].view(m, n)
    weight = torch.randn(n, device=DEV).to(BF)
    h, s = ext().dq_linear_norm(x, *p, bits, g, bias, to, weight, 1e-5)
    y = ext().dq_linear(x, *p, bits, g, bias, None, -1.0, 0)
    close(y, x.double() @ w.t() + bias.double())
    assert torch.equal(s, (y.float() + to.float()).to(BF))
    want = normed(y.double() + to.double(), 1e-5) * weight.double()
    # its own rounding, and a sum of n squares in fp32
    assert float(((h.double() - want).abs() / (want.abs() + 1e-6)).max()) < 4.1e-3


def with_its_ways(bits, m, n, k, g):
    """A product with a bias; with the gate; of up to 48 rows, with a residual and
    with factors of rows.  Returns the first one's kernels."""
    torch.manual_seed(n + m)
    p, w = matrix(bits, n, k, g)
    x = torch.randn(m, k, device=DEV).to(BF)
    x[0] = 0
    bias = torch.randn(n, device=DEV).to(BF)
    plain = x.double() @ w.t()
    names = launched(lambda: close(
        ext().dq_linear(x, *p, bits, g, bias, None, -1.0, 0), plain + bias.double()))
    close(ext().dq_gemv_gateup(x, *p, bits, g, -1.0, 0), gated(plain), 1e-2)
    if m <= 48:
        resid = torch.randn(m, n, device=DEV).to(BF)
        scale = torch.rand(m, device=DEV) + 0.5
        close(ext().dq_linear(x, *p, bits, g, bias, resid, -1.0, 0),
              plain + bias.double() + resid.double())
        want = plain * scale.double().unsqueeze(1)
        y, _ = ext().dq_linear_scaled(x, scale, *p, bits, g, None, resid, 1e-5)
        close(y, want + resid.double())
        close(ext().dq_gateup_scaled(x, scale, *p, bits, g), gated(want), 1e-2)
    return names


@pytest.mark.parametrize("m,n,k,g", [
    (40, 10240, 256, 128), (48, 8200, 2112, 64), (33, 32008, 192, 64),
    (49, 3072, 1024, 64), (64, 2056, 2048, 128), (77, 16384, 2048, 64),
    (81, 1544, 2688, 192), (96, 2048, 2048, 64), (97, 2048, 3072, 64),
    (113, 2504, 2560, 256), (128, 8192, 1024, 128), (49, 2048, 8192, 64),
    (96, 4104, 4224, 128), (112, 1536, 4096, 64), (65, 1032, 14336, 64),
    (80, 10240, 4096, 128)])
def test_eight_waves_along_k(m, n, k, g):
    """8 bits, some tens of rows: 2 to 6 sixteens of rows and two tiles of them,
    2 and 4 waves side by side, parts of k and none, groups that the waves do
    not share evenly, columns that end inside a wave's; bias, residual, gate
    and factors of rows."""
    assert "dq_mid_kernel" in with_its_ways(8, m, n, k, g)


@pytest.mark.parametrize("m,n,k,g", [
    (17, 28680, 1024, 128), (48, 8200, 2112, 64), (33, 32008, 832, 64),
    (25, 1024, 1280, 64), (33, 2008, 896, 128), (50, 4096, 256, 128), (40, 28672, 4096, 128),
    (48, 6144, 4096, 128), (64, 2056, 2048, 128), (77, 16384, 2048, 64),
    (81, 1544, 2688, 192), (90, 6136, 896, 128), (97, 2048, 3072, 64),
    (100, 512, 4992, 128), (113, 2504, 2560, 256), (128, 8192, 1024, 128),
    (65, 1032, 14336, 64), (80, 10240, 4096, 128)])
def test_eight_waves_along_k_of_four_bits(m, n, k, g):
    """The same of 4 bits, whose sums of x waves side by side share and add two
    steps later: one and two steps a group, one turn and many, last turns with
    fewer groups than waves, more row tiles than waves side by side and fewer."""
    assert "dq_mid_kernel" in with_its_ways(4, m, n, k, g)


@pytest.mark.parametrize("bits,m,n,k,g", [
    (8, 17, 5120, 256, 128), (8, 32, 6136, 1024, 64), (8, 32, 6144, 1024, 64),
    (8, 25, 8192, 768, 128), (8, 25, 8200, 768, 128), (8, 17, 8192, 2048, 64),
    (8, 17, 8200, 2048, 64), (8, 64, 28664, 1024, 64), (8, 64, 28672, 1024, 64),
    (8, 50, 28672, 2112, 64), (8, 96, 24576, 2112, 64), (8, 65, 24584, 2112, 64),
    (8, 32, 32768, 512, 64), (8, 32, 32776, 512, 64), (8, 32, 32776, 512, 128),
    (8, 48, 32776, 1216, 64), (8, 33, 32776, 1280, 64), (8, 65, 32776, 1472, 64),
    (8, 65, 32776, 1536, 64), (4, 25, 1024, 768, 64), (4, 90, 8200, 896, 128),
    (4, 200, 4104, 4096, 128), (8, 700, 4100, 6912, 64)])
def test_some_tens_of_rows_by_any_kernel(bits, m, n, k, g):
    """Sizes about the edges of several kernels' ranges, which one of them has at a
    time: all that goes with a product is taken there by whichever it is."""
    with_its_ways(bits, m, n, k, g)


@pytest.mark.parametrize("bits,m,n,k,g", [
    (4, 129, 2048, 2048, 64), (8, 161, 16384, 2048, 64), (4, 200, 4104, 3072, 128),
    (8, 300, 2048, 2048, 128), (4, 511, 1032, 1920, 64), (8, 512, 2056, 2688, 192),
    (4, 385, 520, 4992, 128), (8, 256, 4096, 4096, 64), (4, 512, 3072, 768, 128),
    (8, 768, 2048, 2048, 64), (4, 673, 2048, 2048, 128)])
def test_eight_waves_of_many_rows(bits, m, n, k, g):
    """The same of 129 to 768 rows: up to eight row tiles, last ones of one row."""
    torch.manual_seed(n + m)
    p, w = matrix(bits, n, k, g)
    x = torch.randn(m, k, device=DEV).to(BF)
    bias = torch.randn(n, device=DEV).to(BF)
    plain = x.double() @ w.t()
    assert "dq_mid_kernel" in launched(lambda: close(
        ext().dq_linear(x, *p, bits, g, bias, None, -1.0, 0), plain + bias.double()))
    close(ext().dq_gemv_gateup(x, *p, bits, g, -1.0, 0), gated(plain), 1e-2)


# (bits, gate, rows, n, k, group): taken, and the neighbour that is not
LINES = [
    # rows, columns in eights, one round of workgroups
    ((4, 0, 768, 2048, 2048, 128), (4, 0, 769, 2048, 2048, 128)),
    ((4, 0, 100, 4104, 2048, 128), (4, 0, 100, 4102, 2048, 128)),
    ((8, 0, 96, 32768, 2048, 64), (8, 0, 96, 32776, 2048, 64)),
    ((4, 0, 80, 32768, 1024, 128), (4, 0, 80, 32776, 1024, 128)),
    # a gate's chain, where the other kernel has parts, and above 48 rows
    ((4, 1, 48, 10240, 4096, 128), (4, 1, 48, 10240, 9216, 128)),
    ((4, 1, 40, 4088, 6144, 128), (4, 1, 40, 4104, 6144, 128)),
    ((8, 1, 48, 1024, 6144, 64), (8, 1, 49, 1024, 6144, 64)),
    # few rows: short chains, small matrices, 6144 to 8192 columns
    ((4, 1, 28, 16384, 1280, 128), (4, 1, 28, 16384, 1024, 128)),
    ((8, 1, 28, 4096, 1280, 128), (8, 1, 28, 4096, 1024, 128)),
    ((4, 0, 32, 16384, 1280, 64), (4, 0, 32, 16384, 1024, 64)),
    ((8, 0, 25, 9000, 1024, 64), (8, 0, 24, 9000, 1024, 64)),
    ((8, 0, 49, 3000, 1024, 64), (8, 0, 48, 3000, 1024, 64)),
    ((8, 0, 40, 2016, 1024, 64), (8, 0, 40, 2024, 1024, 64)),
    ((8, 0, 40, 6144, 640, 64), (8, 0, 40, 6136, 640, 64)),
    ((8, 0, 32, 6136, 1536, 64), (8, 0, 32, 6144, 1536, 64)),
    ((8, 0, 32, 8200, 1024, 64), (8, 0, 32, 8192, 1024, 64)),
    ((4, 0, 32, 8200, 2048, 128), (4, 0, 32, 8192, 2048, 128)),
    # short k
    ((8, 0, 200, 2048, 768, 64), (8, 0, 200, 2048, 704, 64)),
    ((8, 0, 32, 9000, 768, 64), (8, 0, 32, 9000, 704, 64)),
    ((8, 0, 64, 6144, 640, 128), (8, 0, 64, 6152, 640, 128)),
    # 16385 to 20480 columns, long k
    ((8, 0, 96, 16384, 1024, 64), (8, 0, 96, 16392, 1024, 64)),
    ((8, 0, 96, 20488, 1024, 64), (8, 0, 96, 20480, 1024, 64)),
    ((4, 0, 55, 16384, 4096, 64), (4, 0, 55, 16392, 4096, 64)),
    ((4, 0, 96, 4096, 12032, 128), (4, 0, 97, 4096, 12032, 128))]


@pytest.mark.parametrize("call,taken", [(c, i == 0) for pair in LINES
                                        for i, c in enumerate(pair)])
def test_eight_waves_at_the_lines(call, taken):
    """On both sides of the lines where other products are the faster ones."""
    bits, gate, m, n, k, g = call
    torch.manual_seed(n + m)
    p, w = matrix(bits, n, k, g)
    x = torch.randn(m, k, device=DEV).to(BF)
    want = x.double() @ w.t()
    got = []
    names = launched(lambda: got.append(
        ext().dq_gemv_gateup(x, *p, bits, g, -1.0, 0) if gate else
        ext().dq_linear(x, *p, bits, g, None, None, -1.0, 0)))
    assert ("dq_mid_kernel" in names) == taken, names
    close(got[0], gated(want) if gate else want, 1e-2 if gate else 5e-3)


def step_of(batch, heads, hidden, inner, T=300):
    """A cache of T keys, and a decode step behind it of two layers of 4 bits."""
    torch.manual_seed(hidden)
    with torch.device(DEV):
        cfg = LlamaConfig(vocab_size=512, hidden_size=hidden, intermediate_size=inner,
                          n_layers=2, n_heads=heads, n_kv_heads=8, head_dim=128)
        m = lfmq.build_model(cfg)
        for p in m.parameters():
            if p.dim() > 1:
                p.normal_(0, p.shape[-1] ** -0.5)
    m = lfmq.quantize(m, lfmq.QuantConfig(scheme="rtn", bits=4, group_size=128,
                                          skip_modules=("lm_head",)))
    cache = m.make_cache(batch, max_seq=T + 8)
    for t in (cache.k_all, cache.v_all):
        t[:, :, :, :T].normal_()
    state = torch.tensor([T, T + 1, 0], dtype=torch.int32, device=DEV)
    ids = torch.randint(512, (batch, 1), device=DEV)
    return cache, lambda: m.forward_decode_step(ids, cache, state, T + 8)


@torch.no_grad()
@pytest.mark.parametrize("batch,heads,hidden,inner", [
    (8, 32, 4096, 14336), (3, 48, 6144, 8192), (16, 32, 2048, 20480)])
def test_a_step_whose_down_projection_is_in_parts(batch, heads, hidden, inner,
                                                  monkeypatch):
    """Its counters are those of decode attention, in each layer and in a graph's
    replays; results to the bit, as a layer's launches are the same then."""
    cache, step = step_of(batch, heads, hidden, inner)
    step()
    found = []
    parts = F.dq_linear_parts
    monkeypatch.setattr(F, "dq_linear_parts",
                        lambda *a: found.append(parts(*a)) or found[-1])
    want = step()
    assert len(found) == 2 and all(y is not None for y in found)
    assert not bool(cache.tickets.any())
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        logits = step()
    for _ in range(3):
        logits.zero_()
        graph.replay()
        assert torch.equal(logits, want)
        assert torch.equal(step(), want)
        assert not bool(cache.tickets.any())
    monkeypatch.setattr(F, "dq_linear_parts", lambda *a: None)
    plain = step()
    # roundings of 2^-9 in two layers' products and the head's
    assert not torch.equal(plain, want)
    assert float((plain.double() - want.double()).norm() / want.double().norm()) < 2e-2


@torch.no_grad()
@pytest.mark.parametrize("batch,inner", [(8, 8192), (3, 16256), (2, 20480)])
def test_a_step_asks_for_parts_only_where_there_may_be_some(batch, inner, monkeypatch):
    """A step of two layers of 2048 without a graph waits for the host, which the
    question takes 5 us a layer."""
    _, step = step_of(batch, 16, 2048, inner)
    asked = []
    monkeypatch.setattr(F, "dq_linear_parts", lambda *a: asked.append(1))
    step()
    assert not asked
