"""Packed products of a prompt against 64 bits (dq_block, dq_short), where their
row tiles, column blocks, stages and parts end.  Tolerances: test_gpu_decode_products."""
import pytest
import torch

from lfmq.ops import hip_ext as ext
from test_gpu_decode_products import BF, DEV, close, gated, launched, matrix

pytestmark = pytest.mark.gpu


# One to three row tiles of 64 to 128, also of sizes in between; column blocks
# that end inside a wave's columns, or between pieces of 16 bytes; one group a
# chunk and several; four chunks up, whole, split, and some tiles split.
@pytest.mark.parametrize("bits,m,n,k,g", [
    (4, 129, 264, 1024, 128), (4, 180, 1041, 2048, 128), (4, 256, 522, 1024, 64), (4, 256, 520, 1024, 64),
    (4, 150, 2062, 5120, 128), (4, 300, 258, 8192, 512), (4, 130, 300, 512, 64),
    (4, 2100, 4352, 1024, 128), (4, 1100, 8450, 1536, 64),
    (8, 129, 264, 512, 64), (8, 256, 1030, 2048, 64), (8, 150, 519, 1024, 64),
    (8, 193, 700, 2048, 128), (8, 2100, 4352, 1024, 64),
    (8, 257, 1030, 2048, 128), (4, 66, 9002, 3072, 64), (4, 49, 28674, 3072, 128)])
def test_many_rows(bits, m, n, k, g):
    torch.manual_seed(m + n)
    p, w = matrix(bits, n, k, g)
    x = torch.randn(m, k, device=DEV).to(BF)
    x[0] = 0
    bias = torch.randn(n, device=DEV).to(BF)
    plain = x.double() @ w.t()
    close(ext().dq_linear(x, *p, bits, g, bias, None, -1.0, 0),
          plain + bias.double())
    if n % 2 == 0:
        close(ext().dq_gemv_gateup(x, *p, bits, g, -1.0, 0), gated(plain),
              1e-2)


# What is large enough for dq_panel: row tiles of 64 to 128; columns that end inside
# a wave's; 16 to 112 groups; several chunks a group; some tiles
# split, the eights of groups of a part then as they fall.
@pytest.mark.parametrize("bits,m,n,k,g", [
    (4, 1100, 8450, 2048, 128), (4, 130, 20002, 6144, 128), (4, 60, 28674, 9216, 128),
    (4, 150, 16390, 8192, 512), (4, 2100, 4352, 3072, 128), (8, 140, 16390, 4608, 64),
    (4, 140, 16391, 4608, 64), (8, 300, 9030, 8192, 128), (8, 700, 4100, 7168, 64)])
def test_many_rows_of_large_products(bits, m, n, k, g):
    assert "dq_panel_kernel" in launched(lambda: test_many_rows(bits, m, n, k, g))


# (k whole, and in parts)
@pytest.mark.parametrize("kernel,bits,m,n,k,g", [
    ("dq_wide_kernel", 4, 8, 8200, 2048, 128), ("dq_mid_kernel", 4, 40, 4104, 4096, 128),
    ("dq_mid_kernel", 4, 100, 4104, 2048, 128), ("dq_mid_kernel", 4, 200, 512, 4096, 128),
    ("dq_mid_kernel", 8, 40, 4104, 4160, 64), ("dq_mid_kernel", 8, 200, 512, 4224, 128),
    ("dq_short_kernel", 4, 40, 4098, 4096, 128),
    ("dq_short_kernel", 4, 100, 4102, 2048, 128),
    ("dq_short_kernel", 8, 100, 4102, 2048, 64),
    ("dq_block_kernel", 4, 200, 514, 4096, 128), ("dq_block_kernel", 8, 200, 514, 4096, 64),
    ("dq_panel_kernel", 4, 300, 8200, 8192, 128),
    ("dq_panel_kernel", 8, 300, 8200, 8192, 64)])
def test_values_that_are_not_finite_stay_in_their_rows(kernel, bits, m, n, k, g):
    torch.manual_seed(0)
    p, w = matrix(bits, n, k, g)
    x = torch.randn(m, k, device=DEV).to(BF)
    x[3, 7], x[m * 2 // 3, k - 96] = float("inf"), float("nan")
    got = []
    assert kernel in launched(lambda: got.append(
        ext().dq_linear(x, *p, bits, g, None, None, -1.0, 0)))
    fine = torch.isfinite(x).all(1)
    assert not bool(torch.isfinite(got[0][~fine]).any())
    close(got[0][fine], x[fine].double() @ w.t())


@pytest.mark.parametrize("bits,m,g", [(4, 8, 128), (8, 16, 64)])
def test_values_that_are_not_finite_and_k_in_parts(bits, m, g):
    n, k = 4096, 14336
    torch.manual_seed(0)
    p, w = matrix(bits, n, k, g)
    x = torch.randn(m, k, device=DEV).to(BF)
    x[3, 7], x[m * 2 // 3, k - 96] = float("inf"), float("nan")
    tickets = torch.zeros(128, dtype=torch.int32, device=DEV)
    y = ext().dq_linear_parts(x, *p, bits, g, None, None, tickets)
    fine = torch.isfinite(x).all(1)
    assert not bool(torch.isfinite(y[~fine]).any())
    close(y[fine], x[fine].double() @ w.t())


@pytest.mark.parametrize("m,n,k,g", [(40, 4104, 4160, 64), (40, 4104, 4224, 128),
                                     (100, 2056, 2112, 64), (200, 512, 4160, 64)])
def test_an_infinite_value_gives_infinite_products(m, n, k, g):
    """8 bits, whose codes less their zeros are exact: what IEEE 754 has for them, and
    nothing of a group that a wave has beside others' (the last of a part)."""
    torch.manual_seed(m)
    p, w = matrix(8, n, k, g)
    x = torch.randn(m, k, device=DEV).to(BF)
    at = torch.arange(m, device=DEV) * (k // g - 1) // (m - 1) * g + 5
    x[torch.arange(m, device=DEV), at] = float("inf")
    got = []
    assert "dq_mid_kernel" in launched(lambda: got.append(
        ext().dq_linear(x, *p, 8, g, None, None, -1.0, 0)))
    sign = w.t()[at].sign()                      # of the product with infinity
    want = torch.where(sign == 0, float("nan"), sign * float("inf"))
    assert torch.equal(got[0].isnan(), want.isnan())
    assert bool((got[0].double() == want)[sign != 0].all())


@pytest.mark.parametrize("bits,n,k,g", [(4, 2062, 2048, 128),
                                        (8, 1040, 1024, 64),
                                        (4, 516, 1536, 64),
                                        (4, 260, 2560, 64),
                                        # dq_panel: whole, and in two parts
                                        (4, 6162, 5120, 128),
                                        (8, 4096, 7168, 64)])
def test_many_rows_by_expert(bits, n, k, g):
    """One to 128 rows a tile, experts without any, tiles that are none; k whole
    (n not in fours), in two and in four parts."""
    torch.manual_seed(n)
    counts = (1, 0, 129, 80, 192, 17, 32, 161)
    p, w = matrix(bits, n, k, g, (len(counts),))
    src = torch.randperm(sum(counts)).to(DEV)
    x = torch.randn(sum(counts), k, device=DEV).to(BF)
    tiles, at, want = [(-1, 0, 0)], 0, []
    for e, c in enumerate(counts):
        tiles += [(e, at + i, min(128, c - i)) for i in range(0, c, 128)]
        want.append(x.double()[src[at:at + c]] @ w[e].t())
        at += c
    tiles = torch.tensor(tiles + [(-1, 0, 0)], dtype=torch.int32, device=DEV)
    want, s32 = torch.cat(want), src.to(torch.int32)
    names = launched(lambda: close(
        ext().moe_linear(x, s32, tiles, *p, bits, g, True, 128), gated(want), 1e-2))
    names |= launched(lambda: close(
        ext().moe_linear(x[src], None, tiles, *p, bits, g, False, 128), want))
    assert ("dq_panel_kernel" in names) == (n * k > 20 << 20), names


# Row tiles of 32 to 128, one to three of them; columns that end inside a wave's;
# k whole and in parts, with more groups to a part than LDS holds and with
# groups of 64's multiples; the residual, which a step of 48 sequences has.
@pytest.mark.parametrize("bits,m,n,k,g", [
    (4, 17, 4098, 4096, 128), (4, 33, 5130, 4160, 64), (8, 48, 4099, 4096, 128),
    (8, 40, 24580, 2112, 64), (4, 49, 2100, 2112, 64), (4, 80, 4098, 1152, 128),
    (4, 64, 5001, 1024, 256), (8, 65, 2062, 2112, 64), (8, 96, 16402, 2112, 64),
    (4, 113, 4098, 1024, 128), (4, 128, 4102, 1152, 64), (8, 97, 2054, 2304, 128),
    (8, 128, 16386, 2048, 64), (8, 77, 32770, 1024, 128), (4, 33, 33026, 2048, 128),
    (4, 33, 4104, 4160, 64), (8, 96, 16400, 2112, 64), (4, 33, 5128, 4160, 64)])
def test_some_rows(bits, m, n, k, g):
    torch.manual_seed(m + n)
    p, w = matrix(bits, n, k, g)
    x = torch.randn(m, k, device=DEV).to(BF)
    x[0] = 0
    bias = torch.randn(n, device=DEV).to(BF)
    plain = x.double() @ w.t()
    # (columns in eights are dq_mid's)
    kernel = "dq_mid_kernel" if n % 8 == 0 else "dq_short_kernel"
    assert kernel in launched(lambda: close(
        ext().dq_linear(x, *p, bits, g, bias, None, -1.0, 0), plain + bias.double()))
    if m <= 48:
        resid = torch.randn(m, n, device=DEV).to(BF)
        close(ext().dq_linear(x, *p, bits, g, None, resid, -1.0, 0),
              plain + resid.double())
    if n % 2 == 0:
        close(ext().dq_gemv_gateup(x, *p, bits, g, -1.0, 0), gated(plain),
              1e-2)


@pytest.mark.parametrize("bits,g,mean", [(4, 128, 0), (4, 128, 1), (8, 64, 0),
                                         (8, 64, 1)])
def test_rows_with_a_common_part(bits, g, mean):
    """What the codes' sums and the zeros' cancel does not cost the fp32 result: 112 or
    224 groups, each added with an error of 2^-24 of sums that are at no time more than
    some times the result (with all zeros' sums at once 24e-6 and 3e-6 for a mean of
    one)."""
    n, k, rows = 4096, 14336, 512
    torch.manual_seed(bits)
    half, per = 1 << bits - 1, 32 // bits
    codes = torch.randint(0, 2 * half, (n, k), device=DEV)
    zeros = half + torch.randint(-half // 4, half // 4 + 1, (n, k // g), device=DEV)
    s = (torch.rand(n, k // g, device=DEV) * 0.02 + 0.01).to(BF)
    w = ((codes.view(n, -1, g) - zeros.unsqueeze(-1)).double()
         * s.double().unsqueeze(-1)).flatten(1)
    pack = lambda t: ext().pack(t.int().contiguous(), bits).unsqueeze(0)
    assert k // g % per == 0
    x = (torch.randn(rows, k, device=DEV) + mean).to(BF)
    tiles = torch.tensor([(0, i, 128) for i in range(0, rows, 128)],
                         dtype=torch.int32, device=DEV)
    got = []
    names = launched(lambda: got.append(ext().moe_linear(
        x, None, tiles, pack(codes), s.unsqueeze(0), pack(zeros), bits, g, False, 128)))
    assert "dq_panel_kernel" in names
    want = x.double() @ w.t()
    assert float((got[0].double() - want).norm() / want.norm()) < 1.5e-6


@torch.no_grad()
def test_rows_by_expert_in_parts_are_all_that_is_kept():
    """k in four parts, whose scratch memory is not the result's."""
    k, n, g, E, each = 2560, 256, 64, 8, 20
    p, w = matrix(4, n, k, g, (E,))
    x = torch.randn(E * each, k, device=DEV).to(BF)
    tiles = torch.tensor([(e, e * each, each) for e in range(E)],
                         dtype=torch.int32, device=DEV)
    y = ext().moe_linear(x, None, tiles, *p, 4, g, False, 128)
    close(y, (x.double().view(E, each, k) @ w.transpose(1, 2)).flatten(0, 1))
    assert y.untyped_storage().nbytes() == y.numel() * 4
