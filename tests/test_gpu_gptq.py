"""GPTQ's column blocks, and the products that carry their errors on."""
import math

import pytest
import torch

from lfmq import QuantConfig
from lfmq.ops import hip_ext as ext
from lfmq.quant.gptq import _block

from gptq_util import gpu_block

pytestmark = pytest.mark.gpu
DEV = "cuda"


# rows of a workgroup: 8, 16 and 32; U by pieces of 16 bytes, and where its
# rows or the matrix do not start on them; results by pieces, and one by one;
# one, two and more groups that start in a block
@pytest.mark.parametrize("n,k,nb,i1,g", [
    (9, 256, 128, 0, 128), (4100, 256, 128, 128, 64), (8200, 192, 64, 128, 32),
    (17, 260, 128, 128, 65), (40, 262, 128, 130, 131), (24, 224, 96, 128, 16)])
def test_block_is_the_tensor_loop(n, k, nb, i1, g):
    cfg = QuantConfig(scheme="gptq", bits=4, group_size=g)
    w = torch.randn(n, k, device=DEV)
    u = torch.randn(k, k, device=DEV).mul_(0.1).triu_()
    u.diagonal().uniform_(0.5, 2.0)
    got = []
    for fn in (_block, gpu_block):
        out = [torch.zeros(n, k, dtype=torch.int32, device=DEV),
               torch.full((n, k // g), 0.4, device=DEV),
               torch.full((n, k // g), 5, dtype=torch.int32, device=DEV)]
        got.append(out + [fn(w, u[i1:i1 + nb, i1:i1 + nb], *out, i1, cfg, g)])
    for a, b in zip(*got):
        assert torch.equal(a, b)


@pytest.mark.parametrize("n,k,nb,i1", [
    (1, 129, 128, 0), (64, 192, 128, 0), (65, 321, 100, 28), (130, 257, 3, 126),
    (200, 512, 128, 256)])
def test_push(n, k, nb, i1):
    """A difference is rounded once, a sum of nb products nb times at most,
    each 2^-24 of the numbers summed.  The block and what is before it stay."""
    w, err = torch.randn(n, k, device=DEV), torch.randn(n, nb, device=DEV)
    u = torch.randn(k, k, device=DEV)
    got = w.clone()
    ext().gptq_push(got, err, u, i1)
    at, ub = i1 + nb, u[i1:i1 + nb].double()
    want = w.double()
    want[:, at:] -= err.double() @ ub[:, at:]
    size = w.abs().double()
    size[:, at:] += nb * (err.abs().double() @ ub[:, at:].abs())
    assert bool(((got - want).abs() <= size * 2 ** -24).all())
    assert torch.equal(got[:, :at], w[:, :at])


def worst_tile(u, w):
    """The largest error of a 64 x 64 tile on or above the diagonal, beside the
    tile of w."""
    n, N = w.shape[0], -(-w.shape[0] // 64)

    def norms(a):
        t = torch.zeros(N * 64, N * 64, dtype=torch.float64, device=w.device)
        t[:n, :n] = a
        return t.view(N, 64, N, 64).square().sum((1, 3)).sqrt()

    return float((norms(u.double() - w) / norms(w))[
        torch.ones(N, N, device=w.device).triu().bool()].max())


# an odd and an even number of steps of one launch, the most of them, and the
# least of two launches
@pytest.mark.parametrize("n", [1100, 1984, 2048, 2049])
def test_inverse_factor_of_either_kind(n):
    """Each rounding moves U by the condition of H, 3600, times 2^-24 at most: of
    sums of n of them 2e-5 of a tile were seen with either kind (and twice that
    with the library's fp32 factors).  Ten times that is too little for a tile
    of the step before, or one left out, or bf16."""
    x = torch.randn(2 * n + 1, n, device=DEV) + torch.randn(n, device=DEV)
    h = x.t() @ x + n * torch.eye(n, device=DEV)
    h = h.tril() + h.tril(-1).t()          # (products of odd sizes are not even)
    u, failed = ext().chol_inverse(h)
    h64 = h.double()
    w = torch.linalg.cholesky(torch.linalg.inv(h64), upper=True)
    assert failed.item() == 0
    assert float(u.tril(-1).abs().max()) == 0.0
    assert worst_tile(u, w) <= 2e-4
    back = u.double() @ h64 @ u.double().t()
    assert float((back - torch.eye(n, device=DEV)).abs().max()) <= 5e-5
    gone = w.clone()
    gone[:64, 64:128] = 0
    assert worst_tile(gone, w) > 2e-4 and worst_tile(w.bfloat16(), w) > 2e-4
    h[n - 1, n - 1] = -h[n - 1, n - 1]
    assert ext().chol_inverse(h)[1].item() == 1


# the most steps of one launch, the least of two
@pytest.mark.parametrize("n", [3072, 3073])
def test_inverse_factor_at_the_line(n):
    test_inverse_factor_of_either_kind(n)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 31, 33, 48, 63, 64])
def test_inverse_factor_of_one_block(n):
    """Every panel of a diagonal block, columns of unequal size.  A rounding
    moves U by the condition times 2^-24 at most, sums of n of them in random
    directions (the scales of rows and columns cancel)."""
    torch.manual_seed(n)
    x = torch.randn(4 * n, n, device=DEV)
    size = torch.exp(2 * torch.randn(n, device=DEV))
    h64 = (x.t() @ x).double()
    tol = 2 * math.sqrt(n) * 2 ** -24 * float(torch.linalg.cond(h64))
    h = (h64 * size * size[:, None]).float()
    u, failed = ext().chol_inverse(h)
    w = torch.linalg.cholesky(torch.linalg.inv(h.double()), upper=True)
    assert failed.item() == 0
    assert float(u.tril(-1).abs().max()) == 0.0
    away = (u.double() - w) * size
    assert float(away.norm() / (w * size).norm()) <= tol
    for i in range(n):
        bad = h.clone()
        bad[i, i] = -bad[i, i]
        assert ext().chol_inverse(bad)[1].item() == 1
    h[n // 2, n // 2] = 2.0 ** 126         # no reciprocal in the normal range
    assert ext().chol_inverse(h)[1].item() == 1


# rows that end inside a workgroup's sixteen and inside a product's 64; a last
# block of 64; one, two and many groups a block; too many rows, and groups that do
# not end with a block, which go block by block
@pytest.mark.parametrize("n,k,g,bits,sym", [
    (1, 256, 128, 4, False), (2048, 512, 128, 4, False), (17, 384, 64, 8, True),
    (4096, 320, 64, 4, False), (1000, 640, 16, 4, True), (4097, 384, 128, 4, False),
    (70, 768, 384, 4, False), (33, 520, 104, 8, False)])
def test_all_columns_are_block_by_block(n, k, g, bits, sym):
    """A launch that takes a block's errors off the next one's columns while it
    carries them on: bit by bit what a launch each leaves."""
    gen = torch.Generator(DEV).manual_seed(n)
    w = torch.randn(n, k, generator=gen, device=DEV)
    if n > 1:
        w[0] *= 1e-39                      # quotients that need divisions
        w[n // 2, 3] = float("inf")
    u = torch.randn(k, k, generator=gen, device=DEV).triu_() * 0.05
    u.diagonal().copy_(torch.rand(k, generator=gen, device=DEV) + 0.5)

    def out():
        return (torch.zeros(n, k, dtype=torch.int32, device=DEV),
                torch.zeros(n, k // g, device=DEV),
                torch.zeros(n, k // g, dtype=torch.int32, device=DEV))

    got, want = out(), out()
    ext().gptq_columns(w.clone(), u, *got, 128, g, bits, sym)
    cfg = QuantConfig(scheme="gptq", bits=bits, group_size=g, sym=sym)
    for i1 in range(0, k, 128):
        i2 = min(i1 + 128, k)
        err = gpu_block(w, u[i1:i2, i1:i2], *want, i1, cfg, g)
        if i2 < k:
            ext().gptq_push(w, err, u, i1)
    finite = torch.isfinite(want[1]).all(1)
    assert int(finite.sum()) == max(n - 1, 1)
    for a, b in zip(got, want):
        assert torch.equal(a[finite], b[finite])


@pytest.mark.parametrize("n,k", [(1, 1), (3, 7), (70, 1030), (5, 2048)])
def test_weights_and_diagonal_of_a_solve(n, k):
    """Columns without inputs: ones on the diagonal, zeros (whatever w holds) in
    the weights; the damping is a mean of k sums in fp32."""
    gen = torch.Generator(DEV).manual_seed(k)
    w = torch.randn(n, k, generator=gen, device=DEV)
    h = torch.rand(k, k, generator=gen, device=DEV) + 0.5
    dead = torch.rand(k, generator=gen, device=DEV) < 0.3
    h.diagonal()[dead] = 0
    w[:, dead] = float("nan")
    kept = w.clone(), h.clone()
    to, d = ext().gptq_prepare(w, h, 0.01)
    assert torch.equal(w.nan_to_num(7.0), kept[0].nan_to_num(7.0))
    assert torch.equal(h, kept[1])
    diag = torch.where(dead, torch.ones_like(h.diagonal()), h.diagonal())
    assert torch.equal(to, torch.where(dead, torch.zeros_like(w), w))
    assert torch.equal(d[0], diag) and torch.equal(d[2] == 0, dead)
    want = diag.double() + 0.01 * diag.double().mean()
    # a sum of k in trees of 64 and 16 and runs of k / 1024, and three roundings
    bound = (26 + k / 1024) * 2 ** -24
    assert float(((d[1].double() - want) / want).abs().max()) <= bound


@pytest.mark.parametrize("act_order", [False, True])
def test_solve_by_the_library_factor(act_order):
    """Pivots that the factor does not take (from 2^125): the library's factor,
    of weights that the columns have not changed.  Without elements beside the
    diagonal nothing is carried on, whatever its size."""
    from lfmq.quant.gptq import gptq_quantize_layer
    torch.manual_seed(3)
    w = torch.randn(40, 256, device=DEV)
    cfg = QuantConfig(scheme="gptq", bits=4, group_size=64, act_order=act_order)
    h = torch.diag(torch.rand(256, device=DEV) + 1)
    h[5, 5] = 0
    h[9, 9] = 3
    want = gptq_quantize_layer(w, h, cfg)
    h[9, 9] = 1.5 * 2.0 ** 125
    assert ext().chol_inverse(h + torch.eye(256, device=DEV))[1].item()
    got = gptq_quantize_layer(w, h, cfg)
    for a, b in zip(got[:3], want[:3]):
        assert torch.equal(a, b)
    assert act_order == (got[3] is not None)
    if act_order:
        assert got[3].dtype == torch.int64 and torch.equal(got[3], want[3])
