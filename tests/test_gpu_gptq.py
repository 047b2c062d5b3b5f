"""GPTQ's column blocks, and the products that carry their errors on."""
import math

import pytest
import torch

from lfmq import QuantConfig
from lfmq.ops import hip_ext as ext
from lfmq.quant.gptq import _block, _gpu_block

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
    for fn in (_block, _gpu_block):
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
