"""GPTQ's column blocks, and the products that carry their errors on."""
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


# the largest of one launch a step, the smallest of two, and one in between
@pytest.mark.parametrize("n", [2048, 2049, 1100])
def test_inverse_factor_of_either_kind(n):
    """First-order bound as in test_gpu_kernels: each rounding moves U by the
    condition of H at most, sums of n of them in random directions."""
    x = torch.randn(2 * n + 1, n, device=DEV) + torch.randn(n, device=DEV)
    h = x.t() @ x + n * torch.eye(n, device=DEV)
    u, failed = ext().chol_inverse(h)
    h64 = h.double()
    w = torch.linalg.cholesky(torch.linalg.inv(h64), upper=True)
    e = torch.linalg.eigvalsh(h64)
    tol = 2 * n ** 0.5 * 2 ** -24 * float(e[-1] / e[0])
    assert failed.item() == 0
    assert float((u.double() - w).norm() / w.norm()) <= tol
    assert float(u.tril(-1).abs().max()) == 0.0
    h[n - 1, n - 1] = -h[n - 1, n - 1]
    assert ext().chol_inverse(h)[1].item() == 1
