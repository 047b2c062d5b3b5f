"""RMS norm of rows kept in registers against 64 bits: widths that end inside a
thread's pieces, each number of them, and what goes to the general kernels."""
import pytest
import torch

from lfmq.ops import hip_ext as ext

pytestmark = pytest.mark.gpu
DEV, BF = "cuda", torch.bfloat16


def close(y, want):
    # a result rounds by 2^-9 of itself; its fp32 factors are off by 2^-20
    assert float(((y.double() - want).abs() / (want.abs() + 1e-6)).max()) < \
        2 ** -8 + 2 ** -18


@pytest.mark.parametrize("width", [8, 512, 2040, 2048, 2056, 4096, 4104, 8200,
                                   14336, 16384, 16392, 1002])
@pytest.mark.parametrize("rows", [1, 37])
def test_rows_in_registers(width, rows):
    x, r, w = (torch.randn(n, width, device=DEV).to(BF) for n in (rows, rows, 1))
    w = w[0]

    def norm(v):
        v = v.double()
        return v * torch.rsqrt((v ** 2).mean(-1, keepdim=True) + 1e-5) * \
            w.double()

    close(ext().rmsnorm(x, w, 1e-5, None), norm(x))
    both = x.float() + r.float()               # exact but for cancelled bits
    close(ext().rmsnorm(x, w, 1e-5, r), norm(both))
    y, new = ext().rmsnorm_residual(x, r, w, 1e-5)
    close(y, norm(both))
    assert torch.equal(new, both.to(BF))


def test_rows_that_do_not_start_on_16_bytes():
    x = torch.randn(3 * 4096 + 1, device=DEV).to(BF)[1:].view(3, 4096)
    w = torch.ones(4096, device=DEV, dtype=BF)
    v = x.double()
    close(ext().rmsnorm(x, w, 1e-5, None),
          v * torch.rsqrt((v ** 2).mean(-1, keepdim=True) + 1e-5))
