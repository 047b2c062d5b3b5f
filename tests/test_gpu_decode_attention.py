"""Decode attention over several ranges of keys: the merge by the launch's own
last workgroup against the merge by a second launch."""
import pytest
import torch

from lfmq.ops import hip_ext as ext
from lfmq.ops import ref

pytestmark = pytest.mark.gpu
DEV, BF = "cuda", torch.bfloat16


@pytest.mark.parametrize("b,T,room,hq,hkv,d", [
    (1, 256, 600, 32, 8, 128), (1, 257, 0, 32, 8, 128), (48, 300, 200, 32, 8, 128),
    (20, 900, 0, 32, 8, 128), (1, 4129, 0, 8, 2, 128), (3, 9000, 7900, 8, 1, 128),
    (1, 16300, 0, 16, 2, 64), (5, 700, 90, 12, 2, 64), (2, 3000, 0, 3, 3, 128),
    # the most ranges of 128 keys, and one key more
    (2, 3072, 5000, 8, 2, 128), (2, 3073, 5000, 8, 2, 128)])
def test_merge_in_the_launch(b, T, room, hq, hkv, d):
    """Same ranges, same order of sums: the same bits, launch after launch on
    other values, with results of other workgroups, of other XCDs most of them,
    read in the launch that writes them."""
    tmax = T + room
    inv = ref.rope_freqs(d, 500000.0).to(DEV)
    tk = torch.zeros(b * hq, dtype=torch.int32, device=DEV)
    st = torch.tensor([T], dtype=torch.int32, device=DEV)
    gen = torch.Generator(DEV).manual_seed(T)
    kc, vc = (torch.empty(b, hkv, tmax, d, dtype=BF, device=DEV)
              for _ in range(2))
    for i in range(12):
        for t in (kc, vc):
            t.normal_(0, 1, generator=gen)
        qkv = torch.randn(b, (hq + 2 * hkv) * d, generator=gen,
                          device=DEV).to(BF)
        one, two = (ext().attn_decode_fused(qkv, kc, vc, tmax, d ** -0.5, inv,
                                            hq, st, t) for t in (tk, None))
        assert torch.equal(one, two), i
    assert int(tk.abs().sum()) == 0
    q = ref.apply_rope(qkv[:, :hq * d].view(b, 1, hq, d).float().cpu(),
                       torch.tensor([T - 1])).view(b, hkv, -1, d).to(DEV)
    k, v = (t[:, :, :T].double() for t in (kc, vc))
    p = torch.softmax(q.double() @ k.transpose(2, 3) * d ** -0.5, -1)
    want = (p @ v).view(b, -1)
    # roundings of q, k and o
    assert float((one.view(b, -1).double() - want).norm() / want.norm()) < 6e-3
