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


# one round of a wave, of four and of eight waves (eight heads of 128 on a key
# head), one key more and less; a last range of one key; the most ranges
@pytest.mark.parametrize("b,T,room,hq,hkv,d", [
    (1, 1, 3, 8, 1, 128), (1, 32, 0, 8, 2, 128), (2, 33, 500, 4, 4, 64),
    (3, 129, 70, 7, 1, 128), (1, 256, 1, 16, 2, 128), (2, 257, 300, 8, 1, 128),
    (1, 1025, 7, 6, 1, 128), (1, 16384, 0, 8, 1, 128), (1, 300, 16200, 8, 1, 128),
    (2, 385, 15, 2, 1, 64)])
def test_rows_past_the_keys(b, T, room, hq, hkv, d):
    """What the cache holds behind the keys, and where the new key goes, is not
    read: NaN there changes nothing.  The new rows are written."""
    tmax = T + room
    inv = ref.rope_freqs(d, 500000.0).to(DEV)
    tk = torch.zeros(b * hq, dtype=torch.int32, device=DEV)
    st = torch.tensor([T], dtype=torch.int32, device=DEV)
    gen = torch.Generator(DEV).manual_seed(T)
    kc, vc = (torch.randn(b, hkv, tmax, d, generator=gen, device=DEV).to(BF)
              for _ in range(2))
    for t in (kc, vc):
        t[:, :, T - 1:] = float("nan")
    qkv = torch.randn(b, (hq + 2 * hkv) * d, generator=gen, device=DEV).to(BF)
    o = ext().attn_decode_fused(qkv, kc, vc, tmax, d ** -0.5, inv, hq, st, tk)
    assert int(tk.abs().sum()) == 0
    assert bool(kc[:, :, T:].isnan().all()) and bool(vc[:, :, T:].isnan().all())
    at = torch.tensor([T - 1])
    rows = qkv.float().cpu()
    q = ref.apply_rope(rows[:, :hq * d].view(b, 1, hq, d), at)
    new = ref.apply_rope(rows[:, hq * d:(hq + hkv) * d].view(b, 1, hkv, d), at)
    k, v = (t[:, :, :T].double() for t in (kc, vc))
    assert float((k[:, :, -1].cpu() - new[:, 0].double()).abs().max()) \
        <= 2 ** -8 * float(new.abs().max())
    assert torch.equal(vc[:, :, T - 1].flatten(1), qkv[:, (hq + hkv) * d:])
    q = q.view(b, hkv, -1, d).to(DEV).double()
    want = (torch.softmax(q @ k.transpose(2, 3) * d ** -0.5, -1) @ v).view(b, -1)
    # roundings of q, k and o, as above
    assert float((o.view(b, -1).double() - want).norm() / want.norm()) < 6e-3


# up to 4 MiB of keys and values by the caches, from there on past them
@pytest.mark.parametrize("b,T,room,hq,hkv,d", [
    (2, 511, 0, 8, 8, 128), (2, 512, 0, 32, 8, 128), (2, 500, 13, 16, 8, 128),
    (3, 1366, 0, 16, 2, 128), (4, 513, 0, 16, 8, 64), (5, 1100, 77, 8, 8, 64)])
def test_keys_past_the_caches(b, T, room, hq, hkv, d):
    test_rows_past_the_keys(b, T, room, hq, hkv, d)
