"""The edges of what the GPU calls take: nothing at all, more than a counter
or an address holds, infinities, numbers below the normal range, tensors that
stand for more than their values, streams and graphs."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
BF = torch.bfloat16


def ext():
    from lfmq.ops import hip_ext
    return hip_ext()


# ------------------------------------------------------------- attention
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
