"""One column block of the GPTQ solve by its kernel alone."""
import torch

from lfmq.ops import hip_ext


def gpu_block(w, ub, codes, scales, zeros, i1, cfg, g) -> torch.Tensor:
    """lfmq.quant.gptq._block in one launch, the same bit by bit."""
    if ub.stride(1) != 1:
        ub = ub.contiguous()
    return hip_ext().gptq_block(w, ub, codes, scales, zeros, i1, g, cfg.bits,
                                cfg.sym)
