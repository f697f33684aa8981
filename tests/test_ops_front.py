"""What the native front of nnfusion_amd.ops refuses, on host tensors: the refusal comes before the library or a device is
asked for anything."""
import pytest
import torch

from nnfusion_amd import ops


def test_w8a8_without_scales_is_refused():
    """The fp16 product with an absent scale vector must not turn into the int32 accumulators: an output buffer given for the
    product holds half of their bytes."""
    a, w = torch.zeros((4, 256), dtype=torch.int8), torch.zeros((32, 256), dtype=torch.int8)
    s_tok, s_ch = torch.ones(4), torch.ones(32)
    out = torch.empty((4, 32), dtype=torch.float16)
    for scales in ((None, s_ch), (s_tok, None), (None, None)):
        for y in (None, out):
            with pytest.raises(TypeError):
                ops.w8a8_gemm(a, scales[0], w, scales[1], out=y)
