"""The K-streaming W8A8 kernel (w8a8_kstream.hip): 2 .. 64 rows and blocks of up to 64.

Sizes at its edges: rows around the blocks of 16, columns that are no multiple of 16 (the last tile is moved back), one to six tiles a
workgroup (five and six with four blocks of rows: their sums meet in two rounds), K that is no multiple of 256 (half the bytes a wavefront and chunk), a single wavefront in the last chunk, chunks that wrap around.
The int32 accumulators are exact; the fp16 results follow from them by the oracle's formula, bit for bit.
"""
import numpy as np
import pytest

import oracle
from nnfusion_amd import datagen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [
    (2, 16, 1024), (16, 4112, 1152), (7, 40, 8192), (9, 8200, 2048), (17, 528, 2176), (32, 8192, 4096), (33, 24576, 1024), (48, 300, 5504), (64, 4100, 1280),
    (65, 520, 2048), (130, 1000, 1152), (200, 2056, 1024), (300, 272, 4096), (1000, 144, 1152), (45, 12296, 1408), (64, 16384, 1024),
    (100, 8208, 1024), (128, 12288, 1152), (64, 24560, 1024), (16, 24560, 1152), (30, 20000, 1024)])
def test_products(gpu, m, n, k):
    import torch

    from nnfusion_amd import ops

    print(f"case w8a8 kstream M={m} N={n} K={k}", flush=True)
    a, s_tok, w, s_ch = datagen.w8a8_case(3, m, n, k)
    t = [torch.from_numpy(np.ascontiguousarray(x)).to(gpu) for x in (a, s_tok, w, s_ch)]
    acc = oracle.w8a8_acc(a, w)
    assert np.array_equal(ops.w8a8_gemm_acc(t[0], t[2]).cpu().numpy(), acc)
    y = ops.w8a8_gemm(*t)
    again = ops.w8a8_gemm(*t)
    torch.cuda.synchronize()
    assert torch.equal(y, again)
    assert np.array_equal(y.cpu().numpy().view(np.uint16), oracle.w8a8_epilogue(acc, s_tok, s_ch).view(np.uint16))
