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


def _operands(m=4, n=32, k=256):
    return (torch.zeros((m, k), dtype=torch.float16), torch.zeros((n, k // 2), dtype=torch.uint8),
            torch.ones((n, k // 128), dtype=torch.float16))


def _strided(t):
    return torch.cat([t, t], dim=1)[:, ::2]


@pytest.mark.parametrize("call", [ops.w4a16_gemm, ops.wna16_gemm])
def test_products_refuse_operands_they_would_misread(call):
    a, wq, s = _operands()
    bad = {
        "fp32 activations": (a.float(), wq, s), "signed weights": (a, wq.to(torch.int8), s), "fp32 scales": (a, wq, s.float()),
        "strided activations": (_strided(a), wq, s), "strided weights": (a, _strided(wq), s), "strided scales": (a, wq, _strided(s)),
        "weights of another K": (a, wq[:, :64].contiguous(), s), "scales of fewer rows": (a, wq, s[:31].contiguous()),
        "scales of another group": (a, wq, s[:, :1].contiguous()),
    }
    for what, operands in bad.items():
        with pytest.raises(AssertionError):
            call(*operands)
            pytest.fail(what)
    for operands, error in (((a[0], wq, s), ValueError), ((a, wq, s[0]), ValueError), ((None, wq, s), TypeError), ((a, wq.numpy(), s), TypeError)):
        with pytest.raises(error):
            call(*operands)
    for group, error in ((1 << 40, OverflowError), (0, AssertionError), ("128", TypeError)):
        with pytest.raises(error):
            call(a, wq, s, group=group)


def test_zero_points_are_checked():
    a, wq, s = _operands()
    good = torch.zeros((32, 1), dtype=torch.uint8)  # two 4-bit zero points of a row
    for z in (good.to(torch.int8), torch.zeros((32, 2), dtype=torch.uint8), good[:31].contiguous(), good.reshape(-1),
              torch.zeros((32, 2), dtype=torch.uint8)[:, ::2]):
        with pytest.raises(AssertionError):
            ops.wna16_gemm(a, wq, s, zero_points=z)


def test_other_calls_refuse_wrong_types():
    a = torch.zeros((4, 64), dtype=torch.float16)
    i8 = torch.zeros((4, 256), dtype=torch.int8)
    scales = torch.ones(4)
    for f in (lambda: ops.w8a8_gemm(i8.to(torch.uint8), scales, i8, scales), lambda: ops.w8a8_gemm(i8, scales.double(), i8, scales),
              lambda: ops.w8a8_gemm(i8, scales, i8, scales.half()), lambda: ops.w8a8_gemm_acc(i8, i8.short()),
              lambda: ops.elementwise("add", a.float(), a.float()), lambda: ops.elementwise("add", a, a.float()),
              lambda: ops.elementwise("add", a, a[:2]), lambda: ops.elementwise("add", a.t(), a.t()),
              lambda: ops.elementwise("add", a, torch.zeros((1, 64), dtype=torch.float16))):
        with pytest.raises(AssertionError):
            f()


@pytest.mark.gpu
def test_status_of_the_library_becomes_an_error(gpu):
    a, wq, s = (t.to(gpu) for t in _operands())
    small = torch.empty(16, dtype=torch.uint8, device=gpu)
    for f, status in ((lambda: ops.w4a16_gemm(a, wq, s, zp=16), -2),
                      (lambda: ops.w4a16_gemm_fused(torch.cat([a] * 64), wq, s, rms_gamma=a[0], workspace=small), -3),
                      (lambda: ops.elementwise("add", a), -1)):
        with pytest.raises(ops.NnfError) as e:
            f()
        assert e.value.status == status


@pytest.mark.gpu
def test_calls_on_a_side_stream_are_ordered_there(gpu):
    """Inputs are written, and results read, by work of the side stream alone: a call that went to another stream would read the
    zeros the input held before (the copy that fills it waits behind some milliseconds of other work of its stream)."""
    gen = torch.Generator(device=gpu).manual_seed(3)
    m, n, k = 45, 1024, 4096
    src = torch.randn((m, k), generator=gen, device=gpu, dtype=torch.float16)
    wq = torch.randint(0, 256, (n, k // 2), generator=gen, device=gpu, dtype=torch.uint8)
    s = torch.rand((n, k // 128), generator=gen, device=gpu).mul_(0.01).add_(0.005).half()
    res = torch.randn((m, n), generator=gen, device=gpu, dtype=torch.float16)
    i8 = torch.randint(-127, 128, (40, k), generator=gen, device=gpu, dtype=torch.int8)
    ones = torch.ones(40, device=gpu)
    busy = torch.randn((4096, 4096), generator=gen, device=gpu)

    def calls(x):
        return (ops.w4a16_gemm(x, wq, s), ops.wna16_gemm(x, wq, s), ops.w4a16_gemm_fused(x, wq, s, rms_gamma=src[0], residual=res),
                ops.wna16_gemm_fused(x, wq, s, residual=res, zp=7), ops.w8a8_gemm(i8, ones, i8, ones), ops.w8a8_gemm_acc(i8, i8),
                ops.elementwise("swish", x), ops.rms_norm(x, src[0]), ops.dequantize(wq, s))

    want = calls(src)
    x = torch.zeros_like(src)
    torch.cuda.synchronize()
    side = torch.cuda.Stream(gpu)
    with torch.cuda.stream(side):
        for _ in range(8):
            busy @ busy
        x.copy_(src)
        got = calls(x)
    side.synchronize()
    assert all(torch.equal(g, w) for g, w in zip(got, want))
