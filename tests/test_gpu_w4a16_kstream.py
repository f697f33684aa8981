"""The K-streaming MFMA kernel: fp16 x int4 products of 2 .. 64 rows and of blocks of up to 64 (w4a16_kstream.hip).

Sizes at its edges: rows around the blocks of 16, one column tile up to six a workgroup, columns that are no multiple of 16 (the
last tile is moved back), a single group for the last chunk, an odd number of groups (scale rows that start in the middle of
a word), all 64 groups of the longest range, ranges of K that end unevenly.  Every product also runs without
synchronisation words (one range of K, or the kernel that served it before).
Tolerance, of the result's RMS: the output's rounding, 2^-11 of up to 5.5 RMS, 2.7e-3, and a bias's and a residual's once more; with
RMSNorm weights times gamma rounded to eleven bits, 2^-11 / sqrt(3) in the 2-norm at most and 5.5 of that, 1.6e-3: 5e-3 (SiLU-gate: two rounded
products multiplied, values up to some ten RMS, 2e-2).
"""
import numpy as np
import pytest

import oracle
from nnfusion_amd import datagen

pytestmark = pytest.mark.gpu

TOL = 5e-3


def _t(gpu, *arrays):
    import torch

    return [None if a is None else torch.from_numpy(np.ascontiguousarray(a)).to(gpu) for a in arrays]


def _check(y, ref, tol=TOL):
    y = y.cpu().numpy().astype(np.float32)
    assert np.isfinite(y).all()
    err = float(np.abs(y - ref.astype(np.float32)).max())
    rms = float(np.sqrt(np.mean(np.asarray(ref, np.float64) ** 2)))
    assert err <= tol * max(rms, 1e-6), (err, rms)


def _ws(gpu, nbytes=64 << 20):
    import torch

    return torch.empty(nbytes, dtype=torch.uint8, device=gpu)


@pytest.mark.parametrize("m,n,k", [
    (17, 16, 1152), (32, 48, 2176), (33, 40, 1152), (48, 4096, 1024), (49, 520, 4096), (64, 4112, 1280), (64, 24576, 1024), (63, 300, 8192),
    (8, 40, 1792), (11, 4096, 1152), (16, 4112, 1408), (13, 2064, 7936), (10, 4096, 3968), (16, 12288, 3712), (8, 24576, 1792),
    (65, 520, 2048), (128, 4104, 1408), (130, 1000, 4096), (257, 1040, 1152), (1000, 272, 1280), (90, 2048, 8448), (200, 1024, 9216), (45, 8200, 2048), (20, 12288, 1280), (40, 640, 11008), (33, 4096, 11008), (64, 1030, 9984), (29, 256, 8448), (50, 2048, 1664)])
@pytest.mark.parametrize("with_sync", [True, False], ids=["sync", "no-sync"])
def test_products(gpu, m, n, k, with_sync):
    import torch

    from nnfusion_amd import ops

    print(f"case kstream M={m} N={n} K={k} sync={with_sync}", flush=True)
    a, wq, s = datagen.w4a16_case(3, m, n, k)
    ta, tw, ts = _t(gpu, a, wq, s)
    sync = ops.sync_flags(gpu) if with_sync else None
    ws = _ws(gpu)
    ref = oracle.w4a16_gemm(a, wq, s, f32_out=True)
    y = ops.wna16_gemm(ta, tw, ts, workspace=ws, sync=sync)
    _check(y, ref)
    again = ops.wna16_gemm(ta, tw, ts, workspace=ws, sync=sync)
    torch.cuda.synchronize()
    assert torch.equal(y, again)
    assert sync is None or int(sync.count_nonzero()) == 0


@pytest.mark.parametrize("zp", [0, 15])
def test_zero_points(gpu, zp):
    from nnfusion_amd import ops

    a, wq, s = datagen.w4a16_case(5, 45, 200, 2304)
    ta, tw, ts = _t(gpu, a, wq, s)
    _check(ops.w4a16_gemm(ta, tw, ts, zp=zp, workspace=_ws(gpu)), oracle.w4a16_gemm(a, wq, s, zp=zp, f32_out=True))


@pytest.mark.parametrize("m,n,k", [(45, 200, 1152), (64, 4128, 2048), (31, 72, 4096), (48, 1024, 9216), (9, 1000, 2688), (16, 4096, 7936), (100, 1032, 2048), (150, 1024, 8704)])
def test_bias_and_residual_in_place(gpu, m, n, k):
    from nnfusion_amd import ops

    a, wq, s = datagen.w4a16_case(7, m, n, k)
    rng = np.random.default_rng(1)
    bias = rng.standard_normal(n).astype(np.float16)
    resid = rng.standard_normal((m, n)).astype(np.float16)
    ta, tw, ts, tb, out = _t(gpu, a, wq, s, bias, resid)
    ops.w4a16_gemm_fused(ta, tw, ts, bias=tb, residual=out, out=out, workspace=_ws(gpu), sync=ops.sync_flags(gpu))
    ref = oracle.add_f16(oracle.add_f16(oracle.w4a16_gemm(a, wq, s), np.broadcast_to(bias, (m, n))), resid)
    _check(out, ref)


@pytest.mark.parametrize("gate", [False, True], ids=["plain", "silu-gate"])
@pytest.mark.parametrize("m,n,k,spread", [(45, 300, 1152, 1.0), (64, 8200, 1024, 1.0), (33, 2048, 8192, 1.0), (20, 40, 2176, 1.0), (48, 512, 2048, 3000.0),
                                              (4, 40, 1152, 1.0), (16, 2050, 2560, 1.0), (9, 8192, 1280, 1.0), (16, 512, 1280, 3000.0), (70, 1030, 1152, 1.0), (200, 512, 2048, 1.0)])
def test_rms_norm(gpu, m, n, k, spread, gate):
    """spread: of the RMSNorm weight.  At 3000 neither gamma times an activation (up to 80) nor gamma times a weight of 15 is an fp16 number."""
    from nnfusion_amd import ops

    a, wq, s = datagen.w4a16_case(9, m, 2 * n if gate else n, k)
    if spread > 1:
        a, s = (a.astype(np.float32) * 20).astype(np.float16), (s.astype(np.float32) / spread).astype(np.float16)
    gamma = (spread * (1.0 + 0.1 * np.random.default_rng(2).standard_normal(k))).astype(np.float16)
    ta, tw, ts, tg = _t(gpu, a, wq, s, gamma)
    y = ops.w4a16_gemm_fused(ta, tw, ts, rms_gamma=tg, act=1 if gate else 0, workspace=_ws(gpu), sync=ops.sync_flags(gpu))
    x = a.astype(np.float64)
    x = x / np.sqrt(np.mean(x * x, axis=1, keepdims=True) + 1e-6) * gamma.astype(np.float64)
    ref = x @ oracle.dequantize_w4(wq, s).astype(np.float64).T
    if gate:
        g, u = ref[:, :n], ref[:, n:]
        ref = g / (1.0 + np.exp(-g)) * u
        # the gate and up products are rounded to fp16 and multiplied: twice the relative error of one, on a result with heavier tails
        _check(y, ref, 4 * TOL)
    else:
        _check(y, ref)


@pytest.mark.parametrize("m,n,k", [(4, 40, 1152), (16, 2050, 2560), (45, 300, 1152)])
def test_small_rms_norm_weight(gpu, m, n, k):
    """gamma of about 2^-14, where a fraction of a weight times it has few bits in fp16 (of a sixteenth six: 4e-3 of the 2-norm).  Bound: weights times
    gamma and the output rounded to eleven bits, 2^-11 / sqrt(3) each at most; the output, 2^-24 apart below 2^-14."""
    from nnfusion_amd import ops

    a, wq, s = datagen.w4a16_case(9, m, n, k)
    gamma = ((1.0 + 0.1 * np.random.default_rng(2).standard_normal(k)) / 16384).astype(np.float16)
    ta, tw, ts, tg = _t(gpu, a, wq, s, gamma)
    y = ops.w4a16_gemm_fused(ta, tw, ts, rms_gamma=tg, workspace=_ws(gpu), sync=ops.sync_flags(gpu)).cpu().numpy().astype(np.float64)
    x = a.astype(np.float64)
    x = x / np.sqrt(np.mean(x * x, axis=1, keepdims=True) + 1e-6) * gamma.astype(np.float64)
    q = oracle.dequantize_w4(wq, np.ones_like(s)).astype(np.float64)
    ref = x @ (q * np.repeat(s.astype(np.float64), 128, axis=1)).T
    assert np.linalg.norm(y - ref) <= (np.sqrt(2 / 3) * 2.0 ** -11 + 2.0 ** -24 / np.sqrt(12 * np.mean(ref ** 2))) * np.linalg.norm(ref)


@pytest.mark.parametrize("m,n,k", [(4, 40, 1152), (16, 2050, 2560), (45, 300, 1152), (70, 72, 1024)])
@pytest.mark.parametrize("form", ["outliers", "small"])
def test_rms_norm_weights_of_any_size(gpu, form, m, n, k):
    """Weights times gamma on both sides of fp16's range.  outliers: one gamma in 64 of 30000 (up to 15 times that a weight), in every other group of
    128 only; small: gamma of 6e-5.  2-norm of the error: a weight times gamma and the output are rounded to eleven bits each, 2^-11 / sqrt(3) at
    most; the output's own spacing of 2^-24 where it is a subnormal number."""
    from nnfusion_amd import ops

    print(f"case gamma {form} M={m} N={n} K={k}", flush=True)
    a, wq, s = datagen.w4a16_case(9, m, n, k)
    rng = np.random.default_rng(6)
    gamma = 6e-5 * (1.0 + 0.1 * rng.standard_normal(k))
    if form == "outliers":
        gamma = gamma / 6e-2
        gamma.reshape(-1, 128)[::2, 5::64] *= 3e7
        s = (s.astype(np.float32) / 16).astype(np.float16)
    gamma = gamma.astype(np.float16)
    ta, tw, ts, tg = _t(gpu, a, wq, s, gamma)
    y = ops.w4a16_gemm_fused(ta, tw, ts, rms_gamma=tg, workspace=_ws(gpu), sync=ops.sync_flags(gpu)).cpu().numpy().astype(np.float64)
    x = a.astype(np.float64)
    x = x / np.sqrt(np.mean(x * x, axis=1, keepdims=True) + 1e-6) * gamma.astype(np.float64)
    q = oracle.dequantize_w4(wq, np.ones_like(s)).astype(np.float64)
    ref = x @ (q * np.repeat(s.astype(np.float64), 128, axis=1)).T
    assert np.abs(ref).max() < 60000.0
    assert np.isfinite(y).all()
    subnormal = 2.0 ** -24 / np.sqrt(12 * np.mean(ref ** 2))
    assert np.linalg.norm(y - ref) <= (np.sqrt(2 / 3) * 2.0 ** -11 + subnormal) * np.linalg.norm(ref)
