"""The K-streaming MFMA kernel on 8-bit weights in groups of 32 / 64 / 128 (w8a16_kstream_q{5,6,7}.hip), and on 4-bit weights whose rows hold an odd
number of groups of 128 (scales of every other row start in the middle of a word).

Sizes at the kernel's edges: rows around the blocks of 16 and blocks of rows, columns that are no multiple of 16, one to six tiles a workgroup
(bytes of zero points come 64 a load, four a tile row with groups of 32), chunks with a single group, long K, odd numbers of columns (groups of
128 in odd numbers go elsewhere then).  Tolerance, of the result's RMS: the output's rounding, 2^-11 of up to 5.5 RMS, 2.7e-3, and a residual's
once more; weights, and weights times gamma, rounded to eleven bits each, 2^-11 / sqrt(3) in the 2-norm at most and 5.5 of that, 2.2e-3: 5e-3
(SiLU-gate: two rounded products multiplied, values up to some ten RMS, 2e-2).
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


def _check(y, ref, tol):
    y = y.cpu().numpy().astype(np.float32)
    assert np.isfinite(y).all()
    err = float(np.abs(y - ref.astype(np.float32)).max())
    rms = float(np.sqrt(np.mean(np.asarray(ref, np.float64) ** 2)))
    assert err <= tol * max(rms, 1e-6), (err, rms)


@pytest.mark.parametrize("zero_points", [True, False], ids=["zero-points", "scalar"])
@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize("bits,m,n,k,form", [
    (8, 2, 40, 1280, "plain"), (8, 16, 4112, 1536, "plain"), (8, 7, 8200, 2816, "residual"), (8, 12, 4096, 11008, "residual"),
    (8, 17, 16, 1024, "plain"), (8, 33, 528, 2048, "residual"), (8, 49, 12288, 1024, "plain"), (8, 16, 24576, 1280, "plain"),
    (8, 100, 1032, 2304, "plain"), (8, 300, 272, 1280, "residual"), (8, 5, 300, 1152, "rms"), (8, 9, 6144, 4096, "rms"), (8, 31, 72, 2432, "rms"),
    (8, 64, 4128, 1280, "rms"), (8, 3, 2056, 1664, "gate"), (8, 16, 300, 8192, "gate"), (8, 45, 4100, 1024, "gate"), (8, 9, 301, 1152, "plain"),
    (4, 5, 300, 1152, "plain"), (4, 20, 4130, 1664, "residual"), (4, 64, 272, 11136, "rms"), (4, 9, 302, 2432, "gate"), (4, 9, 301, 1152, "plain")])
def test_products(gpu, bits, m, n, k, form, group, zero_points):
    import torch

    from nnfusion_amd import ops

    print(f"case kstream_q bits={bits} M={m} N={n} K={k} {form} group={group} zero_points={zero_points}", flush=True)
    zp = 7 if bits == 4 else 119
    gate, rms = form == "gate", form in ("rms", "gate")
    rows = 2 * n if gate else n
    a, wq, s, z = datagen.wna16_case(5, m, rows, k, bits, group, zero_points)
    rng = np.random.default_rng(3)
    gamma = (1.0 + 0.1 * rng.standard_normal(k)).astype(np.float16) if rms else None
    resid = rng.standard_normal((m, n)).astype(np.float16) if form == "residual" else None
    ta, tw, ts, tz, tg, tr = _t(gpu, a, wq, s, z, gamma, resid)
    w = oracle.dequantize_wn(wq, s, bits, group, zp, z).astype(np.float64)
    x = a.astype(np.float64)
    if rms:
        x = x / np.sqrt(np.mean(x * x, axis=1, keepdims=True) + 1e-6) * gamma.astype(np.float64)
    ref = x @ w.T
    if gate:
        ref = ref[:, :n] / (1.0 + np.exp(-ref[:, :n])) * ref[:, n:]
    if resid is not None:
        ref = ref + resid.astype(np.float64)
    if form == "plain":
        y = ops.wna16_gemm(ta, tw, ts, bits, group, zp, tz)
        again = ops.wna16_gemm(ta, tw, ts, bits, group, zp, tz)
    else:
        y = ops.wna16_gemm_fused(ta, tw, ts, bits, group, zp, tz, rms_gamma=tg, residual=tr, act=1 if gate else 0)
        out = tr.clone() if tr is not None else None  # the residual in place
        again = ops.wna16_gemm_fused(ta, tw, ts, bits, group, zp, tz, rms_gamma=tg, residual=out, act=1 if gate else 0, out=out)
    torch.cuda.synchronize()
    assert torch.equal(y, again)
    _check(y, ref, 4 * TOL if gate else TOL)


@pytest.mark.parametrize("bits,group,m,n,k,gate", [(4, 32, 40, 72, 4096, False), (4, 64, 64, 40, 1280, True), (4, 128, 16, 300, 2304, True),
                                                   (8, 32, 5, 300, 1152, False), (8, 128, 45, 72, 4096, False), (8, 64, 9, 302, 2560, True)])
def test_small_rms_norm_weight(gpu, bits, group, m, n, k, gate):
    """A weight's scale times gamma of 7.7e-7 (8 bits: 4.8e-8), where fp16 keeps a few bits of a weight.  The 2-norm of the error: the roundings of
    the weight times its scale, of that times gamma (both away from fp16's ends, by a power of two) and of the output, 2^-11 / sqrt(3) each at most,
    2^-11 in all, twice that behind SiLU-gate (3.2e-3 for a product as it is), and the output's own spacing of 2^-24 where it is a subnormal number."""
    from nnfusion_amd import ops

    print(f"case small gamma bits={bits} group={group} M={m} N={n} K={k} gate={gate}", flush=True)
    zp = 7 if bits == 4 else 119
    a, wq, s, z = datagen.wna16_case(6, m, 2 * n if gate else n, k, bits, group, True)
    s = (s.astype(np.float32) / 16).astype(np.float16)
    if gate: # (the product of the two within the range of fp16)
        s[n:] = (s[n:].astype(np.float32) * 512).astype(np.float16)
    gamma = ((1.0 + 0.1 * np.random.default_rng(4).standard_normal(k)) / 1024).astype(np.float16)
    ta, tw, ts, tz, tg = _t(gpu, a, wq, s, z, gamma)
    x = a.astype(np.float64)
    x = x / np.sqrt(np.mean(x * x, axis=1, keepdims=True) + 1e-6) * gamma.astype(np.float64)
    q = oracle.dequantize_wn(wq, np.ones_like(s), bits, group, zp, z).astype(np.float64)
    ref = x @ (q * np.repeat(s.astype(np.float64), group, axis=1)).T
    if gate:
        ref = ref[:, :n] / (1.0 + np.exp(-ref[:, :n])) * ref[:, n:]
    y = ops.wna16_gemm_fused(ta, tw, ts, bits, group, zp, tz, rms_gamma=tg, act=1 if gate else 0).cpu().numpy().astype(np.float64)
    assert np.linalg.norm(y - ref) <= ((2 if gate else 1) * 2.0 ** -11 + 2.0 ** -24 / np.sqrt(12 * np.mean(ref ** 2))) * np.linalg.norm(ref)


@pytest.mark.parametrize("bits,group,m,n,k,gate", [(4, 32, 40, 72, 1024, False), (4, 64, 45, 40, 1280, True), (4, 128, 64, 300, 1152, False),
                                                   (8, 32, 5, 300, 1152, True), (8, 64, 40, 72, 2304, False), (8, 128, 9, 302, 1024, False)])
@pytest.mark.parametrize("form", ["outliers", "scales", "small"])
def test_rms_norm_weights_and_scales_of_any_size(gpu, form, bits, group, m, n, k, gate):
    """Weights times gamma on both sides of fp16's range (scales: of 4 bits, 1 / 16 of them with 8).  outliers: one gamma in 64 of 3000, scales up
    to 0.1; scales of 150 .. 300 with gamma of 1e-2; scales of 2e-3 .. 4e-3 with gamma of 6e-5.  2-norm of the error: a weight, that times gamma and
    the output are rounded to eleven bits each, 2^-11 / sqrt(3) at most, 2^-11 in all; a gate: of two products multiplied, twice that; the output's
    own spacing of 2^-24 where it is a subnormal number."""
    from nnfusion_amd import ops

    print(f"case gamma {form} bits={bits} group={group} M={m} N={n} K={k} gate={gate}", flush=True)
    zp = 7 if bits == 4 else 119
    a, wq, _, z = datagen.wna16_case(8, m, 2 * n if gate else n, k, bits, group, True)
    rng = np.random.default_rng(5)
    low, high, gamma = {"outliers": (0.05, 0.1, 1.0), "scales": (150.0, 300.0, 1e-2), "small": (2e-3, 4e-3, 6e-5)}[form]
    s = (rng.uniform(low, high, (wq.shape[0], k // group)) / (1 if bits == 4 else 16)).astype(np.float16)
    gamma = gamma * (1.0 + 0.1 * rng.standard_normal(k))
    if form == "outliers":
        gamma[5::64] *= 3000.0
    gamma = gamma.astype(np.float16)
    if gate: # (products of a gate of about one and up: within the range of fp16)
        s[:n] = (s[:n].astype(np.float32) * {"outliers": 2.0 ** -14, "scales": 2.0 ** -8, "small": 2.0 ** 14}[form]).astype(np.float16)
    ta, tw, ts, tz, tg = _t(gpu, a, wq, s, z, gamma)
    x = a.astype(np.float64)
    x = x / np.sqrt(np.mean(x * x, axis=1, keepdims=True) + 1e-6) * gamma.astype(np.float64)
    q = oracle.dequantize_wn(wq, np.ones_like(s), bits, group, zp, z).astype(np.float64)
    ref = x @ (q * np.repeat(s.astype(np.float64), group, axis=1)).T
    if gate:
        ref = ref[:, :n] / (1.0 + np.exp(-ref[:, :n])) * ref[:, n:]
    assert np.abs(ref).max() < 60000.0
    y = ops.wna16_gemm_fused(ta, tw, ts, bits, group, zp, tz, rms_gamma=tg, act=1 if gate else 0).cpu().numpy().astype(np.float64)
    assert np.isfinite(y).all()
    subnormal = 2.0 ** -24 / np.sqrt(12 * np.mean(ref ** 2))
    assert np.linalg.norm(y - ref) <= ((2 if gate else 1) * 2.0 ** -11 + subnormal) * np.linalg.norm(ref)
