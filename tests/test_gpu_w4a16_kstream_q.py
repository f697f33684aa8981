"""The K-streaming MFMA kernel for 4-bit weights in groups of 32 / 64 / 128 with a scalar zero point or one per (row, group)
(w4a16_kstream_q{5,6,7}.hip): products of 2 .. 512 rows, with RMSNorm, residual and SiLU-gate inside.

Sizes at the kernel's edges, as in test_gpu_w4a16_kstream.py: rows around the blocks of 16 and blocks of rows, columns that are no multiple of 16,
one to six tiles a workgroup (scales of four tiles come in one load, of two with groups of 32), chunks with a single group, long K; five tiles of
four blocks of rows with RMSNorm, which take it as a launch ahead.
Tolerance, of the result's RMS: the output's rounding, 2^-11 of up to 5.5 RMS, 2.7e-3, and a residual's or bias's once more; weights, and weights times
gamma, rounded to eleven bits each, 2^-11 / sqrt(3) in the 2-norm at most and 5.5 of that, 2.2e-3: 5e-3 (SiLU-gate: two rounded
products multiplied, values up to some ten RMS, 2e-2; in half a million of them some reach 40 RMS, so the roundings of gate, up and output, 2^-11 of
the value each, count by the value besides).
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


def _check(y, ref, tol, rel=0.0):
    y = y.cpu().numpy().astype(np.float32)
    assert np.isfinite(y).all()
    err = float((np.abs(y - ref.astype(np.float32)) - rel * np.abs(ref)).max())
    rms = float(np.sqrt(np.mean(np.asarray(ref, np.float64) ** 2)))
    assert err <= tol * max(rms, 1e-6), (err, rms)


@pytest.mark.parametrize("zero_points", [True, False], ids=["zero-points", "scalar"])
@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize("m,n,k,form", [
    (2, 40, 1280, "plain"), (16, 4112, 1536, "plain"), (7, 8200, 2816, "residual"), (12, 4096, 11008, "residual"), (17, 16, 1024, "plain"),
    (33, 528, 2048, "residual"), (49, 12288, 1024, "plain"), (64, 24576, 1280, "plain"), (100, 1032, 2304, "plain"), (300, 272, 1280, "residual"),
    (5, 300, 1280, "rms"), (9, 6144, 4096, "rms"), (31, 72, 2304, "rms"), (64, 4128, 1280, "rms"), (3, 2056, 1536, "gate"), (16, 300, 8192, "gate"),
    (45, 8200, 1024, "gate"), (130, 500, 1280, "gate"), (64, 16380, 1152, "rms"), (48, 24560, 1024, "rms"), (40, 12280, 1152, "gate"),
    (64, 20480, 1280, "rms")])
def test_products(gpu, m, n, k, form, group, zero_points):
    import torch

    from nnfusion_amd import ops

    print(f"case kstream_q M={m} N={n} K={k} {form} group={group} zero_points={zero_points}", flush=True)
    gate, rms = form == "gate", form in ("rms", "gate")
    rows = 2 * n if gate else n
    a, wq, s, z = datagen.wna16_case(5, m, rows, k, 4, group, zero_points)
    rng = np.random.default_rng(3)
    gamma = (1.0 + 0.1 * rng.standard_normal(k)).astype(np.float16) if rms else None
    resid = rng.standard_normal((m, n)).astype(np.float16) if form == "residual" else None
    ta, tw, ts, tz, tg, tr = _t(gpu, a, wq, s, z, gamma, resid)
    w = oracle.dequantize_wn(wq, s, 4, group, 7, z).astype(np.float64)
    x = a.astype(np.float64)
    if rms:
        x = x / np.sqrt(np.mean(x * x, axis=1, keepdims=True) + 1e-6) * gamma.astype(np.float64)
    ref = x @ w.T
    if gate:
        ref = ref[:, :n] / (1.0 + np.exp(-ref[:, :n])) * ref[:, n:]
    if resid is not None:
        ref = ref + resid.astype(np.float64)
    if form == "plain":
        y = ops.wna16_gemm(ta, tw, ts, 4, group, 7, tz)
        again = ops.wna16_gemm(ta, tw, ts, 4, group, 7, tz)
    else:
        y = ops.wna16_gemm_fused(ta, tw, ts, 4, group, 7, tz, rms_gamma=tg, residual=tr, act=1 if gate else 0)
        out = tr.clone() if tr is not None else None  # the residual in place
        again = ops.wna16_gemm_fused(ta, tw, ts, 4, group, 7, tz, rms_gamma=tg, residual=out, act=1 if gate else 0, out=out)
    torch.cuda.synchronize()
    assert torch.equal(y, again)
    _check(y, ref, 4 * TOL if gate else TOL, 3 * 2.0 ** -11 if gate else 0.0)
