"""The row-streaming MFMA kernel with K a compile-time constant (w4a16_mrows.hip): activations in blocks of 4, 8 and 16 rows.

Rows on both sides of a block's size, every number of blocks a wavefront brings in (1 .. 8, of which two, four or eight are in
flight), the ends of the run-time K that two to seven rows take to it (1280, 1792, 6400, 7936), a last tile that is moved back, and -- 22016 columns and more -- more outputs a thread than the two whose residual is asked
for ahead.  Tolerance, of the result's RMS: the output's rounding, 2^-11 of up to 5.5 RMS, 2.7e-3, and a residual's once more; with RMSNorm
activations times gamma rounded to eleven bits, 2^-11 / sqrt(3) in the 2-norm at most and 5.5 of that, 1.6e-3: 5e-3 (SiLU-gate: two
rounded products multiplied, values up to some ten RMS, 2e-2).
"""
import numpy as np
import pytest

import oracle
from nnfusion_amd import datagen

pytestmark = pytest.mark.gpu

TOL = 5e-3


def _check(y, ref, tol=TOL):
    y = y.cpu().numpy().astype(np.float32)
    assert np.isfinite(y).all()
    err = float(np.abs(y - ref.astype(np.float32)).max())
    rms = float(np.sqrt(np.mean(np.asarray(ref, np.float64) ** 2)))
    assert err <= tol * max(rms, 1e-6), (err, rms)


@pytest.mark.parametrize("m,n,k", [(4, 40, 1024), (5, 300, 2048), (8, 1000, 3072), (9, 520, 4096), (2, 4104, 6144), (4, 300, 8192), (8, 72, 8192),
                                   (16, 300, 8192), (3, 520, 1280), (7, 300, 1792), (2, 1000, 6400), (7, 300, 7936), (7, 24584, 1024), (16, 22016, 2048), (17, 300, 1024)])
@pytest.mark.parametrize("form", ["plain", "residual", "rms", "rms-residual", "rms-gate"])
def test_blocks_of_activations(gpu, form, m, n, k):
    import torch

    from nnfusion_amd import ops

    print(f"case mrows {form} M={m} N={n} K={k}", flush=True)
    gate = form == "rms-gate"
    n_out = n // 2 // 8 * 8 if gate else n
    a, wq, s = datagen.w4a16_case(11, m, 2 * n_out if gate else n, k)
    rng = np.random.default_rng(m * k + n)
    gamma = (rng.standard_normal(k) * 0.1 + 1).astype(np.float16) if "rms" in form else None
    residual = rng.standard_normal((m, n_out)).astype(np.float16) if "residual" in form else None
    x = oracle.rmsnorm_f16(a, gamma, 1e-6) if gamma is not None else a
    ref = oracle.w4a16_gemm(x, wq, s, f32_out=True).astype(np.float32)
    if gate:
        g, u = ref[:, :n_out], ref[:, n_out:]
        ref = g / (1 + np.exp(-g)) * u
    if residual is not None:
        ref = ref + residual.astype(np.float32)
    t = [None if v is None else torch.from_numpy(np.ascontiguousarray(v)).to(gpu) for v in (a, wq, s, gamma, residual)]
    y = ops.w4a16_gemm_fused(t[0], t[1], t[2], rms_gamma=t[3], residual=t[4], act=1 if gate else 0)
    _check(y, ref, 2e-2 if gate else TOL)
    if residual is not None:  # in place
        ops.w4a16_gemm_fused(t[0], t[1], t[2], rms_gamma=t[3], residual=t[4], out=t[4])
        assert torch.equal(t[4], y)
