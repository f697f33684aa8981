"""Parity of the fp16 x int4 MFMA GEMM (M > 16) and its fused prologue/epilogues against the CPU oracle.

Tolerance: max|y - y_ref| <= 1e-2 * RMS(y_ref) (stated by the task for the fp16 x int4 path).
Full-size shapes are checked on a sample of output columns (the oracle GEMM of the whole matrix would
take minutes on the host), plus size-independent properties.
"""
import numpy as np
import pytest

import oracle
from nnfusion_amd import datagen

pytestmark = pytest.mark.gpu

TOL = 1e-2


def _t(gpu, *arrays):
    import torch

    return [None if a is None else torch.from_numpy(np.ascontiguousarray(a)).to(gpu) for a in arrays]


def _rms(x):
    return float(np.sqrt(np.mean(np.asarray(x, np.float64) ** 2)))


def _check(y, ref, tol=TOL):
    err = float(np.abs(y.astype(np.float32) - ref.astype(np.float32)).max())
    rms = _rms(ref)
    assert err <= tol * max(rms, 1e-6), (err, rms)


# Plans of the MFMA tile GEMM, passed per call through nnf_w4a16_gemm_variant / nnf_w4a16_gemm_fused_variant (struct
# nnf_plan): None = the library's own choice of kernel and plan; otherwise (tile_rows, k_parts[, tile_cols]): tiles of
# 256, 128, 64 or 32 rows by 256 columns (128 where given: products without SiLU-gate), and the number of workgroups that
# share a tile (each a part of K; parts parked in the workspace and added by the second launch)
PLANS = [None, (256, 1, 256), (256, 2, 256), (128, 1, 256), (128, 3, 256), (64, 1, 256), (64, 2, 256), (32, 1), (32, 3),
         (256, 1, 128), (256, 3, 128), (128, 1, 128), (128, 2, 128), (64, 1, 128), (64, 3, 128)]


@pytest.fixture(params=PLANS, ids=lambda p: "auto" if p is None else "rows%d-parts%d" % p[:2] + ("-cols%d" % p[2] if len(p) > 2 else ""))
def plan(request):
    """Keyword arguments for ops.w4a16_gemm_fused / _gemm below."""
    return {} if request.param is None else {"variant": "gemm_mfma", "plan": request.param}


def _gemm(ta, tw, ts, plan_kw, workspace=None):
    from nnfusion_amd import ops

    if plan_kw:
        return ops.w4a16_gemm_variant(ta, tw, ts, plan_kw["variant"], plan=plan_kw["plan"], workspace=workspace)
    return ops.w4a16_gemm(ta, tw, ts, workspace=workspace)


def _big_ws(gpu):
    import torch

    return torch.empty(64 << 20, dtype=torch.uint8, device=gpu)


@pytest.mark.parametrize("m,n,k", [(200, 300, 1024), (64, 520, 2048), (130, 128, 512), (17, 40, 1280)])
def test_gemm_every_tile_plan_matches_oracle(gpu, plan, m, n, k):
    import torch

    from nnfusion_amd import ops

    print(f"case plan={plan} M={m} N={n} K={k}", flush=True)
    a, wq, s = datagen.w4a16_case(2, m, n, k)
    ta, tw, ts = _t(gpu, a, wq, s)
    y = _gemm(ta, tw, ts, plan, workspace=_big_ws(gpu))
    torch.cuda.synchronize()
    _check(y.cpu().numpy(), oracle.w4a16_gemm(a, wq, s, f32_out=True))


@pytest.mark.parametrize("m,n,k", [
    (128, 256, 128), (256, 256, 256), (17, 32, 128), (100, 96, 384), (300, 520, 1024),
    (512, 1024, 2048), (257, 33, 512), (1024, 512, 4096), (2048, 2048, 512),
])
def test_gemm_matches_oracle(gpu, m, n, k):
    import torch

    from nnfusion_amd import ops

    print(f"case M={m} N={n} K={k}", flush=True)
    a, wq, s = datagen.w4a16_case(0, m, n, k)
    ta, tw, ts = _t(gpu, a, wq, s)
    y = ops.w4a16_gemm(ta, tw, ts)
    torch.cuda.synchronize()
    ref = oracle.w4a16_gemm(a, wq, s, f32_out=True)
    _check(y.cpu().numpy(), ref)


def _random_shapes(count):
    rng = np.random.default_rng(777)
    out = []
    for _ in range(count):
        m = int(rng.choice([1, 2, 3, 8, 15, 16, 17, 31, 32, 33, 40, 41, 64, 65, 127, 128, 129, 200, 256, 300, 513]))
        n = int(rng.choice([1, 15, 16, 17, 64, 100, 255, 256, 257, 500, 1000, 1024, 2000, 4096, 5000]))
        k = int(rng.choice([128, 256, 384, 512, 640, 1024, 1152, 2048, 2560, 3072, 4096, 5120, 6144, 7168, 8192, 11008, 14336]))
        if m * n * k > 300 * 2000 * 4096:
            n = 256
        out.append((m, n, k, int(rng.integers(0, 16))))
    return out


@pytest.mark.parametrize("m,n,k,zp", _random_shapes(150))
def test_gemm_random_shapes(gpu, m, n, k, zp):
    """Shapes drawn across the routes of nnf_w4a16_gemm (the row-streaming kernels with a fixed and a run-time K, ranges of
    K, the MFMA GEMV, stream-K tiles of every height), every zero point."""
    import torch

    from nnfusion_amd import ops

    a, wq, s = datagen.w4a16_case(m + 5 * n + 11 * k + zp, m, n, k)
    ta, tw, ts = _t(gpu, a, wq, s)
    y = ops.w4a16_gemm(ta, tw, ts, zp=zp)
    torch.cuda.synchronize()
    ref = oracle.w4a16_gemm(a, wq, s, zp=zp, f32_out=True)
    _check(y.cpu().numpy(), ref)


@pytest.mark.parametrize("m", [1, 5, 16])
def test_gemm_kernel_serves_small_m(gpu, m):
    """The tile GEMM asked for by variant (the library's own choice for these shapes is a GEMV kernel)."""
    import torch

    from nnfusion_amd import ops

    a, wq, s = datagen.w4a16_case(4, m, 320, 512)
    ta, tw, ts = _t(gpu, a, wq, s)
    y = ops.w4a16_gemm_variant(ta, tw, ts, "gemm_mfma", workspace=_big_ws(gpu))
    torch.cuda.synchronize()
    _check(y.cpu().numpy(), oracle.w4a16_gemm(a, wq, s, f32_out=True))


def test_gemm_one_hot_rows_select_weights(gpu):
    """A = rows of the identity  =>  Y[m, n] = fp16((q[n, m] - 8) * s[n, m/128]) exactly:
    pins nibble order, the K-slot permutation shared by the A and W fragments, and scale indexing."""
    import torch

    from nnfusion_amd import ops

    n, k = 160, 256
    _, wq, s = datagen.w4a16_case(5, 1, n, k)
    a = np.eye(k, dtype=np.float16)
    ta, tw, ts = _t(gpu, a, wq, s)
    y = ops.w4a16_gemm(ta, tw, ts).cpu().numpy()
    torch.cuda.synchronize()
    wd = oracle.dequantize_w4(wq, s)  # [n, k]
    np.testing.assert_array_equal(y, wd.T.astype(np.float16))


@pytest.mark.parametrize("m,n,k", [(16, 8192, 8192), (128, 8192, 8192), (1024, 8192, 8192), (4096, 8192, 8192),
                                   (32, 8192, 8192), (16, 22016, 4096), (16, 4096, 11008),
                                   (250, 21000, 1024), (100, 20004, 768), (640, 8192, 4096), (256, 22016, 4096)])
def test_gemm_full_size_sampled_columns(gpu, m, n, k):
    """configs[2] shapes (and batched-decode shapes on the row-streaming kernels: one launch, over ranges of K; and
    products whose tiles fill at least half of the CUs, which run whole tiles, one workgroup each, with ragged rows
    and columns): all M rows, 192 sampled output columns against the oracle; and linearity in A
    on the whole output (Y(2A) == 2 Y(A) bit for bit, as scaling by 2 is exact outside the subnormal range)."""
    import torch

    from nnfusion_amd import ops

    print(f"case M={m} N={n} K={k}", flush=True)
    a, wq, s = datagen.w4a16_case(0, m, n, k)
    ta, tw, ts = _t(gpu, a, wq, s)
    y = ops.w4a16_gemm(ta, tw, ts)
    torch.cuda.synchronize()
    rng = np.random.default_rng(0)
    cols = np.sort(rng.choice(n, 192, replace=False))
    ref = oracle.w4a16_gemm(a, wq[cols], s[cols], f32_out=True)
    _check(y.cpu().numpy()[:, cols], ref)
    # Scaling by two is exact everywhere except where the fp16 result itself is subnormal (no kernel rescales the
    # activations: the nibbles are decoded to exact fp16 integers on the weight side).
    y1 = ops.w4a16_gemm(ta, tw, ts)
    y2 = ops.w4a16_gemm(ta * 2, tw, ts)
    torch.cuda.synchronize()
    normal = y1.abs() >= 2.0 ** -13
    assert torch.equal(y2[normal], (y1 * 2)[normal])


def test_fused_bias_residual(gpu, plan):
    import torch

    from nnfusion_amd import ops

    m, n, k = 200, 288, 512
    a, wq, s = datagen.w4a16_case(6, m, n, k)
    bias = datagen.normal_f16(6, datagen.S_BIAS, (n,))
    res = datagen.normal_f16(6, datagen.S_RES, (m, n))
    ta, tw, ts, tb, tr = _t(gpu, a, wq, s, bias, res)
    ws = _big_ws(gpu)
    y_b = ops.w4a16_gemm_fused(ta, tw, ts, bias=tb, workspace=ws, **plan).cpu().numpy()
    y_r = ops.w4a16_gemm_fused(ta, tw, ts, residual=tr, workspace=ws, **plan).cpu().numpy()
    y_br = ops.w4a16_gemm_fused(ta, tw, ts, bias=tb, residual=tr, workspace=ws, **plan).cpu().numpy()
    torch.cuda.synchronize()
    d = oracle.w4a16_gemm(a, wq, s)  # fp16 tensor of the unfused Dot
    ref_b = oracle.add_f16(d, np.broadcast_to(bias, (m, n)).copy())
    ref_r = oracle.add_f16(d, res)
    ref_br = oracle.add_f16(ref_b, res)
    _check(y_b, ref_b)
    _check(y_r, ref_r)
    _check(y_br, ref_br)


@pytest.mark.parametrize("m,n,k", [(257, 300, 512), (90, 36, 384), (33, 1001, 256)])
def test_fused_bias_residual_ragged_columns(gpu, plan, m, n, k):
    """N not a multiple of 8 (no 16-byte row pieces), M not a multiple of the tile: the element-wise tail of the
    row-major epilogue, with bias and residual."""
    import torch

    from nnfusion_amd import ops

    a, wq, s = datagen.w4a16_case(13, m, n, k)
    bias = datagen.normal_f16(13, datagen.S_BIAS, (n,))
    res = datagen.normal_f16(13, datagen.S_RES, (m, n))
    ta, tw, ts, tb, tr = _t(gpu, a, wq, s, bias, res)
    ws = _big_ws(gpu)
    y = _gemm(ta, tw, ts, plan, workspace=ws).cpu().numpy()
    y_br = ops.w4a16_gemm_fused(ta, tw, ts, bias=tb, residual=tr, workspace=ws, **plan).cpu().numpy()
    torch.cuda.synchronize()
    d = oracle.w4a16_gemm(a, wq, s)
    _check(y, oracle.w4a16_gemm(a, wq, s, f32_out=True))
    _check(y_br, oracle.add_f16(oracle.add_f16(d, np.broadcast_to(bias, (m, n)).copy()), res))


def test_fused_silu_gate_ragged_columns(gpu, plan):
    import torch

    from nnfusion_amd import ops

    m, n, k = 70, 100, 256
    a, wq, s = datagen.w4a16_case(14, m, 2 * n, k)
    ta, tw, ts = _t(gpu, a, wq, s)
    y = ops.w4a16_gemm_fused(ta, tw, ts, act=1, workspace=_big_ws(gpu), **plan).cpu().numpy()
    torch.cuda.synchronize()
    gu = oracle.w4a16_gemm(a, wq, s)
    ref = oracle.silu_mul_f16(np.ascontiguousarray(gu[:, :n]), np.ascontiguousarray(gu[:, n:]))
    err = np.abs(y.astype(np.float32) - ref.astype(np.float32))
    assert y.shape == (m, n)
    assert _rms(err) <= 1e-3 * _rms(ref) and err.max() <= 5e-2 * max(_rms(ref), 1e-3)


def test_fused_rmsnorm_prologue(gpu, plan):
    import torch

    from nnfusion_amd import ops

    m, n, k = 130, 256, 1024
    a, wq, s = datagen.w4a16_case(7, m, n, k)
    gamma = datagen.normal_f16(7, datagen.S_GAMMA, (k,), 1.0, 0.1)
    ta, tw, ts, tg = _t(gpu, a, wq, s, gamma)
    y = ops.w4a16_gemm_fused(ta, tw, ts, rms_gamma=tg, rms_eps=1e-6, workspace=_big_ws(gpu), **plan).cpu().numpy()
    torch.cuda.synchronize()
    xn = oracle.rmsnorm_f16(a, gamma, 1e-6)
    _check(y, oracle.w4a16_gemm(xn, wq, s, f32_out=True))


def test_fused_silu_gate(gpu, plan):
    import torch

    from nnfusion_amd import ops

    m, n, k = 150, 192, 512  # n = intermediate size; weights hold 2n rows (gate then up)
    a, wq, s = datagen.w4a16_case(8, m, 2 * n, k)
    ta, tw, ts = _t(gpu, a, wq, s)
    y = ops.w4a16_gemm_fused(ta, tw, ts, act=1, workspace=_big_ws(gpu), **plan).cpu().numpy()
    torch.cuda.synchronize()
    gu = oracle.w4a16_gemm(a, wq, s)
    g = np.ascontiguousarray(gu[:, :n])
    u = np.ascontiguousarray(gu[:, n:])
    ref = oracle.silu_mul_f16(g, u)
    assert y.shape == (m, n)
    # The stated tolerance applies to the GEMM outputs g and u: delta = 1e-2 * RMS(gu).  It is
    # carried through h = silu(g) * u element-wise: |dh| <= |dh/dg| delta + |dh/du| delta with
    # |dh/dg| <= 1.1 |u| and |dh/du| = |silu(g)|, plus one fp16 rounding of h.
    delta = TOL * _rms(gu)
    g32, u32 = g.astype(np.float32), u.astype(np.float32)
    silu = g32 / (1.0 + np.exp(-g32))
    bound = delta * (1.1 * np.abs(u32) + np.abs(silu)) + np.abs(ref.astype(np.float32)) * 2.0 ** -10 + 1e-6
    err = np.abs(y.astype(np.float32) - ref.astype(np.float32))
    assert np.all(err <= bound), float((err - bound).max())
    # and the typical error is far smaller: RMS of the error within 1e-3 of RMS(h)
    assert _rms(err) <= 1e-3 * _rms(ref)


@pytest.mark.parametrize("m,n,k", [(1, 320, 1024), (5, 320, 1024), (16, 320, 1024), (2, 520, 4096), (24, 320, 2048), (32, 1000, 4096),
                                   (16, 136, 11008), (24, 264, 8192), (7, 320, 3584)])
def test_fused_small_m_goes_through_the_gemv_kernel(gpu, m, n, k):
    """Decode shapes with a prologue / epilogue: the GEMV kernels (M = 1; 2 .. 32 rows in one launch or over ranges of
    K) multiply the RMSNorm weight in themselves and apply rstd, bias, residual and the gate at their flush (over ranges
    of K: in the reduction pass).  The workspace is the one the query asks for: rstd and partial sums, no M x K
    activations and no M x 2N products."""
    import torch

    from nnfusion_amd import ops

    a, wq, s = datagen.w4a16_case(11, m, 2 * n, k)
    gamma = datagen.normal_f16(11, datagen.S_GAMMA, (k,), 1.0, 0.1)
    bias = datagen.normal_f16(11, datagen.S_BIAS, (n,))
    res = datagen.normal_f16(11, datagen.S_RES, (m, n))
    ta, tw, ts, tg, tb, tr = _t(gpu, a, wq, s, gamma, bias, res)
    xn = oracle.rmsnorm_f16(a, gamma, 1e-6)
    # RMSNorm + bias + residual on the first n weight rows
    y = ops.w4a16_gemm_fused(ta, tw[:n].contiguous(), ts[:n].contiguous(), rms_gamma=tg, rms_eps=1e-6, bias=tb,
                             residual=tr).cpu().numpy()
    d = oracle.w4a16_gemm(xn, wq[:n], s[:n])
    ref = oracle.add_f16(oracle.add_f16(d, np.broadcast_to(bias, (m, n)).copy()), res)
    _check(y, ref)
    # RMSNorm + SiLU gate over all 2n rows (gate rows, then up rows)
    yg = ops.w4a16_gemm_fused(ta, tw, ts, rms_gamma=tg, rms_eps=1e-6, act=1).cpu().numpy()
    torch.cuda.synchronize()
    gu = oracle.w4a16_gemm(xn, wq, s)
    # the bound the tolerance of the two products (delta on each of gate and up) leaves on SiLU(gate) * up
    g, u = np.ascontiguousarray(gu[:, :n]), np.ascontiguousarray(gu[:, n:])
    refg = oracle.silu_mul_f16(g, u).astype(np.float32)
    delta = TOL * _rms(gu)
    g32, u32 = g.astype(np.float32), u.astype(np.float32)
    bound = delta * (1.1 * np.abs(u32) + np.abs(g32 / (1.0 + np.exp(-g32)))) + np.abs(refg) * 2.0 ** -10 + 1e-6
    err = np.abs(yg.astype(np.float32) - refg)
    assert _rms(err) <= 1e-3 * _rms(refg) and np.all(err <= bound), float((err - bound).max())


@pytest.mark.parametrize("m", [3, 24, 200])
def test_residual_may_alias_the_output(gpu, m):
    import torch

    from nnfusion_amd import ops

    n, k = 288, 512
    a, wq, s = datagen.w4a16_case(12, m, n, k)
    res = datagen.normal_f16(12, datagen.S_RES, (m, n))
    ta, tw, ts, tr = _t(gpu, a, wq, s, res)
    y = ops.w4a16_gemm_fused(ta, tw, ts, residual=tr, out=tr, workspace=_big_ws(gpu)).cpu().numpy()
    torch.cuda.synchronize()
    _check(y, oracle.add_f16(oracle.w4a16_gemm(a, wq, s), res))


def test_rejects_bad_arguments(gpu):
    import torch

    from nnfusion_amd import ops

    a, wq, s = datagen.w4a16_case(9, 4, 64, 256)
    ta, tw, ts = _t(gpu, a, wq, s)
    with pytest.raises(ops.NnfError) as e:
        ops.w4a16_gemm(ta, tw, ts, zp=16)
    assert e.value.status == -2
    from nnfusion_amd import _lib

    lib = _lib.kernels()
    y = torch.empty((4, 64), dtype=torch.float16, device=gpu)
    args = (ta.data_ptr(), tw.data_ptr(), ts.data_ptr(), y.data_ptr())
    assert lib.nnf_w4a16_gemm(None, *args, 4, 64, 256, 64, 8, None, 0) == -2      # group != 128
    assert lib.nnf_w4a16_gemm(None, *args, 4, 64, 192, 128, 8, None, 0) == -2     # K % group != 0
    assert lib.nnf_w4a16_gemm(None, *args, 0, 64, 256, 128, 8, None, 0) == -1     # empty M
    assert lib.nnf_w4a16_gemm(None, None, *args[1:], 4, 64, 256, 128, 8, None, 0) == -1  # null pointer
    assert lib.nnf_w4a16_gemm(None, args[0] + 2, *args[1:], 4, 64, 256, 128, 8, None, 0) == -1  # misaligned
    assert b"unsupported" in lib.nnf_status_string(-2)


# ---- the fused parts on the kernels that serve a few rows ------------------------------------------------------------
# auto: the library's choice (one row: the row-streaming GEMV; up to 32 rows: the row-streaming MFMA kernel, over ranges
# of K with the reduction pass where K is long; otherwise the MFMA GEMV kernel with a pre-pass and an element-wise
# kernel); gemv_rows / gemv_mfma: that family only, where it takes the shape.
@pytest.mark.parametrize("variant", ["auto", "gemv_rows", "gemv_mfma"])
@pytest.mark.parametrize("m,n,k", [(1, 4096, 4096), (1, 300, 1024), (1, 1000, 11008), (3, 304, 2048), (16, 4096, 4096),
                                   (16, 520, 3584), (8, 1000, 11008), (24, 304, 4096), (24, 1000, 8192), (7, 100, 2176)])
def test_fused_parts_with_few_rows(gpu, variant, m, n, k):
    import torch

    from nnfusion_amd import ops

    print(f"case variant={variant} M={m} N={n} K={k}", flush=True)
    a, wq, s = datagen.w4a16_case(21, m, 2 * n, k)  # 2n weight rows: the gate product uses all, the others the first n
    bias = datagen.normal_f16(21, datagen.S_BIAS, (n,))
    res = datagen.normal_f16(21, datagen.S_RES, (m, n))
    gamma = datagen.normal_f16(21, datagen.S_GAMMA, (k,), 1.0, 0.1)
    ta, tw, ts, tb, tr, tg = _t(gpu, a, wq, s, bias, res, gamma)
    tw1, ts1 = tw[:n].contiguous(), ts[:n].contiguous()
    kw = {} if variant == "auto" else {"variant": variant}
    ws = _big_ws(gpu)

    def run(w, sc, **fused):
        try:
            return ops.w4a16_gemm_fused(ta, w, sc, workspace=ws, **fused, **kw)
        except ops.NnfError as e:
            assert e.status == -2 and variant != "auto"  # this family does not take the shape
            return None

    d = oracle.w4a16_gemm(a, wq[:n], s[:n])  # fp16 tensor of the unfused Dot
    ref_b = oracle.add_f16(d, np.broadcast_to(bias, (m, n)).copy())
    y = run(tw1, ts1, bias=tb)
    if y is None:
        pytest.skip("variant does not serve this shape")
    _check(y.cpu().numpy(), ref_b)
    _check(run(tw1, ts1, residual=tr).cpu().numpy(), oracle.add_f16(d, res))
    _check(run(tw1, ts1, bias=tb, residual=tr).cpu().numpy(), oracle.add_f16(ref_b, res))
    # the residual in place: the output buffer holds it
    out = tr.clone()
    y_in_place = ops.w4a16_gemm_fused(ta, tw1, ts1, bias=tb, residual=out, out=out, workspace=ws, **kw)
    _check(y_in_place.cpu().numpy(), oracle.add_f16(ref_b, res))
    # RMSNorm prologue alone and with everything behind it
    xn = oracle.rmsnorm_f16(a, gamma, 1e-6)
    dn32 = oracle.w4a16_gemm(xn, wq[:n], s[:n], f32_out=True)
    _check(run(tw1, ts1, rms_gamma=tg, rms_eps=1e-6).cpu().numpy(), dn32)
    dn = oracle.w4a16_gemm(xn, wq[:n], s[:n])
    ref_nbr = oracle.add_f16(oracle.add_f16(dn, np.broadcast_to(bias, (m, n)).copy()), res)
    _check(run(tw1, ts1, rms_gamma=tg, rms_eps=1e-6, bias=tb, residual=tr).cpu().numpy(), ref_nbr)
    # SiLU-gate, without and with the prologue
    for x, fused in ((a, {}), (xn, {"rms_gamma": tg, "rms_eps": 1e-6})):
        gu = oracle.w4a16_gemm(x, wq, s)
        g, u = np.ascontiguousarray(gu[:, :n]), np.ascontiguousarray(gu[:, n:])
        ref = oracle.silu_mul_f16(g, u)
        yg = run(tw, ts, act=1, **fused).cpu().numpy()
        assert yg.shape == (m, n)
        delta = TOL * _rms(gu)
        g32, u32 = g.astype(np.float32), u.astype(np.float32)
        silu = g32 / (1.0 + np.exp(-g32))
        bound = delta * (1.1 * np.abs(u32) + np.abs(silu)) + np.abs(ref.astype(np.float32)) * 2.0 ** -10 + 1e-6
        err = np.abs(yg.astype(np.float32) - ref.astype(np.float32))
        assert np.all(err <= bound), float((err - bound).max())
    torch.cuda.synchronize()


@pytest.mark.parametrize("m,n,k", [(11, 981, 8192), (16, 4096, 8192), (8, 300, 8192), (12, 9000, 8192), (24, 304, 8192),
                                   (8, 1000, 11008), (3, 520, 4096), (200, 300, 1024), (1, 4096, 4096), (16, 48, 2304)])
def test_fused_parts_in_the_workspace_the_query_asks_for(gpu, m, n, k):
    """nnf_w4a16_gemm_fused_workspace_bytes does not know which of the optional parts a call will use, and the kernels
    that serve them differ (8 .. 16 rows at K = 8192 run over two ranges of K without the RMSNorm prologue, in one launch
    with it): a workspace of exactly that size serves every combination."""
    import torch

    from nnfusion_amd import ops

    a, wq, s = datagen.w4a16_case(23, m, 2 * n, k)
    bias = datagen.normal_f16(23, datagen.S_BIAS, (n,))
    res = datagen.normal_f16(23, datagen.S_RES, (m, n))
    gamma = datagen.normal_f16(23, datagen.S_GAMMA, (k,), 1.0, 0.1)
    ta, tw, ts, tb, tr, tg = _t(gpu, a, wq, s, bias, res, gamma)
    tw1, ts1 = tw[:n].contiguous(), ts[:n].contiguous()
    d = oracle.w4a16_gemm(a, wq[:n], s[:n])
    ref_b = oracle.add_f16(d, np.broadcast_to(bias, (m, n)).copy())
    _check(ops.w4a16_gemm_fused(ta, tw1, ts1, bias=tb).cpu().numpy(), ref_b)
    _check(ops.w4a16_gemm_fused(ta, tw1, ts1, residual=tr).cpu().numpy(), oracle.add_f16(d, res))
    out = tr.clone()
    _check(ops.w4a16_gemm_fused(ta, tw1, ts1, bias=tb, residual=out, out=out).cpu().numpy(), oracle.add_f16(ref_b, res))
    xn = oracle.rmsnorm_f16(a, gamma, 1e-6)
    _check(ops.w4a16_gemm_fused(ta, tw1, ts1, rms_gamma=tg, rms_eps=1e-6).cpu().numpy(),
           oracle.w4a16_gemm(xn, wq[:n], s[:n], f32_out=True))
    dn = oracle.w4a16_gemm(xn, wq[:n], s[:n])
    _check(ops.w4a16_gemm_fused(ta, tw1, ts1, rms_gamma=tg, rms_eps=1e-6, residual=tr).cpu().numpy(), oracle.add_f16(dn, res))
    assert ops.w4a16_gemm_fused(ta, tw, ts, act=1).shape == (m, n)
    assert ops.w4a16_gemm_fused(ta, tw, ts, act=1, rms_gamma=tg, rms_eps=1e-6).shape == (m, n)
    torch.cuda.synchronize()


# the library's own plan: whole tiles of each shape (fewer than CUs, more than CUs), tiles in 2 .. 16 equal parts, the even
# split; ragged M and N, K with a last superstep of one group
@pytest.mark.parametrize("m,n,k", [(20, 1160, 640), (33, 300, 16256), (64, 4096, 2304), (73, 12288, 1536), (160, 1792, 5504), (200, 257, 11008),
                                   (250, 4111, 640), (315, 9216, 2304), (450, 448, 640), (450, 1800, 7168), (700, 10000, 512), (1000, 256, 5504),
                                   (1800, 2500, 1408), (2500, 16384, 384), (3000, 700, 3072)])
def test_own_plan_matches_whole_tiles(gpu, m, n, k):
    """The plan the library picks against whole tiles of 128 x 128, one workgroup each (the order in which a tile's K is
    added differs: fp32 sums of K terms, then one rounding to fp16; 2e-3 of the RMS is four times that rounding at the
    RMS), with and without synchronisation words (bit for bit), plain, with RMSNorm and residual, with SiLU-gate."""
    import torch

    from nnfusion_amd import datagen, ops

    a, wq, s = datagen.w4a16_case(m + n + k, m, 2 * n, k)
    a, wq, s = (torch.from_numpy(x).to(gpu) for x in (a, wq, s))
    w1, s1 = wq[:n].contiguous(), s[:n].contiguous()
    gen = torch.Generator(device="cpu").manual_seed(n)
    gamma = torch.randn(k, generator=gen).mul(0.1).add(1).half().to(gpu)
    res = torch.randn(m, n, generator=gen).half().to(gpu)
    sync = ops.sync_flags(gpu)
    for w, sc, parts in ((w1, s1, {}), (w1, s1, dict(rms_gamma=gamma, residual=res)), (wq, s, dict(act=1, rms_gamma=gamma))):
        ref = ops.w4a16_gemm_fused(a, w, sc, variant="gemm_mfma", plan=(128, 1, 256 if "act" in parts else 128), **parts).float()
        one = ops.w4a16_gemm_fused(a, w, sc, variant="gemm_mfma", sync=sync, plan=(0, 0, 0), **parts)
        two = ops.w4a16_gemm_fused(a, w, sc, variant="gemm_mfma", plan=(0, 0, 0), **parts)
        assert torch.equal(one, two)
        err = float((one.float() - ref).abs().max())
        assert err <= (2e-2 if "act" in parts else 1e-2) * float(ref.pow(2).mean().sqrt()), err
        assert float((one.float() - ref).pow(2).mean().sqrt()) <= 2e-3 * float(ref.pow(2).mean().sqrt())
        assert not sync.any()


# the row-streaming kernel with K as a run-time value: an odd number of groups per row (scales of odd rows start in the middle
# of a word), one to four groups per wavefront and step, one and two blocks of rows, activations straight in and through
# LDS; fewer tiles than CUs, a last tile moved back by an odd number of rows, several tiles per workgroup
@pytest.mark.parametrize("m,n,k", [(2, 40, 1664), (16, 1002, 1920), (9, 4110, 1920), (20, 300, 1920), (32, 4110, 3968), (3, 520, 3200), (16, 4110, 3968),
                                   (6, 4096, 5504), (16, 30, 4992), (8, 1002, 8064), (13, 9000, 6784), (5, 520, 5120), (31, 1000, 3584),
                                   (33, 300, 1152), (64, 4110, 2048), (45, 1000, 1664), (50, 5000, 1280)])
def test_run_time_k_with_any_number_of_groups(gpu, m, n, k):
    """Plain, with bias and residual, with RMSNorm (activations times gamma beyond fp16 among them) and SiLU-gate, against
    the oracle's product of the same tensors; RMSNorm against the node as a call of its own."""
    import torch

    from nnfusion_amd import datagen, ops

    a, wq, s = datagen.w4a16_case(m + n + k, m, 2 * n, k)
    ref = oracle.wna16_gemm(a, wq, s, 4, 128, zp=8, f32_out=True)
    t = [torch.from_numpy(x).to(gpu) for x in (a, wq, s)]
    w1, s1 = t[1][:n].contiguous(), t[2][:n].contiguous()
    rms = float(np.sqrt((ref.astype(np.float64) ** 2).mean()))
    plain = ops.w4a16_gemm(t[0], w1, s1)
    assert np.abs(plain.float().cpu().numpy() - ref[:, :n]).max() <= 1e-2 * rms
    gen = torch.Generator(device="cpu").manual_seed(k)
    gamma = torch.randn(k, generator=gen).mul(0.1).add(1).half().to(gpu)
    bias, res = torch.randn(n, generator=gen).half().to(gpu), torch.randn(m, n, generator=gen).half().to(gpu)
    y = res.clone()
    ops.w4a16_gemm_fused(t[0], w1, s1, bias=bias, residual=y, out=y)
    assert torch.equal(y, ops.elementwise("add", ops.elementwise("add", plain, bias), res))
    x = (t[0] * 12000).clamp(-6e4, 6e4)
    normed = ops.rms_norm(x, gamma, 1e-5)
    one = ops.w4a16_gemm_fused(x, w1, s1, rms_gamma=gamma, rms_eps=1e-5)
    if k % 256:  # (elsewhere gamma alone joins the activations, rstd the sums: another rounding, and other limits)
        want = ops.w4a16_gemm(normed, w1, s1).float()
        # (one rounding the other way now and then in the activations, then y's own: 2^-11 of up to five RMS each)
        assert float((one.float() - want).abs().max()) <= 5e-3 * float(want.pow(2).mean().sqrt())
    x = x if k % 256 else t[0]
    p = ops.w4a16_gemm(ops.rms_norm(x, gamma, 1e-5), t[1], t[2]).float()
    g = p[:, :n]
    want = g / (1 + torch.exp(-g)) * p[:, n:]
    y = ops.w4a16_gemm_fused(x, t[1], t[2], rms_gamma=gamma, rms_eps=1e-5, act=1).float()
    assert float((y - want).abs().max()) <= 2e-2 * float(want.pow(2).mean().sqrt())


# shapes whose RMSNorm form on the row-streaming kernel writes M x K normalised activations to scratch memory: 33 .. 64 rows, K no
# multiple of 256, 17 .. 32 rows; few weight rows, so that the tile GEMM needs less
@pytest.mark.parametrize("m,n,k", [(50, 107, 1536), (64, 23, 2048), (58, 109, 1792), (32, 126, 3200), (31, 16, 3712), (27, 33, 1280)])
def test_scratch_memory_sized_for_the_tile_gemm_is_accepted(gpu, m, n, k):
    """A program that sized its scratch memory for the tile GEMM (rstd and the parked tiles, a literal in generated code)
    is served there: same results, nothing written beyond; without room for that either the call is refused."""
    import torch

    from nnfusion_amd import _lib, ops

    a, wq, s = datagen.w4a16_case(m + n, m, n, k)
    gamma = datagen.normal_f16(5, datagen.S_GAMMA, (k,), 1.0, 0.1)
    res = datagen.normal_f16(5, datagen.S_RES, (m, n))
    ta, tw, ts, tg, tr = _t(gpu, a, wq, s, gamma, res)
    lib = _lib.kernels()
    sync = ops.sync_flags(gpu)
    parked = lib.nnf_w4a16_gemm_variant_workspace_bytes(m, n, k, 128, ops.VARIANTS["gemm_mfma"], None)
    need = 256 + parked
    assert need < m * k * 2  # (what the row-streaming kernel asks for)
    ref = oracle.add_f16(oracle.w4a16_gemm(oracle.rmsnorm_f16(a, gamma, 1e-6), wq, s), res)
    for words in (None, sync):
        buf = torch.full((need + 4096,), 0x5A, dtype=torch.uint8, device=gpu)
        y = ops.w4a16_gemm_fused(ta, tw, ts, rms_gamma=tg, rms_eps=1e-6, residual=tr, workspace=buf[:need], sync=words)
        _check(y.cpu().numpy(), ref)
        assert bool((buf[need:] == 0x5A).all()) and not sync.any()
        if parked:
            with pytest.raises(ops.NnfError) as e:
                ops.w4a16_gemm_fused(ta, tw, ts, rms_gamma=tg, rms_eps=1e-6, residual=tr, workspace=buf[:need - 16], sync=words)
            assert e.value.status == -3
    # the same kernel by name, given rstd alone
    if k % 256 == 0 and m <= 32:
        y = ops.w4a16_gemm_fused(ta, tw, ts, rms_gamma=tg, rms_eps=1e-6, residual=tr, workspace=buf[:256], variant="gemv_rows")
        _check(y.cpu().numpy(), ref)
        assert bool((buf[need:] == 0x5A).all())


# Tiles of 64 and 128 rows on four wavefronts and on eight: one a CU over odd and even numbers of supersteps, the last one of a
# single group; parts of few and of many supersteps; more tiles than CUs one by one and in the even split (plan without parts:
# tiles that workgroups share in the middle); ragged rows and columns
@pytest.mark.parametrize("m,n,k,rows,parts,cols", [
    (130, 520, 2176, 128, 1, 128), (65, 130, 2048, 128, 1, 128), (200, 300, 512, 128, 1, 128), (100, 384, 4480, 128, 2, 128),
    (256, 1000, 1280, 128, 4, 128), (1000, 5000, 512, 128, 1, 128), (1100, 4700, 2176, 128, 0, 128), (40, 3000, 11136, 128, 0, 128),
    (33, 257, 2432, 64, 1, 128), (64, 640, 2048, 64, 1, 128), (190, 500, 640, 64, 1, 128), (100, 520, 4480, 64, 2, 128),
    (256, 9000, 2176, 64, 0, 128), (256, 9000, 640, 64, 1, 128), (130, 520, 2176, 128, 1, 256), (100, 1000, 4480, 128, 2, 256),
    (100, 2700, 2432, 128, 12, 256), (1100, 9000, 1408, 128, 0, 256), (33, 1000, 2176, 64, 1, 256), (64, 3000, 4480, 64, 12, 256),
    (1, 300, 2176, 128, 1, 128), (1, 300, 2176, 64, 1, 256)])
def test_four_and_eight_wavefronts(gpu, m, n, k, rows, parts, cols):
    """Against float32 products of the same values: rounding the weights (times gamma) and the result to fp16 gives 2-norm errors
    of about 2^-11.5 each, SiLU-gate three such results (1e-3, 2e-3); one and two launches bit for bit."""
    import torch

    from nnfusion_amd import ops

    print(f"case M={m} N={n} K={k} tile={rows}x{cols} parts={parts}", flush=True)
    a, wq, s = datagen.w4a16_case(m + n + k, m, 2 * n, k)
    gamma = datagen.normal_f16(m, datagen.S_GAMMA, (k,), 1.0, 0.1)
    res = datagen.normal_f16(m, datagen.S_RES, (m, n))
    bias = datagen.normal_f16(m, datagen.S_BIAS, (n,))
    a, wq, s, gamma, res, bias = _t(gpu, a, wq, s, gamma, res, bias)
    q = torch.stack((wq & 15, wq >> 4), dim=2).reshape(2 * n, k).float() - 8
    w = q * s.float().repeat_interleave(128, dim=1)
    x = a.float()
    xn = x * torch.rsqrt(x.pow(2).mean(dim=1, keepdim=True) + 1e-6) * gamma.float()
    w1, s1 = wq[:n].contiguous(), s[:n].contiguous()
    gate, up = (xn @ w.t()).split(n, dim=1)
    forms = [(wq, s, dict(act=1, rms_gamma=gamma), torch.nn.functional.silu(gate) * up, 2e-3)]
    if not (rows == 64 and cols == 256):
        forms += [(w1, s1, {}, x @ w[:n].t(), 1e-3), (w1, s1, dict(rms_gamma=gamma, residual=res), xn @ w[:n].t() + res.float(), 1e-3),
                  (w1, s1, dict(bias=bias, residual=res), x @ w[:n].t() + bias.float() + res.float(), 1e-3)]
    sync = ops.sync_flags(gpu)
    for w_, s_, kw, ref, tol in forms:
        plan = (rows, parts, 256 if "act" in kw else cols)
        one = ops.w4a16_gemm_fused(a, w_, s_, variant="gemm_mfma", plan=plan, sync=sync, **kw)
        two = ops.w4a16_gemm_fused(a, w_, s_, variant="gemm_mfma", plan=plan, **kw)
        assert torch.equal(one, two)
        assert float((one.float() - ref).norm() / ref.norm()) <= tol
        assert float((one.float() - ref).abs().max() / ref.pow(2).mean().sqrt()) <= (2e-2 if "act" in kw else TOL)
        assert not sync.any()


# Whole tiles of 128 x 192: even and odd numbers of supersteps, the last tile of rows and columns ragged (columns no multiple of eight
# too: stored an element at a time), N = the plain form's and the SiLU-gate form's outputs, both within the rule
@pytest.mark.parametrize("m,n_plain,n_gate,k", [(300, 11300, 5601, 2560), (257, 11523, 5555, 2816), (700, 6200, 3000, 3072), (513, 9216, 4608, 2560),
                                                (1000, 4608, 2310, 4096), (201, 24500, 12199, 2816)])
def test_tiles_of_192_columns(gpu, m, n_plain, n_gate, k):
    """Against float32 products of the same values, bounds as for the other tiles (test_four_and_eight_wavefronts); with and without
    synchronisation words bit for bit."""
    import torch

    from nnfusion_amd import ops

    print(f"case M={m} N={n_plain}/{n_gate} K={k}", flush=True)
    n = max(n_plain, 2 * n_gate)
    a, wq, s = datagen.w4a16_case(m + n + k, m, n, k)
    gamma = datagen.normal_f16(m, datagen.S_GAMMA, (k,), 1.0, 0.1)
    res = datagen.normal_f16(m, datagen.S_RES, (m, n_plain))
    bias = datagen.normal_f16(m, datagen.S_BIAS, (n_plain,))
    a, wq, s, gamma, res, bias = _t(gpu, a, wq, s, gamma, res, bias)
    q = torch.stack((wq & 15, wq >> 4), dim=2).reshape(n, k).float() - 8
    w = q * s.float().repeat_interleave(128, dim=1)
    x = a.float()
    xn = x * torch.rsqrt(x.pow(2).mean(dim=1, keepdim=True) + 1e-6) * gamma.float()
    wp, sp, wg, sg = (t[:c].contiguous() for c in (n_plain, 2 * n_gate) for t in (wq, s))
    gate, up = (xn @ w[:2 * n_gate].t()).split(n_gate, dim=1)
    plain, normed = x @ w[:n_plain].t(), xn @ w[:n_plain].t()
    sync = ops.sync_flags(gpu)
    for w_, s_, kw, ref, tol in ((wg, sg, dict(act=1, rms_gamma=gamma), torch.nn.functional.silu(gate) * up, 2e-3), (wp, sp, {}, plain, 1e-3),
                                 (wp, sp, dict(rms_gamma=gamma, residual=res), normed + res.float(), 1e-3),
                                 (wp, sp, dict(bias=bias, residual=res), plain + bias.float() + res.float(), 1e-3),
                                 (wp, sp, dict(rms_gamma=gamma, bias=bias), normed + bias.float(), 1e-3)):
        one = ops.w4a16_gemm_fused(a, w_, s_, variant="gemm_mfma", plan=(0, 0, 0), sync=sync, **kw)
        two = ops.w4a16_gemm_fused(a, w_, s_, variant="gemm_mfma", plan=(0, 0, 0), **kw)
        assert torch.equal(one, two)
        assert float((one.float() - ref).norm() / ref.norm()) <= tol
        assert float((one.float() - ref).abs().max() / ref.pow(2).mean().sqrt()) <= (2e-2 if "act" in kw else TOL)
        assert not sync.any()


@pytest.mark.parametrize("m,n_plain,n_gate,k", [(300, 11300, 5601, 2560), (257, 11523, 5555, 2816), (700, 6200, 3000, 3072), (1000, 4608, 2310, 4096)])
def test_tiles_of_192_columns_where_the_wait_runs_out(gpu, m, n_plain, n_gate, k):
    """RMSNorm inside the launch: rows that a workgroup computes itself, its wait for the others being over at once, have the same bits."""
    import torch

    from nnfusion_amd import ops

    print(f"case M={m} N={n_plain}/{n_gate} K={k}", flush=True)
    n = max(n_plain, 2 * n_gate)
    a, wq, s = datagen.w4a16_case(m + n + k, m, n, k)
    gamma = datagen.normal_f16(m, datagen.S_GAMMA, (k,), 1.0, 0.1)
    res = datagen.normal_f16(m, datagen.S_RES, (m, n_plain))
    bias = datagen.normal_f16(m, datagen.S_BIAS, (n_plain,))
    a, wq, s, gamma, res, bias = _t(gpu, a, wq, s, gamma, res, bias)
    wp, sp, wg, sg = (t[:c].contiguous() for c in (n_plain, 2 * n_gate) for t in (wq, s))
    sync = ops.sync_flags(gpu)
    for w_, s_, kw in ((wg, sg, dict(act=1)), (wp, sp, {}), (wp, sp, dict(residual=res)), (wp, sp, dict(bias=bias)), (wp, sp, dict(bias=bias, residual=res))):
        kw = dict(kw, rms_gamma=gamma, variant="gemm_mfma", plan=(0, 0, 0))
        two = ops.w4a16_gemm_fused(a, w_, s_, **kw)
        for spin_limit in (0, -1):
            assert torch.equal(ops.w4a16_gemm_fused(a, w_, s_, sync=sync, spin_limit=spin_limit, **kw), two)
            assert not sync.any()
