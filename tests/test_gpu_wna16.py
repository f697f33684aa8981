"""Parity of nnf_wna16_gemm (4- or 8-bit weights, groups of 32 / 64 / 128, scalar or per-(row, group) zero points; HIP,
through the C ABI) against the CPU oracle.

Tolerance (stated by the task): max|y - y_ref| <= 1e-2 * RMS(y_ref), y_ref = the oracle's fp32-accumulated product with
the weights dequantised as (q - z) * s; a one-hot activation row must return the dequantised weights exactly.
"""
import ctypes

import numpy as np
import pytest

import oracle
from nnfusion_amd import datagen

pytestmark = pytest.mark.gpu

TOL = 1e-2


def _case(seed, m, n, k, bits, group, zp_tensor):
    return datagen.wna16_case(seed, m, n, k, bits, group, zp_tensor)


def _run(gpu, a, wq, s, bits, group, zp, zps):
    import torch

    from nnfusion_amd import ops

    t = [torch.from_numpy(x).to(gpu) for x in (a, wq, s)]
    tz = None if zps is None else torch.from_numpy(zps).to(gpu)
    y = ops.wna16_gemm(*t, bits=bits, group=group, zp=zp, zero_points=tz)
    torch.cuda.synchronize()
    return y.cpu().numpy()


def _check(y, ref):
    rms = float(np.sqrt(np.mean(ref.astype(np.float64) ** 2)))
    err = float(np.abs(y.astype(np.float32) - ref).max())
    assert np.isfinite(y).all()
    assert err <= TOL * max(rms, 1e-6), (err, rms)


SHAPES = [
    # the wavefront-per-row kernel (M <= 16): one row, ragged N, K shorter than one pass of a wavefront, an odd number
    # of groups, the benchmark's shapes
    (1, 4096, 4096), (1, 33, 128), (3, 1000, 512), (16, 257, 2048), (5, 64, 160), (1, 12288, 4096), (8, 300, 11008),
    (16, 4111, 4096), (2, 7, 384),
    # one row, K a multiple of 256: the row-streaming kernel (one, two and three loads per row and
    # wavefront; one, two and four wavefronts per row; fewer rows than wavefronts)
    (1, 300, 1024), (1, 22016, 4096), (1, 4096, 11008), (1, 1000, 8192), (1, 5000, 16384), (1, 257, 2560), (1, 5, 4096),
    # a few rows of 4-bit weights with K = 2048 / 4096 / 8192: the row-streaming MFMA kernel (one, two and four loads per
    # step and wavefront; fewer tiles than CUs, a ragged last tile, several tiles per workgroup)
    (2, 4096, 4096), (5, 300, 2048), (8, 1000, 8192), (16, 48, 8192), (13, 12288, 4096), (16, 9000, 2048),
    (17, 4096, 4096), (32, 1000, 2048), (25, 12288, 4096), (31, 40, 4096),
    # ... with any other K that is a multiple of 256: one piece up to 8192 (two, three, four blocks of 128 per wavefront and
    # step; wavefronts past the end of K), ranges of K above (11008: three; 14336: four; 28672: seven)
    (4, 4096, 3584), (16, 1000, 5120), (9, 300, 7168), (2, 4096, 11008), (16, 4096, 11008), (8, 520, 14336), (5, 64, 28672),
    (16, 33, 2560),
    # the tile kernel: one partial tile, ragged M and N, many tiles, a long K
    (17, 33, 128), (64, 64, 512), (100, 1000, 160), (300, 257, 2048), (128, 4096, 4096), (33, 520, 11008), (1024, 130, 384),
    # 4-bit weights above 16 rows with K a multiple of 256: the stream-K tile GEMM (tiles of 32 x 256, 64 x 128, 128 x 128,
    # 256 x 128, 256 x 256; tiles shared between workgroups and not; ragged M and N)
    (17, 300, 256), (40, 1000, 1024), (100, 257, 2048), (130, 4096, 4096), (700, 3000, 1280), (1100, 2050, 768),
    (1600, 520, 2560), (2000, 8192, 512), (30, 22016, 4096),
    # 8-bit weights above 32 rows (16 at K = 8192): two or three blocks of rows through the row-streaming kernel (two
    # above N = 8192), the last block of one, two and all rows; one block more: the tile kernel
    (33, 4096, 4096), (65, 1000, 2048), (96, 520, 4096), (97, 520, 4096), (48, 300, 8192), (49, 300, 8192), (50, 4111, 4096),
    (64, 9000, 2048), (65, 9000, 2048),
    # enough 128 x 128 tiles to fill the chip: the larger tile kernel; ragged M and N, an odd number of groups
    (2048, 2048, 512), (1100, 4100, 160), (4096, 1030, 384),
    # ... 256 x 128 tiles (one round of them beats two of 128 x 128), 256 x 256 tiles (they fill the chip): ragged M and N
    (1000, 8100, 384), (1990, 8100, 160), (300, 22016, 128),
]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("bits,group,zp_tensor", [
    (4, 32, False), (4, 32, True), (4, 64, False), (4, 64, True), (4, 128, True),
    (8, 32, False), (8, 32, True), (8, 64, True), (8, 128, False), (8, 128, True),
])
def test_wna16_matches_oracle(gpu, m, n, k, bits, group, zp_tensor):
    if k % group:
        pytest.skip("K is not a multiple of the group")
    a, wq, s, zps = _case(m * 131 + n + k + bits + group, m, n, k, bits, group, zp_tensor)
    zp = 7 if bits == 4 else 131
    ref = oracle.wna16_gemm(a, wq, s, bits, group, zp=zp, zero_points=zps, f32_out=True)
    _check(_run(gpu, a, wq, s, bits, group, zp, zps), ref)


@pytest.mark.parametrize("m,n,k", [(4, 70, 640), (40, 70, 640), (2000, 2100, 640), (40, 300, 1024), (300, 520, 768),
                                   (2000, 2100, 512), (1990, 8100, 640)])
@pytest.mark.parametrize("bits,group,zp_tensor", [(4, 32, True), (4, 64, False), (8, 64, True), (8, 128, False), (8, 32, True),
                                                   (4, 64, True), (4, 128, True), (4, 32, False)])
def test_one_hot_rows_return_the_dequantised_weights(gpu, m, n, k, bits, group, zp_tensor):
    """A = e_k: 1 * w is exact in every kernel (m = 2000: the 256 x 128 tiles, m = 1990: the 256 x 256 tiles; K a multiple
    of 256 with 4-bit weights: the stream-K tile GEMM), so the output is fp16((q - z) * s) bit for bit; pins nibble and byte order of weights and zero
    points and the block each scale belongs to, on the device."""
    _, wq, s, zps = _case(5, m, n, k, bits, group, zp_tensor)
    zp = 3 if bits == 4 else 200
    wd = oracle.dequantize_wn(wq, s, bits, group, zp=zp, zero_points=zps)
    ks = [0, 1, 7, 8, 31, 32, 63, 64, 127, 128, 255, 256, 511, 512, 639][:m] if m <= 16 else [(7 * r) % k for r in range(min(m, k))]
    a = np.zeros((m, k), np.float16)
    for r, kk in enumerate(ks):
        a[r, kk] = 1.0
    y = _run(gpu, a, wq, s, bits, group, zp, zps)
    for r, kk in enumerate(ks):
        np.testing.assert_array_equal(y[r], wd[:, kk].astype(np.float16))
    assert not y[len(ks):].any()


@pytest.mark.parametrize("m,k", [(1, 1024), (1, 4096), (1, 11008), (1, 16384), (7, 2048), (16, 4096), (3, 8192), (32, 4096),
                                 (20, 2048), (16, 11008), (6, 5120), (11, 7168), (16, 3584)])
@pytest.mark.parametrize("group,zp_tensor", [(32, True), (64, True), (128, True), (32, False), (64, False)])
def test_one_hot_rows_through_the_row_streaming_kernels(gpu, m, k, group, zp_tensor):
    """4-bit weights with one row and K a multiple of 256, or a few rows and K = 2048 / 4096 / 8192, run on the
    row-streaming kernels: the same pin for their scales and zero points (first and last weight of a group, of a
    wavefront's load, of a wavefront's K segment, of a step, of the row)."""
    n = 700
    _, wq, s, zps = _case(11, 1, n, k, 4, group, zp_tensor)
    wd = oracle.dequantize_wn(wq, s, 4, group, zp=5, zero_points=zps)
    kks = [kk for kk in sorted({0, 1, 31, 32, 63, 64, 127, 128, 255, 256, 511, 512, 1023, 1024, 2047, 2048, 4095, 4096, 6143,
                                6144, 8191, 8192, k // 2 - 1, k // 2, k - 129, k - 33, k - 1}) if kk < k]
    for c in range(0, len(kks), m):
        chunk = kks[c:c + m]
        a = np.zeros((m, k), np.float16)
        for r, kk in enumerate(chunk):
            a[r, kk] = 1.0
        y = _run(gpu, a, wq, s, 4, group, 5, zps)
        for r, kk in enumerate(chunk):
            np.testing.assert_array_equal(y[r], wd[:, kk].astype(np.float16), err_msg="k = %d" % kk)
        assert not y[len(chunk):].any()


@pytest.mark.parametrize("m,k", [(1, 1024), (1, 2048), (1, 2560), (1, 4096), (1, 8192), (1, 11008), (1, 16384), (16, 2048), (7, 4096),
                                 (16, 4096), (3, 8192), (16, 8192), (20, 2048), (32, 4096), (33, 2048), (40, 4096), (24, 8192)])
@pytest.mark.parametrize("group,zp_tensor", [(32, True), (64, True), (128, True), (32, False), (128, False)])
def test_one_hot_rows_through_the_row_streaming_kernels_with_8_bit_weights(gpu, m, k, group, zp_tensor):
    """8-bit weights with one row and K a multiple of 256, or 2 .. 16 rows and K = 2048 / 4096 / 8192 (up to 32 rows at
    2048 / 4096, and a few blocks of that many rows one after the other), run on the
    row-streaming kernels as well (a row is K bytes, a lane meets 16 weights per load): the same pin (first and last
    weight of a group, of a lane, of a wavefront's load, of a wavefront's K segment, of a step, of the row)."""
    n = 700
    _, wq, s, zps = _case(13, 1, n, k, 8, group, zp_tensor)
    wd = oracle.dequantize_wn(wq, s, 8, group, zp=201, zero_points=zps)
    kks = [kk for kk in sorted({0, 1, 15, 16, 31, 32, 63, 64, 127, 128, 255, 256, 511, 512, 1023, 1024, 2047, 2048, 3071, 3072,
                                4095, 4096, 6143, 6144, 8191, 8192, k // 2 - 1, k // 2, k - 129, k - 33, k - 17, k - 1}) if kk < k]
    for c in range(0, len(kks), m):
        chunk = kks[c:c + m]
        a = np.zeros((m, k), np.float16)
        for r, kk in enumerate(chunk):
            a[r, kk] = 1.0
        y = _run(gpu, a, wq, s, 8, group, 201, zps)
        for r, kk in enumerate(chunk):
            np.testing.assert_array_equal(y[r], wd[:, kk].astype(np.float16), err_msg="k = %d" % kk)
        assert not y[len(chunk):].any()


def _random_shapes(count):
    rng = np.random.default_rng(20240607)
    ks = [128, 256, 384, 512, 768, 1024, 1280, 2048, 2560, 3584, 4096, 5120, 7168, 8192, 11008, 14336]
    out = []
    for i in range(count):
        m = int(rng.choice([1, 1, 2, 3, 7, 8, 15, 16, 17, 24, 32, 33, 63, 64, 100, 129, 257, 300]))
        n = int(rng.choice([16, 17, 31, 33, 64, 100, 255, 256, 257, 500, 1000, 1024, 2000, 4096]))
        k = int(rng.choice(ks))
        if m * n * k > 300 * 2000 * 4096:
            n = 256
        out.append((m, n, k, int(rng.choice([4, 4, 4, 8])), int(rng.choice([32, 64, 128])), bool(rng.integers(0, 2)), int(rng.integers(0, 16))))
    return out


@pytest.mark.parametrize("m,n,k,bits,group,zp_tensor,zp", _random_shapes(120))
def test_wna16_random_shapes(gpu, m, n, k, bits, group, zp_tensor, zp):
    """Shapes drawn across the routes of nnf_wna16_gemm (row-streaming kernels with a fixed and a run-time K, ranges of K,
    stream-K tiles, plain kernels), every block parameter and zero point."""
    a, wq, s, zps = _case(m + 3 * n + 7 * k + bits + group, m, n, k, bits, group, zp_tensor)
    zp = zp if bits == 4 else 16 * zp + 3
    ref = oracle.wna16_gemm(a, wq, s, bits, group, zp=zp, zero_points=zps, f32_out=True)
    _check(_run(gpu, a, wq, s, bits, group, zp, zps), ref)


@pytest.mark.parametrize("k", [4096, 8192])
def test_tile_gemm_without_its_workspace_runs_on_the_plain_kernel(gpu, k):
    """Above 16 rows 4-bit weights want the stream-K tile GEMM's workspace; a caller that brings none (or too little)
    gets the same product from the plain tile kernel (K = 8192; at 4096 the K-streaming kernel needs none)."""
    import torch

    from nnfusion_amd import ops

    m, n, group = 130, 1024, 64
    a, wq, s, zps = _case(21, m, n, k, 4, group, True)
    need = ops.wna16_workspace_bytes(m, n, k, 4, group)
    assert need > 0
    t = [torch.from_numpy(x).to(gpu) for x in (a, wq, s, zps)]
    ref = oracle.wna16_gemm(a, wq, s, 4, group, zero_points=zps, f32_out=True)
    for ws_bytes in (need, need - 16, 16):
        y = ops.wna16_gemm(t[0], t[1], t[2], bits=4, group=group, zero_points=t[3],
                           workspace=torch.empty(ws_bytes, dtype=torch.uint8, device=gpu))
        torch.cuda.synchronize()
        _check(y.cpu().numpy(), ref)


@pytest.mark.parametrize("bits,group,zp_tensor", [(4, 32, True), (4, 64, False), (4, 128, True), (8, 32, True), (8, 128, False)])
@pytest.mark.parametrize("m,n,k", [(17, 24592, 2048), (32, 24610, 4096), (20, 24600, 1024), (60, 24592, 1280), (520, 300, 1024), (600, 1100, 1536),
                                   (70, 520, 6400)])
def test_products_beyond_the_k_streaming_kernel(gpu, m, n, k, bits, group, zp_tensor):
    """More columns than six tiles a workgroup hold, more rows, longer K: two blocks of rows on the row-streaming kernels (17 .. 32 rows, K = 2048
    and 4096), the tile GEMM of 4-bit weights, the plain tile kernel of 8-bit ones (which sizes go where: tests/cpp/test_host.cpp)."""
    print(f"case beyond kstream bits={bits} M={m} N={n} K={k} group={group} zero_points={zp_tensor}", flush=True)
    a, wq, s, zps = _case(m + n + k + group, m, n, k, bits, group, zp_tensor)
    zp = 5 if bits == 4 else 83
    _check(_run(gpu, a, wq, s, bits, group, zp, zps), oracle.wna16_gemm(a, wq, s, bits, group, zp=zp, zero_points=zps, f32_out=True))


# 160 x 96, 128 x 128 and 128 x 96 tiles on pairs of wavefronts (tests/cpp/test_host.cpp holds the plan to that): ragged rows and columns, an even and
# an odd number of steps of 128, a last one of 32, 64 and 96 values
@pytest.mark.parametrize("bits,m,n,k", [(8, 300, 10900, 1280), (8, 300, 10900, 1152), (8, 301, 10983, 1184), (4, 158, 21500, 1248),
                                        (8, 1150, 2690, 1280), (8, 1120, 3100, 1056), (8, 1150, 2690, 1152), (4, 1130, 2900, 1056),
                                        (8, 1005, 2560, 1024), (8, 1130, 2562, 1152), (4, 470, 5800, 1120), (4, 505, 5801, 1184)])
def test_tiles_on_pairs_of_wavefronts(gpu, bits, m, n, k):
    print(f"case pairs of wavefronts bits={bits} M={m} N={n} K={k}", flush=True)
    group = 32 if k % 64 else 64
    a, wq, s, zps = _case(m + n + k, m, n, k, bits, group, bits == 8)
    zp = 7 if bits == 4 else 131
    _check(_run(gpu, a, wq, s, bits, group, zp, zps), oracle.wna16_gemm(a, wq, s, bits, group, zp=zp, zero_points=zps, f32_out=True))
    # one-hot rows: the dequantised weights bit for bit, each k from the half of a step that holds it
    a[:] = 0
    ks = [(37 * r) % k for r in range(m)]
    a[np.arange(m), ks] = 1.0
    wd = oracle.dequantize_wn(wq, s, bits, group, zp=zp, zero_points=zps).astype(np.float16)
    np.testing.assert_array_equal(_run(gpu, a, wq, s, bits, group, zp, zps), wd[:, ks].T)


# ... with every form of their block parameters: groups as long as a step, a scalar zero point with 8 bits, zero points two a byte, an odd number of
# them a row
@pytest.mark.parametrize("bits,m,n,k,group,zp_tensor",
                         [(8, 300, 10900, 1280, 128, False), (8, 300, 10900, 1152, 128, True), (8, 301, 10983, 1184, 32, False), (4, 284, 10894, 1920, 32, True),
                          (8, 1150, 2690, 1152, 128, False), (8, 1120, 3100, 1056, 32, False), (4, 834, 4526, 1152, 64, True), (4, 834, 4526, 1152, 128, True),
                          (8, 1005, 2560, 1024, 128, False), (8, 1130, 2562, 1152, 128, True), (4, 515, 4250, 2176, 128, True), (4, 470, 5800, 1120, 32, True)])
def test_block_parameters_of_tiles_on_pairs_of_wavefronts(gpu, bits, m, n, k, group, zp_tensor):
    """Bounds as for the other tiles (test_tiles_on_pairs_of_wavefronts)."""
    print(f"case pairs of wavefronts bits={bits} M={m} N={n} K={k} group={group} zero_points={zp_tensor}", flush=True)
    a, wq, s, zps = _case(m + n + k + group, m, n, k, bits, group, zp_tensor)
    zp = 7 if bits == 4 else 131
    _check(_run(gpu, a, wq, s, bits, group, zp, zps), oracle.wna16_gemm(a, wq, s, bits, group, zp=zp, zero_points=zps, f32_out=True))
    a[:] = 0
    ks = [(37 * r) % k for r in range(m)]
    a[np.arange(m), ks] = 1.0
    wd = oracle.dequantize_wn(wq, s, bits, group, zp=zp, zero_points=zps).astype(np.float16)
    np.testing.assert_array_equal(_run(gpu, a, wq, s, bits, group, zp, zps), wd[:, ks].T)


# one row on the plain GEMV: fewer rows than wavefronts, either side of 24, 28 and 31 a CU, a pass of a few lanes, one pass and many
@pytest.mark.parametrize("n,k", [(1, 128), (33, 384), (1000, 1152), (4096, 2176), (6144, 640), (6145, 384), (7168, 4224),
                                 (7169, 4224), (7936, 640), (7937, 640), (8191, 640), (8192, 640), (300, 16512)])
@pytest.mark.parametrize("bits,group,zp_tensor", [(4, 32, True), (4, 64, False), (8, 32, True), (8, 128, False)])
def test_one_row_on_the_plain_kernel(gpu, n, k, bits, group, zp_tensor):
    a, wq, s, zps = _case(n + k + bits + group, 1, n, k, bits, group, zp_tensor)
    zp = 7 if bits == 4 else 131
    _check(_run(gpu, a, wq, s, bits, group, zp, zps), oracle.wna16_gemm(a, wq, s, bits, group, zp=zp, zero_points=zps, f32_out=True))


# the tile GEMM on odd multiples of 128: a last superstep of half the weights, whose scales and zero points end with the row (the last
# row: with the tensor); tiles of 128 x 128, 64 x 128 and 256 x 128, parts of K that end with it, the shortest K; some that stay on the plain kernel
@pytest.mark.parametrize("m,n,k", [(1000, 1030, 1152), (520, 300, 2176), (530, 700, 4224), (130, 520, 11136), (40, 9000, 8320), (70, 513, 8320),
                                   (1700, 2048, 2176), (2600, 2500, 2176), (900, 767, 1152), (256, 300, 6272), (1320, 304, 2176), (1000, 1032, 1152), (2600, 2504, 2176), (2600, 2500, 2688)])
@pytest.mark.parametrize("group,zp_tensor", [(32, True), (64, True), (128, True), (32, False), (64, False)])
def test_tile_gemm_on_odd_multiples_of_128(gpu, m, n, k, group, zp_tensor):
    """Against float32 products of the dequantised weights; 2-norm of the roundings of weights and result to fp16 about 4e-4 (1e-3)."""
    import torch

    from nnfusion_amd import ops

    print(f"case M={m} N={n} K={k} group={group} zero points={zp_tensor}", flush=True)
    a, wq, s, zps = _case(m + n + k + group, m, n, k, 4, group, zp_tensor)
    a, wq, s = [torch.from_numpy(x).to(gpu) for x in (a, wq, s)]
    q = torch.stack((wq & 15, wq >> 4), dim=2).reshape(n, k).float()
    z = 5.0
    if zp_tensor:
        zt = torch.from_numpy(zps).to(gpu)
        z = torch.stack((zt & 15, zt >> 4), dim=2).reshape(n, -1)[:, :k // group].float().repeat_interleave(group, dim=1)
    ref = a.float() @ ((q - z) * s.float().repeat_interleave(group, dim=1)).t()
    sync = ops.sync_flags(gpu)
    par = dict(bits=4, group=group, zp=5, zero_points=zt if zp_tensor else None)
    for y in (ops.wna16_gemm(a, wq, s, **par), ops.wna16_gemm(a, wq, s, sync=sync, **par)):
        assert float((y.float() - ref).norm() / ref.norm()) <= 1e-3
        assert float((y.float() - ref).abs().max() / ref.pow(2).mean().sqrt()) <= 1e-2
    assert not sync.any()


# ... every shape of its tiles, on four wavefronts and on eight, whole, in parts of K and in the even split (tests/cpp/test_host.cpp holds the plan to that)
@pytest.mark.parametrize("m,n,k", [(17, 12479, 8320), (18, 12368, 10368), (34, 8407, 12160), (99, 8408, 1152), (65, 528, 6272),
                                  (37, 8202, 8832), (65, 11910, 8320), (526, 808, 1152), (65, 512, 7040), (132, 11000, 1152),
                                  (1287, 12016, 1152), (260, 11128, 1152), (65, 11184, 6784), (261, 3746, 11392),
                                  (387, 8296, 1152), (2060, 272, 2176), (523, 13488, 1152), (135, 11914, 11136),
                                  (1566, 10200, 2432), (387, 8291, 2688), (2060, 269, 2688)])
@pytest.mark.parametrize("group,zp_tensor", [(32, True), (64, False), (128, True)])
def test_every_tile_on_odd_multiples_of_128(gpu, m, n, k, group, zp_tensor):
    test_tile_gemm_on_odd_multiples_of_128(gpu, m, n, k, group, zp_tensor)


# (128, False): the kernel of groups of 128 with a scalar zero point, by name
@pytest.mark.parametrize("m,n,k", [(1000, 1032, 1152), (520, 300, 2176), (17, 12479, 8320), (99, 8408, 1152), (260, 11128, 1152), (387, 8296, 1152),
                                   (523, 13488, 1152), (1320, 304, 2176)])
@pytest.mark.parametrize("group,zp_tensor", [(32, True), (64, False), (128, True), (128, False)])
def test_infinities_at_the_end_of_odd_multiples_of_128(gpu, m, n, k, group, zp_tensor):
    """Infinite activations in the last K step of the tile GEMM: infinities of the sign that the sum over K has, NaN where a weight is 0 or
    two of them cancel; other rows as without them.  So with an infinity in RMSNorm's weight, in every row."""
    import torch

    from nnfusion_amd import ops

    print(f"case infinities M={m} N={n} K={k} group={group} zero points={zp_tensor}", flush=True)
    a, wq, s, zps = _case(m + n + k + group, m, n, k, 4, group, zp_tensor)
    bad = a.copy()
    bad[1, k - 1], bad[2, k - 64], bad[m - 1, k - 1], bad[m - 1, k - 2] = np.inf, -np.inf, np.inf, -np.inf
    ta, tb, tw, ts = [torch.from_numpy(x).to(gpu) for x in (a, bad, wq, s)]
    q = torch.stack((tw & 15, tw >> 4), dim=2).reshape(n, k)
    tz = torch.from_numpy(zps).to(gpu) if zp_tensor else None
    z = 5 if tz is None else torch.stack((tz & 15, tz >> 4), dim=2).reshape(n, -1)[:, :k // group].repeat_interleave(group, dim=1).int()
    sign = (q.int() - z).sign().float()

    def same(y, ref):
        assert torch.equal(y.isnan(), ref.isnan()) and torch.equal(y.isposinf(), ref.isposinf()) and torch.equal(y.isneginf(), ref.isneginf())

    forms = [dict(), dict(sync=ops.sync_flags(gpu))]
    for kw in forms:
        if (group, zp_tensor) == (128, False):
            run = lambda x, **more: ops.w4a16_gemm_fused(x, tw, ts, zp=5, variant="gemm_mfma", **kw, **more)
        else:
            run = lambda x: ops.wna16_gemm(x, tw, ts, bits=4, group=group, zp=5, zero_points=tz, **kw)
        y, clean = run(tb), run(ta)
        rows = [r for r in range(m) if r not in (1, 2, m - 1)]
        assert torch.equal(y[rows], clean[rows]) and bool(clean.isfinite().all())
        same(y[1], float("inf") * sign[:, k - 1])
        same(y[2], -float("inf") * sign[:, k - 64])
        same(y[m - 1], float("inf") * sign[:, k - 1] - float("inf") * sign[:, k - 2])
        if (group, zp_tensor) == (128, False):
            gamma = torch.ones(k, dtype=torch.float16, device=gpu)
            gamma[k - 1] = float("inf")
            same(run(ta, rms_gamma=gamma), float("inf") * ta[:, k - 1:].sign().float() * sign[:, k - 1])


def test_default_parameters_are_the_specialised_kernels(gpu):
    import torch

    from nnfusion_amd import ops

    for m, n, k in ((1, 4096, 4096), (16, 1000, 2048), (128, 512, 4096)):
        a, wq, s = datagen.w4a16_case(3, m, n, k)
        t = [torch.from_numpy(x).to(gpu) for x in (a, wq, s)]
        y0 = ops.w4a16_gemm(*t, zp=8)
        y1 = ops.wna16_gemm(*t, bits=4, group=128, zp=8)
        assert torch.equal(y0, y1)
        # ... and a zero-point tensor holding the scalar everywhere takes the plain kernels to the same product
        zps = torch.full((n, (k // 128 + 1) // 2), 0x88, dtype=torch.uint8, device=gpu)
        y2 = ops.wna16_gemm(*t, bits=4, group=128, zero_points=zps)
        torch.cuda.synchronize()
        ref = oracle.wna16_gemm(a, wq, s, 4, 128, zp=8, f32_out=True)
        _check(y2.cpu().numpy(), ref)


def test_wna16_argument_errors(gpu):
    import torch

    from nnfusion_amd import _lib
    from nnfusion_amd.ops import NnfQuant

    lib = _lib.kernels()
    buf = torch.zeros(1 << 16, dtype=torch.uint8, device=gpu)
    p = buf.data_ptr()

    def call(q, m=4, n=64, k=256, a=p):
        qp = None if q is None else ctypes.cast(ctypes.pointer(q), ctypes.c_void_p)
        return lib.nnf_wna16_gemm(None, a, p, p, p, m, n, k, qp, None, 0)

    assert call(None) == -1
    assert call(NnfQuant(4, 64, 8, None), a=None) == -1
    assert call(NnfQuant(4, 64, 8, None), a=p + 2) == -1
    assert call(NnfQuant(4, 64, 8, None), m=0) == -1
    assert call(NnfQuant(3, 64, 8, None)) == -2      # bits
    assert call(NnfQuant(4, 16, 8, None)) == -2      # group
    assert call(NnfQuant(4, 64, 16, None)) == -2     # zero point outside 4 bits
    assert call(NnfQuant(8, 64, 256, None)) == -2    # ... outside 8 bits
    assert call(NnfQuant(8, 128, 0, None), k=192) == -2  # K % group
    assert call(NnfQuant(8, 64, 255, None)) == 0
    torch.cuda.synchronize()


# fixed K (one, two, four blocks per wavefront and step; one and two blocks of rows; activations straight in and through
# LDS), run-time K (two, three, four blocks; wavefronts past the end of K), ranges of K; fewer tiles than CUs, ragged N,
# several tiles per workgroup
FUSED_SHAPES = [(2, 40, 2048), (16, 1000, 2048), (32, 4111, 2048), (3, 520, 4096), (8, 4111, 4096), (17, 300, 4096), (32, 5000, 4096),
                (2, 1000, 8192), (16, 4111, 8192), (2, 300, 3584), (16, 1000, 3584), (9, 520, 5120), (16, 4111, 7168), (6, 33, 2560),
                (5, 520, 11008), (16, 1000, 14336),
                # the nodes one by one behind the tile kernels: whole 16-byte pieces of a row, and one column at a time
                (40, 1000, 1024), (37, 1001, 640)]


@pytest.mark.parametrize("m,n,k", FUSED_SHAPES)
@pytest.mark.parametrize("group,zp_tensor", [(32, True), (64, False), (64, True), (128, True)])
def test_fused_rows_equal_the_nodes(gpu, m, n, k, group, zp_tensor):
    """The nodes around a product inside the row-streaming kernels against the same nodes as calls of their own.  Without
    RMSNorm bit for bit.  With it the sum of squares is added in another order, so a normalised activation may round the
    other way now and then (2^-11 of its value): on a sum of K independent terms that is at most 2^-11 of its RMS (five
    sigma: 2.5e-3), plus the rounding of y itself (2^-11 of up to five RMS)."""
    import torch

    from nnfusion_amd import ops

    a, wq, s, zps = _case(m * 17 + n + k + group, m, 2 * n, k, 4, group, zp_tensor)
    t = [torch.from_numpy(x).to(gpu) for x in (a, wq, s)]
    tz = torch.from_numpy(zps).to(gpu) if zp_tensor else None
    gen = torch.Generator(device="cpu").manual_seed(m + n)
    gamma = torch.randn(k, generator=gen).mul(0.1).add(1).half().to(gpu)
    bias = torch.randn(n, generator=gen).half().to(gpu)
    res = torch.randn(m, n, generator=gen).half().to(gpu)
    q = dict(bits=4, group=group, zp=5)
    half = lambda x: None if x is None else x[:n].contiguous()
    w1, s1, z1 = half(t[1]), half(t[2]), half(tz)
    plain = ops.wna16_gemm(t[0], w1, s1, zero_points=z1, **q)
    y = ops.wna16_gemm_fused(t[0], w1, s1, zero_points=z1, bias=bias, residual=res, **q)
    assert torch.equal(y, ops.elementwise("add", ops.elementwise("add", plain, bias), res))
    inplace = res.clone()
    ops.wna16_gemm_fused(t[0], w1, s1, zero_points=z1, residual=inplace, out=inplace, **q)
    assert torch.equal(inplace, ops.elementwise("add", plain, res))

    def gated(x):
        p = ops.wna16_gemm(x, t[1], t[2], zero_points=tz, **q).float()
        g = p[:, :n]
        return (g / (1 + torch.exp(-g)) * p[:, n:])

    def close(y, ref, tol):
        rms = float(ref.float().pow(2).mean().sqrt())
        assert torch.isfinite(y).all()
        assert float((y.float() - ref.float()).abs().max()) <= tol * rms

    # (fp16 results of values up to some ten RMS, the device's exp)
    close(ops.wna16_gemm_fused(t[0], t[1], t[2], zero_points=tz, act=1, **q), gated(t[0]), 1e-2)
    # activations times gamma beyond the range of fp16 are still normalised
    x = (t[0] * 12000).clamp(-6e4, 6e4)
    normed = ops.rms_norm(x, gamma, 1e-5)
    close(ops.wna16_gemm_fused(x, w1, s1, zero_points=z1, rms_gamma=gamma, rms_eps=1e-5, **q),
          ops.wna16_gemm(normed, w1, s1, zero_points=z1, **q), 5e-3)
    close(ops.wna16_gemm_fused(x, t[1], t[2], zero_points=tz, rms_gamma=gamma, rms_eps=1e-5, act=1, **q), gated(normed), 2e-2)


# blocks of eight rows and of sixteen on either side of their line, weights ahead of the activations (K = 8192) and behind them; five and
# six tiles a workgroup with SiLU-gate at K = 2048
@pytest.mark.parametrize("m,n,k", [(8, 24, 2048), (9, 24, 2048), (8, 520, 4096), (9, 4111, 4096), (8, 520, 8192), (9, 520, 8192), (8, 8224, 2048),
                                   (15, 12288, 2048)])
@pytest.mark.parametrize("group,zp_tensor", [(32, True), (64, False), (128, True)])
def test_fused_rows_in_blocks_of_eight_and_sixteen(gpu, m, n, k, group, zp_tensor):
    test_fused_rows_equal_the_nodes(gpu, m, n, k, group, zp_tensor)


# both sides of the line between RMSNorm ahead of the row-streaming kernels and inside them: rows at K = 4096 (8 and up
# inside) and at K = 2048 (17 and up ahead); every other K ahead
@pytest.mark.parametrize("m,n,k", [(7, 1000, 4096), (17, 520, 4096), (32, 4111, 4096), (17, 520, 2048), (2, 1000, 8192), (16, 4111, 8192),
                                   (4, 520, 3072), (16, 1000, 5120), (9, 300, 6400)])
@pytest.mark.parametrize("group,zp_tensor", [(32, True), (64, False)])
def test_fused_rows_with_rms_norm_ahead(gpu, m, n, k, group, zp_tensor):
    """Where RMSNorm is a pass of its own in front of the kernel, the fused product is the nodes' own arithmetic, bit for bit
    (inside, the sum of squares is added in another order: some rounding of some activation differs)."""
    import torch

    from nnfusion_amd import ops

    a, wq, s, zps = _case(m * 13 + n + k + group, m, n, k, 4, group, zp_tensor)
    a, wq, s = [torch.from_numpy(x).to(gpu) for x in (a, wq, s)]
    q = dict(bits=4, group=group, zp=5, zero_points=torch.from_numpy(zps).to(gpu) if zp_tensor else None)
    gen = torch.Generator(device="cpu").manual_seed(m + k)
    gamma = torch.randn(k, generator=gen).mul(0.1).add(1).half().to(gpu)
    res = torch.randn(m, n, generator=gen).half().to(gpu)
    ref = ops.wna16_gemm(ops.rms_norm(a, gamma, 1e-5), wq, s, **q)
    assert torch.equal(ops.wna16_gemm_fused(a, wq, s, rms_gamma=gamma, rms_eps=1e-5, **q), ref)
    y = ops.wna16_gemm_fused(a, wq, s, rms_gamma=gamma, rms_eps=1e-5, residual=res, out=res.clone(), **q)
    assert torch.equal(y, ops.elementwise("add", ref, res))


def test_fused_rows_with_the_output_over_the_input(gpu):
    """x = product(RMSNorm(x)) written over x: workgroups that finish must not change what others still read."""
    import torch

    from nnfusion_amd import ops

    m, k = 8, 4096
    a, wq, s, zps = _case(77, m, k, k, 4, 64, True)
    t = [torch.from_numpy(x).to(gpu) for x in (a, wq, s, zps)]
    gamma = torch.ones(k, dtype=torch.float16, device=gpu)
    ref = ops.wna16_gemm(ops.rms_norm(t[0], gamma), t[1], t[2], group=64, zero_points=t[3])
    ops.wna16_gemm_fused(t[0], t[1], t[2], group=64, zero_points=t[3], rms_gamma=gamma, out=t[0])
    assert torch.equal(t[0], ref)


# the plain tile kernel over ranges of K: every tile shape, a last range shorter than the others (and one that is no multiple of
# 128), ragged M and N; 4-bit zero points that start at any byte of a row
@pytest.mark.parametrize("m,n,k", [(40, 300, 4000), (100, 257, 15232), (130, 1030, 8192), (249, 256, 11008), (257, 520, 6304), (300, 3000, 5504),
                                   (600, 448, 14336), (1000, 256, 2080)])
@pytest.mark.parametrize("bits,group,zp_tensor", [(8, 32, True), (8, 128, False), (4, 32, True), (4, 64, False)])
def test_tile_kernel_over_ranges_of_k(gpu, m, n, k, bits, group, zp_tensor):
    """With the workspace it prefers against the oracle, and with any smaller one (fewer ranges, or one)."""
    import torch

    from nnfusion_amd import ops

    if k % group:
        pytest.skip("K is not a multiple of the group")
    a, wq, s, zps = _case(m + n + k + bits, m, n, k, bits, group, zp_tensor)
    zp = 7 if bits == 4 else 131
    ref = oracle.wna16_gemm(a, wq, s, bits, group, zp=zp, zero_points=zps, f32_out=True)
    t = [torch.from_numpy(x).to(gpu) for x in (a, wq, s)]
    tz = None if zps is None else torch.from_numpy(zps).to(gpu)
    want = ops.wna16_workspace_bytes(m, n, k, bits, group, tz)
    for nbytes in {want, want // 2, 16}:
        y = ops.wna16_gemm(*t, bits=bits, group=group, zp=zp, zero_points=tz,
                           workspace=torch.empty(max(16, nbytes), dtype=torch.uint8, device=gpu))
        torch.cuda.synchronize()
        _check(y.cpu().numpy(), ref)


def test_reduction_pass_over_more_rows_than_a_grid_has(gpu):
    """A tall, narrow product whose plan takes two ranges of K: the pass that adds them up, above 65535 rows (what other
    launches limit a grid to in y)."""
    import torch

    from nnfusion_amd import ops

    m, n, k, group = 65600, 100, 8192, 128
    assert ops.wna16_workspace_bytes(m, n, k, 8, group) >= 2 * m * n * 4
    gen = torch.Generator(device=gpu).manual_seed(m)
    a = torch.randn((m, k), generator=gen, device=gpu, dtype=torch.float16)
    _, wq, s, _ = _case(17, 1, n, k, 8, group, False)
    y = ops.wna16_gemm(a, torch.from_numpy(wq).to(gpu), torch.from_numpy(s).to(gpu), bits=8, group=group, zp=128)
    rows = [0, 1, 64, 4095, 65533, 65534, 65535, 65536, m - 1]
    _check(y[rows].cpu().numpy(), oracle.wna16_gemm(a[rows].cpu().numpy(), wq, s, 8, group, zp=128, f32_out=True))
    torch.cuda.synchronize()
