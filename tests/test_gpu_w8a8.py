"""W8A8 on the int8 MFMA: the int32 accumulators must be bit-identical to the CPU oracle (pure integer
arithmetic), and the fp16 output identical to fp16((float)acc * s_tok * s_ch) evaluated left to right."""
import numpy as np
import pytest

import oracle
from nnfusion_amd import datagen

pytestmark = pytest.mark.gpu


def _t(gpu, *arrays):
    import torch

    return [torch.from_numpy(np.ascontiguousarray(a)).to(gpu) for a in arrays]


# Kernel families, asked for per call through nnf_w8a8_gemm_variant where the family takes the shape (the library's own
# choice where it does not): "auto"; "skinny": the split-K M <= 16 kernel; "mfma_rows": the row-streaming MFMA kernel
# (2 <= M <= 32, K = 1024 .. 16384 in multiples of 256); otherwise the MFMA tile GEMM with a plan (tile_rows, k_parts):
# tiles of 256 x 256, 256 x 128 (third value: the columns), 128 x 128 or 64 x 256 outputs (0: the library's choice) and the
# number of K ranges (int32 partial sums, added exactly by the reduction pass); "auto-sync": the library's choice given
# synchronisation words (8 .. 32 rows with K from 8192: the row-streaming kernel over two ranges of K in one launch)
@pytest.fixture(params=["auto", "auto-sync", "skinny", "mfma_rows", (0, 0), (256, 1, 256), (256, 2, 256), (256, 1, 128), (256, 3, 128), (256, 0),
                        (128, 1), (128, 3), (64, 1), (64, 2)],
                ids=lambda p: p if isinstance(p, str) else "gemm-rows%d-parts%d" % p[:2] + ("-cols%d" % p[2] if len(p) > 2 else ""))
def path(request):
    return request.param


def _kw(path, m, n, k):
    """Keyword arguments of ops.w8a8_gemm / w8a8_gemm_acc for a fixture value."""
    from nnfusion_amd import ops

    if path == "skinny":
        return {"variant": "gemv_mfma"} if ops.w8a8_variant_supported(m, n, k, "gemv_mfma") else {}
    if path == "mfma_rows":
        return {"variant": "gemv_rows"} if m > 1 and ops.w8a8_variant_supported(m, n, k, "gemv_rows") else {}
    if path == "auto":
        return {}
    if path == "auto-sync":
        import torch

        return {"sync": ops.sync_flags(torch.device("cuda:0"))}
    return {"variant": "gemm_mfma", "plan": path}


def _words_left_zero(kw):
    return "sync" not in kw or int(kw["sync"].count_nonzero()) == 0


def _big_ws(gpu):
    import torch

    return torch.empty(64 << 20, dtype=torch.uint8, device=gpu)


@pytest.mark.parametrize("m,n,k", [
    (1, 64, 128), (1, 1000, 1024), (3, 17, 256), (16, 512, 8192), (32, 300, 512), (100, 257, 384),
    (256, 256, 128), (512, 1024, 2048), (1, 8192, 8192), (32, 4096, 4096),
    # M <= 16 with chunk counts that leave wavefronts partly idle, two passes over K per tile, many tiles
    (5, 200, 2176), (2, 100, 11008), (7, 48, 16384), (9, 1000, 8320), (1, 33000, 1024), (13, 8200, 4096),
    # ... and with K so short that the workgroup has fewer threads than a tile has outputs (two wavefronts, 9 .. 16 rows)
    (14, 4128, 128), (9, 100, 128), (16, 300, 128), (13, 64, 128), (8, 520, 128), (12, 1000, 128),
    # one activation row: rows shared by 1..8 wavefronts, ragged last K segment, fewer rows than wavefronts
    (1, 300, 4096), (1, 4096, 11008), (1, 100, 16384), (1, 50, 2048), (1, 513, 5248), (1, 2000, 24576), (1, 40, 1152),
    # 2 .. 32 rows through the row-streaming MFMA kernel: every K it takes, one and two blocks of 16 rows, ragged N,
    # a single tile, more tiles than CUs
    (2, 512, 2048), (16, 4111, 4096), (17, 1000, 6144), (32, 8192, 8192), (31, 16, 8192), (24, 12288, 4096),
    (8, 40000, 2048), (20, 77, 4096),
    # K that does not fill the last 2-KiB step, K above 8192
    (16, 4111, 11008), (5, 100, 1024), (9, 520, 2560), (32, 300, 7168), (24, 1000, 3584), (12, 2000, 14336), (16, 64, 16384),
    (17, 250, 5376), (32, 4111, 11008), (20, 300, 12288), (24, 100, 9216),
    # two ranges of K given synchronisation words: one to four tiles per workgroup, a last tile moved back, K = 16384
    (8, 4096, 8192), (32, 4111, 8192), (13, 6000, 16384), (24, 8192, 9216),
])
def test_accumulators_bit_exact(gpu, path, m, n, k):
    import torch

    from nnfusion_amd import ops

    print(f"case M={m} N={n} K={k} path={path}", flush=True)
    a, s_tok, w, s_ch = datagen.w8a8_case(0, m, n, k)
    ta, tw, tst, tsc = _t(gpu, a, w, s_tok, s_ch)
    ws = _big_ws(gpu)
    kw = _kw(path, m, n, k)
    acc = ops.w8a8_gemm_acc(ta, tw, workspace=ws, **kw).cpu().numpy()
    y = ops.w8a8_gemm(ta, tst, tw, tsc, workspace=ws, **kw).cpu().numpy()
    torch.cuda.synchronize()
    ref = oracle.w8a8_acc(a, w)
    assert np.array_equal(acc, ref)
    # the epilogue is a closed form of exact inputs: bit-identical fp16
    assert np.array_equal(y.view(np.uint16), oracle.w8a8_epilogue(ref, s_tok, s_ch).view(np.uint16))
    assert _words_left_zero(kw)


def test_extreme_values_do_not_overflow(gpu, path):
    """All operands at -127 / +127 with K = 8192: |acc| = 8192 * 127^2 = 132 128 768 < 2^31."""
    import torch

    from nnfusion_amd import ops

    m, n, k = 4, 48, 8192
    a = np.full((m, k), 127, np.int8)
    a[1] = -127
    w = np.full((n, k), 127, np.int8)
    w[::2] = -127
    ta, tw = _t(gpu, a, w)
    kw = _kw(path, m, n, k)
    acc = ops.w8a8_gemm_acc(ta, tw, workspace=_big_ws(gpu), **kw).cpu().numpy()
    torch.cuda.synchronize()
    assert np.array_equal(acc, oracle.w8a8_acc(a, w))
    assert _words_left_zero(kw)
    assert abs(int(acc[0, 1])) == 8192 * 127 * 127


@pytest.mark.parametrize("m", [512, 4096])
def test_full_size_sampled(gpu, m):
    """configs[3] at N = K = 8192: sampled output columns against the oracle bit for bit, and the
    checksum identity  sum_n acc[m, n] == A[m, :] . (sum_n W[n, :])  over the whole output in int64."""
    import torch

    from nnfusion_amd import ops

    n = k = 8192
    print(f"case M={m}", flush=True)
    a, s_tok, w, s_ch = datagen.w8a8_case(0, m, n, k)
    ta, tw = _t(gpu, a, w)
    acc = ops.w8a8_gemm_acc(ta, tw).cpu().numpy()
    torch.cuda.synchronize()
    cols = np.sort(np.random.default_rng(1).choice(n, 128, replace=False))
    assert np.array_equal(acc[:, cols], oracle.w8a8_acc(a, w[cols]))
    wsum = w.astype(np.int64).sum(axis=0)
    assert np.array_equal(acc.astype(np.int64).sum(axis=1), a.astype(np.int64) @ wsum)


def test_reduction_pass_over_more_rows_than_a_grid_has(gpu):
    """Two ranges of K asked for: the pass that adds them up above 65535 rows (what other launches limit a grid to in y)."""
    import torch

    from nnfusion_amd import ops

    m, n, k = 65537, 20, 512
    a, s_tok, w, s_ch = datagen.w8a8_case(0, m, n, k)
    ta, tw, tst, tsc = _t(gpu, a, w, s_tok, s_ch)
    kw = {"variant": "gemm_mfma", "plan": (256, 2, 128)}
    acc = ops.w8a8_gemm_acc(ta, tw, **kw).cpu().numpy()
    y = ops.w8a8_gemm(ta, tst, tw, tsc, **kw).cpu().numpy()
    torch.cuda.synchronize()
    ref = oracle.w8a8_acc(a, w)
    assert np.array_equal(acc, ref)
    assert np.array_equal(y.view(np.uint16), oracle.w8a8_epilogue(ref, s_tok, s_ch).view(np.uint16))


@pytest.mark.parametrize("m,n,k", [
    # one range of K, the 64-row tile writes its results itself: every remainder of rows and of columns by 2, 4, 8 (stores of 16
    # bytes and single ones), a single column, fewer columns than a wavefront's part of the tile, the shortest K
    (33, 12801, 128), (64, 12802, 256), (47, 12804, 512), (58, 12680, 512), (63, 12672, 384), (34, 1, 128), (40, 31, 128), (64, 257, 256),
    # ranges of K and the reduction pass: whole quads of columns, 1 .. 3 left over, fewer than four
    (33, 1001, 8192), (64, 1002, 8192), (45, 1003, 4096), (50, 1000, 8192), (64, 3, 8192), (60, 4, 8192)])
def test_64_row_tiles_at_ragged_columns(gpu, m, n, k):
    """Bit exact, nothing written beyond the outputs or the workspace the query asks for."""
    import torch

    from nnfusion_amd import _lib, ops

    a, s_tok, w, s_ch = datagen.w8a8_case(2, m, n, k)
    ta, tw, tst, tsc = _t(gpu, a, w, s_tok, s_ch)
    need = _lib.kernels().nnf_w8a8_gemm_workspace_bytes(m, n, k)
    ref = oracle.w8a8_acc(a, w)
    y_ref = oracle.w8a8_epilogue(ref, s_tok, s_ch)
    for dtype, run, want in ((torch.int32, lambda **kw: ops.w8a8_gemm_acc(ta, tw, **kw), ref),
                             (torch.float16, lambda **kw: ops.w8a8_gemm(ta, tst, tw, tsc, **kw), y_ref)):
        out = torch.full((m * n + 512,), 77, dtype=dtype, device=gpu)
        ws = torch.full((need + 4096,), 0x5A, dtype=torch.uint8, device=gpu)
        run(out=out, workspace=ws[:need])
        torch.cuda.synchronize()
        assert np.array_equal(out[:m * n].cpu().numpy().reshape(m, n), want)
        assert bool((out[m * n:] == 77).all()) and bool((ws[need:] == 0x5A).all())


# Whole tiles of 256 x 192, 192 x 256, 128 x 256, 192 x 128 and 128 x 192 (tests/cpp/test_host.cpp holds the plan to that): the last tile of
# rows and of columns ragged, columns no multiple of eight (rows stored an element at a time), one round of tiles and more
@pytest.mark.parametrize("m,n,k", [(1012, 8412, 512), (964, 9008, 1152), (531, 13308, 512), (1411, 5400, 640), (538, 11108, 512), (590, 9984, 1152),
                                   (262, 12544, 512), (455, 8247, 640), (396, 11112, 896), (595, 8476, 896), (1354, 4170, 896)])
def test_tiles_of_192_rows_or_columns(gpu, m, n, k):
    """Accumulators against products in float64 (exact: below 2^53), the fp16 results bit for bit."""
    import torch

    from nnfusion_amd import ops

    print(f"case M={m} N={n} K={k}", flush=True)
    gen = torch.Generator(device=gpu)
    gen.manual_seed(m + n + k)
    a, w = (torch.randint(-127, 128, s, generator=gen, device=gpu, dtype=torch.int8) for s in ((m, k), (n, k)))
    s_tok, s_ch = (torch.rand(s, generator=gen, device=gpu) * 0.009 + 0.001 for s in (m, n))
    ref = (a.double() @ w.double().t()).to(torch.int32)
    assert torch.equal(ops.w8a8_gemm_acc(a, w), ref)
    # ((float)acc * s_tok) * s_ch, rounded to fp32 each time, then to fp16
    y = (ref.float() * s_tok[:, None] * s_ch[None, :]).half()
    assert torch.equal(ops.w8a8_gemm(a, s_tok, w, s_ch), y)
