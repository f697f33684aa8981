"""How the K-streaming kernels are called, whatever their sizes: on a side stream, in a captured graph, with an output that overlaps the activations
(RMSNorm then goes ahead, by way of a copy), with infinities and NaN in one activation row."""
import numpy as np
import pytest

import oracle
from nnfusion_amd import datagen

pytestmark = pytest.mark.gpu

# (bits, group, zero points): groups of 128 with a scalar zero point, others, 8 bits
FORMS = [(4, 128, False), (4, 64, True), (8, 32, True)]


def _t(gpu, *arrays):
    import torch

    return [None if a is None else torch.from_numpy(np.ascontiguousarray(a)).to(gpu) for a in arrays]


def _case(seed, m, n, k, bits, group, zero_points):
    if (bits, group, zero_points) == (4, 128, False):
        return (*datagen.w4a16_case(seed, m, n, k), None)
    return datagen.wna16_case(seed, m, n, k, bits, group, zero_points)


def _products(gpu, m, n, k, bits, group, zero_points):
    """a plain product, one with RMSNorm and one with SiLU-gate, as calls without arguments into buffers of their own; the buffers"""
    import torch

    from nnfusion_amd import ops

    a, wq, s, z = _t(gpu, *_case(4, m, 2 * n, k, bits, group, zero_points))
    gamma = torch.full((k,), 0.75, dtype=torch.float16, device=gpu)
    zp = 7 if bits == 4 else 119
    outs = [torch.zeros(m, n, dtype=torch.float16, device=gpu) for _ in range(3)]
    ws = torch.empty(64 << 20, dtype=torch.uint8, device=gpu)
    sync = ops.sync_flags(gpu)
    w1, s1, z1 = wq[:n], s[:n], None if z is None else z[:n]
    calls = [lambda: ops.wna16_gemm(a, w1, s1, bits, group, zp, z1, out=outs[0], workspace=ws, sync=sync),
             lambda: ops.wna16_gemm_fused(a, w1, s1, bits, group, zp, z1, rms_gamma=gamma, out=outs[1], workspace=ws),
             lambda: ops.wna16_gemm_fused(a, wq, s, bits, group, zp, z, rms_gamma=gamma, act=1, out=outs[2], workspace=ws)]
    return calls, outs, a


@pytest.mark.parametrize("bits,group,zero_points", FORMS)
@pytest.mark.parametrize("m,n,k", [(9, 4096, 2816), (33, 4096, 11008), (100, 1024, 1280)])
def test_side_stream_and_captured_graph(gpu, m, n, k, bits, group, zero_points):
    """The same bits as on the default stream; three replays, each with new activations, after eager work and a synchronization."""
    import torch

    print(f"case kstream calls M={m} N={n} K={k} bits={bits} group={group}", flush=True)
    calls, outs, a = _products(gpu, m, n, k, bits, group, zero_points)
    for call in calls:
        call()
    torch.cuda.synchronize()
    ref = [y.clone() for y in outs]
    for y in outs:
        y.zero_()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for call in calls:
            call()
    side.synchronize()
    assert all(torch.equal(y, r) for y, r in zip(outs, ref))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for call in calls:
            call()
    for _ in range(3):
        a.copy_(a.roll(1, 0))
        for call in calls:
            call()
        torch.cuda.synchronize()
        ref = [y.clone() for y in outs]
        for y in outs:
            y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(y, r) for y, r in zip(outs, ref))


@pytest.mark.parametrize("bits,group,zero_points", FORMS)
@pytest.mark.parametrize("m,k", [(12, 1152), (40, 2048), (40, 1280)])
def test_output_over_the_activations(gpu, m, k, bits, group, zero_points):
    """x = product(RMSNorm(x)) written over x, whole and shifted by eight rows: as with an output elsewhere.  (5e-3 of the RMS: RMSNorm inside the
    kernel and ahead of it round weights times gamma or normalised activations.  4 bits, groups of 128 and a scalar zero point: where the
    product takes normalised activations by way of a copy.)"""
    import torch

    from nnfusion_amd import ops

    if (bits, group, zero_points) == (4, 128, False) and k == 1280:
        pytest.skip("the tile GEMM reads the activations themselves")
    print(f"case overlap M={m} K={k} bits={bits} group={group}", flush=True)
    x, wq, s, z = _t(gpu, *_case(5, m, k, k, bits, group, zero_points))
    gamma = torch.ones(k, dtype=torch.float16, device=gpu)
    zp = 7 if bits == 4 else 119
    ws = torch.empty(64 << 20, dtype=torch.uint8, device=gpu)
    ref = ops.wna16_gemm_fused(x, wq, s, bits, group, zp, z, rms_gamma=gamma, workspace=ws).float()
    for shift in (0, 8):
        buffer = torch.zeros(m + 8, k, dtype=torch.float16, device=gpu)
        buffer[:m] = x
        y = ops.wna16_gemm_fused(buffer[:m], wq, s, bits, group, zp, z, rms_gamma=gamma, out=buffer[shift:shift + m], workspace=ws).float()
        assert float((y - ref).abs().max()) <= 5e-3 * float(ref.pow(2).mean().sqrt())


@pytest.mark.parametrize("bits,group,zero_points", FORMS)
@pytest.mark.parametrize("m,n,k", [(8, 72, 1792), (45, 300, 1280), (70, 40, 1152)])
def test_infinities_and_nan_stay_in_their_row(gpu, m, n, k, bits, group, zero_points):
    """Rows 1, 2 and the last hold an infinity, a NaN and both signs of infinity: their results are what the sums over K give (with
    RMSNorm NaN), every other row is as without them."""
    import torch

    from nnfusion_amd import ops

    print(f"case infinities M={m} N={n} K={k} bits={bits} group={group}", flush=True)
    a, wq, s, z = _case(6, m, n, k, bits, group, zero_points)
    zp = 7 if bits == 4 else 119
    bad = a.copy()
    bad[1, 5], bad[2, k - 1], bad[m - 1, 3], bad[m - 1, 700] = np.inf, np.nan, np.inf, -np.inf
    w = oracle.dequantize_wn(wq, s, bits, group, zp, z).astype(np.float64)
    with np.errstate(invalid="ignore"):
        ref = bad.astype(np.float64) @ w.T
    ta, tb, tw, ts, tz = _t(gpu, a, bad, wq, s, z)
    gamma = torch.ones(k, dtype=torch.float16, device=gpu)
    ws = torch.empty(64 << 20, dtype=torch.uint8, device=gpu)
    rows = [r for r in range(m) if r not in (1, 2, m - 1)]
    clean = ops.wna16_gemm(ta, tw, ts, bits, group, zp, tz, workspace=ws).cpu().numpy()
    y = ops.wna16_gemm(tb, tw, ts, bits, group, zp, tz, workspace=ws).cpu().numpy()
    assert np.array_equal(y[rows], clean[rows])
    for r in (1, 2, m - 1):
        assert np.array_equal(np.isnan(y[r]), np.isnan(ref[r])) and np.array_equal(np.isposinf(y[r]), np.isposinf(ref[r]))
        assert not np.isfinite(y[r]).any()
    clean = ops.wna16_gemm_fused(ta, tw, ts, bits, group, zp, tz, rms_gamma=gamma, workspace=ws).cpu().numpy()
    y = ops.wna16_gemm_fused(tb, tw, ts, bits, group, zp, tz, rms_gamma=gamma, workspace=ws).cpu().numpy()
    assert np.array_equal(y[rows], clean[rows]) and np.isnan(y[[1, 2, m - 1]]).all()


@pytest.mark.parametrize("m,n,k", [(9, 520, 2048), (64, 4100, 1280), (130, 1000, 1152)])
def test_w8a8_side_stream_and_captured_graph(gpu, m, n, k):
    import torch

    from nnfusion_amd import ops

    print(f"case w8a8 kstream calls M={m} N={n} K={k}", flush=True)
    a, s_tok, w, s_ch = _t(gpu, *datagen.w8a8_case(4, m, n, k))
    out = torch.zeros(m, n, dtype=torch.float16, device=gpu)
    ref = ops.w8a8_gemm(a, s_tok, w, s_ch)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        ops.w8a8_gemm(a, s_tok, w, s_ch, out=out)
    side.synchronize()
    assert torch.equal(out, ref)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.w8a8_gemm(a, s_tok, w, s_ch, out=out)
    for _ in range(3):
        a.copy_(a.roll(1, 0))
        ref = ops.w8a8_gemm(a, s_tok, w, s_ch)
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref)
