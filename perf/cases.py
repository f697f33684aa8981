"""The work that programs built on this package have it do, as cases that can be timed and compared.

Every case goes through ``nnfusion_amd.ops`` the way a user's program calls it.  Four kinds:

``linear``  one quantized linear layer, fp16 activations x 4- or 8-bit weights (the QuantDot node);
``decoder`` the linear layers of a stack of Llama-style decoder layers: RMSNorm + QKV, output projection + residual, the
            fused MLP block.  Attention itself is not this package's: its output is an input of the case;
``nodes``   the MLP block of a graph whose gate product is also a result, so that no fusion pattern takes it: RMSNorm, gate, up,
            Swish, Multiply, down, Add as nodes of their own;
``w8a8``    one int8 x int8 linear layer with per-token and per-channel scales, or its raw int32 accumulators.

``keep``: a serving loop that holds its outputs, workspace and synchronisation words (as generated code does); without
it the plain call, which allocates what it needs.  ``graph``: the pass is recorded once into a HIP graph and replayed.

Distributions: activations N(0, 1), weights uniform over their range, scales uniform[0.005, 0.02], zero point 8 (or one
per group, uniform), RMSNorm weights N(1, 0.1); W8A8 operands uniform[-127, 127] and scales uniform[0.001, 0.01].
"""
import math

import torch

from nnfusion_amd import _lib, ops

EPS = 1e-6


def _linear(name, m, n, k, bits=4, group=128, zero_points=False, keep=True):
    return {"name": name, "kind": "linear", "m": m, "n": n, "k": k, "bits": bits, "group": group, "zero_points": zero_points,
            "keep": keep}


def _decoder(name, m, hidden, qkv, attn, inter, layers, bits=4, group=128, zero_points=False, graph=False):
    return {"name": name, "kind": "decoder", "m": m, "hidden": hidden, "qkv": qkv, "attn": attn, "inter": inter,
            "layers": layers, "bits": bits, "group": group, "zero_points": zero_points, "graph": graph}


def listed():
    return [
        # the smallest call there is: one token through one square layer
        _linear("linear_m1", 1, 4096, 4096),
        # single-stream decoding, Llama-7B sizes, called layer by layer
        _decoder("decode_m1", 1, 4096, 12288, 4096, 11008, 4),
        # batched decoding of the same model in a captured graph, as serving loops run it
        _decoder("decode_m16_graph", 16, 4096, 12288, 4096, 11008, 4, graph=True),
        # one of two tensor-parallel shards: the down projection's K (5504) is no multiple of 256
        _decoder("decode_tp2_m6", 6, 4096, 6144, 2048, 5504, 4),
        # a larger, odd decoding batch (continuous batching, speculative verification)
        _decoder("decode_m45", 45, 4096, 12288, 4096, 11008, 2),
        # batched decoding with weights in groups of 64 and a zero point per group (MatMulNBits' asymmetric form)
        _decoder("decode_g64_zp_m8", 8, 4096, 12288, 4096, 11008, 2, group=64, zero_points=True),
        # one chunk of a chunked prefill: 256 tokens through a whole layer
        _decoder("prefill_m256", 256, 4096, 12288, 4096, 11008, 1),
        # a prompt of odd length through an MLP block that stayed unfused, groups of 32 with zero points, plain calls
        {"name": "nodes_g32_zp_m1000", "kind": "nodes", "m": 1000, "hidden": 4096, "inter": 11008, "bits": 4, "group": 32,
         "zero_points": True},
        # the largest product: a long prefill through a square layer
        _linear("prefill_m4096", 4096, 8192, 8192),
        # 8-bit weights with fp16 activations, a ragged prompt, plain call
        _linear("linear_w8_m300", 300, 11008, 4096, bits=8, keep=False),
        # int8 x int8: batched decoding and a ragged prefill
        {"name": "w8a8_m32", "kind": "w8a8", "m": 32, "n": 8192, "k": 8192, "raw": False, "keep": True},
        {"name": "w8a8_m2000", "kind": "w8a8", "m": 2000, "n": 12288, "k": 4096, "raw": False, "keep": True},
    ]


def _log_uniform(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def _quant(rng):
    """Block parameters: the 4-bit / groups-of-128 / scalar-zero-point form most of the time."""
    if rng.random() < 0.6:
        return {"bits": 4, "group": 128, "zero_points": False}
    return {"bits": rng.choice((4, 4, 8)), "group": rng.choice((32, 64, 128)), "zero_points": rng.random() < 0.6}


def _width(rng, low, high):
    """Columns of a layer: usually a multiple of 64, now and then any number."""
    n = int(_log_uniform(rng, low, high))
    return max(low, n // 64 * 64) if rng.random() < 0.75 else n


def draw(rng):
    """One more case of the ranges: 1 .. 4096 tokens, layers of 256 .. 16384 columns and K = 512 .. 16384 (stacks of decoder
    layers: hidden sizes 1024 .. 8192, whole or as one of 2 or 4 shards; up to 512 tokens)."""
    while True:
        kind = rng.choice(("linear", "linear", "linear", "decoder", "decoder", "decoder", "nodes", "w8a8", "w8a8"))
        if kind == "linear":
            case = {"kind": kind, "m": int(_log_uniform(rng, 1, 4097)), "n": _width(rng, 256, 16384),
                    "k": 128 * int(_log_uniform(rng, 4, 129)), **_quant(rng), "keep": rng.random() < 0.7}
        elif kind == "w8a8":
            case = {"kind": kind, "m": int(_log_uniform(rng, 1, 4097)), "n": _width(rng, 256, 16384),
                    "k": 128 * int(_log_uniform(rng, 4, 129)), "raw": rng.random() < 0.2, "keep": rng.random() < 0.7}
        else:
            hidden = 128 * int(_log_uniform(rng, 8, 65))
            shards = rng.choice((1, 1, 2, 4))
            inter = 128 * max(2, int(hidden * rng.uniform(2.5, 4.0) / shards / 128))
            if kind == "nodes":
                case = {"kind": kind, "m": int(_log_uniform(rng, 1, 2049)), "hidden": hidden, "inter": inter, **_quant(rng)}
            else:
                attn = 128 * max(1, hidden // shards // 128)
                kv = 128 * max(1, attn // rng.choice((1, 4)) // 128)
                layers = rng.choice((1, 2, 4))
                case = {"kind": kind, "m": int(_log_uniform(rng, 1, 513)), "hidden": hidden, "qkv": attn + 2 * kv,
                        "attn": attn, "inter": inter, "layers": layers, **_quant(rng), "graph": rng.random() < 0.25}
        w = work(case)
        if w["flops"] <= 3.5e11 and w["bytes"] <= 420e6:
            return case


class _Maker:
    def __init__(self, seed):
        self.dev = torch.device("cuda")
        self.gen = torch.Generator(device=self.dev)
        self.gen.manual_seed(seed)

    def normal(self, shape, mean=0.0, std=1.0):
        t = torch.randn(shape, generator=self.gen, device=self.dev, dtype=torch.float32)
        return t.mul_(std).add_(mean).to(torch.float16)

    def uniform(self, shape, low, high, dtype):
        t = torch.rand(shape, generator=self.gen, device=self.dev, dtype=torch.float32)
        return t.mul_(high - low).add_(low).to(dtype)

    def integers(self, shape, low, high, dtype):
        return torch.randint(low, high, shape, generator=self.gen, device=self.dev, dtype=dtype)

    def weights(self, n, k, case):
        """(wq, scales, zero points or None) of one layer; packed bytes are uniform, so the weights in them are."""
        bits, group = case["bits"], case["group"]
        wq = self.integers((n, k * bits // 8), 0, 256, torch.uint8)
        scales = self.uniform((n, k // group), 0.005, 0.02, torch.float16)
        zp = self.integers((n, (k // group * bits + 7) // 8), 0, 256, torch.uint8) if case["zero_points"] else None
        return wq, scales, zp

    def buffer(self, *shape, dtype=torch.float16):
        return torch.empty(shape, dtype=dtype, device=self.dev)

    def workspace(self, nbytes):
        return torch.empty(max(int(nbytes), 16), dtype=torch.uint8, device=self.dev)


def _scalar_zero_point(case):
    return 8 if case["bits"] == 4 else 128


def _plain(case):
    return case["bits"] == 4 and case["group"] == 128 and not case["zero_points"]


def prepare(case, seed):
    mk = _Maker(seed)
    state = {"case": case}
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        state["a"] = mk.normal((m, k))
        state["w"] = mk.weights(n, k, case)
        if case["keep"]:
            state["out"] = mk.buffer(m, n)
            state["ws"] = mk.workspace(ops.wna16_workspace_bytes(m, n, k, case["bits"], case["group"], state["w"][2]))
            state["sync"] = ops.sync_flags(mk.dev)
    elif kind == "w8a8":
        m, n, k = case["m"], case["n"], case["k"]
        state["a"] = mk.integers((m, k), -127, 128, torch.int8)
        state["b"] = mk.integers((n, k), -127, 128, torch.int8)
        state["s_tok"] = mk.uniform((m,), 0.001, 0.01, torch.float32)
        state["s_ch"] = mk.uniform((n,), 0.001, 0.01, torch.float32)
        if case["keep"]:
            state["out"] = mk.buffer(m, n, dtype=torch.int32 if case["raw"] else torch.float16)
            state["sync"] = ops.sync_flags(mk.dev)
            _, plan = ops._plan_arg(None, state["sync"])
            state["ws"] = mk.workspace(_lib.kernels().nnf_w8a8_gemm_variant_workspace_bytes(m, n, k, 0, plan))
    elif kind == "nodes":
        m, hidden, inter = case["m"], case["hidden"], case["inter"]
        state["x"] = mk.normal((m, hidden))
        state["gamma"] = mk.normal((hidden,), 1.0, 0.1)
        state["gate"], state["up"] = mk.weights(inter, hidden, case), mk.weights(inter, hidden, case)
        state["down"] = mk.weights(hidden, inter, case)
    else:
        _prepare_decoder(state, case, mk)
    return state


def _prepare_decoder(state, case, mk):
    m, hidden, qkv, attn, inter = (case[f] for f in ("m", "hidden", "qkv", "attn", "inter"))
    bits, group = case["bits"], case["group"]
    state["x"] = mk.normal((m, hidden))
    state["layers"] = [
        {"g_in": mk.normal((hidden,), 1.0, 0.1), "qkv": mk.weights(qkv, hidden, case), "attn": mk.normal((m, attn)),
         "o": mk.weights(hidden, attn, case), "g_mlp": mk.normal((hidden,), 1.0, 0.1),
         "gate_up": mk.weights(2 * inter, hidden, case), "down": mk.weights(hidden, inter, case),
         "qkv_out": mk.buffer(m, qkv), "mid": mk.buffer(m, hidden), "out": mk.buffer(m, hidden)}
        for _ in range(case["layers"])]
    lib = _lib.kernels()
    if _plain(case):
        state["sync"] = ops.sync_flags(mk.dev)
        need = [lib.nnf_w4a16_gemm_fused_workspace_bytes(m, n, k, group, 0) +
                lib.nnf_w4a16_gemm_variant_workspace_bytes(m, n, k, group, 0, None) for n, k in ((qkv, hidden), (hidden, attn))]
        need.append(lib.nnf_fused_mlp_w4a16_workspace_bytes(m, hidden, inter, group))
    else:
        zero = [state["layers"][0][w][2] for w in ("qkv", "o", "gate_up", "down")]
        keep, q = zip(*(ops._quant_arg(bits, group, _scalar_zero_point(case), z) for z in zero))
        need = [lib.nnf_wna16_gemm_fused_workspace_bytes(m, qkv, hidden, q[0], 0),
                lib.nnf_wna16_gemm_fused_workspace_bytes(m, hidden, attn, q[1], 0),
                lib.nnf_fused_mlp_wna16_workspace_bytes(m, hidden, inter, q[2], q[3])]
        del keep
    state["ws"] = mk.workspace(max(need))
    if case["graph"]:
        _decoder_pass(state, case)  # what is loaded on first use is loaded outside the capture
        torch.cuda.synchronize()
        state["replay"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["replay"]):
            state["outputs"] = _decoder_pass(state, case)


def _decoder_pass(state, case):
    bits, group, zp, ws = case["bits"], case["group"], _scalar_zero_point(case), state["ws"]
    x = state["x"]
    if _plain(case):
        sync = state["sync"]
        for layer in state["layers"]:
            (wq, sq, _), (wo, so, _) = layer["qkv"], layer["o"]
            (wgu, sgu, _), (wd, sd, _) = layer["gate_up"], layer["down"]
            ops.w4a16_gemm_fused(x, wq, sq, group, zp, rms_gamma=layer["g_in"], rms_eps=EPS, out=layer["qkv_out"],
                                 workspace=ws, sync=sync)
            x = ops.w4a16_gemm_fused(layer["attn"], wo, so, group, zp, residual=x, out=layer["mid"], workspace=ws, sync=sync)
            x = ops.fused_mlp_w4a16(x, layer["g_mlp"], wgu, sgu, wd, sd, EPS, group, zp, out=layer["out"], workspace=ws,
                                    sync=sync)
    else:
        for layer in state["layers"]:
            (wq, sq, zq), (wo, so, zo) = layer["qkv"], layer["o"]
            (wgu, sgu, zgu), (wd, sd, zd) = layer["gate_up"], layer["down"]
            ops.wna16_gemm_fused(x, wq, sq, bits, group, zp, zq, rms_gamma=layer["g_in"], rms_eps=EPS, out=layer["qkv_out"],
                                 workspace=ws)
            x = ops.wna16_gemm_fused(layer["attn"], wo, so, bits, group, zp, zo, residual=x, out=layer["mid"], workspace=ws)
            x = ops.fused_mlp_wna16(x, layer["g_mlp"], wgu, sgu, wd, sd, bits, group, zp, zgu, zd, eps=EPS, out=layer["out"],
                                    workspace=ws)
    return {"qkv": [layer["qkv_out"] for layer in state["layers"]], "x": x}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        wq, scales, zero = state["w"]
        return ops.wna16_gemm(state["a"], wq, scales, case["bits"], case["group"], _scalar_zero_point(case), zero,
                              out=state.get("out"), workspace=state.get("ws"), sync=state.get("sync"))
    if kind == "w8a8":
        if case["raw"]:
            return ops.w8a8_gemm_acc(state["a"], state["b"], out=state.get("out"), workspace=state.get("ws"),
                                     sync=state.get("sync"))
        return ops.w8a8_gemm(state["a"], state["s_tok"], state["b"], state["s_ch"], out=state.get("out"),
                             workspace=state.get("ws"), sync=state.get("sync"))
    if kind == "nodes":
        quant = (case["bits"], case["group"], _scalar_zero_point(case))
        normed = ops.rms_norm(state["x"], state["gamma"], EPS)
        gate = ops.wna16_gemm(normed, *state["gate"][:2], *quant, state["gate"][2])
        up = ops.wna16_gemm(normed, *state["up"][:2], *quant, state["up"][2])
        h = ops.elementwise("multiply", ops.elementwise("swish", gate), up)
        down = ops.wna16_gemm(h, *state["down"][:2], *quant, state["down"][2])
        return {"gate": gate, "y": ops.elementwise("add", down, state["x"])}
    if case["graph"]:
        state["replay"].replay()
        return state["outputs"]
    return _decoder_pass(state, case)


def _weight_bytes(n, k, case):
    groups = k // case["group"]
    zero = n * ((groups * case["bits"] + 7) // 8) if case["zero_points"] else 0
    return n * k * case["bits"] // 8 + n * groups * 2 + zero


def work(case):
    """Weights, inputs and outputs once each; activations between the products of one pass are not counted."""
    m, kind = case["m"], case["kind"]
    if kind == "linear":
        n, k = case["n"], case["k"]
        return {"bytes": _weight_bytes(n, k, case) + 2 * m * (k + n), "flops": 2 * m * n * k}
    if kind == "w8a8":
        n, k = case["n"], case["k"]
        return {"bytes": n * k + m * k + (0 if case["raw"] else 4 * (n + m)) + (4 if case["raw"] else 2) * m * n,
                "flops": 2 * m * n * k}
    hidden, inter = case["hidden"], case["inter"]
    if kind == "nodes":
        weights = 2 * _weight_bytes(inter, hidden, case) + _weight_bytes(hidden, inter, case)
        return {"bytes": weights + 2 * hidden + 2 * m * (2 * hidden + inter), "flops": 6 * m * hidden * inter}
    qkv, attn, layers = case["qkv"], case["attn"], case["layers"]
    weights = (_weight_bytes(qkv, hidden, case) + _weight_bytes(hidden, attn, case) + _weight_bytes(2 * inter, hidden, case) +
               _weight_bytes(hidden, inter, case))
    return {"bytes": layers * (weights + 4 * hidden + 2 * m * (qkv + attn)) + 4 * m * hidden,
            "flops": layers * 2 * m * (qkv * hidden + hidden * attn + 3 * inter * hidden)}


def tolerance(case):
    """Linear layers: fp16 results, weights rounded to fp16 or not before fp32 sums.  Stacks: the same once per product, and
    the rounding of the fp16 tensors between them.  W8A8: exact int32 sums; the fp16 results differ by a rounding at most."""
    if case["kind"] == "w8a8":
        return "exact" if case["raw"] else {"rel": 5e-4, "max": 2e-3}
    if case["kind"] == "linear":
        return {"rel": 2e-3, "max": 1e-2}
    return {"rel": 5e-3, "max": 5e-2}
