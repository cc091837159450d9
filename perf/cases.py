"""The work that a program asks of this framework, as cases that can be timed and compared.

Every case goes through a public entry point: the modules of ``lucid_amd.nn.quantized``, the
functions of ``lucid_amd.quantization``, the model runtimes of ``lucid_amd.bench_configs`` or the
C ABI of ``include/lq_api.h``.  Sizes are those of the repository's own benchmark (4096-wide
square Linears, the 4096 / 11008 block, the 784-256-10 MLP, ResNet-18 at 224 x 224, the six-layer
decoder) and ragged ones of the same ranges.

``listed()`` names the cases, ``draw()`` gives more of the same ranges, ``prepare()`` makes what
a program holds before the call, ``run()`` is one pass, ``exact()`` the same result in 64 bits
with plain torch.
"""

from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import lucid_amd as L
import lucid_amd.nn as nn
import lucid_amd.nn.quantized as nnq
import lucid_amd.nn.quantized.dynamic as nnqd
import lucid_amd.quantization as Q
from lucid_amd import _C, bench_configs
from lucid_amd.graphs import CapturedForward

HIDDEN, FFN = 4096, 11008


def listed():
    return [
        # the smallest program: a dynamically quantized MLP on one batch, module calls and all
        {"name": "mlp_dynamic_b64", "kind": "mlp", "batch": 64, "d_in": 784, "d_hidden": 256, "d_out": 10},
        # a dynamic int8 Linear over a ragged prompt (float in, float out)
        {"name": "dynamic_linear_2000", "kind": "dynamic_linear", "M": 2000, "K": HIDDEN, "N": FFN},
        # a static int8 Linear between two quantized layers: codes in, codes out
        {"name": "static_linear_4096", "kind": "static_linear", "M": 4096, "K": 4096, "N": 4096},
        # a static int8 Linear that gets a float input: the weight-only product, then its grid
        {"name": "float_input_linear_512", "kind": "float_input_linear", "M": 512, "K": HIDDEN, "N": HIDDEN},
        # one decode step's weight-only products of a transformer block, 16 sequences
        {"name": "decode_block_int8_m16", "kind": "decode_block", "M": 16, "hidden": HIDDEN, "ffn": FFN,
         "dtype": "float32"},
        # the same block with 4-bit groups, one sequence in half precision
        {"name": "decode_block_group4_m1", "kind": "decode_block_group", "M": 1, "hidden": HIDDEN, "ffn": FFN,
         "bits": 4, "group": 64, "dtype": "float16"},
        # the default engine's Linear (8-bit groups of 64) over a prompt
        {"name": "group_linear_1024", "kind": "group_linear", "M": 1024, "K": HIDDEN, "N": HIDDEN, "bits": 8,
         "group": 64, "dtype": "float32"},
        # the input gradient through a frozen 4-bit Linear, as adapter training asks for it
        {"name": "group_backward_2048", "kind": "group_backward", "M": 2048, "K": HIDDEN, "N": HIDDEN, "bits": 4,
         "group": 64, "dtype": "float32"},
        # calibrate a range, put a large ragged tensor on its grid and read it back
        {"name": "calibrate_100m", "kind": "calibrate", "rows": 8191, "cols": 12289, "per_channel": False,
         "grid": "qint8"},
        # a residual block's convolution, codes to codes
        {"name": "conv3x3_128_b32", "kind": "conv", "batch": 32, "c_in": 128, "c_out": 128, "height": 28, "width": 28,
         "k": 3, "stride": 1, "groups": 1},
        # a whole static int8 network on one batch of images
        {"name": "resnet18_b32", "kind": "resnet18", "batch": 32, "image": 224},
        # a whole int8 decoder: a prompt, then tokens one at a time
        {"name": "decoder_b8_512_8", "kind": "decoder", "batch": 8, "prompt": 512, "steps": 8},
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _features(rng, lo, hi):
    """Feature counts: mostly multiples of 64 or 16, some odd."""
    n = _log(rng, lo, hi)
    step = rng.choice((64, 64, 16, 1))
    return max(step, n // step * step)


def draw(rng):
    kind = rng.choice(("mlp", "dynamic_linear", "dynamic_linear", "static_linear", "static_linear",
                       "float_input_linear", "float_input_linear", "decode_block", "decode_block",
                       "decode_block_group", "decode_block_group", "group_linear", "group_linear", "group_linear",
                       "group_backward", "group_backward", "calibrate", "calibrate", "conv", "conv", "resnet18",
                       "decoder"))
    dtype = rng.choice(("float32", "float16"))
    if kind == "mlp":
        return {"kind": kind, "batch": _log(rng, 1, 512), "d_in": _features(rng, 64, 4096),
                "d_hidden": _features(rng, 64, 4096), "d_out": _features(rng, 8, 1024)}
    if kind in ("dynamic_linear", "static_linear"):
        K, N = _features(rng, 256, 8192), _features(rng, 256, 4096)
        return {"kind": kind, "M": min(_log(rng, 1, 4096), 2**36 // (K * N)), "K": K, "N": N}
    if kind == "float_input_linear":
        return {"kind": kind, "M": _log(rng, 1, 1024), "K": _features(rng, 256, HIDDEN),
                "N": _features(rng, 256, HIDDEN)}
    if kind == "decode_block":
        h = 64 * _log(rng, 8, 64)
        return {"kind": kind, "M": _log(rng, 1, 16), "hidden": h, "ffn": 16 * rng.randint(h // 8, h // 6),
                "dtype": dtype}
    if kind == "decode_block_group":
        h = 128 * _log(rng, 4, 32)
        return {"kind": kind, "M": _log(rng, 1, 16), "hidden": h, "ffn": 128 * rng.randint(h // 64, h // 48),
                "bits": rng.choice((4, 8)), "group": rng.choice((32, 64, 64, 128)), "dtype": dtype}
    if kind == "group_linear":
        g = rng.choice((32, 64, 64, 128))
        return {"kind": kind, "M": _log(rng, 1, 2048), "K": g * _log(rng, 256 // g, HIDDEN // g),
                "N": _features(rng, 256, HIDDEN), "bits": rng.choice((4, 8)), "group": g,
                "dtype": rng.choice(("float32", "float16", "bfloat16"))}
    if kind == "group_backward":
        g = rng.choice((32, 64, 64, 128))
        return {"kind": kind, "M": _log(rng, 16, 2048), "K": g * _log(rng, 256 // g, HIDDEN // g),
                "N": _features(rng, 256, HIDDEN), "bits": rng.choice((4, 8)), "group": g, "dtype": dtype}
    if kind == "calibrate":
        return {"kind": kind, "rows": _log(rng, 16, 8192), "cols": _log(rng, 64, 12288),
                "per_channel": rng.random() < 0.5, "grid": rng.choice(("qint8", "quint8"))}
    if kind == "conv":
        k = rng.choice((1, 3, 3, 3, 5))
        size = rng.choice((7, 14, 28, 56, rng.randint(7, 60)))
        c = rng.choice((16, 32, 64, 128, 256, 512)) if rng.random() < 0.8 else rng.randint(3, 200)
        c = min(c, 8192 // size)
        return {"kind": kind, "batch": _log(rng, 1, 32), "c_in": c, "c_out": rng.choice((c, 2 * c, 96)),
                "height": size, "width": max(7, size - rng.choice((0, 0, 1, 3))), "k": k,
                "stride": rng.choice((1, 1, 2)), "groups": 1}
    if kind == "resnet18":
        return {"kind": kind, "batch": _log(rng, 1, 32), "image": rng.choice((160, 192, 224))}
    return {"kind": kind, "batch": rng.randint(1, 8), "prompt": _log(rng, 16, 512), "steps": rng.randint(1, 8)}


# ------------------------------------------------------------------------------ inputs

_NP = {torch.float32: np.dtype(np.float32), torch.float16: np.dtype(np.float16), torch.bfloat16: L.bfloat16,
       torch.int8: np.dtype(np.int8), torch.int32: np.dtype(np.int32)}
_CODE = {"float32": _C.F32, "float16": _C.F16}


def _own(t):
    """A torch tensor's values in a tensor of the framework."""
    t = t.contiguous()
    out = L.empty(tuple(t.shape), _NP[t.dtype], "gpu")
    _C.call("lq_memcpy_d2d", out.data_ptr(), t.data_ptr(), t.numel() * t.element_size(), None)
    torch.cuda.current_stream().synchronize()
    return out


class _Shared:
    """A framework tensor's memory, as torch takes it over without a copy."""

    def __init__(self, t, typestr):
        self.tensor = t
        self.__cuda_array_interface__ = {"shape": tuple(t.shape), "typestr": typestr, "data": (t.data_ptr(), False),
                                         "version": 2}


def _view(t):
    """A framework tensor as a torch tensor over the same memory."""
    if t.dtype == L.bfloat16:
        return torch.as_tensor(_Shared(t, "<i2"), device="cuda").view(torch.bfloat16)
    return torch.as_tensor(_Shared(t, t.dtype.str), device="cuda")


def _codes(t):
    """The integer codes of a quantized layer's result."""
    return _view(t.quant_source.codes)


class _Make:
    """Seeded inputs on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, *shape, std=1.0):
        return torch.randn(shape, generator=self.g, device="cuda") * std

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, generator=self.g, device="cuda") * (hi - lo) + lo

    def activations(self, M, K):
        """Rows as a norm leaves them: unit variance, one feature in 64 six times larger."""
        wide = 1.0 + 5.0 * (torch.rand((K,), generator=self.g, device="cuda") < 1 / 64)
        return self.normal(M, K) * wide

    def weight(self, N, *rest):
        """Symmetric per-row int8 codes and scales of a normal weight of variance 1 / fan-in."""
        fan = math.prod(rest)
        codes = (self.normal(N, *rest) * 32).round().clamp(-127, 127).to(torch.int8)
        return codes, self.uniform(0.8, 1.2, N) / (32 * math.sqrt(fan))

    def words(self, N, K, bits, group):
        """Packed group-wise codes with the scales and biases of such a weight."""
        words = torch.randint(-2**31, 2**31, (N, K * bits // 32), generator=self.g, device="cuda",
                              dtype=torch.int64).to(torch.int32)
        scales = self.uniform(0.8, 1.2, N, K // group) * (6 / (2**bits - 1) / math.sqrt(K))
        biases = scales * (-(2**bits - 1) / 2) + self.normal(N, K // group, std=0.05 / math.sqrt(K))
        return words, scales, biases


def _layer(layer, m, bias, out_scale=None, out_zero=None):
    """Fill a quantized layer's buffers, as loading a state dict does."""
    codes, scale = m
    layer.register_buffer("weight_int8", _own(codes))
    layer.register_buffer("weight_scale", _own(scale))
    layer.register_buffer("weight_zero_point", _own(torch.zeros_like(scale)))
    layer.register_buffer("bias", _own(bias))
    if out_scale is not None:
        layer.register_buffer("scale", L.tensor(np.float32(out_scale), device="gpu"))
        layer.register_buffer("zero_point", L.tensor(np.float32(out_zero), device="gpu"))
    return layer


_stream = None


def _the_stream():
    """The one stream that this program's graphs run on."""
    global _stream
    if _stream is None:
        _stream = ctypes.c_void_p()
        _C.call("lq_stream_create", ctypes.byref(_stream))
    return _stream


X_SCALE, X_ZERO = 6 / 127, 118.0  # the activation grid of the static layers
Y_SCALE, Y_ZERO = 4 / 127, 3.0
BLOCK = (("q", 0), ("k", 0), ("v", 0), ("o", 0), ("gate", 1), ("up", 1), ("down", 2))


def _block_shapes(case):
    """(rows in, features out) of a transformer block's seven products."""
    h, f = case["hidden"], case["ffn"]
    return [((h, h), (h, f), (f, h))[i] for _, i in BLOCK]


def _inputs(case, seed):
    """A case's plain inputs, from the seed alone: torch tensors by name."""
    r, kind = _Make(seed), case["kind"]
    if kind == "mlp":
        dims = (case["d_in"], case["d_hidden"], case["d_out"])
        return {"x": r.activations(case["batch"], dims[0]),
                "w": [r.weight(dims[i + 1], dims[i]) for i in range(2)],
                "b": [r.normal(dims[i + 1], std=0.1) for i in range(2)]}
    if kind in ("dynamic_linear", "static_linear", "float_input_linear"):
        return {"x": r.activations(case["M"], case["K"]), "w": r.weight(case["N"], case["K"]),
                "b": r.normal(case["N"], std=0.1)}
    if kind == "decode_block":
        dt = getattr(torch, case["dtype"])
        return {"x": [r.activations(case["M"], case["hidden"]).to(dt), r.activations(case["M"], case["ffn"]).to(dt)],
                "w": [r.weight(n, k) for k, n in _block_shapes(case)],
                "b": [r.normal(n, std=0.1) for _, n in _block_shapes(case)]}
    if kind == "decode_block_group":
        dt = getattr(torch, case["dtype"])
        return {"x": [r.activations(case["M"], case["hidden"]).to(dt), r.activations(case["M"], case["ffn"]).to(dt)],
                "w": [r.words(n, k, case["bits"], case["group"]) for k, n in _block_shapes(case)],
                "b": [r.normal(n, std=0.1) for _, n in _block_shapes(case)]}
    if kind in ("group_linear", "group_backward"):
        dt = getattr(torch, case["dtype"])
        back = kind == "group_backward"
        return {"x": (r.normal(case["M"], case["N"]) if back else r.activations(case["M"], case["K"])).to(dt),
                "w": r.words(case["N"], case["K"], case["bits"], case["group"]),
                "b": r.normal(case["N"], std=0.1)}
    if kind == "calibrate":
        return {"x": r.activations(case["rows"], case["cols"]) + 0.1}
    if kind == "conv":
        c, o, k = case["c_in"], case["c_out"], case["k"]
        return {"x": r.normal(case["batch"], c, case["height"], case["width"]).abs(), "w": r.weight(o, c, k, k),
                "b": r.normal(o, std=0.1)}
    if kind == "resnet18":
        return {"x": r.normal(case["batch"], 3, case["image"], case["image"])}
    n = case["prompt"] + case["steps"]
    return {"tokens": torch.randint(0, bench_configs.VOCAB, (case["batch"], n), generator=r.g, device="cuda",
                                    dtype=torch.int32)}


_models = {}


def _decoder():
    """The decoder's quantized Linears and float embeddings (one model a process, as a server holds it)."""
    if "decoder" not in _models:
        _per_channel_engine()
        dec, glue = bench_configs.decoder(np.random.default_rng(44))
        _models["decoder"] = (Q.quantize_dynamic(dec), glue)
    return _models["decoder"]


def _resnet18():
    """The calibrated, converted ResNet-18 (one model a process)."""
    if "resnet18" not in _models:
        from lucid_amd.nn.layers import manual_seed

        _per_channel_engine()
        manual_seed(5)
        rng = np.random.default_rng(5)
        fused = Q.fuse_modules(bench_configs.resnet18(rng), bench_configs.resnet18_fuse_groups()).to("gpu")
        prepared = Q.prepare(fused, Q.get_minmax_qconfig())
        for _ in range(2):
            prepared(L.tensor(rng.standard_normal((8, 3, 224, 224)).astype(np.float32), device="gpu"))
        _models["resnet18"] = Q.convert(prepared)
    return _models["resnet18"]


def _per_channel_engine():
    """The models run on the per-channel int8 layers, not on the group-wise ones."""
    import lucid_amd.backends as backends

    backends.quantized.engine = "reference"


def prepare(case, seed):
    kind, given = case["kind"], _inputs(case, seed)
    s = {"kind": kind}
    if kind == "mlp":
        lin = [_layer(nnqd.Linear(w[0].shape[1], w[0].shape[0]), w, b) for w, b in zip(given["w"], given["b"])]
        s.update(model=nn.Sequential(lin[0], nn.ReLU(), lin[1]), x=_own(given["x"]))
        s["model"](s["x"])
    elif kind == "dynamic_linear":
        s.update(model=_layer(nnqd.Linear(case["K"], case["N"]), given["w"], given["b"]), x=_own(given["x"]))
        s["model"](s["x"])
    elif kind in ("static_linear", "float_input_linear"):
        s.update(model=_layer(nnq.Linear(case["K"], case["N"]), given["w"], given["b"], Y_SCALE, 128.0 + Y_ZERO))
        x = _own(given["x"])
        s["x"] = nnq.Quantize(X_SCALE, X_ZERO)(x) if kind == "static_linear" else x
        s["model"](s["x"])
    elif kind in ("decode_block", "decode_block_group"):
        _prepare_block(case, given, s)
    elif kind == "group_linear":
        words, scales, biases = given["w"]
        m = nnq.QuantizedLinearMLX(case["K"], case["N"], bits=case["bits"], group_size=case["group"])
        m.register_buffer("packed_weight", _own(words))
        m.register_buffer("scales", _own(scales))
        m.register_buffer("biases", _own(biases))
        m.register_buffer("bias", _own(given["b"]))
        s.update(model=m, x=_own(given["x"]))
    elif kind == "group_backward":
        s.update(given=given, args=(case["M"], case["N"], case["K"], case["group"], case["bits"]),
                 dtype=_CODE[case["dtype"]])
    elif kind == "calibrate":
        grid = getattr(Q, case["grid"])
        obs = (Q.PerChannelMinMaxObserver(ch_axis=0, qdtype=grid) if case["per_channel"]
               else Q.MinMaxObserver(qdtype=grid))
        s.update(x=_own(given["x"]), observer=obs, grid=grid, axis=0 if case["per_channel"] else None)
        obs(s["x"])
    elif kind == "conv":
        k = case["k"]
        m = nnq.ConvReLU2d(case["c_in"], case["c_out"], k, stride=case["stride"], padding=k // 2,
                           groups=case["groups"])
        s["model"] = _layer(m, given["w"], given["b"], Y_SCALE, Y_ZERO)
        s["x"] = nnq.Quantize(5 / 255, 0.0)(_own(given["x"]))
        s["model"](s["x"])
    elif kind == "resnet18":
        net = bench_configs.Int8ResNet(_resnet18(), case["batch"], case["image"])
        s["x"] = _own(given["x"])
        s["forward"] = CapturedForward(net, s["x"])
    else:
        _prepare_decoder(case, given, s)
    torch.cuda.synchronize()
    return s


def _prepare_block(case, given, s):
    """The seven products of a decode step, captured once as a serving loop captures them."""
    M, kind, dt = case["M"], case["kind"], _CODE[case["dtype"]]
    lib, calls, keep, ys = _C.lib(), [], [given], []
    for (_, i), (K, N), w, b in zip(BLOCK, _block_shapes(case), given["w"], given["b"]):
        x = given["x"][1 if i == 2 else 0]
        y = torch.empty((M, N), dtype=x.dtype, device="cuda")
        ys.append(y)
        if kind == "decode_block_group":
            words, scales, biases = w
            size = lib.lq_group_matmul_workspace_size(M, N, K, case["group"])
            ws = torch.empty((max(size, 16),), dtype=torch.uint8, device="cuda")
            calls.append(("lq_group_matmul", x.data_ptr(), dt, K, words.data_ptr(), scales.data_ptr(),
                          biases.data_ptr(), b.data_ptr(), y.data_ptr(), N, M, N, K, case["group"], case["bits"], 1, 0,
                          ws.data_ptr(), size))
            keep.append(ws)
            continue
        codes, scale = w
        if M <= 2:  # one or two rows read the weight as it is stored, more the packed copy
            size = lib.lq_gemv_w8_workspace_size(M, N, K)
            ws = torch.empty((max(size, 16),), dtype=torch.uint8, device="cuda")
            calls.append(("lq_gemv_w8", x.data_ptr(), dt, K, codes.data_ptr(), K, scale.data_ptr(), None, b.data_ptr(),
                          y.data_ptr(), N, M, N, K, 0, ws.data_ptr(), size))
            keep.append(ws)
        else:
            packed = torch.empty((lib.lq_packed_weights_size(N, K),), dtype=torch.int8, device="cuda")
            _C.call("lq_pack_weights_i8", codes.data_ptr(), K, N, K, packed.data_ptr(), None)
            size = lib.lq_gemv_w8_packed_workspace_size(M, N, K)
            ws = torch.empty((max(size, 16),), dtype=torch.uint8, device="cuda")
            calls.append(("lq_gemv_w8_packed", x.data_ptr(), dt, K, packed.data_ptr(), scale.data_ptr(), None,
                          b.data_ptr(), y.data_ptr(), N, M, N, K, 0, ws.data_ptr(), size))
            keep += [ws, packed]
    torch.cuda.synchronize()
    s["graph"] = bench_configs.Graph(lambda st: [_C.call(*c, st) for c in calls], _the_stream())
    s.update(keep=keep, ys=ys)


def _prepare_decoder(case, given, s):
    qdec, glue = _decoder()
    B, T, n = case["batch"], case["prompt"], case["steps"]
    rt = bench_configs.Int8Decoder(qdec, glue, batch=B, max_prompt=T)
    rt.set_prompt(given["tokens"][:, :T].cpu().numpy())
    steps = given["tokens"][:, T:].t().contiguous()
    st = _the_stream()
    torch.cuda.synchronize()

    def score(stream):  # the prompt, then given tokens one at a time, as scoring a continuation does
        rt.prefill(stream)
        for i in range(n):
            _C.call("lq_memcpy_d2d", rt.next.data_ptr(), steps[i].data_ptr(), 4 * B, stream)
            rt.decode(stream)

    s["graph"] = bench_configs.Graph(score, st)
    cache = [_view(t)[:, :, :T + n] for kv in rt.cache for t in kv]
    s.update(runtime=rt, steps=steps, outputs=[_view(rt.logits), *cache])


def run(s):
    kind = s["kind"]
    if kind in ("mlp", "dynamic_linear", "group_linear"):
        return _view(s["model"](s["x"]))
    if kind in ("static_linear", "float_input_linear", "conv"):
        return _codes(s["model"](s["x"]))
    if kind in ("decode_block", "decode_block_group"):
        s["graph"].launch()
        return s["ys"]
    if kind == "group_backward":
        g, (M, N, K, group, bits) = s["given"], s["args"]
        words, scales, biases = g["w"]
        dx = torch.empty((M, K), dtype=g["x"].dtype, device="cuda")
        _C.call("lq_group_matmul", g["x"].data_ptr(), s["dtype"], N, words.data_ptr(), scales.data_ptr(),
                biases.data_ptr(), None, dx.data_ptr(), K, M, N, K, group, bits, 0, 0, None, 0, None)
        return dx
    if kind == "calibrate":
        obs = s["observer"]
        obs(s["x"])
        scale, zero = obs.calculate_qparams()
        q = Q.quantize(s["x"], scale, zero, s["grid"], ch_axis=s["axis"])
        y = Q.dequantize(q, scale, zero, ch_axis=s["axis"])
        return [_view(q), _view(y)]
    if kind == "resnet18":
        return _view(s["forward"]())
    s["graph"].launch()
    return s["outputs"]


# ------------------------------------------------------------------------------ work


def _group_bytes(N, K, case):
    return N * K * case["bits"] / 8 + 8 * N * (K / case["group"]) + 4 * N


def work(case):
    kind = case["kind"]
    size = {"float32": 4, "float16": 2, "bfloat16": 2}.get(case.get("dtype"), 4)
    if kind == "mlp":
        d = (case["d_in"], case["d_hidden"], case["d_out"])
        w = d[0] * d[1] + d[1] * d[2]
        return {"bytes": 4 * case["batch"] * (d[0] + d[2]) + w + 8 * (d[1] + d[2]), "flops": 2 * case["batch"] * w}
    if kind in ("dynamic_linear", "static_linear", "float_input_linear"):
        M, K, N = case["M"], case["K"], case["N"]
        a, c = {"dynamic_linear": (4, 4), "static_linear": (1, 1), "float_input_linear": (4, 1)}[kind]
        return {"bytes": a * M * K + N * K + 12 * N + c * M * N, "flops": 2 * M * N * K}
    if kind in ("decode_block", "decode_block_group"):
        M, shapes = case["M"], _block_shapes(case)
        w = sum(_group_bytes(n, k, case) if "group" in case else n * k + 8 * n for k, n in shapes)
        return {"bytes": w + size * M * (case["hidden"] + case["ffn"] + sum(n for _, n in shapes)),
                "flops": 2 * M * sum(k * n for k, n in shapes)}
    if kind in ("group_linear", "group_backward"):
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": size * M * (K + N) + _group_bytes(N, K, case), "flops": 2 * M * N * K}
    if kind == "calibrate":
        n = case["rows"] * case["cols"]
        return {"bytes": n * (4 + (1 if case["grid"] == "qint8" else 2) + 4), "flops": 6 * n}
    if kind == "conv":
        p, k, st = case["k"] // 2, case["k"], case["stride"]
        oh, ow = (case["height"] + 2 * p - k) // st + 1, (case["width"] + 2 * p - k) // st + 1
        n, c, o = case["batch"], case["c_in"], case["c_out"]
        return {"bytes": n * c * case["height"] * case["width"] + o * c * k * k + n * o * oh * ow,
                "flops": 2 * n * oh * ow * o * c * k * k}
    if kind == "resnet18":
        return {"bytes": case["batch"] * (12 * case["image"] ** 2 + 4000) + 11.7e6,
                "flops": case["batch"] * 3.63e9 * (case["image"] / 224) ** 2}
    d, f, v, ly = bench_configs.D_MODEL, bench_configs.FFN, bench_configs.VOCAB, bench_configs.LAYERS
    B, T, n = case["batch"], case["prompt"], case["steps"]
    w = ly * (4 * d * d + 2 * d * f)
    flops = 2 * B * (T + n) * w + 2 * B * (1 + n) * d * v + 2 * ly * B * d * (T * T + n * (2 * T + n))
    return {"bytes": (1 + n) * (w + d * v) + 4 * ly * B * d * (T + n) * (n + 1) + 4 * B * v, "flops": flops}


# ------------------------------------------------------------------------------ tolerance


def tolerance(case):
    kind = case["kind"]
    if kind in ("static_linear", "calibrate", "conv"):
        return "exact"  # integer sums and one rounding after another: the codes are the codes
    if kind in ("mlp", "dynamic_linear"):
        return {"rel": 1e-5, "max": 1e-3}  # exact sums of codes, 32-bit scales and biases
    if kind == "float_input_linear":
        # codes of 32-bit sums (1e-5 of them off the 64-bit ones): a sum on a rounding edge may fall either way
        return {"differ": min(1e-2, max(4e-5, 1.5 / (case["M"] * case["N"])))}
    if kind == "resnet18":
        return {"rel": 2e-2}  # the float average pool's last bit can move a code of the last grid
    if kind == "decoder":
        return {"rel": 3e-2}  # 16-bit attention, and each layer's codes follow the layer before
    return {"rel": {"float32": 5e-6, "float16": 1.2e-3, "bfloat16": 1e-2}[case["dtype"]],
            "max": {"float32": 1e-4, "float16": 6e-3, "bfloat16": 5e-2}[case["dtype"]]}


# ------------------------------------------------------------------------------ 64 bits


def _range_grid(lo, hi, qmin, qmax):
    """Affine scale and zero point of a range that holds zero."""
    lo, hi = lo.clamp(max=0), hi.clamp(min=0)
    scale = ((hi - lo) / (qmax - qmin)).clamp(min=1e-8)
    return scale, (qmin - (lo / scale).round()).clamp(qmin, qmax)


def _quantized(x, scale, zero, qmin, qmax):
    return ((x / scale).round() + zero).clamp(qmin, qmax)


def _dynamic(x, w, b):
    """A dynamic int8 Linear in 64 bits."""
    codes, ws = w
    s, z = _range_grid(x.min(), x.max(), 0, 255)
    q = _quantized(x, s, z, 0, 255) - z
    return (q @ codes.double().t()) * (s * ws.double()) + b.double()


def _unpacked(w, case):
    """A packed group-wise weight in 64 bits, its scales and biases at the activation's precision."""
    words, scales, biases = w
    bits, dt = case["bits"], getattr(torch, case["dtype"])
    shifts = torch.arange(0, 32, bits, device=words.device, dtype=torch.int32)
    codes = (words.unsqueeze(-1) >> shifts) & (2**bits - 1)
    codes = codes.reshape(words.shape[0], -1, case["group"]).double()
    full = codes * scales.to(dt).double().unsqueeze(-1) + biases.to(dt).double().unsqueeze(-1)
    return full.reshape(words.shape[0], -1)


def _host(t):
    """A buffer of a framework module as torch holds it."""
    return torch.from_numpy(np.ascontiguousarray(t.numpy())).cuda()


def _conv64(x, w, stride, pad):
    """A convolution in 64 bits as a product over unfolded patches, image by image."""
    N, _, H, W = x.shape
    O, _, k, _ = w.shape
    oh, ow = (H + 2 * pad - k) // stride + 1, (W + 2 * pad - k) // stride + 1
    flat = w.reshape(O, -1)
    return torch.stack([(flat @ torch.nn.functional.unfold(x[i:i + 1], k, padding=pad, stride=stride)[0])
                        .reshape(O, oh, ow) for i in range(N)])


def exact(case, seed):
    kind = case["kind"]
    if kind in ("resnet18", "decoder"):
        return _exact_resnet18(case, seed) if kind == "resnet18" else _exact_decoder(case, seed)
    given = _inputs(case, seed)
    if kind == "mlp":
        h = _dynamic(given["x"].double(), given["w"][0], given["b"][0]).clamp(min=0)
        return _dynamic(h, given["w"][1], given["b"][1])
    if kind == "dynamic_linear":
        return _dynamic(given["x"].double(), given["w"], given["b"])
    if kind in ("static_linear", "float_input_linear"):
        x, (codes, ws) = given["x"].double(), given["w"]
        if kind == "static_linear":
            s = float(np.float32(X_SCALE))
            x = (_quantized(x, s, X_ZERO, 0, 255) - X_ZERO) * s
        y = x @ (codes.double() * ws.double()[:, None]).t() + given["b"].double()
        return (_quantized(y, float(np.float32(Y_SCALE)), 128 + Y_ZERO, 0, 255) - 128).to(torch.int8)
    if kind == "decode_block":
        return [given["x"][1 if i == 2 else 0].double() @ (c.double() * ws.double()[:, None]).t() + b.double()
                for (_, i), (c, ws), b in zip(BLOCK, given["w"], given["b"])]
    if kind == "decode_block_group":
        dt = getattr(torch, case["dtype"])
        return [given["x"][1 if i == 2 else 0].double() @ _unpacked(w, case).t() + b.to(dt).double()
                for (_, i), w, b in zip(BLOCK, given["w"], given["b"])]
    if kind == "group_linear":
        dt = getattr(torch, case["dtype"])
        return given["x"].double() @ _unpacked(given["w"], case).t() + given["b"].to(dt).double()
    if kind == "group_backward":
        return given["x"].double() @ _unpacked(given["w"], case)
    if kind == "calibrate":
        return None  # codes, and the codes' values: each is one rounding of a 32-bit number
    s = float(np.float32(5 / 255))
    x = _quantized(given["x"].double(), s, 0.0, 0, 255) * s
    codes, ws = given["w"]
    y = _conv64(x, codes.double() * ws.double().reshape(-1, 1, 1, 1), case["stride"], case["k"] // 2)
    y = (y + given["b"].double().reshape(-1, 1, 1)).clamp(min=0)
    return (_quantized(y, float(np.float32(Y_SCALE)), Y_ZERO, 0, 255) - 128).to(torch.int8)


def _exact_resnet18(case, seed):
    """The converted network's layers in 64 bits, from its buffers."""
    net, x = _resnet18(), _inputs(case, seed)["x"].double()

    def grid(m):
        return m.scale.item(), m.zero_point.item()

    def on_grid(y, m):
        s, z = grid(m)
        return (_quantized(y, s, z, 0, 255) - z) * s

    def weighted(x, m, relu):
        w = _host(m.weight_int8).double() * _host(m.weight_scale).double().reshape(-1, 1, 1, 1)
        y = _conv64(x, w, m.stride[0], m.kernel_size[0] // 2)
        if m.bias is not None:
            y = y + _host(m.bias).double().reshape(-1, 1, 1)
        return on_grid(y.clamp(min=0) if relu else y, m)

    x = weighted(on_grid(x, net.quant), net.conv1, True)
    x = torch.nn.functional.max_pool2d(x, 3, 2, 1)
    for i in range(1, 5):
        for blk in getattr(net, "layer%d" % i):
            y = weighted(weighted(x, blk.conv1, True), blk.conv2, False)
            skip = x if blk.downsample is None else weighted(x, blk.downsample[0], False)
            x = on_grid((y + skip).clamp(min=0), blk.skip)
    w = _host(net.fc.weight_int8).double() * _host(net.fc.weight_scale).double()[:, None]
    return on_grid(x.mean((2, 3)) @ w.t() + _host(net.fc.bias).double(), net.fc)


def _exact_decoder(case, seed):
    """The decoder's layers in 64 bits, each dynamic Linear on its own live range."""
    qdec, glue = _decoder()
    tokens = _inputs(case, seed)["tokens"].long()
    B, T, n = case["batch"], case["prompt"], case["steps"]
    D, H = bench_configs.D_MODEL, bench_configs.HEADS
    tok, pos = (torch.from_numpy(glue[k]).cuda().double() for k in ("tok", "pos"))

    def weight(m):
        return (_host(m.weight_int8), _host(m.weight_scale)), _host(m.bias)

    layers = [[weight(getattr(m, k)) for k in ("qkv", "out", "up", "down")] for m in qdec.layers]
    head = weight(qdec.head)
    cache = [[torch.zeros((B, H, 0, D // H), dtype=torch.float64, device="cuda") for _ in range(2)] for _ in layers]

    def norm(h):
        c = h - h.mean(-1, keepdim=True)
        return c / (c.square().mean(-1, keepdim=True) + 1e-5).sqrt()

    def step(ids, at):
        m = ids.shape[1]
        h = (tok[ids] + pos[at:at + m]).reshape(B * m, D)
        for (qkv, out, up, down), kv in zip(layers, cache):
            q, k, v = _dynamic(norm(h), *qkv).reshape(B, m, 3, H, D // H).permute(2, 0, 3, 1, 4)
            kv[0], kv[1] = torch.cat((kv[0], k), 2), torch.cat((kv[1], v), 2)
            seen = torch.arange(at + m, device="cuda")[None] <= at + torch.arange(m, device="cuda")[:, None]
            a = (q @ kv[0].transpose(2, 3).contiguous()) / math.sqrt(D // H)
            a = a.masked_fill(~seen, -math.inf).softmax(-1) @ kv[1]
            h = h + _dynamic(a.transpose(1, 2).reshape(B * m, D), *out)
            g = _dynamic(norm(h), *up)
            g = 0.5 * g * (1 + torch.tanh(0.7978845608028654 * (g + 0.044715 * g**3)))
            h = h + _dynamic(g, *down)
        return _dynamic(norm(h.reshape(B, m, D)[:, -1]), *head)

    logits = step(tokens[:, :T], 0)
    for i in range(n):
        logits = step(tokens[:, T + i:T + i + 1], T + i)
    return [logits, *(t for kv in cache for t in kv)]
