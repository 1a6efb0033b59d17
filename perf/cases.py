"""The work that a user of this framework has it do, as cases that can be timed and compared.

Every case is a short program over the public entry points of `itexhip`, the calls in the order in which the op kernels
enqueue them, on buffers that the program keeps (weights prepacked once, outputs and intermediates from its arena).
`listed()` are the cases with names, `draw()` gives more of the same ranges.

kind            one pass
chain           QuantizeV2 (given range) -> quantized MatMul [BiasAdd, Relu, Requantize] -> Dequantize
decode          per-token dynamic quantization and the two linears of a feed-forward block, 1 to 16 tokens
dynamic_linear  per-tensor dynamic quantization of float activations -> linear [BiasAdd, Dequantize], a served batch
linear          a linear on quantized activations [BiasAdd, Requantize], a prompt's worth of tokens
ffn             an encoder's feed-forward block: QuantizeV2 -> linear + GELU -> QuantizeV2 -> linear + residual
attention       head split, Q.K^T with scale and mask, P.V, quantization of the context, head merge
bottleneck      three convolutions of a residual block, the last one with the residual Sum
stem            the first convolution of a vision network, 3 input channels
separable       depthwise 3x3 convolution -> pointwise convolution
elementwise     the ops around unfused products: dynamic-range QuantizeV2 and Dequantize of a float tensor, range and
                per-channel Requantize of int32 accumulators
ragged_linear   a linear whose K no matrix kernel likes (not a multiple of 16)
"""
import importlib
import math

import numpy as np
import torch

hip = importlib.import_module("intel-extension-for-tensorflow_amd").itexhip

_TORCH = {hip.FLOAT: torch.float32, hip.BFLOAT16: torch.bfloat16, hip.HALF: torch.float16, hip.QINT8: torch.int8,
          hip.QUINT8: torch.uint8, hip.QINT32: torch.int32}
_TYPES = {"float": hip.FLOAT, "bfloat16": hip.BFLOAT16, "half": hip.HALF, "qint8": hip.QINT8, "quint8": hip.QUINT8}
_BYTES = {"float": 4, "bfloat16": 2, "half": 2, "qint8": 1, "quint8": 1}


def listed():
    return [
        # a single quantized linear between float tensors: three short launches, the smallest thing a graph runs
        dict(name="chain_128x1024x1024", kind="chain", M=128, K=1024, N=1024),
        # one new token through the feed-forward block of an 8B-parameter decoder
        dict(name="decode_mlp_1", kind="decode", M=1, K=4096, N=14336),
        # a larger served batch, float activations in and out
        dict(name="batch_64x4096x14336", kind="dynamic_linear", M=64, K=4096, N=14336, out="float"),
        # a prompt of 2048 tokens through one projection of the same decoder
        dict(name="prefill_2048x4096x14336", kind="linear", M=2048, K=4096, N=14336, out="qint8"),
        # BERT-base feed-forward block, 32 sequences of 128 tokens
        dict(name="ffn_4096x768x3072", kind="ffn", M=4096, K=768, N=3072),
        # BERT-base attention, 128 sequences of 128 tokens
        dict(name="attention_128x128", kind="attention", B=128, S=128, H=12, D=64, out="float"),
        # the same heads over 14 x 14 image patches and a class token: nothing is a multiple of 16
        dict(name="attention_32x197", kind="attention", B=32, S=197, H=12, D=64, out="bfloat16"),
        # ResNet-50, first stage, 32 images
        dict(name="bottleneck_32x56x56", kind="bottleneck", B=32, H=56, W=56, C=256, F=64),
        # ... and its first layer
        dict(name="stem_32x224x224", kind="stem", B=32, H=224, W=224, C=3, O=64, window=7),
        # MobileNet's first separable block, 32 images
        dict(name="separable_32x112x112", kind="separable", B=32, H=112, W=112, C=32, O=64, stride=1),
        # one activation tensor through the stand-alone ops
        dict(name="elementwise_8192x4096", kind="elementwise", rows=8192, depth=4096, type="qint8"),
        # a linear on 1001 features
        dict(name="ragged_1000x1001x1000", kind="ragged_linear", M=1000, K=1001, N=1000, out="float"),
    ]


def _log(rng, lo, hi, multiple=1):
    """A size between lo and hi, even over its logarithm, a multiple of `multiple`."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(multiple, int(round(v / multiple)) * multiple)


def draw(rng):
    kind = rng.choice(["chain", "decode", "dynamic_linear", "linear", "ffn", "attention", "bottleneck", "stem", "separable",
                       "elementwise", "ragged_linear"])
    if kind == "chain":
        return dict(kind=kind, M=_log(rng, 1, 512), K=_log(rng, 64, 4096, 16), N=_log(rng, 10, 4096))
    if kind == "decode":
        return dict(kind=kind, M=rng.randint(1, 16), K=_log(rng, 512, 4096, 16), N=_log(rng, 1024, 14336, 16))
    if kind == "dynamic_linear":
        return dict(kind=kind, M=_log(rng, 17, 512), K=_log(rng, 512, 4096, 16), N=_log(rng, 512, 14336, 4),
                    out=rng.choice(["float", "bfloat16", "half"]))
    if kind == "linear":
        return dict(kind=kind, M=_log(rng, 128, 2048), K=_log(rng, 256, 4096, 16), N=_log(rng, 256, 14336, 8),
                    out=rng.choice(["qint8", "quint8"]))
    if kind == "ffn":
        return dict(kind=kind, M=_log(rng, 64, 4096), K=rng.choice([512, 768, 1024]), N=rng.choice([2048, 3072, 4096]))
    if kind == "attention":
        s = _log(rng, 16, 384)
        h, d = rng.choice([8, 12, 16]), rng.choice([32, 64])
        return dict(kind=kind, B=_log(rng, 1, max(1, min(128, (1 << 21) // (s * s)))), S=s, H=h, D=d,
                    out=rng.choice(["float", "bfloat16", "half"]))
    if kind == "bottleneck":
        hw, f = rng.choice([(56, 64), (28, 128), (14, 256), (7, 512), (48, 64), (25, 128)])
        return dict(kind=kind, B=_log(rng, 1, 32), H=hw, W=hw, C=4 * f, F=f)
    if kind == "stem":
        hw = rng.choice([96, 128, 160, 192, 224, 225])
        return dict(kind=kind, B=_log(rng, 1, 32), H=hw, W=hw, C=rng.choice([1, 3, 4]), O=rng.choice([32, 64]),
                    window=rng.choice([3, 7]))
    if kind == "separable":
        hw, c = rng.choice([(112, 32), (112, 64), (56, 128), (28, 256), (14, 512), (75, 64), (38, 144)])
        return dict(kind=kind, B=_log(rng, 1, 32 if hw < 112 or c < 64 else 16), H=hw, W=hw, C=c, O=rng.choice([1, 2]) * c,
                    stride=rng.choice([1, 2]))
    if kind == "elementwise":
        depth = rng.choice([1, 64, 197, 1000, 4096])
        return dict(kind=kind, rows=_log(rng, 1 << 12, 1 << 24) // depth + 1, depth=depth, type=rng.choice(["qint8", "quint8"]))
    m, k = _log(rng, 8, 1000), 2 * _log(rng, 32, 500) + 1
    return dict(kind=kind, M=m, K=k, N=_log(rng, 8, 1000), out=rng.choice(["float", "quint8"]))


# ---------------------------------------------------------------------------------------------------------------------
# what a program has in hand before the call
# ---------------------------------------------------------------------------------------------------------------------
class _Source:
    """Random tensors on the GPU, all from one seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(*shape, device="cuda", generator=self.g)

    def bytes(self, low, high, dtype, *shape):
        return torch.randint(low, high, shape, dtype=dtype, device="cuda", generator=self.g)


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _weight(src, K, N):
    """Symmetric per-output-channel qint8 weight from N(0, 0.02), prepacked, with its ranges and a float bias."""
    w = src.normal(K, N) * 0.02
    r = w.abs().amax(0)
    wq = torch.round(w * (127.0 / r)).clamp_(-127, 127).to(torch.int8)
    return dict(wq=wq, min_b=-r, max_b=r, bias=src.normal(N) * 0.01, **_pack(wq, K, N))


def _pack(wq, K, N):
    packed = torch.empty(max(16, hip.qgemm_packed_bytes(K, N)), dtype=torch.int8, device="cuda")
    colsum = torch.empty(N, dtype=torch.int32, device="cuda")
    hip.qgemm_prepack_b(wq, False, K, N, packed, colsum, _stream())
    return dict(packed=packed, colsum=colsum)


def _buffer(kind, *shape):
    return torch.empty(*shape, dtype=_TORCH[kind], device="cuda")


def _min_first(lo, hi):
    """(min, max, scale, addend) of the MIN_FIRST quint8 form of QuantizeV2 for a tensor's range, as its op computes them."""
    f32 = np.float32
    lo, hi = min(f32(0.0), f32(float(lo))), max(f32(0.0), f32(float(hi)))
    scale = f32(255.0 / float(hi - lo))
    return float(lo), float(hi), float(scale), float(f32(-lo) * scale)


def _min_first_linear(t_out, lo, hi, **kw):
    return hip.matmul_params(t_in=hip.QUINT8, t_out=t_out, input_mode=hip.MIN_FIRST, min_a=lo, max_a=hi, **kw)


def _conv_weight(src, shape, fan_in):
    """qint8 filter with the output scale that maps its int32 accumulators to the 8-bit range, and a scaled bias."""
    n = shape[-1] * (shape[-2] if shape[-1] == 1 else 1)
    scale = torch.full((n,), 1.0 / (74.0 * 40.0 * math.sqrt(fan_in)) * 24.0, device="cuda") * (0.75 + 0.5 * torch.rand(n, device="cuda", generator=src.g))
    return src.bytes(-127, 128, torch.int8, *shape), scale, src.normal(n) * 4.0


def _epilogue(n, *elt):
    ep = hip.Epilogue()
    ep.n_scales, ep.n_eltwise = n, len(elt)
    for i, (alg, alpha, beta) in enumerate(elt):
        ep.elt[i].alg, ep.elt[i].alpha, ep.elt[i].beta = alg, alpha, beta
    return ep


def _same(size, window, stride):
    """TensorFlow's SAME rule: output extent and leading padding."""
    out = -(-size // stride)
    return out, max((out - 1) * stride + window - size, 0) // 2


def prepare(case, seed):
    src, kind = _Source(seed), case["kind"]
    s = dict(case)
    s["stream"] = _stream()
    if kind in ("chain", "linear", "ragged_linear"):
        M, K, N = case["M"], case["K"], case["N"]
        s["w"] = _weight(src, K, N)
        x = src.normal(M, K)
        if kind == "linear":   # trained activations have a few large values
            x = torch.where(torch.rand(M, K, device="cuda", generator=src.g) < 1e-3, x * 20.0, x)
        lo, hi, s["scale"], s["addend"] = _min_first(x.min(), x.max())
        out_type = hip.QUINT8 if kind == "chain" else _TYPES[case["out"]]
        # a sample of the float result fixes the frozen output range, as a calibration run does
        y = x[:64] @ (s["w"]["wq"].float() * (s["w"]["max_b"] / 127.0)) + s["w"]["bias"]
        r = float(y.abs().max())
        kw = dict(has_dequantize=True)
        if out_type in (hip.QINT8, hip.QUINT8):
            kw = dict(has_requantize=True, min_out=-r if out_type == hip.QINT8 else 0.0, max_out=r)
        if out_type == hip.QUINT8:
            kw["activation"] = hip.ACT_RELU
        s["p"] = _min_first_linear(out_type, lo, hi, **kw)
        s["xq"] = _buffer(hip.QUINT8, M, K)
        s["q"] = _buffer(out_type, M, N)
        if kind == "chain":
            s["x"] = x
            s["y"] = _buffer(hip.FLOAT, M, N)
            s["y_scale"] = float(np.float32(r) / np.float32(255.0))
        else:   # the activations come quantized from the layer before
            hip.quantize(x, s["xq"], M * K, hip.QUINT8, s["scale"], s["addend"], s["stream"])
    elif kind == "decode":
        M, K, N = case["M"], case["K"], case["N"]
        s["x"] = src.normal(M, K)
        s["up"], s["down"] = _weight(src, K, N), _weight(src, N, K)
        s["p"] = _min_first_linear(hip.FLOAT, 0.0, 0.0, has_dequantize=True)
        s["xq"], s["hq"] = _buffer(hip.QUINT8, M, K), _buffer(hip.QUINT8, M, N)
        s["x_min"], s["x_max"], s["h_min"], s["h_max"] = (_buffer(hip.FLOAT, M) for _ in range(4))
        s["h"], s["y"] = _buffer(hip.FLOAT, M, N), _buffer(hip.FLOAT, M, K)
    elif kind == "dynamic_linear":
        M, K, N = case["M"], case["K"], case["N"]
        s["x"], s["w"] = src.normal(M, K), _weight(src, K, N)
        s["p"] = _min_first_linear(_TYPES[case["out"]], 0.0, 0.0, has_dequantize=True)
        s["xq"], s["y"] = _buffer(hip.QUINT8, M, K), _buffer(_TYPES[case["out"]], M, N)
        s["state"] = torch.zeros(hip.DYNAMIC_STATE_FLOATS, dtype=torch.float32, device="cuda")
        s["range"] = s["state"][2:]
    elif kind == "ffn":
        M, K, N = case["M"], case["K"], case["N"]
        s["x"], s["residual"] = src.normal(M, K), src.normal(M, K)
        s["up"], s["down"] = _weight(src, K, N), _weight(src, N, K)
        lo, hi, s["x_scale"], s["x_addend"] = _min_first(s["x"].min(), s["x"].max())
        s["p_up"] = _min_first_linear(hip.FLOAT, lo, hi, has_dequantize=True, activation=hip.ACT_GELU_APPROX)
        h = torch.nn.functional.gelu(s["x"][:64] @ (s["up"]["wq"].float() * (s["up"]["max_b"] / 127.0)) + s["up"]["bias"], approximate="tanh")
        lo, hi, s["h_scale"], s["h_addend"] = _min_first(h.min(), h.max())
        s["p_down"] = _min_first_linear(hip.FLOAT, lo, hi, has_dequantize=True, add_position=1)
        s["xq"], s["hq"] = _buffer(hip.QUINT8, M, K), _buffer(hip.QUINT8, M, N)
        s["h"], s["y"] = _buffer(hip.FLOAT, M, N), _buffer(hip.FLOAT, M, K)
    elif kind == "attention":
        B, S, H, D = (case[k] for k in "BSHD")
        t = _TYPES[case["out"]]
        for name in "qkv":   # the projections' outputs, token by token, and the heads' copies
            s[name] = (src.normal(B, S, H, D) * 30.0).round_().clamp_(-127, 127).to(torch.int8)
            s[name + "h"] = _buffer(hip.QINT8, B, H, S, D)
        # attention weights of 0 .. 1 on the qint8 grid (the softmax between the two products is the user's own op)
        s["probs"] = (torch.rand(B, H, S, S, device="cuda", generator=src.g).pow_(8) * 127.0).round_().to(torch.int8)
        s["mul"] = torch.tensor([D ** -0.5], device="cuda").to(_TORCH[t])
        length = torch.randint(max(1, S // 2), S + 1, (B, 1, 1, 1), device="cuda", generator=src.g)
        s["mask"] = torch.where(torch.arange(S, device="cuda").view(1, 1, 1, S) < length, 0.0, -10000.0).to(_TORCH[t]).contiguous()
        s["p_scores"], shape = hip.bmm_params((B, H, S, D), (B, H, S, D), False, True, t, float(36.0 / (127.0 * 127.0)),
                                              [(hip.BIN_MUL, s["mul"], (1,)), (hip.BIN_ADD, s["mask"], (B, 1, 1, S))])
        s["scores"] = _buffer(t, *shape)
        s["p_context"], shape = hip.bmm_params((B, H, S, S), (B, H, S, D), False, False, t, float(6.0 / (127.0 * 127.0)))
        s["context"] = _buffer(t, *shape)
        s["cq"], s["merged"] = _buffer(hip.QINT8, B, H, S, D), _buffer(hip.QINT8, B, S, H, D)
        s["c_scale"] = float(np.float32(127.0) / np.float32(0.25 * S))
    elif kind == "bottleneck":
        B, H, W, C, F = (case[k] for k in ("B", "H", "W", "C", "F"))
        s["x"] = src.normal(B, H, W, C).mul_(40.0).clamp_(0, 255).to(torch.uint8)   # after a ReLU
        for name, shape, fan in (("reduce", (1, 1, C, F), C), ("middle", (3, 3, F, F), 9 * F), ("expand", (1, 1, F, C), F)):
            w, scale, bias = _conv_weight(src, shape, fan)
            s[name] = dict(scale=scale, bias=bias, **_pack(w, shape[0] * shape[1] * shape[2], shape[3]))
        s["geometry"] = hip.ConvGeometry(B, H, W, F, 3, 3, H, W, 1, 1, 1, 1, 1, 1)
        relu = (hip.ELT_RELU, 0.0, 0.0)
        s["ep_f"], s["ep_sum"] = _epilogue(F, relu), _epilogue(C, (hip.ELT_SUM, 0.5, 0.0), relu)
        s["a"], s["b"], s["y"] = _buffer(hip.QUINT8, B * H * W, F), _buffer(hip.QUINT8, B * H * W, F), _buffer(hip.QUINT8, B * H * W, C)
    elif kind == "stem":
        B, H, W, C, O, k = (case[key] for key in ("B", "H", "W", "C", "O", "window"))
        s["x"] = src.bytes(0, 256, torch.uint8, B, H, W, C)
        w, s["scale"], s["bias"] = _conv_weight(src, (k, k, C, O), k * k * C)
        (OH, pt), (OW, pl) = _same(H, k, 2), _same(W, k, 2)
        # 4 channels, window rows of whole 16-byte vectors, the spatial padding written into the copy: as the op kernel lays it out
        kw = (k + 3) // 4 * 4
        hn = max(pt + H, (OH - 1) * 2 + k)
        wn = (max(pl + W, (OW - 1) * 2 + kw) + 3) // 4 * 4
        s["pad"], s["copy"] = (pt, pl, hn, wn), _buffer(hip.QUINT8, B, hn, wn, 4)
        wp = torch.empty(k, kw, 4, O, dtype=torch.int8, device="cuda")
        hip.pad_nhwc8(w, k, k, C, O, 0, 0, kw, 4, O, wp, s["stream"])
        s.update(_pack(wp, k * kw * 4, O))
        s["geometry"] = hip.ConvGeometry(B, hn, wn, 4, k, kw, OH, OW, 2, 2, 1, 1, 0, 0)
        s["ep"], s["y"] = _epilogue(O, (hip.ELT_RELU, 0.0, 0.0)), _buffer(hip.QUINT8, B, OH, OW, O)
    elif kind == "separable":
        B, H, W, C, O, st = (case[key] for key in ("B", "H", "W", "C", "O", "stride"))
        s["x"] = src.normal(B, H, W, C).mul_(40.0).clamp_(0, 255).to(torch.uint8)
        s["dw"], s["dw_scale"], s["dw_bias"] = _conv_weight(src, (3, 3, C, 1), 9)
        w, s["pw_scale"], s["pw_bias"] = _conv_weight(src, (1, 1, C, O), C)
        s.update(_pack(w, C, O))
        (OH, pt), (OW, pl) = _same(H, 3, st), _same(W, 3, st)
        s["geometry"] = hip.ConvGeometry(B, H, W, C, 3, 3, OH, OW, st, st, 1, 1, pt, pl)
        clip = (hip.ELT_CLIP, 0.0, 200.0)   # Relu6 at the output's scale
        s["ep_dw"], s["ep_pw"] = _epilogue(C, clip), _epilogue(O, clip)
        s["rows"] = B * OH * OW
        s["a"], s["y"] = _buffer(hip.QUINT8, s["rows"], C), _buffer(hip.QUINT8, s["rows"], O)
    elif kind == "elementwise":
        rows, depth, t = case["rows"], case["depth"], _TYPES[case["type"]]
        x = src.normal(rows, depth)
        s["x"] = torch.where(torch.rand(rows, depth, device="cuda", generator=src.g) < 1e-4, x * 50.0, x)
        s["t"], s["mode"] = t, hip.SCALED if t == hip.QINT8 else hip.MIN_FIRST
        s["state"] = torch.zeros(hip.DYNAMIC_STATE_FLOATS, dtype=torch.float32, device="cuda")
        s["q"], s["y"] = _buffer(t, rows, depth), _buffer(hip.FLOAT, rows, depth)
        r = max(abs(float(s["x"].min())), abs(float(s["x"].max())))
        s["y_scale"] = float(np.float32(r) / np.float32(127.0))
        s["acc"] = (src.normal(rows, depth) * float(1 << 20)).round_().to(torch.int32)
        s["lo"], s["hi"] = (torch.zeros(depth, dtype=torch.int32, device="cuda") for _ in range(2))
        s["scales"] = (0.75 + 0.5 * torch.rand(depth, device="cuda", generator=src.g)) * (127.0 / 5.0 / (1 << 20))
        s["aq"] = _buffer(hip.QINT8, rows, depth)
    return s


# ---------------------------------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------------------------------
def _linear(p, x, w, M, K, N, out, stream, addend=None):
    hip.qmatmul(p, x, w["packed"], w["colsum"], M, K, N, w["min_b"], w["max_b"], N, w["bias"], out, stream, addend=addend)


def run(s):
    kind, st = s["kind"], s["stream"]
    if kind == "chain":
        M, K, N = s["M"], s["K"], s["N"]
        hip.quantize(s["x"], s["xq"], M * K, hip.QUINT8, s["scale"], s["addend"], st)
        _linear(s["p"], s["xq"], s["w"], M, K, N, s["q"], st)
        hip.dequantize(s["q"], s["y"], M * N, hip.QUINT8, s["y_scale"], 0, st)
        return s["y"]
    if kind == "linear":
        _linear(s["p"], s["xq"], s["w"], s["M"], s["K"], s["N"], s["q"], st)
        return s["q"]
    if kind == "ragged_linear":
        w = s["w"]
        hip.qmatmul_unpacked(s["p"], s["xq"], w["wq"], False, s["M"], s["K"], s["N"], w["min_b"], w["max_b"], s["N"], w["bias"],
                             s["q"], st)
        return s["q"]
    if kind == "decode":
        M, K, N, up, down = s["M"], s["K"], s["N"], s["up"], s["down"]
        hip.quantize_dynamic_rows(s["x"], s["xq"], M, K, hip.QUINT8, hip.MIN_FIRST, 0.01, s["x_min"], s["x_max"], st)
        hip.qmatmul_per_row(s["p"], s["xq"], up["packed"], up["colsum"], M, K, N, s["x_min"], s["x_max"], up["min_b"], up["max_b"],
                            N, up["bias"], s["h"], st)
        hip.quantize_dynamic_rows(s["h"], s["hq"], M, N, hip.QUINT8, hip.MIN_FIRST, 0.01, s["h_min"], s["h_max"], st)
        hip.qmatmul_per_row(s["p"], s["hq"], down["packed"], down["colsum"], M, N, K, s["h_min"], s["h_max"], down["min_b"],
                            down["max_b"], K, down["bias"], s["y"], st)
        return dict(h=s["h"], y=s["y"])
    if kind == "dynamic_linear":
        M, K, N, w = s["M"], s["K"], s["N"], s["w"]
        hip.quantize_dynamic(s["x"], s["xq"], M * K, hip.QUINT8, hip.MIN_FIRST, 0.01, s["state"], st)
        hip.qmatmul_device_range(s["p"], s["xq"], w["packed"], w["colsum"], M, K, N, s["range"], w["min_b"], w["max_b"], N, w["bias"],
                                 s["y"], st)
        return s["y"]
    if kind == "ffn":
        M, K, N = s["M"], s["K"], s["N"]
        hip.quantize(s["x"], s["xq"], M * K, hip.QUINT8, s["x_scale"], s["x_addend"], st)
        _linear(s["p_up"], s["xq"], s["up"], M, K, N, s["h"], st)
        hip.quantize(s["h"], s["hq"], M * N, hip.QUINT8, s["h_scale"], s["h_addend"], st)
        _linear(s["p_down"], s["hq"], s["down"], M, N, K, s["y"], st, addend=s["residual"])
        return dict(h=s["h"], y=s["y"])
    if kind == "attention":
        B, S, H, D = s["B"], s["S"], s["H"], s["D"]
        for name in "qkv":
            hip.transpose(s[name], s[name + "h"], 1, (B, S, H, D), (0, 2, 1, 3), st)
        hip.qbatch_matmul(s["p_scores"], s["qh"], s["kh"], s["scores"], st)
        hip.qbatch_matmul(s["p_context"], s["probs"], s["vh"], s["context"], st)
        if s["context"].dtype == torch.float32:
            hip.quantize(s["context"], s["cq"], B * H * S * D, hip.QINT8, s["c_scale"], 0.0, st)
        elif s["context"].dtype == torch.bfloat16:
            hip.quantize_bf16(s["context"], s["cq"], B * H * S * D, hip.QINT8, s["c_scale"], 0.0, st)
        else:   # QuantizeV2 does not read half: the context stays half
            return dict(scores=s["scores"], context=s["context"])
        hip.transpose(s["cq"], s["merged"], 1, (B, H, S, D), (0, 2, 1, 3), st)
        return dict(scores=s["scores"], merged=s["merged"])
    if kind == "bottleneck":
        C, F, rows = s["C"], s["F"], s["B"] * s["H"] * s["W"]
        r, m, e = s["reduce"], s["middle"], s["expand"]
        hip.qgemm(s["x"], hip.QUINT8, r["packed"], r["colsum"], rows, C, F, r["scale"], r["bias"], s["ep_f"], hip.QUINT8, s["a"], st)
        hip.qconv2d(s["a"], hip.QUINT8, s["geometry"], m["packed"], m["colsum"], F, m["scale"], m["bias"], s["ep_f"], hip.QUINT8, s["b"], st)
        hip.qgemm_sum(s["b"], hip.QUINT8, e["packed"], e["colsum"], rows, F, C, e["scale"], e["bias"], s["ep_sum"], s["x"], hip.QUINT8,
                      hip.QUINT8, s["y"], st)
        return s["y"]
    if kind == "stem":
        pt, pl, hn, wn = s["pad"]
        hip.pad_nhwc8(s["x"], s["B"], s["H"], s["W"], s["C"], pt, pl, hn, wn, 4, s["copy"], st)
        hip.qconv2d(s["copy"], hip.QUINT8, s["geometry"], s["packed"], s["colsum"], s["O"], s["scale"], s["bias"], s["ep"], hip.QUINT8,
                    s["y"], st)
        return s["y"]
    if kind == "separable":
        hip.qdepthwise_conv2d(s["x"], hip.QUINT8, s["geometry"], 1, s["dw"], s["dw_scale"], s["dw_bias"], s["ep_dw"], hip.QUINT8, s["a"], st)
        hip.qgemm(s["a"], hip.QUINT8, s["packed"], s["colsum"], s["rows"], s["C"], s["O"], s["pw_scale"], s["pw_bias"], s["ep_pw"],
                  hip.QUINT8, s["y"], st)
        return s["y"]
    rows, depth = s["rows"], s["depth"]
    n = rows * depth
    hip.quantize_dynamic(s["x"], s["q"], n, s["t"], s["mode"], 0.01, s["state"], st)
    hip.dequantize(s["q"], s["y"], n, s["t"], s["y_scale"], 0, st)
    hip.minmax_i32_per_channel(s["acc"], rows, depth, s["lo"], s["hi"], st)
    hip.requantize_per_channel(s["acc"], s["aq"], rows, depth, hip.QINT8, s["scales"], st)
    return dict(q=s["q"], y=s["y"], lo=s["lo"], hi=s["hi"], aq=s["aq"])


# ---------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without, and how far two correct results may lie apart
# ---------------------------------------------------------------------------------------------------------------------
def work(case):
    """Bytes: each input and weight read once, each returned tensor written once; tensors between two calls of a pass are
    counted where they are returned too.  flops: multiplications and additions of the products."""
    kind = case["kind"]
    if kind in ("chain", "linear", "ragged_linear", "dynamic_linear", "ffn", "decode"):
        M, K, N = case["M"], case["K"], case["N"]
        if kind == "chain":
            return dict(bytes=4 * M * K + K * N + 12 * N + 4 * M * N, flops=2 * M * K * N)
        if kind == "decode":
            return dict(bytes=8 * M * K + 2 * K * N + 12 * (N + K) + 4 * M * N, flops=4 * M * K * N)
        if kind == "ffn":
            return dict(bytes=12 * M * K + 2 * K * N + 12 * (N + K) + 4 * M * N, flops=4 * M * K * N)
        x = 4 if kind == "dynamic_linear" else 1
        return dict(bytes=x * M * K + K * N + 12 * N + _BYTES[case["out"]] * M * N, flops=2 * M * K * N)
    if kind == "attention":
        B, S, H, D = (case[k] for k in "BSHD")
        e = _BYTES[case["out"]]
        last = 2 if case["out"] == "half" else 1
        return dict(bytes=3 * B * S * H * D + B * H * S * S * (1 + e) + e * B * S + last * B * S * H * D, flops=4 * B * H * S * S * D)
    if kind == "bottleneck":
        rows, C, F = case["B"] * case["H"] * case["W"], case["C"], case["F"]
        return dict(bytes=2 * rows * C + 2 * C * F + 9 * F * F + 8 * (2 * F + C), flops=2 * rows * F * (2 * C + 9 * F))
    if kind == "stem":
        B, H, W, C, O, k = (case[key] for key in ("B", "H", "W", "C", "O", "window"))
        rows = B * -(-H // 2) * -(-W // 2)
        return dict(bytes=B * H * W * C + k * k * C * O + 8 * O + rows * O, flops=2 * rows * k * k * C * O)
    if kind == "separable":
        B, H, W, C, O, st = (case[key] for key in ("B", "H", "W", "C", "O", "stride"))
        rows = B * -(-H // st) * -(-W // st)
        return dict(bytes=B * H * W * C + 9 * C + C * O + 8 * (C + O) + rows * O, flops=2 * rows * C * (9 + O))
    return dict(bytes=14 * case["rows"] * case["depth"] + 12 * case["depth"], flops=0)


def tolerance(case):
    """The integer sums are exact and every float step that follows is fixed (one fp32 operation after another, round to
    nearest even), so two correct implementations give the same bits.  The GELU is the exception: its exp may round
    otherwise, which moves a few of the values between the two linears across a quantization step (against a GELU in
    64 bits: 1e-5 of the block's output, at most 8e-4 of its root mean square in one value)."""
    if case["kind"] == "ffn":
        return {"rel": 4e-5, "max": 4e-3}
    return "exact"
