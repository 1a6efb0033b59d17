"""The 3x3 depthwise convolution at the edges of its tiles (4 output rows x 2 columns, or x 1 with stride 2), against int64
sums and the epilogue's separately rounded fp32 steps in numpy, bit for bit."""
import numpy as np
import pytest

from tests.test_gpu_stream import awkward_floats, finish

pytestmark = pytest.mark.gpu


def sums(x, w, stride, top, left, oh, ow):
    B, H, W, C = x.shape
    p = np.zeros((B, top + H + oh * stride + 3, left + W + ow * stride + 3, C), np.int64)
    p[:, top:top + H, left:left + W] = x
    return sum(p[:, i:i + (oh - 1) * stride + 1:stride, j:j + (ow - 1) * stride + 1:stride] * w[i, j, :, 0].astype(np.int64)
               for i in range(3) for j in range(3))


@pytest.mark.parametrize("B,H,W,C", [(1, 1, 1, 4), (2, 4, 2, 8), (1, 5, 3, 12), (3, 9, 7, 32), (2, 17, 33, 20), (1, 8, 64, 64)])
@pytest.mark.parametrize("stride,top,left", [(1, 1, 1), (1, 0, 2), (2, 0, 0), (2, 1, 1), (2, 2, 0)])
@pytest.mark.parametrize("signed_in", [False, True])
def test_edges(hip, dev, B, H, W, C, stride, top, left, signed_in):
    import torch
    f = np.float32
    oh, ow = -(-H // stride), -(-W // stride)
    rng = np.random.default_rng(H * 31 + W + C + stride)
    x = rng.integers(-128, 128, (B, H, W, C)).astype(np.int8) if signed_in else rng.integers(0, 256, (B, H, W, C)).astype(np.uint8)
    w = rng.integers(-128, 128, (3, 3, C, 1)).astype(np.int8)
    scale = (rng.random(C).astype(f) + f(0.5)) * f(0.004)
    bias = (rng.standard_normal(C) * 9).astype(f)
    acc = sums(x, w, stride, top, left, oh, ow)
    d = lambda a: torch.from_numpy(a).to(dev)
    g = hip.ConvGeometry(B, H, W, C, 3, 3, oh, ow, stride, stride, 1, 1, top, left)
    inf = float("inf")
    for T, dt, lo_t, hi_t in ((hip.QUINT8, np.uint8, 0, 255), (hip.QINT8, np.int8, -128, 127), (hip.FLOAT, f, -inf, inf)):
        for elts, lo, hi, has_bias, has_scale in (((), -inf, inf, True, True), (((hip.ELT_RELU, 0.0, 0.0),), 0.0, inf, False, True),
                                                  (((hip.ELT_CLIP, -2.5, 77.0),), -2.5, 77.0, True, False)):
            ep = hip.Epilogue()
            ep.n_scales, ep.n_eltwise = (C if has_scale else 0), len(elts)
            for i, e in enumerate(elts):
                ep.elt[i].alg, ep.elt[i].alpha, ep.elt[i].beta = e
            out = torch.full((acc.size * np.dtype(dt).itemsize + 32,), 0x55, dtype=torch.uint8, device=dev)
            hip.qdepthwise_conv2d(d(x), hip.QINT8 if signed_in else hip.QUINT8, g, 1, d(w), d(scale) if has_scale else None,
                                  d(bias) if has_bias else None, ep, T, out)
            torch.cuda.synchronize()
            v = acc.astype(f)
            v = v * scale if has_scale else v
            v = v + bias if has_bias else v
            v = np.minimum(np.maximum(v, f(lo)), f(hi))
            ref = v if T == hip.FLOAT else np.rint(np.clip(v, f(lo_t), f(hi_t))).astype(dt)
            got = out.cpu().numpy()
            assert (got[-32:] == 0x55).all()
            np.testing.assert_array_equal(got[:-32].view(dt).reshape(ref.shape), ref)


@pytest.mark.parametrize("B,H,W,C", [(3, 57, 59, 40), (5, 111, 113, 68)])
@pytest.mark.parametrize("signed_in", [False, True])
def test_more_outputs_per_thread(hip, dev, B, H, W, C, signed_in):
    """At stride 1 a small launch has one output position per thread; sizes that get 4 rows and 4 rows x 2 columns."""
    test_edges(hip, dev, B, H, W, C, 1, 1, 1, signed_in)


@pytest.mark.parametrize("post", ["none", "relu", "clip"])
@pytest.mark.parametrize("signed_out", [False, True])
@pytest.mark.parametrize("stride", [1, 2])
def test_rounding_and_saturation(hip, dev, post, signed_out, stride):
    """The conversion instructions of the epilogue on values that come in as biases (scale 0)."""
    import torch
    C, O = 16384, 3 // stride
    bias = awkward_floats(C)
    inf = float("inf")
    lo, hi = {"none": (-inf, inf), "relu": (0.0, inf), "clip": (-3.5, 90.0)}[post]
    ep = hip.Epilogue()
    ep.n_scales, ep.n_eltwise = 1, 0 if post == "none" else 1
    ep.elt[0].alg, ep.elt[0].alpha, ep.elt[0].beta = (hip.ELT_RELU, 0.0, 0.0) if post == "relu" else (hip.ELT_CLIP, lo, hi)
    x = torch.randint(0, 256, (1, 3, 3, C), dtype=torch.uint8, device=dev)
    w = torch.randint(-127, 128, (3, 3, C, 1), dtype=torch.int8, device=dev)
    out = torch.full((O * O, C), 0x55, dtype=torch.uint8, device=dev)
    hip.qdepthwise_conv2d(x, hip.QUINT8, hip.ConvGeometry(1, 3, 3, C, 3, 3, O, O, stride, stride, 1, 1, 1, 1), 1, w,
                          torch.zeros(1, device=dev), torch.from_numpy(bias).to(dev), ep, hip.QINT8 if signed_out else hip.QUINT8, out)
    torch.cuda.synchronize()
    ref = finish(np.zeros((O * O, C)), np.float32(0), bias, None, 0.0, lo, hi, signed_out)
    np.testing.assert_array_equal(out.cpu().numpy().view(ref.dtype), ref)
