"""The small-M kernel as a convolution (few rows, a long K, channels in whole 64s) and with a sum in a MatMul of many rows, against
int64 sums and the epilogue's separately rounded fp32 steps, bit for bit, with the bytes behind the result untouched."""
import numpy as np
import pytest

from tests.test_gpu_ragged_rows import convert
from tests.test_oracle_conv import ref_int_conv

pytestmark = pytest.mark.gpu
F = np.float32


def epilogue(hip, n, *elts):
    ep = hip.Epilogue()
    ep.n_scales, ep.n_eltwise = n, len(elts)
    for i, e in enumerate(elts):
        ep.elt[i].alg, ep.elt[i].alpha, ep.elt[i].beta = e
    return ep


def finish(v, elts, hip, addend):
    for alg, alpha, beta in elts:
        v = (v + F(alpha) * addend.astype(F)) if alg == hip.ELT_SUM else np.maximum(v, F(0)) if alg == hip.ELT_RELU else np.clip(v, F(alpha), F(beta))
    return np.ascontiguousarray(v)


def packed_weight(torch, hip, dev, w, K, N):
    packed, colsum = torch.empty(hip.qgemm_packed_bytes(K, N), dtype=torch.int8, device=dev), torch.empty(N, dtype=torch.int32, device=dev)
    hip.qgemm_prepack_b(torch.from_numpy(w.reshape(K, N)).to(dev), False, K, N, packed, colsum)
    return packed, colsum


# (batch, height, width, channels), filter, output channels, stride, dilation, padding in front, output
@pytest.mark.parametrize("shape,k,O,stride,dil,pad,out", [
    ((1, 7, 7, 64), (3, 3), 48, (1, 1), (1, 1), (1, 1), (7, 7)),          # 9 chunk pairs
    ((1, 1, 1, 576), (1, 1), 16, (1, 1), (1, 1), (0, 0), (1, 1)),         # one position
    ((2, 8, 6, 640), (1, 1), 80, (2, 3), (1, 1), (0, 0), (4, 2)),
    ((3, 5, 9, 192), (3, 3), 32, (2, 1), (1, 1), (1, 1), (3, 9)),
    ((1, 9, 10, 128), (5, 5), 112, (1, 1), (2, 1), (4, 2), (9, 10)),
    ((4, 4, 4, 256), (2, 3), 64, (1, 1), (1, 2), (0, 0), (3, 1)),
    ((1, 6, 5, 64), (3, 3), 64, (1, 1), (3, 2), (7, 9), (15, 20)),        # windows that lie outside as a whole
    ((33, 2, 4, 64), (1, 11), 528, (1, 1), (1, 1), (0, 5), (2, 4)),       # 153 blocks of 32 x 32
    ((8, 7, 10, 192), (3, 3), 528, (1, 1), (1, 1), (1, 1), (7, 10)),      # 306
    ((8, 7, 10, 512), (3, 3), 1072, (1, 1), (1, 1), (1, 1), (7, 10))])    # 612
@pytest.mark.parametrize("signed_in", [False, True])
def test_convolutions(hip, dev, shape, k, O, stride, dil, pad, out, signed_in):
    import torch
    rng = np.random.default_rng(sum(shape) + O)
    (B, H, W, C), (kh, kw), (oh, ow) = shape, k, out
    K, M = kh * kw * C, B * oh * ow
    x = rng.integers(-128, 128, shape).astype(np.int8) if signed_in else rng.integers(0, 256, shape).astype(np.uint8)
    w = rng.integers(-127, 128, (kh, kw, C, O)).astype(np.int8)
    behind = [max((n - 1) * s + (q - 1) * d + 1 - size - p, 0) for n, s, q, d, size, p in zip(out, stride, k, dil, (H, W), pad)]
    acc = ref_int_conv(x, w, stride, dil, ((pad[0], behind[0]), (pad[1], behind[1])))[:, :oh, :ow].reshape(M, O)
    scale, bias = (rng.random(O).astype(F) + F(0.5)) * F(50.0 / (74.0 * 74.0 * np.sqrt(K))), (rng.standard_normal(O) * 20).astype(F)
    v0 = acc.astype(F) * scale + bias
    packed, colsum = packed_weight(torch, hip, dev, w, K, O)
    g = hip.ConvGeometry(B, H, W, C, kh, kw, oh, ow, *stride, *dil, *pad)
    dx, ds, db = (torch.from_numpy(a).to(dev) for a in (x, scale, bias))
    add8, addf = rng.integers(0, 256, (M, O)).astype(np.uint8), rng.standard_normal((M, O)).astype(F)
    relu, clip, total = (hip.ELT_RELU, 0.0, 0.0), (hip.ELT_CLIP, -7.5, 50.0), (hip.ELT_SUM, 0.5, 0.0)
    for T, esz, elts, addend, addend_type in ((hip.QUINT8, 1, (relu,), None, 0), (hip.QINT8, 1, (), None, 0), (hip.FLOAT, 4, (clip,), None, 0),
                                              (hip.BFLOAT16, 2, (), None, 0), (hip.QUINT8, 1, (total, relu), add8, hip.QUINT8),
                                              (hip.FLOAT, 4, (relu, total), addf, hip.FLOAT)):
        y = torch.full((M * O * esz + 64,), 0x5a, dtype=torch.uint8, device=dev)
        args = [dx, hip.QINT8 if signed_in else hip.QUINT8, g, packed, colsum, O, ds, db, epilogue(hip, O, *elts)]
        if addend is None:
            hip.qconv2d(*args, T, y)
        else:
            hip.qconv2d_sum(*args, torch.from_numpy(addend).to(dev), addend_type, T, y)
        pieces = -(-M // 32) * -(-O // 32)
        tile = addend is not None and K <= (576 if pieces <= 256 else 1152 if pieces <= 512 else 4800)
        assert hip.last_kernel()[0] == ("tile" if tile else "small_m")
        got = y.cpu().numpy()
        assert (got[M * O * esz:] == 0x5a).all()
        np.testing.assert_array_equal(got[:M * O * esz], convert(torch, hip, finish(v0, elts, hip, addend), T).ravel())


# up to 256, 512 and 768 blocks of 32 x 32, and the K from which on; beyond 512 up to 4 MB of input for each XCD
@pytest.mark.parametrize("B,hw,C,k,O,kernel", [(1, 16, 512, 1, 1024, "tile"), (1, 16, 576, 1, 1024, "small_m"), (1, 16, 1024, 1, 1040, "tile"),
                                               (1, 16, 1088, 1, 1040, "small_m"), (1, 16, 1088, 1, 2064, "tile"), (1, 16, 4096, 1, 2064, "tile"),
                                               (1, 16, 4160, 1, 2064, "small_m"), (1, 16, 4160, 1, 3088, "tile"), (1, 5, 592, 1, 64, "tile"),
                                               (11, 9, 4480, 1, 576, "small_m"), (12, 9, 4480, 1, 576, "tile")])
def test_line_to_the_tile_kernel(hip, dev, B, hw, C, k, O, kernel):
    import torch
    g = hip.ConvGeometry(B, hw, hw, C, k, k, hw, hw, 1, 1, 1, 1, 0, 0)
    rng = torch.Generator().manual_seed(O)
    x = torch.randint(0, 256, (B, hw, hw, C), dtype=torch.uint8, generator=rng).to(dev)
    packed, colsum = packed_weight(torch, hip, dev, torch.randint(-127, 128, (k * k * C, O), dtype=torch.int8, generator=rng).numpy(), k * k * C, O)
    scale, bias = torch.rand(O, generator=rng).to(dev) * 1e-3, torch.randn(O, generator=rng).to(dev) * 20
    got = []
    for shape in (-1, 2):
        hip.force_tile_shape(conv=shape)
        y = torch.empty(B * hw * hw * O, dtype=torch.uint8, device=dev)
        hip.qconv2d(x, hip.QUINT8, g, packed, colsum, O, scale, bias, epilogue(hip, O, (hip.ELT_RELU, 0.0, 0.0)), hip.QUINT8, y)
        assert hip.last_kernel()[0] == (kernel if shape < 0 else "tile")
        got.append(y)
    assert torch.equal(*got)


@pytest.mark.parametrize("M,N,K,kernel", [(129, 64, 768, "tile"), (129, 64, 784, "small_m"), (260, 512, 1536, "tile"), (260, 512, 1552, "small_m"),
                                          (2048, 60, 1040, "small_m"), (513, 512, 1552, "tile")])
@pytest.mark.parametrize("addend_type", ["float", "quint8"])
def test_matmul_with_a_sum(hip, dev, M, N, K, kernel, addend_type):
    import torch
    rng = np.random.default_rng(M + N)
    x, w = rng.integers(0, 256, (M, K)).astype(np.uint8), rng.integers(-127, 128, (K, N)).astype(np.int8)
    scale, bias = (rng.random(N).astype(F) + F(0.5)) * F(0.001), (rng.standard_normal(N) * 9).astype(F)
    addend = rng.standard_normal((M, N)).astype(F) * F(30) if addend_type == "float" else rng.integers(0, 256, (M, N)).astype(np.uint8)
    packed, colsum = packed_weight(torch, hip, dev, w, K, N)
    elts = ((hip.ELT_SUM, 0.5, 0.0), (hip.ELT_RELU, 0.0, 0.0))
    T, esz = (hip.FLOAT, 4) if addend_type == "float" else (hip.QUINT8, 1)
    y = torch.full((M * N * esz + 64,), 0x5a, dtype=torch.uint8, device=dev)
    dx, ds, db, da = (torch.from_numpy(a).to(dev) for a in (x, scale, bias, addend))
    hip.qgemm_sum(dx, hip.QUINT8, packed, colsum, M, K, N, ds, db, epilogue(hip, N, *elts), da, T, T, y)
    assert hip.last_kernel()[0] == kernel
    got = y.cpu().numpy()
    assert (got[M * N * esz:] == 0x5a).all()
    v = (x.astype(np.int64) @ w.astype(np.int64)).astype(F) * scale + bias
    np.testing.assert_array_equal(got[:M * N * esz], convert(torch, hip, finish(v, elts, hip, addend), T).ravel())
