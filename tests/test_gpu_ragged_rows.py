"""The tile kernel's vector epilogue on output rows that are no whole 16-byte vectors or start off a 16-byte boundary: every
result type and tile shape, the last piece of a row in parts; and the small-M kernel beyond 128 rows, and with longer runs of K.  Against int64 sums and the
epilogue's separately rounded fp32 steps, bit for bit, with the bytes around the result untouched."""
import numpy as np
import pytest

from oracle import pyoracle as orc
from tests.test_gpu_matmul import V2_DEQ, V2_REQ_S8, make_acts, make_layer

pytestmark = pytest.mark.gpu


def convert(torch, hip, v, T):
    if T == hip.FLOAT:
        return v.view(np.uint8)
    if T in (hip.BFLOAT16, hip.HALF):
        return torch.from_numpy(v).to(torch.bfloat16 if T == hip.BFLOAT16 else torch.float16).view(torch.uint8).numpy()
    lo, hi, dt = {hip.QINT8: (-128, 127, np.int8), hip.QUINT8: (0, 255, np.uint8)}[T]
    return np.rint(np.clip(v, np.float32(lo), np.float32(hi))).astype(dt).view(np.uint8)


@pytest.mark.parametrize("M,K,N", [(130, 64, 1), (129, 48, 15), (200, 64, 17), (257, 112, 63), (131, 192, 66), (300, 80, 100), (260, 128, 391), (513, 64, 259)])
@pytest.mark.parametrize("shape", [-1, 0, 1, 2, 3, 4, 5])
def test_rows_of_any_length(hip, dev, M, K, N, shape):
    import torch
    f = np.float32
    rng = np.random.default_rng(M + K + N)
    x, w = rng.integers(0, 256, (M, K)).astype(np.uint8), rng.integers(-128, 128, (K, N)).astype(np.int8)
    scale, bias = (rng.random(N).astype(f) + f(0.5)) * f(0.003), (rng.standard_normal(N) * 9).astype(f)
    v0 = (x.astype(np.int64) @ w.astype(np.int64)).astype(f) * scale + bias
    packed, colsum = torch.empty(hip.qgemm_packed_bytes(K, N), dtype=torch.int8, device=dev), torch.empty(N, dtype=torch.int32, device=dev)
    hip.qgemm_prepack_b(torch.from_numpy(w).to(dev), False, K, N, packed, colsum)
    d = [torch.from_numpy(a).to(dev) for a in (x, scale, bias)]
    hip.force_tile_shape(matmul=shape)
    for T, esz in ((hip.FLOAT, 4), (hip.BFLOAT16, 2), (hip.HALF, 2), (hip.QINT8, 1), (hip.QUINT8, 1)):
        for elts, v in (((), v0), (((hip.ELT_RELU, 0.0, 0.0),), np.maximum(v0, f(0))), (((hip.ELT_CLIP, -7.5, 50.0),), np.clip(v0, f(-7.5), f(50)))):
            ep = hip.Epilogue()
            ep.n_scales, ep.n_eltwise = N, len(elts)
            for i, e in enumerate(elts):
                ep.elt[i].alg, ep.elt[i].alpha, ep.elt[i].beta = e
            off = (M + len(elts)) % 5 * esz
            out = torch.full((M * N * esz + 64,), 0x5a, dtype=torch.uint8, device=dev)
            hip.qgemm_tile(d[0], hip.QUINT8, packed, colsum, M, K, N, d[1], d[2], ep, T, out[off:])
            assert hip.last_kernel()[0] == "tile"
            got = out.cpu().numpy()
            assert (got[:off] == 0x5a).all() and (got[off + M * N * esz:] == 0x5a).all()
            np.testing.assert_array_equal(got[off:off + M * N * esz], convert(torch, hip, np.ascontiguousarray(v), T).ravel())


@pytest.mark.parametrize("N", [44, 100])
@pytest.mark.parametrize("K,shapes", [(192, (0, 1, 2, 3, 4)), (80, (3, 4))])
def test_sums_on_rows_of_any_length(hip, dev, N, K, shapes):
    """8-bit rows of whole words, 32-bit and 16-bit results off a 16-byte boundary: the addend's row segments, the ragged last
    channels, the sum before and after the activation, and in place."""
    import torch
    f, M = np.float32, 260
    rng = np.random.default_rng(N + K)
    x, w = rng.integers(0, 256, (M, K)).astype(np.uint8), rng.integers(-128, 128, (K, N)).astype(np.int8)
    scale, bias = (rng.random(N).astype(f) + f(0.5)) * f(0.003), (rng.standard_normal(N) * 9).astype(f)
    v0 = (x.astype(np.int64) @ w.astype(np.int64)).astype(f) * scale + bias
    packed, colsum = torch.empty(hip.qgemm_packed_bytes(K, N), dtype=torch.int8, device=dev), torch.empty(N, dtype=torch.int32, device=dev)
    hip.qgemm_prepack_b(torch.from_numpy(w).to(dev), False, K, N, packed, colsum)
    d = [torch.from_numpy(a).to(dev) for a in (x, scale, bias)]
    addends = {hip.QUINT8: rng.integers(0, 256, (M, N)).astype(np.uint8), hip.QINT8: rng.integers(-128, 128, (M, N)).astype(np.int8),
               hip.FLOAT: (rng.standard_normal((M, N)) * 30).astype(f)}
    total, relu = (hip.ELT_SUM, 0.75, 0.0), (hip.ELT_RELU, 0.0, 0.0)
    for T, off in ((hip.QUINT8, 0), (hip.QINT8, 4), (hip.FLOAT, 4), (hip.BFLOAT16, 2)):
        esz = {hip.FLOAT: 4, hip.BFLOAT16: 2}.get(T, 1)
        for t_add, add in addends.items():
            for elts in ((total, relu), (relu, total)):
                v = v0
                for e in elts:
                    v = v + f(0.75) * add.astype(f) if e is total else np.maximum(v, f(0))
                want = convert(torch, hip, np.ascontiguousarray(v), T).ravel()
                ep = hip.Epilogue()
                ep.n_scales, ep.n_eltwise = N, 2
                for i, e in enumerate(elts):
                    ep.elt[i].alg, ep.elt[i].alpha, ep.elt[i].beta = e
                add_d = torch.from_numpy(add).to(dev)
                for shape in shapes:
                    hip.force_tile_shape(matmul=shape)
                    out = torch.full((M * N * esz + 64,), 0x5a, dtype=torch.uint8, device=dev)
                    to = out[off:off + M * N * esz]
                    hip.qgemm_sum(d[0], hip.QUINT8, packed, colsum, M, K, N, d[1], d[2], ep, add_d, t_add, T, to)
                    # (tiles wider than 128: the vector epilogue has them, the element-wise one does not)
                    assert hip.last_kernel()[:3] == ("tile", *[(256, 256), (256, 192), (256, 128), (128, 128), (64, 64)][shape])
                    got = out.cpu().numpy()
                    assert (got[:off] == 0x5a).all() and (got[off + M * N * esz:] == 0x5a).all()
                    np.testing.assert_array_equal(got[off:off + M * N * esz], want)
                    if esz == 1 and t_add != hip.FLOAT:   # the addend is the output's buffer
                        to.copy_(add_d.view(torch.uint8).ravel())
                        hip.qgemm_sum(d[0], hip.QUINT8, packed, colsum, M, K, N, d[1], d[2], ep, to, t_add, T, to)
                        got = out.cpu().numpy()
                        assert (got[:off] == 0x5a).all() and (got[off + M * N * esz:] == 0x5a).all()
                        np.testing.assert_array_equal(got[off:off + M * N * esz], want)


@pytest.mark.parametrize("M,N,K", [(129, 70, 784), (140, 33, 1040), (512, 100, 784), (513, 64, 848), (1024, 30, 976), (17, 50, 1600), (64, 200, 3088),
                                   (260, 700, 1040), (2048, 50, 2064), (100, 2040, 1040), (64, 2100, 272),
                                   (9, 4112, 2576), (16, 4100, 5120), (5, 8208, 3088), (13, 8208, 4608)])
def test_small_m_kernel_on_more_rows_and_wavefronts(hip, dev, M, N, K):
    layer, w, bias = make_layer(hip, dev, K, N, seed=K + N)
    x, xq, mn, mx = make_acts(M, K, seed=M + K)
    r = float(np.abs(x @ w + bias).max())
    for kw in (V2_DEQ, V2_REQ_S8):
        np.testing.assert_array_equal(layer.run(xq, kw, mn, mx, -r, r, path="fused"), layer.oracle(xq, kw, mn, mx, -r, r))
        assert hip.last_kernel()[0] == "small_m"


@pytest.mark.parametrize("M,N,K,kernel", [(129, 64, 768, "tile"), (129, 64, 784, "small_m"), (129, 65, 512, "tile"), (129, 65, 528, "small_m"), (512, 256, 768, "tile"), (512, 256, 784, "small_m"),
                                          (512, 257, 784, "tile"), (1024, 128, 784, "small_m"), (1024, 129, 784, "tile"), (1024, 256, 1024, "tile"),
                                          (1024, 256, 1040, "small_m"), (1024, 257, 1040, "tile"), (2048, 64, 784, "small_m"), (2049, 32, 784, "tile"), (64, 4096, 128, "small_m"),
                                          (64, 4160, 128, "tile"), (128, 2048, 1552, "small_m"), (128, 2112, 1552, "tile"), (65, 2700, 5168, "small_m"), (97, 2080, 5168, "tile"),
                                          (96, 2112, 512, "tile"), (96, 2112, 528, "small_m")])
def test_line_between_the_kernels(hip, dev, M, N, K, kernel):
    layer, _, _ = make_layer(hip, dev, K, N, seed=K + N)
    _, xq, mn, mx = make_acts(M, K, seed=M + K)
    np.testing.assert_array_equal(layer.run(xq, V2_DEQ, mn, mx, path="fused"), layer.oracle(xq, V2_DEQ, mn, mx))
    assert hip.last_kernel()[0] == kernel
