"""The unpacked MatMul in 32 x 32 tiles (few tiles, a [K, N] weight), at the edges of its tiles, of a wavefront's 128 k and of the rounds
of all its wavefronts, from operands at odd addresses: against the CPU oracle bit for bit, the bytes behind the result untouched, and
the same as the 64 x 64 tiles give."""
import numpy as np
import pytest

from oracle import pyoracle as orc
from tests.test_gpu_matmul import V1_S32, V2_DEQ, V2_REQ_U8_RELU, make_acts, make_layer, tdt

pytestmark = pytest.mark.gpu

SHAPES = [(1, 47, 1), (3, 65, 2), (16, 127, 15), (17, 129, 16), (31, 128, 17), (32, 255, 31), (33, 257, 32), (65, 511, 33), (64, 513, 47),
          (2, 640, 49), (40, 1023, 64), (7, 1025, 65), (95, 1153, 3), (1, 2049, 300), (300, 147, 1), (511, 301, 510), (256, 1001, 1000)]


def run(hip, dev, layer, p, xq, M, K, N, t_out, off):
    import torch
    a = torch.full((M * K + 32,), 0x33, dtype=torch.uint8, device=dev)
    w = torch.full((K * N + 32,), 0x33, dtype=torch.uint8, device=dev)
    a[off:off + M * K] = torch.from_numpy(xq.view(np.uint8).ravel()).to(dev)
    w[3 * off:3 * off + K * N] = torch.from_numpy(np.ascontiguousarray(layer.wq).view(np.uint8).ravel()).to(dev)
    size = torch.empty(0, dtype=tdt(t_out)).element_size()
    out = torch.full((M * N * size + 64,), 0x55, dtype=torch.uint8, device=dev)
    hip.qmatmul_unpacked(p, a[off:], w[3 * off:], False, M, K, N, layer.min_b_d, layer.max_b_d, layer.min_b.size, layer.bias_d, out)
    got = out.cpu()
    assert (got[M * N * size:] == 0x55).all()
    return got[:M * N * size].view(tdt(t_out)).view(M, N).numpy()


@pytest.mark.parametrize("M,K,N", SHAPES)
@pytest.mark.parametrize("kw", [V2_DEQ, V2_REQ_U8_RELU, V1_S32, dict(V2_DEQ, input_mode=orc.SCALED)])
def test_edges(hip, dev, M, K, N, kw):
    layer, w, bias = make_layer(hip, dev, K, N, seed=K + N)
    x, xq, mn, mx = make_acts(M, K, seed=M, mode=kw["input_mode"])
    r = float(np.abs(x @ w + bias).max())
    ref = layer.oracle(xq, kw, mn, mx, -r, r)
    p = hip.matmul_params(t_in=orc.QUINT8 if xq.dtype == np.uint8 else orc.QINT8, min_a=mn, max_a=mx, min_out=-r, max_out=r, **kw)
    for off in (0, 1):
        got = run(hip, dev, layer, p, xq, M, K, N, kw["t_out"], off)
        assert hip.last_kernel() == ("unpacked", 2 if K > 512 else 1)
        np.testing.assert_array_equal(got, ref)
    hip.force_tile_shape(matmul=0)
    np.testing.assert_array_equal(run(hip, dev, layer, p, xq, M, K, N, kw["t_out"], 3), ref)


# 32 x 32 tiles up to 512 with K <= 512 and up to 256 with more; two groups of wavefronts share a 64 x 64 tile from K = 257 on
@pytest.mark.parametrize("M,K,N,groups", [(512, 301, 1024, 1), (544, 301, 1024, 2), (512, 511, 1024, 1), (256, 513, 1024, 2), (512, 255, 1056, 1)])
def test_line_to_the_larger_tiles(hip, dev, M, K, N, groups):
    layer, _, _ = make_layer(hip, dev, K, N, seed=K + N)
    _, xq, mn, mx = make_acts(M, K, seed=M)
    p = hip.matmul_params(t_in=orc.QUINT8, min_a=mn, max_a=mx, **V2_DEQ)
    np.testing.assert_array_equal(run(hip, dev, layer, p, xq, M, K, N, V2_DEQ["t_out"], 0), layer.oracle(xq, V2_DEQ, mn, mx))
    assert hip.last_kernel() == ("unpacked", groups)
