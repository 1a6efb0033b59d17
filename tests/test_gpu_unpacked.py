"""The quantized MatMul on operands as TensorFlow stores them (itexhip_qmatmul_unpacked): any K, both weight layouts,
against the CPU oracle, bit for bit."""
import numpy as np
import pytest

from oracle import pyoracle as orc
from tests.test_gpu_matmul import V1_S32, V2_DEQ, V2_REQ_U8_RELU, make_acts, make_layer, tdt

pytestmark = pytest.mark.gpu

# edges of the 64 x 64 tile and of the 256-long K step, tensors of fewer than 16 bytes, pieces cut by the end of either
# operand in the last rows, several steps
SHAPES = [(1, 1, 1), (1, 3, 1000), (5, 15, 3), (2, 8, 70), (3, 17, 16), (64, 256, 64), (65, 257, 63), (63, 255, 65),
          (130, 1001, 70), (17, 13, 129), (200, 530, 33)]


@pytest.mark.parametrize("M,K,N", SHAPES)
@pytest.mark.parametrize("kw,transpose_b", [(V2_DEQ, False), (V2_REQ_U8_RELU, False), (V1_S32, False),
                                            (dict(V2_DEQ, input_mode=orc.SCALED), True),
                                            (dict(V1_S32, input_mode=orc.SCALED), True)])
def test_unpacked_matmul_vs_oracle(hip, dev, M, K, N, kw, transpose_b):
    import torch
    layer, w, bias = make_layer(hip, dev, K, N, seed=K + N)
    x, xq, mn, mx = make_acts(M, K, seed=M, mode=kw["input_mode"])
    r_out = float(np.abs(x @ w + bias).max())
    ref = layer.oracle(xq, kw, mn, mx, -r_out, r_out)
    t_in = orc.QUINT8 if xq.dtype == np.uint8 else orc.QINT8
    p = hip.matmul_params(t_in=t_in, min_a=mn, max_a=mx, min_out=-r_out, max_out=r_out, **kw)
    w_d = torch.from_numpy(np.ascontiguousarray(layer.wq.T) if transpose_b else layer.wq).to(dev)
    out = torch.empty((M, N), dtype=tdt(kw["t_out"]), device=dev)
    out.view(torch.uint8).fill_(0x55)
    hip.qmatmul_unpacked(p, torch.from_numpy(xq).to(dev), w_d, transpose_b, M, K, N, layer.min_b_d, layer.max_b_d,
                         layer.min_b.size, layer.bias_d, out)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(out.cpu().numpy(), ref)


# both sides of the line up to which two groups share a tile's K steps (256 tiles); an odd number of steps and a single one,
# where the second group has none
@pytest.mark.parametrize("M,K,N", [(1024, 257, 1024), (1025, 257, 1024), (1020, 513, 1023), (77, 1025, 190), (129, 255, 65), (64, 1281, 64)])
@pytest.mark.parametrize("kw,transpose_b", [(V2_DEQ, False), (V2_REQ_U8_RELU, False), (dict(V2_DEQ, input_mode=orc.SCALED), True)])
def test_split_of_k_steps(hip, dev, M, K, N, kw, transpose_b):
    test_unpacked_matmul_vs_oracle(hip, dev, M, K, N, kw, transpose_b)
    tiles = -(-M // 64) * -(-N // 64)
    assert hip.last_kernel() == ("unpacked", 2 if tiles <= 256 and (transpose_b or K > 256) else 1)


# sizes that go one thread per output by themselves, through the tile kernel as well, and sizes on both sides of the line
@pytest.mark.parametrize("M,K,N", [(5, 15, 3), (2, 8, 70), (3, 17, 16), (17, 13, 129), (1, 17, 200), (200, 33, 1), (65, 9, 66), (300, 36, 8), (300, 39, 8), (300, 46, 8), (300, 47, 8)])
@pytest.mark.parametrize("kw,transpose_b", [(V2_DEQ, False), (V2_REQ_U8_RELU, False), (dict(V2_DEQ, input_mode=orc.SCALED), True)])
@pytest.mark.parametrize("shape", [-1, 0])
def test_both_kernels(hip, dev, M, K, N, kw, transpose_b, shape):
    hip.force_tile_shape(matmul=shape)
    test_unpacked_matmul_vs_oracle(hip, dev, M, K, N, kw, transpose_b)
    assert hip.last_kernel()[0] == ("unpacked" if shape == 0 or K == 47 else "per_output")


def test_more_rows_than_tiles_in_a_launch(hip, dev):
    """2^30 rows of one value and one column: 2^24 tiles of 64 rows, one more launch than 2^32 threads allow."""
    import torch
    M = 1 << 30
    if torch.cuda.mem_get_info()[0] < 8 * M:
        pytest.skip("needs 8 GiB")
    p = hip.matmul_params(t_in=hip.QINT8, t_out=hip.QINT8, input_mode=hip.SCALED, min_a=-127.0, max_a=127.0, has_requantize=True,
                          min_out=-127.0, max_out=127.0)
    a = torch.arange(64, dtype=torch.int8, device=dev).repeat(M // 64)
    w = torch.ones(1, dtype=torch.int8, device=dev)
    lo, hi = torch.full((1,), -127.0, device=dev), torch.full((1,), 127.0, device=dev)
    out = torch.full((M,), -1, dtype=torch.int8, device=dev)
    hip.qmatmul_unpacked(p, a, w, False, M, 1, 1, lo, hi, 1, torch.zeros(1, device=dev), out)
    torch.cuda.synchronize()
    assert torch.equal(out, a)


def test_more_outputs_than_threads_in_a_launch(hip, dev):
    """K * N < 16 with more than 2^32 outputs: one thread per output element, several per thread.  The first 128 rows hold every
    input value once; every later row must be a copy of one of them."""
    import torch
    rows, N = (1 << 32) // 15 // 128 + 1000, 15
    M = rows * 128
    if torch.cuda.mem_get_info()[0] < 24 * M:
        pytest.skip("needs 7 GiB")
    p = hip.matmul_params(t_in=hip.QINT8, t_out=hip.QINT8, input_mode=hip.SCALED, min_a=-127.0, max_a=127.0, has_requantize=True,
                          min_out=-127.0, max_out=127.0)
    a = torch.arange(128, dtype=torch.int8, device=dev).repeat(rows)
    w = torch.arange(-7, 8, dtype=torch.int8, device=dev)
    lo, hi = torch.full((1,), -16.0, device=dev), torch.full((1,), 16.0, device=dev)
    out = torch.full((rows, 128, N), -1, dtype=torch.int8, device=dev)
    hip.qmatmul_unpacked(p, a, w, False, M, 1, N, lo, hi, 1, torch.zeros(N, device=dev), out)
    torch.cuda.synchronize()
    want = (torch.arange(128).view(-1, 1) * torch.arange(-7, 8).view(1, -1) * (16.0 / 127.0))
    assert float((out[0].cpu().float() - want.round()).abs().max()) <= 1.0   # the sizes are the point here, not the rounding
    assert bool((out == out[:1]).all())
