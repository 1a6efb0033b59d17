"""The quantized BatchMatMul where rows are no multiple of a vector load: loads at any byte address, pieces cut by the end of
a row, 16-bit results on rows of any length, whole matrices per XCD.  Against the CPU oracle, bit for bit."""
import numpy as np
import pytest

from oracle import pyoracle as orc
from tests.test_gpu_bmm import check, to16

pytestmark = pytest.mark.gpu

# the shortest operands that take vector loads (K = 16, 4 columns), remainders of the 64-wide tile and of a 16-byte piece,
# 128-row tiles, batches around a multiple of 8
SHAPES = [((3,), 4, 16, 4), ((8,), 5, 17, 7), ((9,), 63, 31, 65), ((64,), 65, 79, 33), ((2, 4), 130, 197, 64), ((70,), 33, 16, 35)]


@pytest.mark.parametrize("B,M,K,N", SHAPES)
@pytest.mark.parametrize("adj_x,adj_y", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("t_out", [orc.FLOAT, orc.BFLOAT16, orc.HALF])
def test_rows_of_any_length(hip, dev, B, M, K, N, adj_x, adj_y, t_out):
    import torch
    rng = np.random.default_rng(M + K * 5 + N)
    x = rng.integers(-128, 128, B + ((K, M) if adj_x else (M, K))).astype(np.int8)
    y = rng.integers(-128, 128, B + ((N, K) if adj_y else (K, N))).astype(np.int8)
    add = rng.standard_normal((1,) * len(B) + (1, N)).astype(np.float32)
    mul = rng.standard_normal(B + (M, 1)).astype(np.float32)
    binary = [(orc.BIN_MUL, mul), (orc.BIN_ADD, add)]
    if t_out != orc.FLOAT:
        binary = [(alg, to16(torch, v, t_out)) for alg, v in binary]
    check(hip, dev, x, y, adj_x, adj_y, binary[1:], t_out, x_off=3, y_off=1)   # an operand broadcast over the rows
    check(hip, dev, x, y, adj_x, adj_y, binary, t_out)
    check(hip, dev, x, y, adj_x, adj_y, (), t_out, x_off=1)


@pytest.mark.parametrize("t_out", [orc.FLOAT, orc.BFLOAT16])
def test_large_tiles(hip, dev, t_out):
    """At least 1024 tiles of 128 rows, which unaligned operands leave to the 64 x 64 ones."""
    rng = np.random.default_rng(3)
    x = rng.integers(-128, 128, (520, 131, 37)).astype(np.int8)
    for n in (3 * 21, 131):
        y = rng.integers(-128, 128, (520, 37, n)).astype(np.int8)
        check(hip, dev, x, y, t_out=t_out, y_off=2)


@pytest.mark.parametrize("adj_x,adj_y", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N", [(5, 7), (4, 6), (2, 9), (70, 65)])
@pytest.mark.parametrize("t_out", [orc.FLOAT, orc.BFLOAT16])
def test_empty_reduction(hip, dev, adj_x, adj_y, M, N, t_out):
    """K = 0 with the null operands of empty tensors: the empty sum, scaled, and the fused operands."""
    import torch
    rng = np.random.default_rng(M + N)
    x, y = (np.zeros(s, np.int8) for s in ((3, 0, M) if adj_x else (3, M, 0), (3, N, 0) if adj_y else (3, 0, N)))
    mul, add = rng.standard_normal((3, M, 1)).astype(np.float32), rng.standard_normal((1, 1, N)).astype(np.float32)
    td = torch.float32 if t_out == orc.FLOAT else torch.bfloat16
    mul, add = torch.from_numpy(mul).to(dev, td), torch.from_numpy(add).to(dev, td)
    fused = [(hip.BIN_ADD, add, (1, 1, N)), (hip.BIN_MUL, mul, (3, M, 1))]
    for binary, want in (((), torch.zeros(3, M, N, dtype=td, device=dev)), (fused[:1], add.expand(3, M, N)), (fused, add * mul)):
        p, shape = hip.bmm_params(x.shape, y.shape, adj_x, adj_y, t_out, 0.5, binary)
        out = torch.full(shape, 7.0, dtype=td, device=dev)
        hip.qbatch_matmul(p, None, None, out)
        torch.cuda.synchronize()
        assert torch.equal(out, want)


# one operand with rows too short for a vector load beside one with any rows: 1 to 3 columns of y, 1 to 3 columns of an adjoint
# x, K < 16 on the side that runs along k
@pytest.mark.parametrize("M,K,N,adj_x,adj_y", [(70, 64, 1, False, False), (66, 130, 3, False, False), (130, 37, 2, True, False),
                                               (3, 70, 68, True, False), (1, 129, 35, True, False), (2, 16, 131, True, True),
                                               (68, 9, 40, False, False), (37, 15, 5, True, True), (3, 8, 2, True, False)])
@pytest.mark.parametrize("t_out", [orc.FLOAT, orc.HALF])
def test_one_narrow_operand(hip, dev, M, K, N, adj_x, adj_y, t_out):
    import torch
    rng = np.random.default_rng(M * 3 + K + N)
    x = rng.integers(-128, 128, (9,) + ((K, M) if adj_x else (M, K))).astype(np.int8)
    y = rng.integers(-128, 128, (9,) + ((N, K) if adj_y else (K, N))).astype(np.int8)
    binary = [(orc.BIN_MUL, rng.standard_normal((1, 1, N)).astype(np.float32)), (orc.BIN_ADD, rng.standard_normal((9, M, 1)).astype(np.float32))]
    if t_out != orc.FLOAT:
        binary = [(alg, to16(torch, v, t_out)) for alg, v in binary]
    for fused in ((), binary[:1], binary):
        check(hip, dev, x, y, adj_x, adj_y, fused, t_out)
        check(hip, dev, x, y, adj_x, adj_y, fused, t_out, x_off=1, y_off=3)


@pytest.mark.parametrize("B0,B1,M", [(4096, 4099, 1), (3, 5, 70000 * 64 + 1), (2, 33000, 1)])
def test_launches_of_any_extent(hip, dev, B0, B1, M):
    """2^24 matrices and more, more tiles of a matrix than one grid dimension behind the first takes, and both ends of the
    split of the matrices over two grid dimensions: outer products over a broadcast batch, K = N = 1."""
    import torch
    g = torch.Generator(device=dev).manual_seed(M + B1)
    x = torch.randint(-128, 128, (B0, 1, M, 1), dtype=torch.int8, device=dev, generator=g)
    y = torch.randint(-128, 128, (1, B1, 1, 1), dtype=torch.int8, device=dev, generator=g)
    p, shape = hip.bmm_params(tuple(x.shape), tuple(y.shape), False, False, hip.FLOAT, 0.25)
    out = torch.full(shape, 0.125, device=dev)
    hip.qbatch_matmul(p, x, y, out)
    torch.cuda.synchronize()
    assert torch.equal(out, x.float() * y.float() * 0.25)


@pytest.mark.parametrize("N", [32, 64, 96, 128, 131])
@pytest.mark.parametrize("off", [0, 1, 16, 32])
def test_16_bit_rows(hip, dev, N, off):
    """16-bit results whose rows are whole 64-byte pieces or not, by their length or by the address of the output (elements)."""
    import torch
    g = torch.Generator(device=dev).manual_seed(N + off)
    x = torch.randint(-128, 128, (8, 69, 64), dtype=torch.int8, device=dev, generator=g)
    y = torch.randint(-128, 128, (8, N, 64), dtype=torch.int8, device=dev, generator=g)
    p, shape = hip.bmm_params(tuple(x.shape), tuple(y.shape), False, True, hip.BFLOAT16, 0.03125)
    n = 8 * 69 * N
    buf = torch.full((n + 128,), 7.0, dtype=torch.bfloat16, device=dev)
    hip.qbatch_matmul(p, x, y, buf[off:])
    torch.cuda.synchronize()
    want = (torch.bmm(x.cpu().float(), y.cpu().float().transpose(1, 2)) * 0.03125).bfloat16()
    assert torch.equal(buf[off:off + n].cpu().view(shape), want)
    assert bool((buf[:off] == 7.0).all()) and bool((buf[off + n:] == 7.0).all())
