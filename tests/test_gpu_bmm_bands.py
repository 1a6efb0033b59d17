"""The quantized BatchMatMul by bands of 16 output rows: remainders of a band, of a 16-column tile, of a k tile and of a 16-byte
vector, rows cut into parts, operands and results at odd addresses, broadcast batches.  Against the CPU oracle, bit for bit."""
import numpy as np
import pytest

from oracle import pyoracle as orc
from tests.test_gpu_bmm import check, run, to16

pytestmark = pytest.mark.gpu
ALL = [orc.FLOAT, orc.BFLOAT16, orc.HALF]


def operands(torch, rng, N, t_out, B=1):
    mul, add = np.float32([0.375]), rng.standard_normal((B, 1, 1, N)).astype(np.float32)
    binary = [(orc.BIN_MUL, mul), (orc.BIN_ADD, add)]
    return binary if t_out == orc.FLOAT else [(alg, to16(torch, v, t_out)) for alg, v in binary]


# P.V over more than 192 k: one row to several bands per wavefront, the first and last columns of a tile, one to six k tiles
@pytest.mark.parametrize("M", [1, 15, 17, 70, 200])
@pytest.mark.parametrize("K,N", [(193, 16), (200, 17), (208, 20), (240, 31), (256, 48), (257, 50), (320, 64), (383, 64), (384, 20), (193, 79)])
@pytest.mark.parametrize("t_out", ALL)
def test_products_over_many_k(hip, dev, M, K, N, t_out):
    import torch
    rng = np.random.default_rng(M * 7 + K + N)
    x, y = rng.integers(-128, 128, (2, 3, M, K)).astype(np.int8), rng.integers(-128, 128, (2, 3, K, N)).astype(np.int8)
    # (few tiles of 16-bit rows that are no whole vectors and over 64 columns are the tiles')
    kernel = "bmm_tiles" if t_out != orc.FLOAT and (K, N) == (193, 79) else "bmm_bands"
    check(hip, dev, x, y, t_out=t_out)
    assert hip.last_kernel()[0] == kernel
    check(hip, dev, x, y, binary=operands(torch, rng, N, t_out, 2)[::-1], t_out=t_out, x_off=3, y_off=1)
    check(hip, dev, x, y[:1], binary=operands(torch, rng, N, t_out)[1:], t_out=t_out, x_off=16)
    assert hip.last_kernel()[0] == kernel


# Q.K^T of at least 1024 tiles of 128 rows: rows of whole vectors and others, one to eleven column tiles, D of one and two k tiles
@pytest.mark.parametrize("M,K,N", [(65, 64, 16), (66, 16, 17), (80, 32, 20), (81, 64, 33), (65, 80, 47), (70, 48, 64), (129, 64, 99), (65, 32, 161)])
@pytest.mark.parametrize("t_out", ALL)
def test_many_matrices(hip, dev, M, K, N, t_out):
    import torch
    rng = np.random.default_rng(M * 7 + K + N)
    x, y = rng.integers(-128, 128, (129, 8, M, K)).astype(np.int8), rng.integers(-128, 128, (129, 8, N, K)).astype(np.int8)
    # (16-bit rows of up to 64 columns that are no whole vectors are the tiles')
    kernel = ("bmm_tiles", 21) if t_out != orc.FLOAT and N % 8 and N <= 64 else ("bmm_bands", 1)
    check(hip, dev, x, y, adj_y=True, binary=operands(torch, rng, N, t_out, 129), t_out=t_out)
    assert hip.last_kernel() == kernel
    check(hip, dev, x, y[:, :1], adj_y=True, binary=operands(torch, rng, N, t_out)[:1] if N == 20 else (), t_out=t_out)
    # (nor fp32 rows whose last 32 columns are more than half full, without operands)
    assert hip.last_kernel() == (("bmm_tiles", 21) if t_out == orc.FLOAT and N == 17 else kernel)


# both sides of the lines between the bands and the tiles: y along k, then y transposed on the way
@pytest.mark.parametrize("B,M,K,N,adj_y,t_out,n_ops,kernel", [
    (1030, 70, 64, 61, True, orc.BFLOAT16, 1, "bmm_tiles"), (1030, 70, 64, 67, True, orc.BFLOAT16, 1, "bmm_bands"),
    (345, 257, 64, 67, True, orc.HALF, 0, "bmm_tiles"), (345, 256, 64, 67, True, orc.HALF, 0, "bmm_tiles"), (520, 256, 64, 67, True, orc.HALF, 0, "bmm_bands"),
    (700, 70, 64, 169, True, orc.FLOAT, 0, "bmm_bands"), (515, 70, 64, 169, True, orc.FLOAT, 0, "bmm_tiles"), (515, 70, 64, 193, True, orc.FLOAT, 0, "bmm_tiles"),
    (300, 192, 64, 169, True, orc.FLOAT, 0, "bmm_bands"), (300, 193, 64, 169, True, orc.FLOAT, 0, "bmm_tiles"), (515, 129, 96, 61, True, orc.FLOAT, 0, "bmm_tiles"),
    (515, 129, 112, 61, True, orc.FLOAT, 0, "bmm_bands"), (700, 70, 192, 159, True, orc.FLOAT, 0, "bmm_bands"), (515, 70, 192, 179, True, orc.FLOAT, 0, "bmm_tiles"),
    (515, 70, 64, 193, True, orc.FLOAT, 1, "bmm_bands"),
    (64, 130, 192, 100, False, orc.BFLOAT16, 0, "bmm_tiles"), (64, 130, 208, 100, False, orc.BFLOAT16, 0, "bmm_bands"),
    (86, 130, 192, 100, False, orc.BFLOAT16, 0, "bmm_bands"), (64, 130, 192, 96, False, orc.BFLOAT16, 0, "bmm_bands"),
    (64, 130, 192, 72, False, orc.BFLOAT16, 2, "bmm_tiles"), (64, 130, 192, 80, False, orc.FLOAT, 0, "bmm_bands"),
    (64, 130, 192, 84, False, orc.FLOAT, 0, "bmm_tiles"),
    (40, 130, 199, 84, False, orc.HALF, 1, "bmm_tiles"), (43, 130, 199, 84, False, orc.HALF, 1, "bmm_bands"),
    (2049, 20, 70, 52, False, orc.HALF, 1, "bmm_tiles"), (2048, 20, 70, 52, False, orc.HALF, 1, "bmm_bands"),
    (2049, 20, 70, 48, False, orc.HALF, 1, "bmm_bands"), (2049, 20, 70, 52, False, orc.HALF, 0, "bmm_bands"),
    # (what the device holds at once: 1024 workgroups, 768 where the LDS of a CU takes three)
    (769, 64, 272, 64, False, orc.HALF, 0, "bmm_tiles"), (1025, 64, 256, 64, False, orc.HALF, 0, "bmm_bands"), (768, 64, 272, 64, False, orc.HALF, 0, "bmm_bands"),
    (998, 65, 272, 64, False, orc.HALF, 0, "bmm_tiles"), (999, 65, 272, 64, False, orc.HALF, 0, "bmm_bands"), (998, 129, 272, 64, False, orc.HALF, 0, "bmm_bands"),
    (1025, 20, 208, 56, False, orc.FLOAT, 0, "bmm_tiles"), (1025, 20, 192, 64, False, orc.FLOAT, 0, "bmm_bands"),
    (1025, 20, 321, 40, False, orc.BFLOAT16, 1, "bmm_tiles"), (1025, 20, 320, 40, False, orc.BFLOAT16, 1, "bmm_bands"), (1025, 20, 321, 32, False, orc.BFLOAT16, 1, "bmm_bands"),
    (340, 130, 191, 50, False, orc.HALF, 0, "bmm_tiles"), (340, 130, 193, 50, False, orc.HALF, 0, "bmm_bands"), (342, 130, 191, 50, False, orc.HALF, 0, "bmm_bands"),
    (340, 130, 191, 48, False, orc.HALF, 0, "bmm_bands"), (42, 130, 256, 100, False, orc.HALF, 0, "bmm_tiles"),
    (43, 130, 256, 100, False, orc.HALF, 0, "bmm_bands"), (42, 130, 256, 104, False, orc.HALF, 0, "bmm_bands"), (256, 60, 190, 70, False, orc.BFLOAT16, 0, "bmm_tiles"),
    (2049, 20, 199, 52, False, orc.FLOAT, 1, "bmm_tiles"), (2049, 20, 199, 48, False, orc.FLOAT, 1, "bmm_bands")])
def test_lines_to_the_tiles(hip, dev, B, M, K, N, adj_y, t_out, n_ops, kernel):
    import torch
    rng = np.random.default_rng(M + K + N)
    x = rng.integers(-128, 128, (B, M, K)).astype(np.int8)
    y = rng.integers(-128, 128, (B, N, K) if adj_y else (B, K, N)).astype(np.int8)
    ops = [(alg, v.reshape(v.shape[1:] if v.ndim > 1 else v.shape)) for alg, v in operands(torch, rng, N, t_out)][:n_ops]
    check(hip, dev, x, y, adj_y=adj_y, binary=ops, t_out=t_out)
    assert hip.last_kernel()[0] == kernel


def test_results_beyond_the_memory_side_cache(hip, dev):
    """fp32 rows without operands: bands for 235 MB, tiles for each half, the same results."""
    import torch
    B, M, K, N = 1100, 280, 16, 191
    x, y = (torch.randint(-128, 128, s, dtype=torch.int8, device=dev) for s in ((B, M, K), (B, N, K)))
    whole, halves = torch.empty(B, M, N, device=dev), torch.empty(2, B // 2, M, N, device=dev)
    hip.qbatch_matmul(hip.bmm_params((B, M, K), (B, N, K), False, True, hip.FLOAT, 0.01)[0], x, y, whole)
    assert hip.last_kernel()[0] == "bmm_bands"
    p, _ = hip.bmm_params((B // 2, M, K), (B // 2, N, K), False, True, hip.FLOAT, 0.01)
    for i in range(2):
        hip.qbatch_matmul(p, x[i * B // 2:], y[i * B // 2:], halves[i])
        assert hip.last_kernel()[0] == "bmm_tiles"
    assert torch.equal(whole, halves.view(B, M, N))


@pytest.mark.parametrize("K,N,parts,t_out", [(64, 288, 2, orc.HALF), (32, 320, 2, orc.BFLOAT16), (200, 160, 2, orc.FLOAT), (193, 144, 2, orc.FLOAT)])
def test_rows_in_parts(hip, dev, K, N, parts, t_out):
    """Rows of whole 64-byte pieces above 512 bytes, the last part shorter than the others."""
    import torch
    rng = np.random.default_rng(N)
    adj_y = t_out != orc.FLOAT
    x = rng.integers(-128, 128, ((400, 70, K) if adj_y else (9, 70, K))).astype(np.int8)
    y = rng.integers(-128, 128, ((400, N, K) if adj_y else (9, K, N))).astype(np.int8)
    check(hip, dev, x, y, adj_y=adj_y, binary=[(alg, v.reshape(v.shape[1:] if v.ndim > 1 else v.shape)) for alg, v in operands(torch, rng, N, t_out)],
          t_out=t_out)
    assert hip.last_kernel() == ("bmm_bands", parts)


@pytest.mark.parametrize("t_out", ALL)
@pytest.mark.parametrize("N", [64, 67])
def test_results_at_any_address(hip, dev, t_out, N):
    """A result that starts off a 16-byte boundary, with the elements around it untouched."""
    import torch
    rng = np.random.default_rng(N)
    x, y = rng.integers(-128, 128, (130, 37, 200)).astype(np.int8), rng.integers(-128, 128, (130, 200, N)).astype(np.int8)
    want = run(hip, dev, x, y, 2.0, 3.0, t_out=t_out)
    xd, yd = torch.from_numpy(x).to(dev), torch.from_numpy(y).to(dev)
    p, _ = hip.bmm_params(x.shape, y.shape, False, False, t_out, float(np.float32(6.0) / np.float32(127 * 127)))
    dt = torch.float32 if t_out == orc.FLOAT else torch.int16
    for off in range(1, 16 // dt.itemsize):
        out = torch.full((want.size + 16,), -77, dtype=dt, device=dev)
        hip.qbatch_matmul(p, xd, yd, out[off:])
        assert hip.last_kernel()[0] == "bmm_bands"
        got = out.cpu().numpy()
        assert (got[:off] == -77).all() and (got[off + want.size:] == -77).all()
        np.testing.assert_array_equal(got[off:off + want.size].view(want.dtype), want.ravel())
