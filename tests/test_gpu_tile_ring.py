"""The tile kernel with a ring of eight LDS stages (64 x 64 tiles, one per CU) and its 128 x 64 tiles: K loops shorter than the
ring, as long as it and longer, K a multiple of 64 and not, ragged rows and channels, rows that are whole 16-byte vectors and not,
the vector and (no bias, a sum of rows that are not whole words) the element-wise epilogue; and the sizes at which the choice of a tile
shape changes.  Bit-equal to the oracle."""
import numpy as np
import pytest

from oracle import pyoracle as orc
from tests.test_gpu_matmul import V2_DEQ, V2_REQ_S8, make_acts, make_layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [4, 5])
@pytest.mark.parametrize("K", [16, 64, 112, 128, 192, 384, 448, 464, 512, 576, 1088])
def test_k_loops_around_the_ring(hip, dev, shape, K):
    hip.force_tile_shape(matmul=shape)
    for M, N, kw in [(70, 80, V2_DEQ), (130, 132, V2_DEQ), (129, 67, V2_DEQ), (193, 144, V2_REQ_S8)]:
        layer, w, bias = make_layer(hip, dev, K, N, seed=K + N + shape)
        x, xq, mn, mx = make_acts(M, K, seed=M + K)
        r = float(np.abs(x @ w + bias).max())
        ref = layer.oracle(xq, kw, mn, mx, -r, r)
        whole = N % 4 == 0   # every row a multiple of 16 bytes
        for path in ("tile", "fused"):
            np.testing.assert_array_equal(layer.run(xq, kw, mn, mx, -r, r, path=path), ref)
            if path == "fused" and M <= 128:
                assert hip.last_kernel()[0] == "small_m"
            elif shape == 5 and whole:
                assert hip.last_kernel() == ("tile", 128, 64, 8)
            else:   # (128 x 64 tiles take whole vectors alone)
                assert hip.last_kernel() == ("tile", 64, 64, 8 if K > 768 else 4)


@pytest.mark.parametrize("K", [752, 768, 784, 832, 896, 960, 1040])
def test_k_where_the_ring_of_64x64_tiles_changes(hip, dev, K):
    """Four stages up to 12 steps of 64, eight beyond."""
    hip.force_tile_shape(matmul=4)
    for M, N, kw in [(70, 80, V2_DEQ), (129, 67, V2_DEQ), (193, 144, V2_REQ_S8)]:
        layer, w, bias = make_layer(hip, dev, K, N, seed=K + N)
        x, xq, mn, mx = make_acts(M, K, seed=M + K)
        r = float(np.abs(x @ w + bias).max())
        np.testing.assert_array_equal(layer.run(xq, kw, mn, mx, -r, r, path="tile"), layer.oracle(xq, kw, mn, mx, -r, r))
        assert hip.last_kernel() == ("tile", 64, 64, 8 if K > 768 else 4)


@pytest.mark.parametrize("M,K,N,tile", [(1024, 512, 1024, (64, 64, 4)), (1025, 512, 1024, (64, 64, 4)),       # 256 and 272 tiles of 64 x 64
                                        (1024, 896, 1024, (64, 64, 8)), (1025, 896, 1024, (128, 64, 8)),
                                        (2048, 768, 1024, (128, 64, 8)), (2049, 768, 1024, (128, 128, 4)),    # 256 and 272 of 128 x 64
                                        (2048, 752, 1024, (64, 64, 4)), (2048, 784, 1021, (64, 64, 4)),       # clamped loads, rows of odd length
                                        (1920, 832, 544, (64, 64, 4)), (1840, 832, 544, (128, 64, 8)),        # 15 tile rows against 30 or 29
                                        (4224, 1552, 256, (64, 64, 4)), (4160, 1552, 256, (128, 64, 8)),      # clamped loads, 33 against 66 or 65
                                        (384, 1536, 2880, (128, 64, 8)), (384, 1472, 2880, (64, 64, 4)),      # 3 against 6, N >= M
                                        (120, 1040, 8224, (128, 64, 8))])                                      # one tile row
def test_where_the_shape_changes(hip, dev, M, K, N, tile):
    layer, _, _ = make_layer(hip, dev, K, N, seed=K + N)
    _, xq, mn, mx = make_acts(M, K, seed=M + K)
    np.testing.assert_array_equal(layer.run(xq, V2_DEQ, mn, mx, path="fused"), layer.oracle(xq, V2_DEQ, mn, mx))
    assert hip.last_kernel() == ("tile", *tile)


@pytest.mark.parametrize("M,K,N,kernel", [(16, 64, 8256, "small_m"), (17, 64, 8192, "small_m"), (17, 64, 8256, "tile"),       # 128 and 129 tiles
                                          (32, 48, 8256, "small_m"), (32, 64, 8257, "small_m"),                              # rows of odd length
                                          (32, 240, 16384, "tile"), (32, 256, 16384, "small_m"), (32, 256, 16448, "tile"),   # 256 and 257
                                          (32, 752, 16448, "tile"), (32, 768, 16448, "small_m"), (32, 768, 16384, "tile"),
                                          (33, 64, 8192, "small_m"), (33, 64, 8256, "tile"), (65, 64, 4096, "small_m"),
                                          (65, 64, 4160, "tile"), (128, 1040, 4160, "tile"), (128, 64, 4161, "small_m"),
                                          (128, 128, 4161, "tile"), (128, 112, 4161, "small_m"), (128, 2000, 4161, "tile"),  # rows of odd length
                                          (129, 64, 64, "tile")])
def test_line_between_the_small_m_and_the_tile_kernel(hip, dev, M, K, N, kernel):
    layer, _, _ = make_layer(hip, dev, K, N, seed=K + N)
    _, xq, mn, mx = make_acts(M, K, seed=M + K)
    np.testing.assert_array_equal(layer.run(xq, V2_DEQ, mn, mx, path="fused"), layer.oracle(xq, V2_DEQ, mn, mx))
    assert hip.last_kernel()[0] == kernel


@pytest.mark.parametrize("K", [448, 2048])
def test_addend_in_the_ring_kernels(hip, dev, K):
    """The float addend is staged through the transposition buffer, which lies in the ring."""
    import torch
    M, N = 200, 196
    layer, _, _ = make_layer(hip, dev, K, N, seed=K)
    _, xq, mn, mx = make_acts(M, K, seed=K)
    addend = np.random.default_rng(K).standard_normal((M, N)).astype(np.float32)
    base = layer.oracle(xq, V2_DEQ, mn, mx)
    p = hip.matmul_params(t_in=orc.QUINT8, min_a=mn, max_a=mx, add_position=1, **V2_DEQ)
    x_d, a_d = torch.from_numpy(xq).to(dev), torch.from_numpy(addend).to(dev)
    for shape in (4, 5):
        hip.force_tile_shape(matmul=shape)
        out = torch.empty((M, N), dtype=torch.float32, device=dev)
        hip.qmatmul(p, x_d, layer.packed, layer.colsum, M, K, N, layer.min_b_d, layer.max_b_d, N, layer.bias_d, out, addend=a_d)
        np.testing.assert_array_equal(out.cpu().numpy(), base + addend)


@pytest.mark.parametrize("shape,tile", [(3, (128, 128)), (4, (64, 64))])
@pytest.mark.parametrize("K", [64, 112, 512, 752, 768, 784, 832, 1088])
@pytest.mark.parametrize("sum_alpha", [None, 0.5])
def test_element_wise_epilogue(hip, dev, shape, tile, K, sum_alpha):
    """Without a bias, or with a sum over rows that no vector load reads: 8-bit, 16-bit and 32-bit results."""
    import torch
    from tests.test_gpu_ragged_rows import convert
    f, M, N = np.float32, 150, 203
    rng = np.random.default_rng(K)
    x, w = rng.integers(0, 256, (M, K)).astype(np.uint8), rng.integers(-128, 128, (K, N)).astype(np.int8)
    scale, bias = (rng.random(N).astype(f) + f(0.5)) * f(0.05 / np.sqrt(K)), (rng.standard_normal(N) * 9).astype(f)
    add = (rng.standard_normal((M, N)) * 30).astype(f)
    v = (x.astype(np.int64) @ w.astype(np.int64)).astype(f) * scale
    v = np.maximum(v if sum_alpha is None else (v + bias) + f(sum_alpha) * add, f(0))
    packed, colsum = torch.empty(hip.qgemm_packed_bytes(K, N), dtype=torch.int8, device=dev), torch.empty(N, dtype=torch.int32, device=dev)
    hip.qgemm_prepack_b(torch.from_numpy(w).to(dev), False, K, N, packed, colsum)
    xd, sd, bd, ad = (torch.from_numpy(a).to(dev) for a in (x, scale, bias, add))
    elts = ([] if sum_alpha is None else [(hip.ELT_SUM, sum_alpha, 0.0)]) + [(hip.ELT_RELU, 0.0, 0.0)]
    ep = hip.Epilogue()
    ep.n_scales, ep.n_eltwise = N, len(elts)
    for i, e in enumerate(elts):
        ep.elt[i].alg, ep.elt[i].alpha, ep.elt[i].beta = e
    ring = tile + (8 if tile == (64, 64) and K > 768 else 4,)
    for T, esz in ((hip.QUINT8, 1), (hip.QINT8, 1), (hip.BFLOAT16, 2), (hip.FLOAT, 4)):
        for force in (shape, 0):   # (a forced 256 x 256 is not for this epilogue: it tells which one ran)
            hip.force_tile_shape(matmul=force)
            out = torch.full((M * N * esz + 16,), 0x5a, dtype=torch.uint8, device=dev)
            if sum_alpha is None:
                hip.qgemm_tile(xd, hip.QUINT8, packed, colsum, M, K, N, sd, None, ep, T, out)
            else:
                hip.qgemm_sum(xd, hip.QUINT8, packed, colsum, M, K, N, sd, bd, ep, ad, hip.FLOAT, T, out)
            if force == shape:
                assert hip.last_kernel() == ("tile", *ring)
            else:
                assert hip.last_kernel()[1] < 256
            got = out.cpu().numpy()
            assert (got[M * N * esz:] == 0x5a).all()
            np.testing.assert_array_equal(got[:M * N * esz], convert(torch, hip, np.ascontiguousarray(v), T).ravel())
