"""The kernel for a short K, many rows and an 8-bit result, at the sizes where its tiles and pieces end, against int64 products
and the epilogue's separately rounded fp32 steps in numpy, bit for bit.  Convolutions: against the patch-matrix path."""
import numpy as np
import pytest

from oracle import pyoracle as orc
from tests.test_gpu_conv import check_implicit_conv
from tests.test_gpu_matmul import V2_REQ_S8, V2_REQ_U8_RELU, make_acts, make_layer
from tests.test_oracle_conv import ref_int_conv

pytestmark = pytest.mark.gpu
ANY_SIZE = 16   # force_tile_shape: this kernel whatever the size of the call


def reference(x, w, scale, bias, addend, sum_scale, lo, hi, signed_out):
    return finish(x.astype(np.int64) @ w.astype(np.int64), scale, bias, addend, sum_scale, lo, hi, signed_out)


def finish(acc, scale, bias, addend, sum_scale, lo, hi, signed_out):
    f = np.float32
    with np.errstate(invalid="ignore", over="ignore"):   # signalling NaN
        v = acc.astype(f) * scale
        v = v + bias
    if addend is not None:
        v = v + f(sum_scale) * addend.astype(f)
    v = np.fmin(np.fmax(v, f(lo)), f(hi))   # NaN: the bound
    v = np.fmin(np.fmax(v, f(-128 if signed_out else 0)), f(127 if signed_out else 255))
    return np.rint(v).astype(np.int8 if signed_out else np.uint8)


def run(hip, dev, M, K, N, post, add_type, signed_in, signed_out, seed):
    import torch
    rng = np.random.default_rng(seed)
    x = rng.integers(-128, 128, (M, K)).astype(np.int8) if signed_in else rng.integers(0, 256, (M, K)).astype(np.uint8)
    w = rng.integers(-127, 128, (K, N)).astype(np.int8)
    scale = (rng.random(N).astype(np.float32) + np.float32(0.5)) * np.float32(60.0 / (74.0 * 74.0 * np.sqrt(K)))
    bias = (rng.standard_normal(N) * 20).astype(np.float32)
    inf = float("inf")
    lo, hi = {"none": (-inf, inf), "relu": (0.0, inf), "clip": (-3.5, 90.0)}[post]
    ep = hip.Epilogue()
    ep.n_scales = N
    elts, addend = [], None
    if add_type is not None:
        elts.append((hip.ELT_SUM, 0.375, 0.0))
        addend = rng.integers(-128, 128, (M, N)).astype(np.int8) if add_type == hip.QINT8 else rng.integers(0, 256, (M, N)).astype(np.uint8)
    if post != "none":
        elts.append((hip.ELT_RELU, 0.0, 0.0) if post == "relu" else (hip.ELT_CLIP, lo, hi))
    ep.n_eltwise = len(elts)
    for i, (alg, a, b) in enumerate(elts):
        ep.elt[i].alg, ep.elt[i].alpha, ep.elt[i].beta = alg, a, b
    d = lambda a: torch.from_numpy(a).to(dev)
    packed = torch.empty(hip.qgemm_packed_bytes(K, N), dtype=torch.int8, device=dev)
    colsum = torch.empty(N, dtype=torch.int32, device=dev)
    hip.qgemm_prepack_b(d(w), False, K, N, packed, colsum)
    out = torch.full((M * N + 64,), 0x55, dtype=torch.uint8, device=dev)
    T_in, T_out = hip.QINT8 if signed_in else hip.QUINT8, hip.QINT8 if signed_out else hip.QUINT8
    if addend is None:
        hip.qgemm(d(x), T_in, packed, colsum, M, K, N, d(scale), d(bias), ep, T_out, out)
    else:
        hip.qgemm_sum(d(x), T_in, packed, colsum, M, K, N, d(scale), d(bias), ep, d(addend), add_type, T_out, out)
    assert hip.last_kernel()[0] == "short_k"
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert (got[M * N:] == 0x55).all()
    ref = reference(x, w, scale, bias, addend, 0.375, lo, hi, signed_out)
    np.testing.assert_array_equal(got[:M * N].view(ref.dtype).reshape(M, N), ref)


# one row tile and its remainders, one piece of K and the ends of a 32-deep chunk, a group of chunks and a weight that takes
# one wavefront column per workgroup, one piece of channels, remainders of 32 and 64, several workgroups along N
@pytest.mark.parametrize("M,K,N", [(129, 16, 16), (160, 32, 48), (161, 48, 64), (191, 64, 80), (300, 96, 256), (1025, 144, 272),
                                   (257, 176, 144), (140, 512, 528), (133, 1136, 64)])
@pytest.mark.parametrize("post", ["none", "relu", "clip"])
@pytest.mark.parametrize("signed_out", [False, True])
def test_ragged_sizes(hip, dev, M, K, N, post, signed_out):
    hip.force_tile_shape(matmul=ANY_SIZE)
    for i, add_type in enumerate((None, hip.QUINT8, hip.QINT8)):
        run(hip, dev, M, K, N, post, add_type, bool(i & 1), signed_out, M + K + N + i)


@pytest.mark.parametrize("M,K,N", [(131073, 64, 64), (70001, 48, 96), (27203, 32, 320)])
def test_several_tiles_per_wavefront(hip, dev, M, K, N):
    """Sizes that take this kernel by themselves, a row more than whole tiles."""
    run(hip, dev, M, K, N, "relu", None, False, False, 1)
    run(hip, dev, M, K, N, "relu", hip.QUINT8, False, False, 2)


@pytest.mark.parametrize("M,K,N", [(98305, 256, 48), (131100, 192, 80), (100001, 144, 64)])
def test_longer_k_by_itself(hip, dev, M, K, N):
    """Just inside the lines from which a longer K takes this kernel, a row more than whole tiles."""
    run(hip, dev, M, K, N, "relu", None, False, False, 3)


@pytest.mark.parametrize("M,K,N", [(32801, 64, 64), (10945, 112, 192), (16500, 128, 256), (16500, 160, 208), (16500, 192, 256), (16500, 256, 256)])
def test_small_launches_with_a_residual(hip, dev, M, K, N):
    """Just inside the lines from which a call with a residual takes this kernel."""
    run(hip, dev, M, K, N, "relu", hip.QUINT8, False, False, 4)


# every count of 32-deep chunks that a wavefront holds at once and the first one beyond, several row tiles per wavefront, the
# last chunk whole or half
@pytest.mark.parametrize("K", [16, 64, 80, 128, 144, 192, 208, 256, 272])
@pytest.mark.parametrize("add", [False, True])
def test_chunk_counts(hip, dev, K, add):
    hip.force_tile_shape(matmul=ANY_SIZE)
    run(hip, dev, 133001, K, 16, "clip", hip.QUINT8 if add else None, False, K % 32 != 0, seed=K)


def test_clip_with_bounds_the_wrong_way_round(hip, dev):
    """min(max(v, lo), hi) is hi everywhere then, for this kernel's sizes as for others."""
    import torch
    M, K, N = 40000, 32, 64
    ep = hip.Epilogue()
    ep.n_scales, ep.n_eltwise = N, 1
    ep.elt[0].alg, ep.elt[0].alpha, ep.elt[0].beta = hip.ELT_CLIP, 9.0, 4.0
    packed = torch.empty(hip.qgemm_packed_bytes(K, N), dtype=torch.int8, device=dev)
    colsum = torch.empty(N, dtype=torch.int32, device=dev)
    hip.qgemm_prepack_b(torch.ones(K, N, dtype=torch.int8, device=dev), False, K, N, packed, colsum)
    x = torch.arange(256, dtype=torch.uint8, device=dev).repeat(M * K // 256)
    out = torch.zeros(M, N, dtype=torch.uint8, device=dev)
    hip.qgemm(x, hip.QUINT8, packed, colsum, M, K, N, torch.full((N,), 0.01, device=dev), torch.zeros(N, device=dev), ep, hip.QUINT8, out)
    torch.cuda.synchronize()
    assert bool((out == 4).all())


@pytest.mark.parametrize("shape,wshape,strides,dil,lead", [
    ((2, 9, 10, 16), (3, 3, 16, 48), (1, 1), (1, 1), None), ((1, 8, 7, 32), (3, 2, 32, 64), (2, 1), (1, 2), None),
    ((2, 6, 6, 48), (2, 2, 48, 112), (1, 1), (1, 1), None), ((3, 13, 11, 16), (5, 5, 16, 80), (2, 2), (1, 1), (3, 1)),
    ((1, 12, 12, 128), (1, 1, 128, 160), (2, 2), (1, 1), None), ((1, 3, 3, 16), (3, 3, 16, 16), (1, 1), (1, 1), None),
    ((4, 33, 31, 32), (3, 3, 32, 64), (1, 1), (1, 1), (0, 0))])
@pytest.mark.parametrize("signed_in", [False, True])
def test_convolutions(hip, dev, shape, wshape, strides, dil, lead, signed_in):
    hip.force_tile_shape(conv=ANY_SIZE)
    check_implicit_conv(hip, dev, shape, wshape, strides, dil, lead, signed_in, np.random.default_rng(sum(shape) + signed_in), "short_k")


# no padding: every count of chunks that a wavefront holds at once, window rows of 4 channels among them
@pytest.mark.parametrize("wshape,strides", [((1, 1, 32, 48), (1, 1)), ((2, 2, 16, 64), (1, 1)), ((2, 3, 16, 64), (2, 1)), ((2, 2, 32, 80), (1, 2)),
                                            ((3, 3, 16, 64), (1, 1)), ((3, 4, 16, 64), (2, 2)), ((7, 8, 4, 64), (2, 2)), ((4, 4, 16, 32), (1, 1)),
                                            ((3, 3, 32, 64), (1, 1))])
def test_convolutions_without_padding(hip, dev, wshape, strides):
    hip.force_tile_shape(conv=ANY_SIZE)
    check_implicit_conv(hip, dev, (3, 23, 24, wshape[2]), wshape, strides, (1, 1), (0, 0), False, np.random.default_rng(sum(wshape)), "short_k")


@pytest.mark.parametrize("kw", [V2_REQ_S8, V2_REQ_U8_RELU, dict(V2_REQ_S8, input_mode=orc.SCALED),
                                dict(V2_REQ_U8_RELU, input_mode=orc.SCALED)], ids=["s8", "u8_relu", "s8_scaled", "u8_relu_scaled"])
@pytest.mark.parametrize("per_channel", [False, True])
@pytest.mark.parametrize("M,K,N", [(300, 96, 272), (161, 48, 80), (140, 400, 528)])
def test_parameters_derived_in_the_kernel(hip, dev, kw, per_channel, M, K, N):
    """itexhip_qmatmul and itexhip_qmatmul_device_range with one weight range and one per channel, against the oracle."""
    import torch
    layer, w, bias = make_layer(hip, dev, K, N, seed=K + N, per_channel=per_channel)
    x, xq, mn, mx = make_acts(M, K, seed=M, mode=kw["input_mode"])
    r_out = float(np.abs(np.maximum(x @ w + bias, 0) if kw.get("activation") else x @ w + bias).max())
    lo = 0.0 if kw["t_out"] == orc.QUINT8 else -r_out
    t_in = orc.QUINT8 if xq.dtype == np.uint8 else orc.QINT8
    p = hip.matmul_params(t_in=t_in, min_a=mn, max_a=mx, min_out=lo, max_out=r_out, **kw)
    ep = hip.qmatmul_epilogue_desc(p, layer.min_b.size)
    # the chains this kernel takes: none, or one ReLU
    assert [(ep.elt[i].alg, ep.elt[i].alpha) for i in range(ep.n_eltwise)] in ([], [(hip.ELT_RELU, 0.0)])
    ref = layer.oracle(xq, kw, mn, mx, lo, r_out)
    hip.force_tile_shape(matmul=ANY_SIZE)
    np.testing.assert_array_equal(layer.run(xq, kw, mn, mx, lo, r_out, path="fused"), ref)
    assert hip.last_kernel()[0] == "short_k"
    p = hip.matmul_params(t_in=t_in, min_a=77.0, max_a=-3.0, min_out=lo, max_out=r_out, **kw)   # min_a / max_a unused
    range_a = torch.tensor([mn, mx], dtype=torch.float32, device=dev)
    out = torch.full((M, N), 0x55, dtype=torch.uint8, device=dev)
    hip.qmatmul_device_range(p, torch.from_numpy(xq).to(dev), layer.packed, layer.colsum, M, K, N, range_a, layer.min_b_d,
                             layer.max_b_d, layer.min_b.size, layer.bias_d, out)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(out.cpu().numpy().view(ref.dtype), ref)


@pytest.mark.parametrize("post", ["none", "relu", "clip"])
@pytest.mark.parametrize("signed_add", [False, True])
@pytest.mark.parametrize("signed_out", [False, True])
@pytest.mark.parametrize("O", [48, 144])
def test_convolutions_with_a_residual(hip, dev, post, signed_add, signed_out, O):
    """Every post-op of a convolution, and of a MatMul on its patch matrix, without an addend, with one and with one that is the
    output's own buffer."""
    import torch
    rng = np.random.default_rng(O + signed_add)
    B, H, W, C = 3, 11, 10, 32
    M, K = B * H * W, 9 * C
    x, w = rng.integers(0, 256, (B, H, W, C)).astype(np.uint8), rng.integers(-127, 128, (3, 3, C, O)).astype(np.int8)
    acc = ref_int_conv(x, w, (1, 1), (1, 1), ((1, 1), (1, 1))).reshape(M, O)
    scale = ((rng.random(O) + 0.5) * 8e-4).astype(np.float32)
    bias = (rng.standard_normal(O) * 20).astype(np.float32)
    addend = rng.integers(-128, 128, (M, O)).astype(np.int8) if signed_add else rng.integers(0, 256, (M, O)).astype(np.uint8)
    T_add, T_out = (hip.QINT8 if s else hip.QUINT8 for s in (signed_add, signed_out))
    inf = float("inf")
    lo, hi = {"none": (-inf, inf), "relu": (0.0, inf), "clip": (-3.5, 90.0)}[post]
    d = lambda a: torch.from_numpy(a).to(dev)
    g = hip.ConvGeometry(B, H, W, C, 3, 3, H, W, 1, 1, 1, 1, 1, 1)
    packed = torch.empty(hip.qgemm_packed_bytes(K, O), dtype=torch.int8, device=dev)
    colsum = torch.empty(O, dtype=torch.int32, device=dev)
    hip.qgemm_prepack_b(d(w.reshape(K, O)), False, K, O, packed, colsum)
    xd, sc, bi = d(x), d(scale), d(bias)
    cols = torch.empty((M, K), dtype=torch.uint8, device=dev)
    hip.im2col8(xd, g, K, cols)
    hip.force_tile_shape(matmul=ANY_SIZE, conv=ANY_SIZE)
    for add in (False, True):
        ep = hip.Epilogue()
        elts = ([(hip.ELT_SUM, 0.375, 0.0)] if add else []) + {"none": [], "relu": [(hip.ELT_RELU, 0.0, 0.0)], "clip": [(hip.ELT_CLIP, lo, hi)]}[post]
        ep.n_scales, ep.n_eltwise = O, len(elts)
        for i, e in enumerate(elts):
            ep.elt[i].alg, ep.elt[i].alpha, ep.elt[i].beta = e
        ref = finish(acc, scale, bias, addend if add else None, 0.375, lo, hi, signed_out)
        for in_place in (False, True) if add else (False,):
            for conv in (False, True):
                out = d(addend.view(np.uint8)) if in_place else torch.full((M, O), 0x55, dtype=torch.uint8, device=dev)
                src = out if in_place else d(addend)
                if conv and add:
                    hip.qconv2d_sum(xd, hip.QUINT8, g, packed, colsum, O, sc, bi, ep, src, T_add, T_out, out)
                elif conv:
                    hip.qconv2d(xd, hip.QUINT8, g, packed, colsum, O, sc, bi, ep, T_out, out)
                elif add:
                    hip.qgemm_sum(cols, hip.QUINT8, packed, colsum, M, K, O, sc, bi, ep, src, T_add, T_out, out)
                else:
                    hip.qgemm(cols, hip.QUINT8, packed, colsum, M, K, O, sc, bi, ep, T_out, out)
                torch.cuda.synchronize()
                assert hip.last_kernel()[0] == "short_k"
                np.testing.assert_array_equal(out.cpu().numpy().view(ref.dtype), ref, err_msg=str((add, in_place, conv)))


def test_residual_in_place_several_tiles_per_wavefront(hip, dev):
    """The addend of a tile is read while the tile before it is stored: one buffer for both, at a size that takes this kernel by
    itself."""
    import torch
    M, K, N = 100003, 64, 256
    g = torch.Generator(device=dev).manual_seed(5)
    x, both = (torch.randint(0, 256, (M, n), dtype=torch.uint8, device=dev, generator=g) for n in (K, N))
    w = torch.randint(-127, 128, (K, N), dtype=torch.int8, device=dev, generator=g)
    packed = torch.empty(hip.qgemm_packed_bytes(K, N), dtype=torch.int8, device=dev)
    colsum = torch.empty(N, dtype=torch.int32, device=dev)
    hip.qgemm_prepack_b(w, False, K, N, packed, colsum)
    ep = hip.Epilogue()
    ep.n_scales, ep.n_eltwise = 1, 2
    for i, e in enumerate([(hip.ELT_SUM, 0.375, 0.0), (hip.ELT_RELU, 0.0, 0.0)]):
        ep.elt[i].alg, ep.elt[i].alpha, ep.elt[i].beta = e
    scale, bias = torch.full((1,), 1e-3, device=dev), torch.full((N,), 20.0, device=dev)
    v = (x.float() @ w.float()) * scale   # every sum below 2^24: exact in fp32 in any order
    v = v + bias
    want = (v + 0.375 * both.float()).clamp(0, 255).round().to(torch.uint8)
    hip.qgemm_sum(x, hip.QUINT8, packed, colsum, M, K, N, scale, bias, ep, both, hip.QUINT8, hip.QUINT8, both)
    assert hip.last_kernel() == ("short_k", 2, True)
    torch.cuda.synchronize()
    assert torch.equal(both, want)


@pytest.mark.parametrize("M,K,N,group", [(133003, 64, 1008, 2), (400003, 16, 144, 1), (139003, 32, 976, 1), (123003, 240, 976, 4),
                                         (139003, 272, 912, 4), (1003, 304, 80, 2), (1003, 400, 80, 4)])
def test_residual_forms(hip, dev, M, K, N, group):
    """Past 96 or 256 MB of activations, residual and result, and a K past 384, a residual takes loads in groups instead of held
    chunks."""
    import torch
    hip.force_tile_shape(matmul=ANY_SIZE)
    g = torch.Generator(device=dev).manual_seed(K)
    x = torch.randint(0, 256, (M, K), dtype=torch.uint8, device=dev, generator=g)
    add = torch.randint(-128, 128, (M, N), dtype=torch.int8, device=dev, generator=g)
    w = torch.randint(-127, 128, (K, N), dtype=torch.int8, device=dev, generator=g)
    packed = torch.empty(hip.qgemm_packed_bytes(K, N), dtype=torch.int8, device=dev)
    colsum = torch.empty(N, dtype=torch.int32, device=dev)
    hip.qgemm_prepack_b(w, False, K, N, packed, colsum)
    ep = hip.Epilogue()
    ep.n_scales, ep.n_eltwise = 1, 1
    ep.elt[0].alg, ep.elt[0].alpha = hip.ELT_SUM, 0.375
    scale, bias = torch.full((1,), 1e-3, device=dev), torch.full((N,), 20.0, device=dev)
    v = (x.float() @ w.float()) * scale   # every sum below 2^24: exact in fp32 in any order
    v = v + bias
    want = (v + 0.375 * add.float()).clamp(-128, 127).round().to(torch.int8)
    out = torch.empty((M, N), dtype=torch.int8, device=dev)
    hip.qgemm_sum(x, hip.QUINT8, packed, colsum, M, K, N, scale, bias, ep, add, hip.QINT8, hip.QINT8, out)
    assert hip.last_kernel() == ("short_k", group, False)
    torch.cuda.synchronize()
    assert torch.equal(out, want)


@pytest.mark.parametrize("image,K,N,form", [((3000007,), 16, 128, (1, False)), ((2000003,), 48, 272, (2, False)), ((2000003,), 112, 256, (4, False)),
                                            ((1700003,), 144, 128, (4, False)), ((1700003,), 240, 160, (4, False)),
                                            ((2200003,), 48, 128, (2, True)), ((2200003,), 48, 160, (2, True)),     # below the line, three columns
                                            ((2300003,), 48, 160, (2, False)), ((1500007,), 16, 240, (1, True)),    # past theirs, four columns
                                            ((260009,), 64, 480, (2, False)), ((260009,), 64, 448, (2, True)),      # two chunks over 8 columns, 7
                                            ((700001,), 16, 480, (1, False)), ((700001,), 16, 448, (1, True)),      # one
                                            ((1200007,), 176, 208, (6, True)), ((5000011,), 32, 64, (1, True)),     # a longer K, one column
                                            ((1000, 53, 51), 80, 160, (4, False)), ((1000, 53, 51), 80, 128, (3, True)),
                                            ((540, 29, 31), 16, 832, (4, False)), ((500, 29, 31), 16, 832, (1, True))])
def test_results_past_the_caches(hip, dev, image, K, N, form):
    """From 128 to 448 MB of activations and result on, some sizes take loads in groups instead of held chunks; a MatMul, or a 1 x 1
    convolution."""
    import torch
    M = int(np.prod(image))
    g = torch.Generator(device=dev).manual_seed(K)
    x = torch.randint(0, 256, (M, K), dtype=torch.uint8, device=dev, generator=g)
    w = torch.randint(-127, 128, (K, N), dtype=torch.int8, device=dev, generator=g)
    packed = torch.empty(hip.qgemm_packed_bytes(K, N), dtype=torch.int8, device=dev)
    colsum = torch.empty(N, dtype=torch.int32, device=dev)
    hip.qgemm_prepack_b(w, False, K, N, packed, colsum)
    ep = hip.Epilogue()
    ep.n_scales = 1
    scale, bias = torch.full((1,), 1e-3, device=dev), torch.full((N,), 20.0, device=dev)
    v = (x.float() @ w.float()) * scale   # every sum below 2^24: exact in fp32 in any order
    want = (v + bias).clamp(-128, 127).round().to(torch.int8)
    out = torch.empty((M, N), dtype=torch.int8, device=dev)
    if len(image) == 1:
        hip.qgemm(x, hip.QUINT8, packed, colsum, M, K, N, scale, bias, ep, hip.QINT8, out)
    else:
        B, H, W = image
        geometry = hip.ConvGeometry(B, H, W, K, 1, 1, H, W, 1, 1, 1, 1, 0, 0)
        hip.qconv2d(x, hip.QUINT8, geometry, packed, colsum, N, scale, bias, ep, hip.QINT8, out)
    assert hip.last_kernel() == ("short_k", *form)
    torch.cuda.synchronize()
    assert torch.equal(out, want)


def awkward_floats(n):
    """n fp32 values: ties around every 8-bit result with their neighbours, infinities, NaN, denormals, random bit patterns."""
    f = np.float32
    ties = np.arange(-131, 259).astype(f) + f(0.5)
    special = np.array([np.inf, -np.inf, np.nan, -np.nan, 0.0, -0.0, 1e-45, -1e-45, 3.4e38, -3.4e38, 2.0 ** 31, -2.0 ** 31], f)
    v = np.concatenate([ties, np.nextafter(ties, f(-1e9)), np.nextafter(ties, f(1e9)), special])
    patterns = np.random.default_rng(9).integers(0, 1 << 32, n - v.size, dtype=np.uint64).astype(np.uint32).view(f)
    return np.concatenate([v, patterns])


@pytest.mark.parametrize("post", ["none", "relu", "clip"])
@pytest.mark.parametrize("signed_out", [False, True])
def test_rounding_and_saturation(hip, dev, post, signed_out):
    """The conversion instructions of the epilogue on values that come in as biases (scale 0)."""
    import torch
    M, K, N = 40, 16, 16384
    bias = awkward_floats(N)
    ep = hip.Epilogue()
    ep.n_scales, ep.n_eltwise = 1, 0 if post == "none" else 1
    inf = float("inf")
    lo, hi = {"none": (-inf, inf), "relu": (0.0, inf), "clip": (-3.5, 90.0)}[post]
    ep.elt[0].alg, ep.elt[0].alpha, ep.elt[0].beta = (hip.ELT_RELU, 0.0, 0.0) if post == "relu" else (hip.ELT_CLIP, lo, hi)
    x = torch.randint(0, 256, (M, K), dtype=torch.uint8, device=dev)
    w = torch.randint(-127, 128, (K, N), dtype=torch.int8, device=dev)
    packed = torch.empty(hip.qgemm_packed_bytes(K, N), dtype=torch.int8, device=dev)
    colsum = torch.empty(N, dtype=torch.int32, device=dev)
    hip.qgemm_prepack_b(w, False, K, N, packed, colsum)
    out = torch.full((M, N), 0x55, dtype=torch.uint8, device=dev)
    hip.force_tile_shape(matmul=ANY_SIZE)
    hip.qgemm(x, hip.QUINT8, packed, colsum, M, K, N, torch.zeros(1, device=dev), torch.from_numpy(bias).to(dev), ep,
              hip.QINT8 if signed_out else hip.QUINT8, out)
    torch.cuda.synchronize()
    ref = finish(np.zeros((M, N)), np.float32(0), bias, None, 0.0, lo, hi, signed_out)
    np.testing.assert_array_equal(out.cpu().numpy().view(ref.dtype), ref)
