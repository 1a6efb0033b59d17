"""The kernel for a short K, many rows and an 8-bit result, at the sizes where its tiles and pieces end, against int64 products
and the epilogue's separately rounded fp32 steps in numpy, bit for bit.  Convolutions: against the patch-matrix path."""
import numpy as np
import pytest

from tests.test_gpu_conv import check_implicit_conv

pytestmark = pytest.mark.gpu
ANY_SIZE = 16   # force_tile_shape: this kernel whatever the size of the call


def reference(x, w, scale, bias, addend, sum_scale, lo, hi, signed_out):
    f = np.float32
    v = (x.astype(np.int64) @ w.astype(np.int64)).astype(f) * scale
    v = v + bias
    if addend is not None:
        v = v + f(sum_scale) * addend.astype(f)
    v = np.minimum(np.maximum(v, f(lo)), f(hi))
    v = np.clip(v, f(-128 if signed_out else 0), f(127 if signed_out else 255))
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


@pytest.mark.parametrize("M,K,N", [(131073, 64, 64), (70001, 48, 96), (20003, 32, 320)])
def test_several_tiles_per_wavefront(hip, dev, M, K, N):
    """Sizes that take this kernel by themselves, a row more than whole tiles."""
    run(hip, dev, M, K, N, "relu", None, False, False, 1)
    run(hip, dev, M, K, N, "relu", hip.QUINT8, False, False, 2)


@pytest.mark.parametrize("shape,wshape,strides,dil,lead", [
    ((2, 9, 10, 16), (3, 3, 16, 48), (1, 1), (1, 1), None), ((1, 8, 7, 32), (3, 2, 32, 64), (2, 1), (1, 2), None),
    ((2, 6, 6, 48), (2, 2, 48, 112), (1, 1), (1, 1), None), ((3, 13, 11, 16), (5, 5, 16, 80), (2, 2), (1, 1), (3, 1)),
    ((1, 12, 12, 128), (1, 1, 128, 160), (2, 2), (1, 1), None), ((1, 3, 3, 16), (3, 3, 16, 16), (1, 1), (1, 1), None),
    ((4, 33, 31, 32), (3, 3, 32, 64), (1, 1), (1, 1), (0, 0))])
@pytest.mark.parametrize("signed_in", [False, True])
def test_convolutions(hip, dev, shape, wshape, strides, dil, lead, signed_in):
    hip.force_tile_shape(conv=ANY_SIZE)
    check_implicit_conv(hip, dev, shape, wshape, strides, dil, lead, signed_in, np.random.default_rng(sum(shape) + signed_in))
