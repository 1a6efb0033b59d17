"""The 3 x 3 Conv2D kernel that keeps its input rows in LDS, at the sizes where its tiles, runs, rows and images end, against
int64 sums and the epilogue's separately rounded fp32 steps in numpy, bit for bit."""
import numpy as np
import pytest

from tests.test_gpu_stream import awkward_floats, finish
from tests.test_oracle_conv import ref_int_conv

pytestmark = pytest.mark.gpu
DIRECT = 17   # force_tile_shape: this kernel wherever it can take the call


def run(hip, dev, shape, O, pad, out_hw, post, signed_in, signed_out, seed, scalar_scale=False, kernel="direct", scale=None, bias=None):
    import torch
    rng = np.random.default_rng(seed)
    B, H, W, C = shape
    (pt, pl), (oh, ow) = pad, out_hw
    x = rng.integers(-128, 128, shape).astype(np.int8) if signed_in else rng.integers(0, 256, shape).astype(np.uint8)
    w = rng.integers(-127, 128, (3, 3, C, O)).astype(np.int8)
    trailing = max(oh + 2 - H - pt, 0), max(ow + 2 - W - pl, 0)
    acc = ref_int_conv(x, w, (1, 1), (1, 1), ((pt, trailing[0]), (pl, trailing[1])))[:, :oh, :ow].reshape(B * oh * ow, O)
    if scale is None:
        scale = ((rng.random(1 if scalar_scale else O) + 0.5) * 60.0 / (74.0 * 74.0 * np.sqrt(9 * C))).astype(np.float32)
    if bias is None:
        bias = (rng.standard_normal(O) * 20).astype(np.float32)
    inf = float("inf")
    lo, hi = {"none": (-inf, inf), "relu": (0.0, inf), "clip": (-3.5, 90.0)}[post]
    ep = hip.Epilogue()
    ep.n_scales, ep.n_eltwise = scale.size, 0 if post == "none" else 1
    if post != "none":
        ep.elt[0].alg, ep.elt[0].alpha, ep.elt[0].beta = (hip.ELT_RELU, 0.0, 0.0) if post == "relu" else (hip.ELT_CLIP, lo, hi)
    d = lambda a: torch.from_numpy(a).to(dev)
    packed = torch.empty(hip.qgemm_packed_bytes(9 * C, O), dtype=torch.int8, device=dev)
    colsum = torch.empty(O, dtype=torch.int32, device=dev)
    hip.qgemm_prepack_b(d(w.reshape(9 * C, O)), False, 9 * C, O, packed, colsum)
    n = B * oh * ow * O
    out = torch.full((n + 64,), 0x55, dtype=torch.uint8, device=dev)
    g = hip.ConvGeometry(B, H, W, C, 3, 3, oh, ow, 1, 1, 1, 1, pt, pl)
    hip.qconv2d(d(x), hip.QINT8 if signed_in else hip.QUINT8, g, packed, colsum, O, d(scale), d(bias), ep,
                hip.QINT8 if signed_out else hip.QUINT8, out)
    assert hip.last_kernel()[0] == kernel
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert (got[n:] == 0x55).all()
    ref = finish(acc, scale, bias, None, 0.0, lo, hi, signed_out)
    np.testing.assert_array_equal(got[:n].view(ref.dtype).reshape(ref.shape), ref)


def same(h, w):
    return (1, 1), (h, w)


# one position, a tile and its remainder, images smaller than a tile, runs that cross several images, rows longer than 256
# pieces and shorter, every count of 32 channels in and of wavefronts side by side
@pytest.mark.parametrize("shape,O", [((1, 1, 1, 32), 32), ((1, 4, 8, 64), 64), ((1, 3, 11, 64), 32), ((9, 2, 3, 128), 128),
                                     ((5, 7, 7, 96), 96), ((3, 1, 40, 32), 64), ((2, 40, 1, 128), 160), ((1, 3, 130, 96), 256),
                                     ((2, 5, 200, 64), 64), ((40, 25, 25, 64), 192)])
@pytest.mark.parametrize("signed_in", [False, True])
def test_sizes(hip, dev, shape, O, signed_in):
    hip.force_tile_shape(conv=DIRECT)
    run(hip, dev, shape, O, *same(shape[1], shape[2]), "relu", signed_in, not signed_in, sum(shape) + O)


@pytest.mark.parametrize("pad,out_hw", [((0, 0), (7, 9)), ((0, 1), (9, 10)), ((2, 2), (11, 13)), ((1, 0), (8, 7)), ((1, 1), (5, 6))])
def test_padding(hip, dev, pad, out_hw):
    """Windows that all lie inside, reach into one side, are padded by more than one, or leave rows and columns unused."""
    hip.force_tile_shape(conv=DIRECT)
    run(hip, dev, (3, 9, 11, 64), 64, pad, out_hw, "none", False, False, 5)


@pytest.mark.parametrize("post", ["none", "relu", "clip"])
@pytest.mark.parametrize("signed_out", [False, True])
@pytest.mark.parametrize("C", [32, 64, 96, 128])
def test_post_ops(hip, dev, post, signed_out, C):
    hip.force_tile_shape(conv=DIRECT)
    run(hip, dev, (2, 13, 14, C), 64, *same(13, 14), post, False, signed_out, C, scalar_scale=signed_out)


@pytest.mark.parametrize("post", ["none", "relu", "clip"])
@pytest.mark.parametrize("signed_out", [False, True])
@pytest.mark.parametrize("where", ["bias", "scale"])
def test_infinities_and_nan(hip, dev, post, signed_out, where):
    """Ties, infinities, NaN and random bit patterns as biases (scale 0) and as scales (sums of either sign and 0)."""
    O = 4096
    v = awkward_floats(O)
    hip.force_tile_shape(conv=DIRECT)
    run(hip, dev, (1, 5, 7, 32), O, *same(5, 7), post, where == "scale", signed_out, 3,
        **(dict(bias=v, scale=np.zeros(1, np.float32)) if where == "bias" else dict(scale=v, bias=np.zeros(O, np.float32))))


@pytest.mark.parametrize("shape,O,kernel", [((13, 56, 56, 64), 64, "direct"), ((13, 28, 28, 128), 128, "direct"), ((1, 190, 190, 64), 64, "direct"),
                                            ((4, 64, 64, 128), 160, "direct"), ((1, 300, 300, 64), 64, "tile"), ((1, 177, 177, 96), 96, "tile"),
                                            ((4, 288, 288, 32), 96, "short_k")])
def test_without_force(hip, dev, shape, O, kernel):
    """Several runs per CU, and the calls on either side of the lines to the other kernels."""
    run(hip, dev, shape, O, *same(shape[1], shape[2]), "relu", False, False, 9, kernel=kernel)
