"""Element counts that are no whole groups of 4, whose last elements the vector kernels finish themselves, and requantization with
depths that are no multiple of 4: bit for bit against the fp32 steps in numpy, with the elements behind the result untouched."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32


def saturate(v, signed):
    lo, hi = (-128, 127) if signed else (0, 255)
    return np.rint(np.clip(v, F(lo), F(hi))).astype(np.int8 if signed else np.uint8)


def result(torch, dev, n, dtype):
    """n elements and a guard behind them."""
    size = np.dtype(dtype).itemsize
    out = torch.full((n * size + 64,), 0x5a, dtype=torch.uint8, device=dev)

    def get():
        b = out.cpu().numpy()
        assert (b[n * size:] == 0x5a).all()
        return b[:n * size].view(dtype)
    return out, get


@pytest.mark.parametrize("n", [1, 3, 4, 5, 6, 7, 1023, 2049, 4098, 16385, 131071, 131073, 524290])
@pytest.mark.parametrize("signed", [False, True])
def test_quantize_and_dequantize(hip, dev, n, signed):
    import torch
    rng = np.random.default_rng(n)
    x = (rng.standard_normal(n) * 40).astype(F)
    t, dt = (hip.QINT8, np.int8) if signed else (hip.QUINT8, np.uint8)
    dx = torch.from_numpy(x).to(dev)
    scale, addend = F(1.7), F(3.25)
    out, get = result(torch, dev, n, dt)
    hip.quantize(dx, out, n, t, float(scale), float(addend))
    q = saturate(x * scale + addend, signed)
    np.testing.assert_array_equal(get(), q)
    y, get = result(torch, dev, n, F)
    hip.dequantize(torch.from_numpy(q).to(dev), y, n, t, 0.3, 7)
    np.testing.assert_array_equal(get(), (q.astype(F) - F(7)) * F(0.3))
    # the range of a tensor whose largest or smallest element is among the last ones
    for last in (1000.0, -1000.0):
        x[-1] = last
        out, get = result(torch, dev, n, dt)
        state = torch.zeros(hip.DYNAMIC_STATE_FLOATS, dtype=torch.float32, device=dev)
        hip.quantize_dynamic(torch.from_numpy(x).to(dev), out, n, t, hip.SCALED, 0.01, state)
        s = state[:6].cpu().numpy()
        assert s[0] == x.min() and s[1] == x.max()
        np.testing.assert_array_equal(get(), saturate(x * s[4] + s[5], signed))


@pytest.mark.parametrize("n", [5, 1030, 131071])
def test_nan_among_the_last_elements(hip, dev, n):
    """It has no part in the range; a tensor of nothing else has the range that one of whole groups of 4 has."""
    import torch
    for m, fill in ((n, 2.0), (n, np.nan), (n // 4 * 4, np.nan)):
        x = np.full(m, fill, F)
        x[-1] = np.nan
        state = torch.zeros(hip.DYNAMIC_STATE_FLOATS, dtype=torch.float32, device=dev)
        hip.quantize_dynamic(torch.from_numpy(x).to(dev), torch.empty(m, dtype=torch.int8, device=dev), m, hip.QINT8, hip.SCALED, 0.01, state)
        lo, hi = state[:2].cpu().tolist()
        assert (lo, hi) == ((2.0, 2.0) if fill == 2.0 else (float("inf"), -float("inf")))


# either side of the count from which on groups of any depth go together; scales at any address
@pytest.mark.parametrize("rows,depth", [(7, 1), (5, 3), (333, 197), ((1 << 21) - 1, 1), ((1 << 21) + 1, 1), ((1 << 21) + 3, 1), ((1 << 20) + 1, 2),
                                        (700001, 3), (419431, 5), (299999, 7), (10647, 197), (2097, 1001), (512, 4098), (600, 4096), (3, 700001)])
@pytest.mark.parametrize("signed", [False, True])
def test_requantize(hip, dev, rows, depth, signed):
    import torch
    rng = np.random.default_rng(rows + depth)
    n = rows * depth
    x = rng.integers(-60000, 60000, (rows, depth)).astype(np.int32)
    x.flat[0], x.flat[-1] = np.iinfo(np.int32).max, np.iinfo(np.int32).min
    scales = (rng.random(depth).astype(F) + F(0.5)) * F(0.002)
    dx = torch.from_numpy(x).to(dev)
    t, dt = (hip.QINT8, np.int8) if signed else (hip.QUINT8, np.uint8)
    for off in (0, 1):
        ds = torch.zeros(depth + off, dtype=torch.float32, device=dev)
        ds[off:] = torch.from_numpy(scales).to(dev)
        out, get = result(torch, dev, n, dt)
        hip.requantize_per_channel(dx, out, rows, depth, t, ds[off:])
        np.testing.assert_array_equal(get().reshape(rows, depth), saturate(x.astype(F) * scales, signed))
    out, get = result(torch, dev, n, dt)
    hip.requantize(dx, out, n, t, 0.002)
    np.testing.assert_array_equal(get().reshape(rows, depth), saturate(x.astype(F) * F(0.002), signed))
