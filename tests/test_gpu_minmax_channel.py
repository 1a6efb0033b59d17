"""Per-channel range of int32 accumulators and dynamic quantization at the sizes where their work is divided."""
import numpy as np
import pytest

from oracle import pyoracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,depth,off", [
    (1, 4, 0), (3, 8, 0), (2049, 4, 0), (4096, 252, 0), (4097, 256, 0), (700, 260, 0), (33, 4100, 0), (129, 64, 1),
    (8193, 12, 0), (5000, 1, 1), (4099, 255, 0), (300, 257, 0), (70000, 197, 0), (513, 1000, 1),
    (8, 4, 0), (9, 4, 0), (5, 260, 0), (8, 1003, 0), (9, 1003, 1), (257, 4, 0), (264, 4, 0), (7, 1, 1)])
def test_channel_ranges(hip, dev, rows, depth, off):
    """Groups of 4 channels and single ones, fewer and more than a workgroup's channels, unaligned tensors, chunk edges."""
    import torch
    rng = np.random.default_rng(rows + depth)
    x = rng.integers(-2 ** 31, 2 ** 31, (rows, depth), dtype=np.int64).astype(np.int32)
    raw = torch.zeros(x.size + 4, dtype=torch.int32, device=dev)
    x_d = raw[off:off + x.size]
    x_d.copy_(torch.from_numpy(x.ravel()))
    mn, mx = (torch.zeros(depth, dtype=torch.int32, device=dev) for _ in range(2))
    hip.minmax_i32_per_channel(x_d, rows, depth, mn, mx)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(mn.cpu().numpy(), x.min(0))
    np.testing.assert_array_equal(mx.cpu().numpy(), x.max(0))
