"""Per-channel range of int32 accumulators where one workgroup has all rows of its channels and nothing is initialised: both
sides of the lines to the launches that initialise, on outputs that hold other values."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,depth", [(1, 5), (8, 300), (9, 3), (9, 8), (17, 2), (255, 17), (256, 33), (257, 15), (511, 36), (512, 64), (513, 4),
                                        (4095, 4096), (4096, 4100), (4097, 4096), (1, 1), (3, 1), (24576, 1), (24575, 1), (24580, 1),
                                        (1024, 4096), (1025, 4100), (4096, 4096), (4096, 4128), (1025, 6528), (1025, 6560), (1024, 16384), (1024, 16416), (1280, 13088), (1281, 13088), (4096, 8192), (4096, 8224), (536, 4652), (1024, 5120), (1024, 5124), (1024, 5092), (512, 16380), (512, 10236), (512, 10244), (256, 20476), (256, 20484), (256, 12287), (256, 12289), (128, 24575), (128, 24577),
                                        (512, 16388), (256, 16383), (256, 16385), (20, 65500), (20, 131200)])
@pytest.mark.parametrize("off", [0, 1])
def test_range(hip, dev, rows, depth, off):
    import torch
    rng = np.random.default_rng(rows + depth)
    x = rng.integers(-2 ** 31, 2 ** 31, rows * depth, dtype=np.int64).astype(np.int32)
    x[rng.integers(0, x.size)] = np.iinfo(np.int32).min
    x[rng.integers(0, x.size)] = np.iinfo(np.int32).max
    buf = torch.zeros(x.size + 4, dtype=torch.int32, device=dev)
    buf[off:off + x.size] = torch.from_numpy(x).to(dev)
    lo, hi = torch.full((depth + 2,), -9, dtype=torch.int32, device=dev), torch.full((depth + 2,), 9, dtype=torch.int32, device=dev)
    for _ in range(2):   # the second call finds the first one's results
        hip.minmax_i32_per_channel(buf[off:], rows, depth, lo[1:], hi[1:])
    torch.cuda.synchronize()
    got_lo, got_hi = lo.cpu().numpy(), hi.cpu().numpy()
    assert got_lo[0] == got_lo[-1] == -9 and got_hi[0] == got_hi[-1] == 9
    np.testing.assert_array_equal(got_lo[1:-1], x.reshape(rows, depth).min(0))
    np.testing.assert_array_equal(got_hi[1:-1], x.reshape(rows, depth).max(0))
