"""Zero-padded copy to 4 channels (itexhip_pad_nhwc8): 16-byte loads at any address, moved inside the tensor at its two ends,
pixels cleared at the row's ends."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# tensors of 15, 16 and a few more bytes, rows of fewer than 4 pixels, leading padding of 0 .. 9 pixels, trailing padding
@pytest.mark.parametrize("c", [1, 2, 3, 4])
@pytest.mark.parametrize("n,h,w,lead,out_hw", [(1, 1, 5, (0, 0), (1, 8)), (1, 1, 4, (0, 3), (1, 8)), (1, 2, 8, (1, 1), (4, 12)),
                                               (1, 1, 16, (0, 0), (1, 16)), (3, 5, 1, (2, 2), (8, 4)), (2, 7, 3, (0, 9), (7, 16)),
                                               (2, 9, 33, (3, 2), (15, 40)), (5, 31, 30, (2, 3), (35, 36))])
@pytest.mark.parametrize("shift", [0, 1])
def test_pad_to_four_channels(hip, dev, c, n, h, w, lead, out_hw, shift):
    import torch
    x = np.random.default_rng(c + w).integers(1, 256, (n, h, w, c)).astype(np.uint8)
    ref = np.zeros((n, *out_hw, 4), np.uint8)
    ref[:, lead[0]:lead[0] + h, lead[1]:lead[1] + w, :c] = x
    buf = torch.full((x.size + shift,), 0xaa, dtype=torch.uint8, device=dev)
    buf[shift:].copy_(torch.from_numpy(x.reshape(-1)))
    out = torch.full(ref.shape, 0x55, dtype=torch.uint8, device=dev)
    hip.pad_nhwc8(buf.data_ptr() + shift, n, h, w, c, lead[0], lead[1], out_hw[0], out_hw[1], 4, out)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(out.cpu().numpy(), ref)
