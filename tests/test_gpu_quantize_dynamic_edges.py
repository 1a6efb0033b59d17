"""QuantizeV2 against the tensor's own range where the second pass divides its work: one step, several steps, remainders."""
import numpy as np
import pytest

from oracle import pyoracle as orc

pytestmark = pytest.mark.gpu

STEP = 256 * 4 * 4   # elements a workgroup quantizes per step


@pytest.mark.parametrize("n", [200003, STEP * 2048 - 4, STEP * 2048 + 1, STEP * 2048 * 2 + STEP + 7])
@pytest.mark.parametrize("qint8", [True, False])
def test_whole_tensor(hip, dev, n, qint8):
    import torch
    x = np.random.default_rng(n).standard_normal(n).astype(np.float32)
    x[n - 1], x[n // 2] = -7.5, 6.25     # the extremes, one of them in the last, partial group
    T, mode = (orc.QINT8, orc.SCALED) if qint8 else (orc.QUINT8, orc.MIN_FIRST)
    state = torch.zeros(hip.DYNAMIC_STATE_FLOATS, dtype=torch.float32, device=dev)
    q = torch.full((n + 16,), 0x55, dtype=torch.uint8, device=dev)
    hip.quantize_dynamic(torch.from_numpy(x).to(dev), q, n, T, mode, 0.01, state)
    torch.cuda.synchronize()
    st, ref, omn, omx = orc.quantize_v2(x, float(x.min()), float(x.max()), T, mode, ensure_minimum_range=0.01)
    assert st == orc.OK
    got = q.cpu().numpy()
    np.testing.assert_array_equal(got[:n].view(ref.dtype), ref)
    assert (got[n:] == 0x55).all()
    np.testing.assert_array_equal(state[2:4].cpu().numpy(), np.array([omn[0], omx[0]], np.float32))


# a thread holds 1, 2 or 4 groups of 4 elements: rows at those limits, beyond them, and of lengths that are read one by one
@pytest.mark.parametrize("rows,cols", [(3, 4), (2, 4092), (1, 4096), (2, 4100), (3, 8192), (2, 8196), (16, 14336), (1, 16384),
                                       (2, 16388), (2, 40004), (3, 1), (2, 4097)])
@pytest.mark.parametrize("qint8", [True, False])
def test_per_row(hip, dev, rows, cols, qint8):
    import torch
    rng = np.random.default_rng(rows * cols)
    x = rng.standard_normal((rows, cols)).astype(np.float32)
    x[:, cols // 2], x[:, cols - 1] = 6.25 + np.arange(rows), -7.5 - np.arange(rows)   # the extremes, one at the row's end
    T, mode = (orc.QINT8, orc.SCALED) if qint8 else (orc.QUINT8, orc.MIN_FIRST)
    q = torch.full((rows * cols + 16,), 0x55, dtype=torch.uint8, device=dev)
    lo, hi = (torch.empty(rows, dtype=torch.float32, device=dev) for _ in range(2))
    hip.quantize_dynamic_rows(torch.from_numpy(x).to(dev), q, rows, cols, T, mode, 0.01, lo, hi)
    torch.cuda.synchronize()
    st, ref, omn, omx = orc.quantize_v2(x, x.min(1), x.max(1), T, mode, axis=0, ensure_minimum_range=0.01)
    assert st == orc.OK
    got = q.cpu().numpy()
    np.testing.assert_array_equal(got[:rows * cols].view(ref.dtype).reshape(rows, cols), ref)
    assert (got[rows * cols:] == 0x55).all()
    np.testing.assert_array_equal(lo.cpu().numpy(), omn)
    np.testing.assert_array_equal(hi.cpu().numpy(), omx)
