"""The quantized Transpose where the walk follows the input's order instead of the output's."""
import numpy as np
import pytest

from tests.test_gpu_shape_ops import run_transpose

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,perm", [
    ((3, 197, 12, 64), (0, 2, 1, 3)), ((3, 12, 197, 64), (0, 2, 1, 3)),   # head split and merge
    ((2, 7, 3, 5, 16), (0, 3, 1, 2, 4)), ((5, 4, 3, 2, 16), (3, 1, 0, 2, 4)),
    ((2, 3, 2, 3, 2, 3, 20), (5, 3, 1, 0, 2, 4, 6)), ((9, 11, 3), (1, 0, 2)), ((11, 9, 513), (1, 0, 2))])
@pytest.mark.parametrize("dtype", [np.int8, np.int32])
def test_walk_order(hip, dev, shape, perm, dtype):
    x = np.random.default_rng(sum(shape)).integers(-128, 128, shape).astype(dtype)
    np.testing.assert_array_equal(run_transpose(hip, dev, x, perm), np.transpose(x, perm))
