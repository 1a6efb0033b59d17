"""The quantized Transpose walked in either tensor's order, one and two units per thread."""
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


# runs of one unit (16 bytes of int8, one int32) and of a few: rows that share lines, destinations a power of two apart, remainders of a workgroup, bytes on both sides of 2^20
@pytest.mark.parametrize("shape,perm", [
    ((64, 7, 16), (1, 0, 2)), ((1000, 32, 16), (1, 0, 2)), ((32, 1000, 16), (1, 0, 2)), ((256, 128, 16), (1, 0, 2)),
    ((101, 67, 16), (1, 0, 2)), ((50, 9, 80, 16), (2, 1, 0, 3)), ((100, 20, 32), (1, 0, 2)), ((20, 100, 48), (1, 0, 2)),
    ((33, 16, 4), (1, 0, 2)), ((200, 3, 70, 4), (2, 0, 1, 3)), ((3, 1, 64, 16), (2, 1, 0, 3)), ((16, 16), (1, 0)),
    ((1024, 1024), (1, 0)), ((1025, 1024), (1, 0)), ((70, 16, 1), (1, 0, 2))])
@pytest.mark.parametrize("dtype", [np.int8, np.int32])
def test_short_runs(hip, dev, shape, perm, dtype):
    x = np.random.default_rng(sum(shape)).integers(-128, 128, shape).astype(dtype)
    np.testing.assert_array_equal(run_transpose(hip, dev, x, perm), np.transpose(x, perm))


# tensors that an L2 does not hold, in the input's order: single bytes, ints and 16-byte units, runs, more than 4 dimensions;
# and one whose destinations lie a multiple of 4 KB apart, which stays in the output's
@pytest.mark.parametrize("shape,perm,dtype", [
    ((267, 133, 24, 64), (3, 2, 0, 1), np.int8), ((36, 50, 246, 16), (3, 0, 1, 2), np.int32), ((146, 408, 38, 16), (2, 0, 1, 3), np.int8),
    ((128, 128, 12, 64), (0, 2, 1, 3), np.int8), ((10, 83, 21, 12, 38), (4, 1, 2, 0, 3), np.int32), ((3, 64, 768, 256), (3, 1, 2, 0), np.int8)])
def test_large(hip, dev, shape, perm, dtype):
    x = np.random.default_rng(sum(shape)).integers(-128, 128, shape, dtype=np.int8).astype(dtype)
    np.testing.assert_array_equal(run_transpose(hip, dev, x, perm), np.transpose(x, perm))
