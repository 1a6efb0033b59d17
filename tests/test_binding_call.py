"""The C extension behind the binding's wrappers: it takes the plain forms of arguments, raises what the library refuses, and
leaves every other form to the ctypes prototypes without having called anything.  No GPU: the library's checks end the calls."""
import ctypes as C
import re

import numpy as np
import pytest
import torch

ENTRIES = """quantize quantize_bf16 dequantize dequantize16 requantize requantize_per_channel minmax_i32_per_channel minmax_f32
qgemm qgemm_tile qgemv qgemm_sum qmatmul qmatmul_per_row qmatmul_device_range qmatmul_unpacked quantize_dynamic
quantize_dynamic_static quantize_dynamic_rows qbatch_matmul pad_nhwc8 qconv2d qconv2d_sum qdepthwise_conv2d transpose""".split()


def test_every_prototype_has_its_entry(hip):
    assert sorted(n[1:] for n, f in vars(hip).items() if n.startswith("_") and hasattr(f, "argtypes")) == sorted(ENTRIES)
    assert all(callable(getattr(hip._call, n)) for n in ENTRIES)


def test_plain_forms_are_taken(hip):
    t = torch.empty(4)
    for buf in (None, 0, 64, t, (1 << 47) + 5):
        assert hip._call.quantize(buf, buf, 0, hip.QUINT8, 1.5, 0, None) is True
    p = hip.matmul_params()
    assert hip._call.qmatmul(p, t, t, t, 0, 64, 16, t, t, 16, t, None, t, 0) is True
    ep, g = hip.Epilogue(), hip.ConvGeometry()
    with pytest.raises(hip.ItexHipError, match="implicit GEMM"):   # both structures arrive
        hip._call.qconv2d(t, hip.QUINT8, g, t, t, 16, t, t, ep, hip.QUINT8, t, 0)


def test_the_library_refuses(hip):
    for n, match in ((-1, "negative"), (1 << 33, "null")):
        with pytest.raises(hip.ItexHipError, match=match) as e:
            hip._call.quantize(None, None, n, hip.QUINT8, 1.0, 0.0, 0)
        assert e.value.code == hip.INVALID_ARGUMENT
    with pytest.raises(hip.ItexHipError):
        hip.transpose(64, 64, 1, (2, 2), (0, 0))


class Raises:
    def data_ptr(self):
        raise RuntimeError("no storage")


def test_other_forms_are_left_alone(hip):
    ok = [None, None, -1, hip.QUINT8, 1.0, 0.0, 0]    # -1: a call that got through would raise
    for at, bad in [(0, np.int64(64)), (0, "x"), (0, 1.0), (0, 1 << 70), (2, np.int64(-1)), (2, -1.0), (2, 1 << 64), (3, 1 << 33),
                    (3, True), (4, "x"), (4, np.float32(1)), (5, None), (6, object())]:
        args = list(ok)
        args[at] = bad
        assert hip._call.quantize(*args) is False, (at, bad)
    assert hip._call.quantize(*ok[:-1]) is False
    assert hip._call.qmatmul(hip.Epilogue(), *([0] * 13)) is False             # another structure
    assert hip._call.qmatmul(np.zeros(64, np.int32), *([0] * 13)) is False
    for dims, perm in [([2, 2], (0, 1)), ((2, 2), (0,)), ((2, 2.0), (0, 1)), ((1,) * 9, tuple(range(9)))]:
        assert hip._call.transpose(0, 0, 1, dims, perm, 0) is False
    with pytest.raises(RuntimeError, match="no storage"):
        hip._call.quantize(Raises(), *ok[1:])


def test_arguments_are_those_of_the_wrapper(hip):
    """Each wrapper hands the extension what it hands the prototype, in the prototype's order."""
    import inspect
    for name in ENTRIES:
        if name in ("transpose", "qgemm", "qgemm_tile", "qgemv"):
            continue   # (the last three below)
        src = " ".join(inspect.getsource(getattr(hip, name)).split())
        fast = re.search(r"_call\.%s\((.*?)\): _check" % name, src).group(1)
        slow = re.search(r"_check\(_%s\((.*)\)\)$" % name, src).group(1)
        plain = re.sub(r"\b(_addr|C\.byref)\(|\bint\((?!bool)", "(", slow)
        while re.search(r"(?<![\w])\((\w+)\)", plain):
            plain = re.sub(r"(?<![\w])\((\w+)\)", r"\1", plain)
        assert fast == plain, name
    for name in ("qgemm", "qgemm_tile", "qgemv"):
        wrapper = getattr(hip, name)
        src = " ".join(inspect.getsource(wrapper).split())
        params = ", ".join(inspect.signature(wrapper).parameters)
        assert re.search(r"_call\.%s\((.*?)\): _gemm_call" % name, src).group(1) == params
        assert re.search(r"_gemm_call\((.*)\)$", src).group(1) == "_%s, %s" % (name, params)
