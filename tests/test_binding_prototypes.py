"""The prototyped entry points of the ctypes binding: their signatures are the header's, and they take and refuse the same
arguments as the calls that wrap every argument themselves.  No GPU: empty tensors end in the library's checks."""
import ctypes as C
import os
import re

import numpy as np
import pytest
import torch

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "itexhip.h")


def c_type(declaration):
    if "*" in declaration:
        return C.c_void_p
    return {"int": C.c_int, "int32_t": C.c_int, "int64_t": C.c_int64, "float": C.c_float}[declaration.split()[0]]


def test_signatures_match_the_header(hip):
    text = open(HEADER).read()
    bound = {n: f for n, f in vars(hip).items() if n.startswith("_") and hasattr(f, "argtypes")}
    assert len(bound) == 25
    for name, fn in bound.items():
        args = re.search(r"int itexhip%s\(([^;]*)\);" % name, text).group(1)
        assert tuple(fn.argtypes) == tuple(c_type(a.strip()) for a in args.split(",")), name


@pytest.mark.parametrize("buf", [None, 0, np.int64(64), torch.empty(4), (1 << 47) + 5])
def test_addresses(hip, buf):
    want = hip._ptr(buf).value
    got = hip._addr(buf)
    assert (got or None) == want
    hip.quantize(buf, buf, 0, hip.QUINT8, np.float32(1.5), 0, 0)
    hip.dequantize(buf, buf, np.int64(0), hip.QUINT8, 1, np.int32(3), None)


def test_refusals(hip):
    for bad in ("x", object()):
        with pytest.raises((TypeError, ValueError)):
            hip.quantize(bad, None, 0, hip.QUINT8, 1.0)
    with pytest.raises((TypeError, C.ArgumentError)):
        hip.quantize(None, None, 0, hip.QUINT8, "x")
    with pytest.raises(C.ArgumentError):
        hip.quantize(None, None, 0, 12.0, 1.0)
    with pytest.raises(hip.ItexHipError, match="negative"):
        hip.quantize(None, None, -1, hip.QUINT8, 1.0)
    with pytest.raises(hip.ItexHipError, match="null"):
        hip.quantize(None, None, 1 << 33, hip.QUINT8, 1.0)   # 64 bits arrive
