"""Two copies of the binding in one process (it has several import names, and ITEXHIP_LIB chooses a library per copy): each calls
its own library, raises its own error and takes its own structures.  No GPU: the library's checks end the calls."""
import importlib.util
import os
import shutil

import pytest


def load_copy(hip, name):
    spec = importlib.util.spec_from_file_location(name, hip.__file__)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


@pytest.mark.parametrize("other_library", [False, True])
def test_copies_do_not_share_state(hip, monkeypatch, tmp_path, other_library):
    first = load_copy(hip, "first")
    if other_library:
        lib = shutil.copy(first.LIB_PATH, tmp_path / "libitexhip.so")
        monkeypatch.setenv("ITEXHIP_LIB", str(lib))
    second = load_copy(hip, "second")
    assert os.path.samefile(first.LIB_PATH, second.LIB_PATH) != other_library
    for copy, other in ((first, second), (second, first)):
        with pytest.raises(copy.ItexHipError, match="negative"):
            copy.quantize(None, None, -1, copy.QUINT8, 1.0)
        rest = [0, 0, 0, 0, 64, 16, 0, 0, 16, 0, 0, 0, 0]
        assert copy._call.qmatmul(copy.matmul_params(), *rest) is True
        assert copy._call.qmatmul(other.matmul_params(), *rest) is False
    if other_library:   # the message is the library's own
        for copy, n in ((first, -1), (second, 1)):
            with pytest.raises(copy.ItexHipError):
                copy.quantize(None, None, n, copy.QUINT8, 1.0)
        assert b"negative" in first.raw().itexhip_last_error() and b"null" in second.raw().itexhip_last_error()


def test_without_the_extension(hip, monkeypatch):
    """No extension for this Python: the same calls through the ctypes prototypes."""
    import importlib.machinery
    monkeypatch.setattr(importlib.machinery, "EXTENSION_SUFFIXES", [".no-such-abi.so"])
    plain = load_copy(hip, "plain")
    assert plain._call.quantize(None, None, 0, plain.QUINT8, 1.0, 0.0, 0) is False
    plain.quantize(None, None, 0, plain.QUINT8, 1.0)
    plain.qmatmul(plain.matmul_params(), 0, 0, 0, 0, 64, 16, 0, 0, 16, 0, 0)
    plain.transpose(64, 64, 1, (0, 2), (1, 0))
    with pytest.raises(plain.ItexHipError, match="negative"):
        plain.quantize(None, None, -1, plain.QUINT8, 1.0)


def test_build_without_python_headers(hip, monkeypatch, tmp_path):
    import sysconfig
    import __graft_entry__ as entry
    build = entry._load_build_module()
    monkeypatch.setattr(build, "LIB", str(tmp_path))
    built = build.build_call(verbose=False)
    assert os.path.basename(built).startswith("itexhip_call.") and os.path.basename(built) != "itexhip_call.so"
    monkeypatch.setattr(sysconfig, "get_paths", lambda: {"include": str(tmp_path)})
    assert build.build_call(verbose=False) is None
