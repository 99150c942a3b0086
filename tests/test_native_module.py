"""Which module the functions of qgemm_amd go through: the one built for this Python, with every entry they call; where there is
none they say so once and take ctypes."""
import importlib.machinery
import types
import warnings

import pytest

from qgemm_amd import lib, ops


@pytest.fixture(autouse=True)
def _fresh(monkeypatch):
    monkeypatch.delenv("QGEMM_LIBRARY", raising=False)
    monkeypatch.setattr(ops, "_native_module", None)
    monkeypatch.setattr(lib, "_torch_ext", None)


def _raise(e):
    raise e


@pytest.mark.parametrize("load", [lambda: types.ModuleType("qgemm_python"), lambda: _raise(ImportError("undefined symbol"))],
                         ids=["an older module", "a module that does not load"])
def test_a_module_that_cannot_be_used(load, monkeypatch):
    monkeypatch.setattr(ops, "load_torch_extension", load)
    with pytest.warns(RuntimeWarning, match="ctypes"):
        assert ops._native() is False
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert ops._native() is False


def test_the_built_module_is_used():
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert ops._native() is lib.load_torch_extension()


def test_modules_of_other_pythons_are_left_alone(tmp_path, monkeypatch):
    lib.load_library()
    monkeypatch.setattr(lib, "_HERE", str(tmp_path))
    (tmp_path / "qgemm_python.cpython-27-other.so").write_bytes(b"not for this Python")
    with pytest.raises(ImportError, match="is missing"):
        lib.load_torch_extension()
    loaded = []
    monkeypatch.setattr(importlib.util, "spec_from_file_location", lambda name, path: loaded.append(path) or _raise(ImportError("seen")))
    for ending in reversed(importlib.machinery.EXTENSION_SUFFIXES):        # (the last one written is the one this Python prefers)
        (tmp_path / ("qgemm_python" + ending)).write_bytes(b"")
        with pytest.raises(ImportError, match="seen"):
            lib.load_torch_extension()
        assert loaded[-1].endswith("qgemm_python" + ending)
