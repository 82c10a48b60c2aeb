"""Where the CPython module of the shortest calls is missing, the package makes
them through ctypes: the same statuses, messages and refusals; and building
without the interpreter's headers leaves the module out."""
import os
import sys
import sysconfig

import pytest

import honei_amd._lib as L
import test_py_bands
import test_py_calls
from honei_amd import build


@pytest.fixture
def through_ctypes(monkeypatch):
    monkeypatch.setitem(sys.modules, "honei_amd._calls", None)      # its import fails
    monkeypatch.delattr("honei_amd._calls", raising=False)
    monkeypatch.setattr(L, "_calls_module", None)
    assert L.calls().__name__ == "honei_amd._calls_ctypes"


@pytest.mark.parametrize("name,count", [("product_bmdv_q1", 6), ("defect_q1", 7), ("jacobi_q1", 7), ("ell_spmv", 5),
                                        ("ell_jacobi", 6)])
def test_refused_arguments(through_ctypes, name, count):
    test_py_calls.test_refused_arguments(name, count)


@pytest.mark.parametrize("dtype", ["float", "double"])
def test_status_and_message(through_ctypes, dtype):
    test_py_calls.test_status_and_message(dtype)


@pytest.mark.parametrize("name,before", [("product_bmdv_q1_double", ()), ("defect_q1_float", (48,))])
def test_list_of_bands(through_ctypes, name, before):
    test_py_bands.test_list_of_bands(name, before)


def test_band_pointers_follow_the_bands(through_ctypes, monkeypatch):
    test_py_bands.test_band_pointers_follow_the_bands(monkeypatch)


def test_module_carries_the_abi_tag(tmp_path):
    (tmp_path / "_calls.so").write_bytes(b"")
    made = build.build_calls(str(tmp_path))
    assert made == str(tmp_path / ("_calls" + sysconfig.get_config_var("EXT_SUFFIX"))) and os.path.getsize(made)
    assert not (tmp_path / "_calls.so").exists()
    assert L.calls().__name__ == "honei_amd._calls"


def test_no_headers(tmp_path, monkeypatch):
    monkeypatch.setattr(build.sysconfig, "get_paths", lambda: {"include": str(tmp_path / "none")})
    assert build.build_calls(str(tmp_path), verbose=False) is None and not os.listdir(tmp_path)


def test_no_compiler(tmp_path, monkeypatch):
    monkeypatch.setattr(build.shutil, "which", lambda name: None)
    assert build.build_calls(str(tmp_path), verbose=False) is None and not os.listdir(tmp_path)
