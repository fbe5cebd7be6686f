"""CPU checks that a library or an extension built from earlier sources is told
apart: the library with a message that says to rebuild it, the extension by
leaving every call to the Python paths."""

import ctypes
import importlib.util
import types

import pytest

from hyquant_amd import _lib
from hyquant_amd import decode_d_stage as dd


@pytest.mark.parametrize("version,match", [(_lib.ABI_VERSION, "hyq_append_rows.*rebuild"), (_lib.ABI_VERSION - 1, "ABI.*rebuild")])
def test_older_library_is_refused_by_name(monkeypatch, version, match):
    old = types.SimpleNamespace(hyq_abi_version=lambda: version)
    for name in _lib.EXPORTS:
        if name not in ("hyq_append_rows", "hyq_abi_version"):
            setattr(old, name, types.SimpleNamespace())
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(ctypes, "CDLL", lambda path: old)
    monkeypatch.setattr(_lib.os.path, "exists", lambda path: True)
    with pytest.raises(RuntimeError, match=match):
        _lib.lib()


def test_older_extension_is_left_alone(monkeypatch):
    P = _lib.DecodeParams

    def set_entry(hybrid):
        raise AssertionError("bound")

    old = types.SimpleNamespace(layout=lambda: (ctypes.sizeof(P), P.seg_n.offset, P.dtype_flags.offset), set_entry=set_entry)
    spec = types.SimpleNamespace(loader=types.SimpleNamespace(exec_module=lambda m: None))
    monkeypatch.setattr(dd, "_FX", None)
    monkeypatch.setattr("os.path.exists", lambda path: True)
    monkeypatch.setattr(importlib.util, "spec_from_file_location", lambda *a: spec)
    monkeypatch.setattr(importlib.util, "module_from_spec", lambda s: old)
    assert dd._load_fast_ext() is False
