"""The native per-call host path against the library it is bound to: a library
or a binding of another version, and one that lacks a function, are refused with
FlashAttentionExtensionError before any function is called."""
import ctypes

import pytest

from flash_attention_v100 import _lib


class _Other:
    """The loaded library with some functions replaced or missing."""

    def __init__(self, lib, without=(), **funcs):
        for n in _lib.EXPORTS:
            if n not in without:
                setattr(self, n, funcs.get(n, getattr(lib, n)))


def _version(v):
    return ctypes.CFUNCTYPE(ctypes.c_int32)(lambda: v)


def test_binds_to_its_own_library():
    mod = _lib._host()
    _lib._bind_host(mod, _lib.load())


def test_refuses_another_version():
    mod, lib = _lib._host(), _lib.load()
    other = _Other(lib, fa_abi_version=_version(_lib.ABI_VERSION + 1))
    with pytest.raises(_lib.FlashAttentionExtensionError, match="ABI version"):
        _lib._bind_host(mod, other)
    with pytest.raises(_lib.FlashAttentionExtensionError, match="ABI version"):
        _lib._check_library(other, "other.so")
    _lib._bind_host(mod, lib)


def test_refuses_other_structs(monkeypatch):
    class Longer(ctypes.Structure):
        _fields_ = _lib.FwdArgs._fields_ + [("more", ctypes.c_int64)]

    mod = _lib._host()
    monkeypatch.setattr(_lib, "FwdArgs", Longer)
    with pytest.raises(_lib.FlashAttentionExtensionError, match="bytes"):
        _lib._bind_host(mod, _lib.load())


def test_refuses_a_library_without_a_function():
    lib = _lib.load()
    _lib._check_library(lib, _lib.LIB_PATH)
    with pytest.raises(_lib.FlashAttentionExtensionError, match="fa_fwd_cols"):
        _lib._check_library(_Other(lib, without=("fa_fwd_cols",)), "older.so")


def test_refuses_null_addresses():
    mod = _lib._host()
    sizes = ctypes.sizeof(_lib.FwdArgs), ctypes.sizeof(_lib.BwdArgs)
    addr = ctypes.cast(_lib.load().fa_abi_version, ctypes.c_void_p).value
    with pytest.raises(ValueError):
        mod.bind(addr, *sizes, 0, 0, 0, 0, 0, 0)
    with pytest.raises(TypeError):
        mod.bind(addr, *sizes)
