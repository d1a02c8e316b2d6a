"""The vector-call entry points (csrc/pyentry.cpp): every function of the C ABI
that returns a number, the same results as through ctypes, and argument errors
raised before the call."""
from __future__ import annotations

import ctypes
import sysconfig

import pytest

from braidinfer_amd import _lib


def test_every_entry_is_bound():
    mod = _lib._load_entries()
    for name in _lib.exported_symbols():
        if name != "bfa_last_error":
            assert callable(getattr(mod, name)), name


@pytest.mark.parametrize("args", [(1, 1024, 4096, 128), (64, 4096, 6144, 128), (300, 512, 800, 80)])
def test_same_results_as_ctypes(args):
    name = "bfa_fused_rmsnorm_qkv_workspace_size"
    assert _lib.entry(name)(*args) == getattr(_lib.load(), name)(*args)


def test_errors_and_their_text():
    with pytest.raises(ValueError, match="bad dtype"):
        _lib.call("bfa_silu_and_mul", None, None, 9, 1, 8, 16, 8, None)
    fn = _lib.entry("bfa_get_tuning")
    with pytest.raises(TypeError):
        fn()
    with pytest.raises(TypeError):
        fn("0")
    with pytest.raises(OverflowError):
        fn(1 << 40)
    assert fn(0) == -1 and fn(ctypes.c_int(0)) == -1


@pytest.mark.parametrize("offset", [0, 2])
def test_what_ctypes_takes_for_a_pointer(offset):
    """The host's check that x is 16-byte aligned tells which address arrived (a
    call of no tokens ends there)."""
    memory = (ctypes.c_char * 64)()
    base = (ctypes.addressof(memory) + 15) // 16 * 16
    array = (ctypes.c_char * 8).from_address(base + offset)
    fn, raw = _lib.entry("bfa_linear"), _lib.load().bfa_linear

    def rc(f, x):
        return f(x, _lib.BF16, 0, 64, 64, base, 8, 64, None, 0, 0, _lib.BF16, None, 0, 8, _lib.F32, None, _lib.BF16,
                 8, None, 0, None)

    for x in (base + offset, ctypes.c_void_p(base + offset), array, ctypes.byref(array), ctypes.pointer(array),
              ctypes.cast(array, ctypes.POINTER(ctypes.c_int))):
        assert rc(fn, x) == rc(raw, x) == (-1 if offset else 0)

    class Held:
        _as_parameter_ = base + offset

    assert rc(fn, Held()) == rc(raw, Held()) == (-1 if offset else 0)
    for x in ("text", object(), 1.5):
        with pytest.raises(TypeError):
            rc(fn, x)


def test_the_module_is_this_interpreters_own(monkeypatch, tmp_path):
    """Its name carries the ABI tag, and without one for this interpreter the calls
    go through ctypes, to the same results."""
    assert _lib.ENTRY_PATH.name == "_bfa_entry" + sysconfig.get_config_var("EXT_SUFFIX")
    size = _lib.workspace_size("bfa_linear_workspace_size", 300, 2048, 1024, 0)
    monkeypatch.setattr(_lib, "_entries", None)
    monkeypatch.setattr(_lib, "ENTRY_PATH", tmp_path / "_bfa_entry.cpython-27.so")
    assert _lib.entry("bfa_linear") is _lib.load().bfa_linear
    assert _lib.workspace_size("bfa_linear_workspace_size", 300, 2048, 1024, 0) == size
    with pytest.raises(ValueError, match="bad dtype"):
        _lib.call("bfa_silu_and_mul", None, None, 9, 1, 8, 16, 8, None)


def test_a_build_without_python_headers(monkeypatch, tmp_path):
    """The library is the product: it builds where the module cannot."""
    from braidinfer_amd import build

    monkeypatch.setattr(build.sysconfig, "get_paths", lambda: {"include": str(tmp_path)})
    assert build._build_entry() is None
