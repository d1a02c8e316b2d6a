"""The vector-call entry points (csrc/pyentry.cpp): every function of the C ABI
that returns a number, the same results as through ctypes, and argument errors
raised before the call."""
from __future__ import annotations

import ctypes

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
