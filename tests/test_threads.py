"""Scratch buffers, between host threads and where memory ends.  A buffer is kept
per (device, stream) and a call queues several kernels over it with the GIL
released, so two threads on one stream must not interleave theirs; the partial
sums of a linear layer above 64 tokens are optional.  On the CPU, with entry points
that only record; the GPU counterpart is tests/test_gpu_threads.py."""
from __future__ import annotations

import threading
import time
from types import SimpleNamespace

import pytest
import torch

from braidinfer_amd import _lib
from braidinfer_amd.kernels import _qkv
from braidinfer_amd.layers import CascadeAttention, linear


class Recorder:
    """Stands in for the entry points: notes which scratch pointers are in use,
    holds each for a while, and keeps the sizes it was given."""

    def __init__(self, ptr_arg):
        self.ptr_arg, self.busy, self.shared, self.sizes = ptr_arg, set(), 0, []
        self.lock = threading.Lock()

    def __call__(self, *args):
        ptr = args[self.ptr_arg]
        with self.lock:
            self.shared += ptr in self.busy
            self.busy.add(ptr)
            self.sizes.append(args[self.ptr_arg + 1])
        time.sleep(0.02)
        with self.lock:
            self.busy.discard(ptr)
        return 0


@pytest.fixture
def host(monkeypatch):
    """The drivers on CPU tensors, every thread on stream 7 of device 0."""
    dev = torch.device("cpu", 0)
    monkeypatch.setattr(_lib, "require_device", lambda *t: dev)
    monkeypatch.setattr(_lib, "stream_of", lambda d: 7)
    monkeypatch.setattr(_lib, "status_word", lambda d: torch.zeros(1, dtype=torch.int32))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(_lib, "_workspaces", {})

    def entries(size, **fns):
        ns = SimpleNamespace(**fns)
        for name in ("bfa_linear", "bfa_cascade_attention", "bfa_fused_rmsnorm_qkv"):
            setattr(ns, name + "_workspace_size", lambda *a: size)
        monkeypatch.setattr(_lib, "_entries", ns)
        monkeypatch.setattr(_qkv, "_fused_fn", fns.get("bfa_fused_rmsnorm_qkv"))

    return entries


def _in_threads(fn, n=4):
    errors = []

    def run():
        try:
            fn()
        except BaseException as e:  # reported in the main thread
            errors.append(e)

    threads = [threading.Thread(target=run) for _ in range(n)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(30)
    assert not errors and not any(t.is_alive() for t in threads), errors


def _linear():
    x = torch.zeros(300, 64, dtype=torch.bfloat16)
    return lambda: linear(x, x[:64])


def _qkv_call():
    x = torch.zeros(300, 64, dtype=torch.bfloat16)
    return lambda: _qkv.fused_rmsnorm_qkv(x, x[0], x[:192], 1, 1, 1e-6, mixed_rounding=True,
                                          qkv_dtype=torch.bfloat16, out_dtype=torch.bfloat16)


def _cascade():
    att = CascadeAttention(2, 64, 0.125, 1, 16)
    kv = torch.zeros(4, 2, 1, 16, 64, dtype=torch.bfloat16)
    q = torch.zeros(3, 2, 64, dtype=torch.bfloat16)
    return lambda: att.forward(q, torch.arange(3), kv, [], 0)


@pytest.mark.parametrize("name,make,ptr_arg", [("bfa_linear", _linear, 19), ("bfa_fused_rmsnorm_qkv", _qkv_call, 30),
                                               ("bfa_cascade_attention", _cascade, 31)])
def test_one_call_at_a_time_on_a_buffer(host, name, make, ptr_arg):
    rec = Recorder(ptr_arg)
    host(4096, **{name: rec})
    _in_threads(make())
    assert rec.sizes == [4096] * 4 and rec.shared == 0


def test_the_lock_is_given_back_after_an_error(host):
    def fail(*args):
        return -1

    host(4096, bfa_linear=fail)
    call = _linear()

    def run():
        with pytest.raises(ValueError):
            call()

    _in_threads(run)
    rec = Recorder(19)
    host(8192, bfa_linear=rec)
    call()
    assert rec.sizes[0] >= 8192


@pytest.mark.parametrize("tokens,served", [(300, True), (64, False)])
def test_linear_without_memory_for_its_partial_sums(host, monkeypatch, tokens, served):
    def full(self, nbytes):
        raise torch.cuda.OutOfMemoryError("no memory")

    rec = Recorder(19)
    host(4096, bfa_linear=rec)
    monkeypatch.setattr(_lib.Scratch, "reserve", full)
    x = torch.zeros(300, 64, dtype=torch.bfloat16)
    if served:
        linear(x[:tokens], x[:64])
        assert rec.sizes == [0]
    else:
        with pytest.raises(torch.cuda.OutOfMemoryError):
            linear(x[:tokens], x[:64])
