"""Host threads on one stream: calls of several kernels over the stream's scratch
buffer (a linear layer with split tiles, the QKV operand and its projection, split
attention) return what they return alone."""
from __future__ import annotations

import threading

import pytest
import torch

from braidinfer_amd import _lib
from braidinfer_amd.layers import CascadeAttention, RotaryEmbedding, linear, qwen3_attention_input
from oracle import torch_ref as R
from tests.helpers import gen, randn
from tests.test_gpu_cascade import build_case

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _linear(g):
    x, w = randn(g, 300, 2048).to(DEV), randn(g, 1024, 2048, std=0.03).to(DEV)
    assert _lib.workspace_size("bfa_linear_workspace_size", 300, 2048, 1024, _lib.LINEAR_PLAIN) > 0
    return lambda: linear(x, w)


def _qkv(g):
    x, ln, w = randn(g, 200, 1024).to(DEV), randn(g, 1024, mean=1.0).to(DEV), randn(g, 1024, 1024, std=0.03).to(DEV)
    qn, kn = randn(g, 128, mean=1.0, std=0.1).to(DEV), randn(g, 128, mean=1.0, std=0.1).to(DEV)
    pos, table = torch.arange(200, device=DEV), R.cos_sin_cache(128, 4096, 1e4).to(DEV)
    return lambda: torch.cat(qwen3_attention_input(x, ln, w, None, 4, 2, 1e-6, pos, table, qn, kn), -1)


def _attention(g):
    chunks, kv, total = build_case(int(torch.randint(1000, (1,), generator=g)), 8, 2, [200, 300, 100], [0, 0, 0],
                                   pages=60)
    att = CascadeAttention(8, 128, 128 ** -0.5, 2, 16, rotary_emb=RotaryEmbedding(128, 128, 4096, 1e6).to(DEV))
    q, qpos, kv = randn(g, 40, 8, 128).to(DEV), torch.arange(total - 40, total, device=DEV), kv.to(DEV)
    levels = att.create_cascade_levels(chunks)
    return lambda: att.forward(q, qpos, kv, levels, 0)


@pytest.mark.parametrize("make", [_linear, _qkv, _attention])
def test_threads_share_a_stream(make):
    calls = [make(gen(700 + i)) for i in range(4)]
    alone = [c() for c in calls]
    torch.cuda.synchronize()
    start, wrong = threading.Barrier(4), []

    def run(i):
        start.wait()
        outs = [calls[i]() for _ in range(30)]
        torch.cuda.synchronize()
        wrong.extend(i for o in outs if not torch.equal(o, alone[i]))

    threads = [threading.Thread(target=run, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not wrong and not any(t.is_alive() for t in threads)
