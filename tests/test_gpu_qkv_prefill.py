"""The QKV projection above 64 tokens for head_dim 64 and 128 (qkv_prefill.hip):
every tile size one token short of and past its rows, whole and split over K,
both epilogue families, against the oracle; and the paged append through output
rows and caches that do not take 16-byte stores."""
from __future__ import annotations

import pytest
import torch

import braidinfer_amd
from braidinfer_amd import _lib
from braidinfer_amd.kernels import FusedRMSNormQKVMixedPrecision, PagedKVAppend
from braidinfer_amd.layers import llama_attention_input, qwen3_attention_input
from oracle import torch_ref as R
from tests.helpers import assert_close, bits, randn
from tests.test_gpu_fused_append import call, check, make_case, run_case, to_dev
from tests.test_gpu_qkv import make

pytestmark = pytest.mark.gpu
DEV = "cuda"

TILE_TOKENS = (256, 192, 160, 128, 256, 192, 128, 64)


@pytest.mark.parametrize("tile", range(8))
@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("d,hq,hkv", [(64, 7, 1), (128, 3, 1)])
def test_tiles(tuning, tile, splits, d, hq, hkv):
    """9 heads of 64 and 5 of 128: the last column tile is partly empty."""
    tuning("GEMM_TILE", tile)
    tuning("GEMM_SPLITS", splits)
    for edge in (-1, 1):
        t, h = max(2 * TILE_TOKENS[tile] + edge, 65), 256
        g, x, ln, w, b = make(500 + tile + d, t, h, hq, hkv, d)
        pos = torch.randint(-50, 4096, (t,), generator=g)
        cache = R.cos_sin_cache(d, 4096, 1e4)
        got = llama_attention_input(x.to(DEV), ln.to(DEV), w.to(DEV), hq, hkv, 1e-5, pos.to(DEV), cache.to(DEV))
        for y, exp, name in zip(got, R.llama_attention_input(x, ln, w, hq, hkv, 1e-5, pos, cache), "qkv"):
            assert_close(y, exp, what=f"llama {name} tile={tile} t={t}")
        # q/k norm weights near 1: RoPE's inputs stay of order 1, where a flip of
        # the bf16 rounding before it is inside the plain tolerance
        qn, kn = randn(g, d, mean=1.0, std=0.1), randn(g, d, mean=1.0, std=0.1)
        got = qwen3_attention_input(x.to(DEV), ln.to(DEV), w.to(DEV), b.to(DEV), hq, hkv, 1e-6, pos.to(DEV),
                                    cache.to(DEV), qn.to(DEV), kn.to(DEV))
        ref = R.qwen3_attention_input(x, ln, w, b, hq, hkv, 1e-6, pos, cache, qn, kn)
        for y, exp, name in zip(got, ref, "qkv"):
            assert_close(y, exp, what=f"qwen3 {name} tile={tile} t={t}", slack=2.0 ** -7 * exp.float().abs() + 2e-2)
    braidinfer_amd.check_device_status()


@pytest.mark.parametrize("d,hq,hkv,split_tiles", [(64, 27, 2, 32), (128, 11, 2, 14)])
def test_whole_and_split_tiles_in_one_call(tuning, d, hq, hkv, split_tiles):
    """18 row tiles of 64 tokens, the last one ragged, by 16 (31 heads of 64: half
    of the last one empty) or 15 column tiles of 128: 256 whole ones, the others
    split in three; with and without q/k norm, and with the append."""
    tuning("GEMM_TILE", 7)
    tuning("GEMM_SPLITS", 3)
    t, h = 1100, 256
    n = (hq + 2 * hkv) * d
    size = _lib.workspace_size("bfa_fused_rmsnorm_qkv_workspace_size", t, h, n, d)
    assert size == t * h * 2 + split_tiles * 3 * 64 * 128 * 4
    g, x, ln, w, b = make(570 + d, t, h, hq, hkv, d)
    pos = torch.randint(-50, 4096, (t,), generator=g)
    cache = R.cos_sin_cache(d, 4096, 1e4)
    got = llama_attention_input(x.to(DEV), ln.to(DEV), w.to(DEV), hq, hkv, 1e-5, pos.to(DEV), cache.to(DEV))
    for y, exp, name in zip(got, R.llama_attention_input(x, ln, w, hq, hkv, 1e-5, pos, cache), "qkv"):
        assert_close(y, exp, what=f"llama {name} d={d}")
    qn, kn = randn(g, d, mean=1.0, std=0.1), randn(g, d, mean=1.0, std=0.1)
    got = qwen3_attention_input(x.to(DEV), ln.to(DEV), w.to(DEV), b.to(DEV), hq, hkv, 1e-6, pos.to(DEV),
                                cache.to(DEV), qn.to(DEV), kn.to(DEV))
    ref = R.qwen3_attention_input(x, ln, w, b, hq, hkv, 1e-6, pos, cache, qn, kn)
    for y, exp, name in zip(got, ref, "qkv"):  # the slack of test_tiles
        assert_close(y, exp, what=f"qwen3 {name} d={d}", slack=2.0 ** -7 * exp.float().abs() + 2e-2)
    for qwen in (False, True):
        check(make_case(580 + d + qwen, t, hidden=h, hq=hq, hkv=hkv, d=d, qwen=qwen), f"append d={d} qwen={qwen}")
    braidinfer_amd.check_device_status()


@pytest.mark.parametrize("d", [64, 128])
def test_fp16(d):
    t, h, hq, hkv = 130, 256, 4, 2
    g, x, ln, w, b = make(540 + d, t, h, hq, hkv, d, dtype=torch.float16)
    pos = torch.randint(0, 4096, (t,), generator=g)
    cache = R.cos_sin_cache(d, 4096, 1e4)
    got = llama_attention_input(x.to(DEV), ln.to(DEV), w.to(DEV), hq, hkv, 1e-5, pos.to(DEV), cache.to(DEV))
    for y, exp, name in zip(got, R.llama_attention_input(x, ln, w, hq, hkv, 1e-5, pos, cache), "qkv"):
        assert_close(y, exp, what=f"fp16 llama {name} d={d}")
    got = FusedRMSNormQKVMixedPrecision.forward(x.to(DEV), ln.to(DEV), w.to(DEV), b.to(DEV), hq, hkv, eps=1e-6)
    for y, exp, name in zip(got, R.split_qkv(R.qkv_mixed_precision(x, ln, w, b, 1e-6), hq, hkv), "qkv"):
        assert_close(y, exp, what=f"fp16 mixed {name} d={d}")


@pytest.mark.parametrize("qwen", [False, True])
@pytest.mark.parametrize("splits", [1, 2])
def test_append_rows_of_8_bytes(tuning, qwen, splits):
    """A cache whose strides are multiples of 4 elements only, and an output
    whose row stride is: the same bits as through the wide stores."""
    tuning("GEMM_SPLITS", splits)
    c = make_case(560 + qwen, 150, hidden=256, hq=4, hkv=2, d=64, qwen=qwen)
    fused, plain, got, exp, skipped = run_case(c)
    assert not skipped and torch.equal(bits(got), bits(exp)) and torch.equal(bits(fused), bits(plain))
    to_dev(c)
    pages, _, hkv, ps, d = c["cache"].shape
    wide = torch.zeros(pages, 2, hkv, ps, d + 4, dtype=torch.bfloat16, device=DEV)
    view = wide[..., :d]
    view.copy_(c["cache"])
    n = plain.shape[1]
    out = torch.zeros(150, n + 4, dtype=torch.bfloat16, device=DEV)[:, :n]
    call(c, PagedKVAppend(view, c["kv_indices"].to(DEV), c["cache_pos"].to(DEV), c["ps"]), out=out)
    assert torch.equal(bits(view.cpu().contiguous()), bits(exp))
    assert torch.equal(bits(out.cpu().contiguous()), bits(plain))
