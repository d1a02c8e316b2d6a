"""The linear layers' GEMM above 64 tokens (linear_gemm.hip): every tile size at
the edges of its tiles, split over K and whole, against the oracle; the general
dtype and masked forms; and a caller without a workspace."""
from __future__ import annotations

import pytest
import torch

from braidinfer_amd import _lib
from braidinfer_amd.kernels import attention_output
from braidinfer_amd.layers import gate_up_silu_and_mul, linear, linear_add_residual
from oracle import torch_ref as R
from tests.helpers import assert_close, gen, randn

pytestmark = pytest.mark.gpu
DEV = "cuda"

# tokens per tile of each planner tile
TILE_TOKENS = (256, 192, 160, 128, 256, 192, 128, 64)


@pytest.mark.parametrize("tile", range(8))
@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("edge", [-1, 1])
def test_tiles(tuning, tile, splits, edge):
    """One token short of and one past a whole row of tiles; 4 K stages over 3
    splits (1, 1 and 2 stages, fewer than the ring holds)."""
    tuning("GEMM_TILE", tile)
    tuning("GEMM_SPLITS", splits)
    t, k, n = max(2 * TILE_TOKENS[tile] + edge, 65), 256, 392
    g = gen(4000 + tile)
    x, w, r = randn(g, t, k), randn(g, n, k, std=0.03), randn(g, t, n, std=2.0)
    # one bf16 ulp of the projection, as for the other linear paths: its rounding
    # precedes the addition
    slack = 2.0 ** -7 * R.linear(x, w).float().abs()
    assert_close(linear_add_residual(x.to(DEV), w.to(DEV), r.to(DEV)), R.linear_add_residual(x, w, r),
                 what=f"residual tile={tile}", slack=slack, max_slack_frac=1e-3)
    w2 = randn(g, 2 * n, k, std=0.05)
    exp = R.gate_up_silu_and_mul(x, w2)
    # silu and up are rounded before their product: two more ulps at most
    assert_close(gate_up_silu_and_mul(x.to(DEV), w2.to(DEV)), exp, what=f"gate_up tile={tile}",
                 slack=2.0 ** -6 * exp.float().abs(), max_slack_frac=1e-4)


@pytest.mark.parametrize("splits", [1, 2])
def test_general_forms(tuning, splits):
    """n not a multiple of 8, a bias in fp32, fp16 operands, and the fp32 -> fp16
    rounding of the attention output."""
    tuning("GEMM_SPLITS", splits)
    g = gen(4100)
    t, k, n = 77, 192, 203
    x, w, b = randn(g, t, k), randn(g, n, k, std=0.03), torch.randn(n, generator=g)
    assert_close(linear(x.to(DEV), w.to(DEV), b.to(DEV)), R.linear(x, w, b), what="odd n, fp32 bias")
    xh, wh = x.half(), w.half()
    assert_close(linear(xh.to(DEV), wh.to(DEV)), R.linear(xh, wh), what="fp16")
    r = randn(g, t, n)
    y = attention_output(x.to(DEV), w.to(DEV), r.to(DEV))
    assert_close(y, (x.float() @ w.float().t() + r.float()).half().to(x.dtype), what="attention output")


@pytest.mark.parametrize("tile", range(8))
@pytest.mark.parametrize("splits", [1, 3])
def test_general_forms_on_every_tile(tuning, tile, splits):
    """The general epilogue, one token past a tile: rows that do not take 16-byte
    stores (n odd, and a multiple of 4) with a bias or an fp32 residual, SwiGLU of
    an odd width, and the attention output's fp16 sum on rows that do."""
    tuning("GEMM_TILE", tile)
    tuning("GEMM_SPLITS", splits)
    g = gen(4300 + tile)
    t, k = TILE_TOKENS[tile] + 1, 192
    x = randn(g, t, k)
    for n in (299, 300):
        w, b = randn(g, n, k, std=0.03), torch.randn(n, generator=g)
        assert_close(linear(x.to(DEV), w.to(DEV), b.to(DEV)), R.linear(x, w, b), what=f"bias n={n} tile={tile}")
        r = torch.randn(t, n, generator=g)
        assert_close(linear_add_residual(x.to(DEV), w.to(DEV), r.to(DEV)),
                     (R.linear(x, w).float() + r).to(x.dtype), what=f"fp32 residual n={n} tile={tile}",
                     # one bf16 ulp of the projection: its rounding precedes the addition
                     slack=2.0 ** -7 * R.linear(x, w).float().abs(), max_slack_frac=1e-3)
    w2 = randn(g, 2 * 203, k, std=0.05)
    exp = R.gate_up_silu_and_mul(x, w2)
    # silu and up are rounded before their product: two more ulps at most
    assert_close(gate_up_silu_and_mul(x.to(DEV), w2.to(DEV)), exp, what=f"gate_up tile={tile}",
                 slack=2.0 ** -6 * exp.float().abs(), max_slack_frac=1e-4)
    w, r = randn(g, 328, k, std=0.03), randn(g, t, 328)
    assert_close(attention_output(x.to(DEV), w.to(DEV), r.to(DEV)),
                 (x.float() @ w.float().t() + r.float()).half().to(x.dtype), what=f"attention output tile={tile}")


@pytest.mark.parametrize("n", [2000, 2003])
def test_whole_and_split_tiles_in_one_call(tuning, n):
    """18 x 16 tiles of 64 x 128: 256 whole ones, 32 split in three, the last row and
    column tiles ragged; n = 2003 through the general epilogue."""
    tuning("GEMM_TILE", 7)
    tuning("GEMM_SPLITS", 3)
    g = gen(4400 + n)
    t, k = 1100, 256
    assert _lib.workspace_size("bfa_linear_workspace_size", t, k, n, _lib.LINEAR_PLAIN) == 32 * 3 * 64 * 128 * 4
    x, w, r = randn(g, t, k), randn(g, n, k, std=0.03), randn(g, t, n, std=2.0)
    slack = 2.0 ** -7 * R.linear(x, w).float().abs()  # one bf16 ulp of the projection, as in test_tiles
    assert_close(linear_add_residual(x.to(DEV), w.to(DEV), r.to(DEV)), R.linear_add_residual(x, w, r),
                 what=f"residual n={n}", slack=slack, max_slack_frac=1e-3)
    inter = n // 2
    assert _lib.workspace_size("bfa_linear_workspace_size", t, k, inter, 1) == 32 * 3 * 64 * 128 * 4
    w2 = randn(g, 2 * inter, k, std=0.05)
    exp = R.gate_up_silu_and_mul(x, w2)
    assert_close(gate_up_silu_and_mul(x.to(DEV), w2.to(DEV)), exp, what=f"gate_up n={inter}",
                 slack=2.0 ** -6 * exp.float().abs(), max_slack_frac=1e-4)


def test_without_workspace():
    """A caller that brings no workspace gets the unsplit plan: the same result
    up to the order of the fp32 sums, so at most one bf16 rounding apart."""
    g = gen(4200)
    t, k, n = 96, 2048, 256
    x, w = randn(g, t, k).to(DEV), randn(g, n, k, std=0.03).to(DEV)
    assert _lib.workspace_size("bfa_linear_workspace_size", t, k, n, _lib.LINEAR_PLAIN) > 0
    out = torch.empty(t, n, dtype=x.dtype, device=DEV)
    _lib.call("bfa_linear", _lib.ptr(x), _lib.BF16, t, k, k, _lib.ptr(w), n, k, None, 0, _lib.LINEAR_PLAIN,
              _lib.BF16, None, 0, n, _lib.F32, _lib.ptr(out), _lib.BF16, n, None, 0, _lib.stream_of(x.device))
    exp = R.linear(x.cpu(), w.cpu())
    assert_close(out, exp, what="no workspace")
    assert_close(linear(x, w), exp, what="split")
