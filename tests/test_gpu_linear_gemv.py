"""The linear layers' one-launch weight stream (linear_gemv.hip) against the
oracle: every token-block count at its edges, K steps short of, at and past a
batch of every wave, widths that leave the last workgroup partly empty, and the
general dtypes."""
from __future__ import annotations

import pytest
import torch

from braidinfer_amd.kernels import attention_output
from braidinfer_amd.layers import gate_up_silu_and_mul, linear, linear_add_residual
from oracle import torch_ref as R
from tests.helpers import assert_close, gen, randn

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("t", [1, 4, 5, 16, 17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("k,n", [(64, 24), (704, 200), (2112, 37)])
def test_streams(tuning, t, k, n):
    """1, 11 and 33 K steps for 4 waves: no full batch, one and a remainder, and
    several."""
    tuning("LINEAR_GEMV", 1)
    g = gen(5000 + t + k)
    x, w, r, b = randn(g, t, k), randn(g, n, k, std=0.03), randn(g, t, n, std=2.0), randn(g, n, std=0.5)
    assert_close(linear(x.to(DEV), w.to(DEV), b.to(DEV)), R.linear(x, w, b), what=f"bias t={t} k={k}")
    # one bf16 ulp of the projection: its rounding precedes the addition
    slack = 2.0 ** -7 * R.linear(x, w).float().abs()
    assert_close(linear_add_residual(x.to(DEV), w.to(DEV), r.to(DEV)), R.linear_add_residual(x, w, r),
                 what=f"residual t={t} k={k}", slack=slack, max_slack_frac=2e-3)
    w2 = randn(g, 2 * n, k, std=0.05)
    exp = R.gate_up_silu_and_mul(x, w2)
    # silu and up are rounded before their product: two more ulps at most
    assert_close(gate_up_silu_and_mul(x.to(DEV), w2.to(DEV)), exp, what=f"gate_up t={t} k={k}",
                 slack=2.0 ** -6 * exp.float().abs(), max_slack_frac=1e-3)


@pytest.mark.parametrize("t,k,n,inter", [(1, 8192, 512, 64), (16, 9216, 300, 48), (3, 4096, 64, 4096),
                                         (2, 2048, 64, 4100)])
def test_planned_forms(t, k, n, inter):
    """The forms that the planner picks: 8 waves from 128 K steps, one weight block
    for gate_up of up to 4 tokens from 32 MiB."""
    g = gen(5100 + t)
    x, w = randn(g, t, k), randn(g, n, k, std=0.03)
    assert_close(linear(x.to(DEV), w.to(DEV)), R.linear(x, w), what=f"plain t={t} k={k}")
    w2 = randn(g, 2 * inter, k, std=0.03)
    exp = R.gate_up_silu_and_mul(x, w2)
    assert_close(gate_up_silu_and_mul(x.to(DEV), w2.to(DEV)), exp, what=f"gate_up t={t} k={k}",
                 slack=2.0 ** -6 * exp.float().abs(), max_slack_frac=1e-3)


def test_general_dtypes_and_strided_rows():
    g = gen(5200)
    t, k, n = 7, 256, 50
    x, w, r = randn(g, t, k), randn(g, n, k, std=0.03), randn(g, t, n)
    xh, wh = x.half(), w.half()
    assert_close(linear(xh.to(DEV), wh.to(DEV)), R.linear(xh, wh), what="fp16")
    y = attention_output(x.to(DEV), w.to(DEV), r.to(DEV))
    assert_close(y, (x.float() @ w.float().t() + r.float()).half().to(x.dtype), what="attention output")
    wide = torch.zeros(t, k + 8, dtype=x.dtype, device=DEV)
    wide[:, :k] = x.to(DEV)
    assert torch.equal(linear(wide[:, :k], w.to(DEV)), linear(x.to(DEV), w.to(DEV)))
