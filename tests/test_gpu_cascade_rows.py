"""The flat form of cascade attention at the edges of its row blocks, with one and
two 16-row blocks per wave (CASCADE_FLAT 1 at these sizes, and 2), against the
oracle and bit for bit against each other; and what its softmax does with scores that keep growing
along the keys, with scores of 2^34, and with a negative or zero scale, against
64 bits."""
from __future__ import annotations

import pytest
import torch

from braidinfer_amd.layers import CascadeAttention, RotaryEmbedding
from tests.helpers import assert_close, gen, randn
from tests.test_gpu_cascade import _check_case, build_case

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("tokens,hq,hkv,d", [(128, 16, 8, 128), (129, 16, 8, 128), (161, 4, 1, 128),
                                             (128, 32, 4, 64), (129, 32, 4, 64), (145, 16, 2, 64)])
@pytest.mark.parametrize("causal,knorm", [(True, False), (False, True)])
@pytest.mark.parametrize("flat", [1, 2])
def test_row_blocks(tuning, tokens, hq, hkv, d, causal, knorm, flat):
    tuning("CASCADE_FLAT", flat)
    _check_case(f"rows {tokens} {hq} {hkv} {d}", tokens, hq, hkv, [48, 130, 64, tokens], [0, 77, -5, 0], causal,
                knorm, d=d)


@pytest.mark.parametrize("tokens,hq,hkv,d", [(25, 4, 1, 128), (97, 4, 2, 128), (161, 4, 1, 128), (145, 16, 2, 64),
                                             (600, 16, 8, 128)])
@pytest.mark.parametrize("causal", [True, False])
def test_one_and_two_blocks_agree(tuning, tokens, hq, hkv, d, causal):
    """Which wave takes a row changes none of its sums; the planner's own choice
    (600 tokens: two blocks) is one of the two."""
    chunks, kv, total = build_case(97, hq, hkv, [700, 130, tokens], [0, 0, 0], pages=120, d=d)
    q = randn(gen(98), tokens, hq, d, std=2.0)
    qpos = torch.arange(total - tokens, total)
    att = CascadeAttention(hq, d, d ** -0.5, hkv, 16, rotary_emb=RotaryEmbedding(d, d, 4096, 1e6).to(DEV))
    levels = att.create_cascade_levels(chunks)
    outs = []
    for flat in (1, 2, None) if tokens * hq > 96 * hkv else (1, 2):
        tuning("CASCADE_FLAT", flat)
        outs.append(att.forward(q.to(DEV), qpos.to(DEV), kv.to(DEV), levels, 0, causal_mask=causal).cpu())
    assert all(torch.equal(o, outs[0]) for o in outs)


@pytest.mark.parametrize("tokens", [100, 300])
@pytest.mark.parametrize("wg", [8, 64])
@pytest.mark.parametrize("flat", [1, 2])
def test_growing_scores_and_sign(tuning, tokens, wg, flat):
    """Keys that grow along the walk move the running maximum in every tile (by
    less and by more than the step that rescales); P is rounded to bf16 as
    everywhere, so the plain tolerance holds.  (-q, -scale) is (q, scale)."""
    tuning("CASCADE_FLAT", flat)
    tuning("CASCADE_FLAT_WG", wg)
    hq, hkv, d, ps = 8, 4, 128, 16
    chunks, kv, total = build_case(91, hq, hkv, [400, 300, 200], [0, 0, 0], pages=90)
    for i, c in enumerate(chunks):
        c.cached_position_start -= 1000
        c.global_position_start -= 1000
        for j, p in enumerate(c.page_table):
            kv[p, 0] *= 0.05 + 0.1 * (i + j / 20.0)
    rope = RotaryEmbedding(d, d, 4096, 1e6).to(DEV)
    q = randn(gen(92), tokens, hq, d, std=3.0)
    qpos = torch.arange(total - tokens, total)
    outs = []
    for s in (1.0, -1.0):
        att = CascadeAttention(hq, d, s * d ** -0.5, hkv, ps, rotary_emb=rope)
        levels = att.create_cascade_levels(chunks)
        outs.append(att.forward((q * s).to(DEV), qpos.to(DEV), kv.to(DEV), levels, 0).cpu())
    assert torch.equal(outs[0], outs[1])
    ks, vs = [], []
    for c in chunks:
        k, v = (kv[c.page_table, i].double().transpose(1, 2).reshape(-1, hkv, d)[: c.kv_length] for i in (0, 1))
        ks.append(k)
        vs.append(v)
    k, v = torch.cat(ks).repeat_interleave(hq // hkv, 1), torch.cat(vs).repeat_interleave(hq // hkv, 1)
    sc = torch.einsum("thd,khd->htk", q.double(), k) * d ** -0.5
    hide = torch.arange(total)[None, :] > qpos[:, None]
    exp = torch.einsum("htk,khd->thd", torch.softmax(sc.masked_fill(hide, float("-inf")), -1), v)
    assert_close(outs[0].reshape(tokens, hq, d), exp, what=f"growing scores tokens={tokens} wg={wg}")


@pytest.mark.parametrize("tokens,flat", [(100, 1), (300, 2)])
@pytest.mark.parametrize("causal", [True, False])
def test_zero_scale(tuning, tokens, flat, causal):
    """Every score is 0: the mean of the visible values, with partly filled pages
    and a causal edge inside a tile."""
    tuning("CASCADE_FLAT", 1)
    hq, hkv, d, ps = 8, 4, 128, 16
    chunks, kv, total = build_case(93, hq, hkv, [130, 77, tokens], [0, 0, 0], pages=60)
    q = randn(gen(94), tokens, hq, d)
    qpos = torch.arange(total - tokens, total)
    att = CascadeAttention(hq, d, 0.0, hkv, ps, rotary_emb=RotaryEmbedding(d, d, 4096, 1e6).to(DEV))
    out = att.forward(q.to(DEV), qpos.to(DEV), kv.to(DEV), att.create_cascade_levels(chunks), 0, causal_mask=causal)
    v = torch.cat([kv[c.page_table, 1].double().transpose(1, 2).reshape(-1, hkv, d)[: c.kv_length] for c in chunks])
    seen = torch.arange(1, total + 1).view(-1, 1, 1)
    mean = (v.cumsum(0) / seen)[qpos] if causal else v.mean(0, keepdim=True).expand(tokens, -1, -1)
    assert_close(out.reshape(tokens, hq, d), mean.repeat_interleave(hq // hkv, 1), what=f"scale 0 causal={causal}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tokens,flat", [(100, 1), (300, 2)])
def test_scores_of_any_size(tuning, tokens, flat, dtype):
    """Scores up to 2^34 (2^28 in fp16), further apart than any exponential: each
    query returns the value of its largest visible key."""
    tuning("CASCADE_FLAT", flat)
    hq, hkv, d, ps = 8, 4, 128, 16
    chunks, kv, total = build_case(95, hq, hkv, [200, 90, tokens], [0, 0, 0], pages=60)
    kv = kv.to(dtype)
    g = gen(96)
    sign = (torch.randint(0, 2, (d,), generator=g) * 2 - 1).to(dtype)
    # keys of 128 sizes 1 to 2 apart by 2^-7, shuffled along the walk
    size = 1 + torch.randint(0, 128, (total,), generator=g) / 128.0
    big = 2.0 ** (15 if dtype == torch.bfloat16 else 12)
    pos = 0
    for c in chunks:
        for j in range(c.kv_length):
            kv[c.page_table[j // ps], 0, :, j % ps] = big * size[pos] * sign
            pos += 1
    q = (big * sign).expand(tokens, hq, d).contiguous()
    qpos = torch.arange(total - tokens, total)
    att = CascadeAttention(hq, d, d ** -0.5, hkv, ps, rotary_emb=RotaryEmbedding(d, d, 4096, 1e6).to(DEV))
    out = att.forward(q.to(DEV), qpos.to(DEV), kv.to(DEV), att.create_cascade_levels(chunks), 0).cpu()
    v = torch.cat([kv[c.page_table, 1].double().transpose(1, 2).reshape(-1, hkv, d)[: c.kv_length] for c in chunks])
    exp = torch.empty(tokens, hkv, d, dtype=torch.float64)
    for t in range(tokens):
        seen = size[: int(qpos[t]) + 1]
        exp[t] = v[: seen.numel()][seen == seen.max()].mean(0)  # equal keys share the weight
    assert_close(out.reshape(tokens, hq, d), exp.repeat_interleave(hq // hkv, 1), what=f"scores of any size {dtype}")


def test_positions_at_the_end_of_32_bits(tuning):
    """Keys from -2^31 on (the flat form keeps key positions in 32 bits): a query
    below all of them sees none, one at -2^31 + 5 sees six."""
    tuning("CASCADE_FLAT", 1)
    hq, hkv, d, ps, tokens = 8, 4, 128, 16, 100
    chunks, kv, total = build_case(99, hq, hkv, [130, 70], [0, 0], pages=30)
    att = CascadeAttention(hq, d, 0.0, hkv, ps, rotary_emb=RotaryEmbedding(d, d, 4096, 1e6).to(DEV))
    levels = att.create_cascade_levels(chunks)
    q = randn(gen(100), tokens, hq, d).to(DEV)
    qpos = torch.full((tokens,), -2 ** 31 + 5, device=DEV)
    qpos[:50] = -2 ** 31 - 7
    att._plan(levels, att._chunk_meta(levels), q.device)[1].add_(-2 ** 31)  # the plan's key positions, as kept
    out = att.forward(q, qpos, kv.to(DEV), levels, 0).reshape(tokens, hq, d)
    CascadeAttention._plans.clear()  # (the changed plan among them)
    v = kv[chunks[0].page_table[0], 1, :, :6].double().mean(1).repeat_interleave(hq // hkv, 0)
    assert not out[:50].any()
    assert_close(out[50:], v.expand(50, -1, -1), what="the first six keys")
