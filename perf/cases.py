"""Performance cases of the per-layer kernels: what one decoder layer of an engine
that uses this package calls, at the sizes of its three model shapes.

Five kinds of case, each one pass through the package's public entry points:

* ``qkv``   the attention input (RMSNorm + QKV projection [+ q/k norm] + RoPE, with
  the paged KV append when ``append``), ``llama_attention_input`` or
  ``qwen3_attention_input``;
* ``mlp``   add+RMSNorm, gate_up + SiLU*mul, down projection + residual;
* ``attn``  cascade attention over a paged cache whose chunks were moved, the new
  tokens' own keys last;
* ``rows``  the memory-bound row operations: embedding gather, add+RMSNorm, RoPE of
  a packed q/k, paged append, SiLU*mul;
* ``layer`` one whole decoder layer made of these, as a HIP graph when ``graph``
  (how a serving loop runs decode steps).

Weights and activations are drawn on the GPU from the seed: N(0, 1) activations,
N(0, 0.02)-scaled weights, N(1, 0.1) norm weights.
"""
from __future__ import annotations

import functools
import math
from types import SimpleNamespace

import torch

from braidinfer_amd.kernels import PagedKVAppend, append_to_paged_kv_cache_custom
from braidinfer_amd.layers import (CascadeAttention, RMSNorm, RotaryEmbedding, VocabParallelEmbedding,
                                   gate_up_silu_and_mul, linear_add_residual, llama_attention_input,
                                   qwen3_attention_input, silu_and_mul)

PAGE = 16
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
# hidden, q heads, kv heads, head_dim, intermediate, vocabulary, rope theta, table length, eps, q/k norm
MODELS = {
    "tinyllama": SimpleNamespace(h=2048, hq=32, hkv=4, d=64, inter=5632, vocab=32000, theta=1e4, maxpos=4096,
                                 eps=1e-5, qk_norm=False),
    "qwen3": SimpleNamespace(h=1024, hq=16, hkv=8, d=128, inter=3072, vocab=151936, theta=1e6, maxpos=40960,
                             eps=1e-6, qk_norm=True),
    "llama3": SimpleNamespace(h=4096, hq=32, hkv=8, d=128, inter=14336, vocab=128256, theta=5e5, maxpos=8192,
                              eps=1e-5, qk_norm=False),
}


def listed():
    return [
        # a handful of interactive users on a small fp16 checkpoint: latency of one call
        dict(name="qkv_tinyllama_t5_fp16", kind="qkv", model="tinyllama", dtype="fp16", tokens=5, append=False),
        # one user's decode step, the whole layer replayed as the graph a serving loop keeps
        dict(name="layer_qwen3_t1_graph", kind="layer", model="qwen3", dtype="bf16", tokens=1, context=3000, graph=True),
        # a full decode batch: one new token of 64 sequences, k and v appended to their pages
        dict(name="qkv_llama3_t64_append", kind="qkv", model="llama3", dtype="bf16", tokens=64, append=True),
        # an ordinary prompt of odd length
        dict(name="qkv_qwen3_t700_append", kind="qkv", model="qwen3", dtype="bf16", tokens=700, append=True),
        # a long prefill
        dict(name="qkv_llama3_t8192", kind="qkv", model="llama3", dtype="bf16", tokens=8192, append=False),
        # the MLP of a partly filled decode batch
        dict(name="mlp_llama3_t40", kind="mlp", model="llama3", dtype="bf16", tokens=40),
        # the MLP of a chunked prefill / a short prompt
        dict(name="mlp_llama3_t300", kind="mlp", model="llama3", dtype="bf16", tokens=300),
        # the MLP of a long prefill, the largest piece of work of a layer
        dict(name="mlp_llama3_t6000", kind="mlp", model="llama3", dtype="bf16", tokens=6000),
        # one token decoded over a few thousand cached keys
        dict(name="attn_qwen3_t1", kind="attn", model="qwen3", dtype="bf16", tokens=1, context=4000),
        # a short question over cached context chunks
        dict(name="attn_tinyllama_t24", kind="attn", model="tinyllama", dtype="bf16", tokens=24, context=2000),
        # a prompt chunk over a long cached context
        dict(name="attn_qwen3_t1000", kind="attn", model="qwen3", dtype="bf16", tokens=1000, context=8000),
        # the row operations of a long prefill
        dict(name="rows_llama3_t8192", kind="rows", model="llama3", dtype="bf16", tokens=8192),
    ]


def _spread(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["qkv", "qkv", "mlp", "mlp", "attn", "attn", "rows", "layer"])
    case = dict(kind=kind, model=rng.choice(sorted(MODELS)), dtype=rng.choice(["bf16", "bf16", "bf16", "fp16"]))
    if kind == "qkv":
        case.update(tokens=_spread(rng, 1, 8192), append=rng.random() < 0.5)
    elif kind == "mlp":
        case.update(tokens=_spread(rng, 1, 6000))
    elif kind == "attn":
        case.update(tokens=_spread(rng, 1, 1000), context=_spread(rng, 200, 8000))
        if case["model"] == "tinyllama":
            case["context"] = min(case["context"], 3000)
    elif kind == "rows":
        case.update(tokens=_spread(rng, 1, 8192))
    else:
        case.update(tokens=_spread(rng, 1, 512), context=_spread(rng, 200, 3000), graph=False)
        case["graph"] = case["tokens"] <= 16
    return case


# ------------------------------------------------------------------- inputs


class _Draw:
    """Seeded inputs on the GPU."""

    def __init__(self, seed, dtype):
        self.dev = torch.device("cuda", torch.cuda.current_device())
        self.g = torch.Generator(device=self.dev).manual_seed(seed)
        self.dtype = dtype

    def randn(self, *shape, std=1.0, mean=0.0):
        return torch.randn(*shape, generator=self.g, device=self.dev).mul_(std).add_(mean).to(self.dtype)

    def ints(self, lo, hi, n):
        return torch.randint(lo, hi, (n,), generator=self.g, device=self.dev)

    def perm(self, n):
        return torch.randperm(n, generator=self.g, device=self.dev)


@functools.lru_cache(maxsize=None)
def _rope(model):
    """The model's rotary module, made once per model as a program does."""
    m = MODELS[model]
    return RotaryEmbedding(m.d, m.d, m.maxpos, m.theta).cuda()


@functools.lru_cache(maxsize=None)
def _table(model):
    """The rotary table in plain torch: cos | sin of position times inverse frequency, fp32."""
    m = MODELS[model]
    inv = 1.0 / (m.theta ** (torch.arange(0, m.d, 2, dtype=torch.float32) / m.d))
    ang = torch.einsum("i,j -> ij", torch.arange(m.maxpos, dtype=torch.float32), inv)
    return torch.cat((ang.cos(), ang.sin()), dim=-1).cuda()


def _norm(weight, eps):
    n = RMSNorm(weight.numel(), eps=eps).to(weight.device)
    with torch.no_grad():
        n.weight.data = weight
    return n


def _qkv_inputs(r, m, t):
    n = (m.hq + 2 * m.hkv) * m.d
    x = SimpleNamespace(x=r.randn(t, m.h), ln=r.randn(m.h, std=0.1, mean=1.0), w=r.randn(n, m.h, std=0.02))
    if m.qk_norm:
        x.qn = r.randn(m.d, std=0.1, mean=1.0)
        # key-norm weights of widely different magnitude
        u = torch.rand(m.d, generator=r.g, device=r.dev)
        x.kn = torch.exp(u * math.log(100.0) + math.log(0.05)).to(r.dtype)
    return x


def _pages_of_batch(r, t):
    """Page tables of t sequences with one new token each (CSR), every sequence on pages of its own."""
    lens = r.ints(0, 15 * PAGE, t)
    per = lens // PAGE + 1
    indptr = torch.cat([torch.zeros(1, dtype=torch.int64, device=r.dev), per.cumsum(0)]).to(torch.int32)
    pages = 16 * t
    return pages, r.perm(pages)[: int(indptr[-1])].to(torch.int32), indptr, lens


def _chunks(case, r, m):
    """A system prompt and context chunks in shuffled pages, every second context chunk moved, and the new
    tokens' chunk: (chunks, pages in all, keys in all)."""
    t, ctx = case["tokens"], case["context"]
    host = torch.Generator().manual_seed(ctx)  # the lengths belong to the case, the pages and moves to the seed
    lengths, left = [min(ctx, 100)], ctx - min(ctx, 100)
    while left > 0:
        n = min(left, int(torch.randint(90, 400, (1,), generator=host)))
        lengths.append(n)
        left -= n
    lengths.append(t)
    need = sum(-(-n // PAGE) for n in lengths)
    pages = need + need // 4 + 8
    perm = r.perm(pages).tolist()
    span = min(2000, m.maxpos // 4)
    moves = r.ints(-span, span, len(lengths)).tolist()
    chunks, used, pos = [], 0, 0
    for i, n in enumerate(lengths):
        npg = -(-n // PAGE)
        moved = 0 < i < len(lengths) - 1 and i % 2 == 1
        delta = moves[i] if moved else 0
        chunks.append(SimpleNamespace(page_table=perm[used:used + npg], kv_length=n, cached_position_start=pos,
                                      global_position_start=pos + delta,
                                      chunk_type=SimpleNamespace(value="system_prompt" if i == 0 else "context")))
        used += npg
        pos += n
    return chunks, pages, pos


def _attn_inputs(case, r, m):
    t = case["tokens"]
    chunks, pages, keys = _chunks(case, r, m)
    a = SimpleNamespace(chunks=chunks, keys=keys, kv=r.randn(pages, 2, m.hkv, PAGE, m.d))
    a.qpos = torch.arange(keys - t, keys, device=r.dev)
    a.table = torch.tensor(chunks[-1].page_table, dtype=torch.int32, device=r.dev)
    a.cpos = torch.arange(t, device=r.dev)
    return a


def prepare(case, seed):
    m, t = MODELS[case["model"]], case["tokens"]
    r = _Draw(seed, DTYPES[case["dtype"]])
    s = SimpleNamespace(case=case, m=m, kind=case["kind"])
    if s.kind == "qkv":
        s.q = _qkv_inputs(r, m, t)
        s.rope = _rope(case["model"])
        s.pos = r.ints(0, m.maxpos, t)
        s.append = None
        if case["append"]:
            if t <= 64:
                pages, table, indptr, lens = _pages_of_batch(r, t)
                seqs = dict(kv_indptr=indptr, batch_indices=torch.arange(t, device=r.dev))
            else:
                pages, lens, seqs = 2 * -(-t // PAGE), torch.arange(t, device=r.dev), {}
                table = r.perm(pages)[: -(-t // PAGE)].to(torch.int32)
            s.cache = r.randn(pages, 2, m.hkv, PAGE, m.d)
            s.append = PagedKVAppend(s.cache, table, lens, PAGE, **seqs)
    elif s.kind == "mlp":
        s.x, s.res = r.randn(t, m.h), r.randn(t, m.h)
        s.norm = _norm(r.randn(m.h, std=0.1, mean=1.0), m.eps)
        s.gate_up, s.down = r.randn(2 * m.inter, m.h, std=0.02), r.randn(m.h, m.inter, std=0.02)
    elif s.kind == "attn":
        s.a = _attn_inputs(case, r, m)
        s.query = r.randn(t, m.hq, m.d)
        s.att = CascadeAttention(m.hq, m.d, m.d ** -0.5, m.hkv, PAGE, rotary_emb=_rope(case["model"]))
        s.levels = s.att.create_cascade_levels(s.a.chunks)
        s.k_norm = None
        if m.qk_norm:
            u = torch.rand(m.d, generator=r.g, device=r.dev)
            s.k_norm = _norm(torch.exp(u * math.log(100.0) + math.log(0.05)).to(r.dtype), m.eps)
    elif s.kind == "rows":
        s.embed = VocabParallelEmbedding(m.vocab, m.h).to(r.dev)
        with torch.no_grad():
            s.embed.weight.data = r.randn(m.vocab, m.h, std=0.02)
        s.ids = r.ints(0, m.vocab, t)
        s.x = r.randn(t, m.h)
        s.norm = _norm(r.randn(m.h, std=0.1, mean=1.0), m.eps)
        s.packed = r.randn(t, (m.hq + 2 * m.hkv) * m.d)
        s.pos = r.ints(0, m.maxpos, t)
        s.rope = _rope(case["model"])
        s.table = r.perm(2 * -(-t // PAGE))[: -(-t // PAGE)].to(torch.int32)
        s.cpos = torch.arange(t, device=r.dev)
        s.cache = r.randn(2 * -(-t // PAGE), 2, m.hkv, PAGE, m.d)
        s.gate_up = r.randn(t, 2 * m.inter)
    else:
        s.q = _qkv_inputs(r, m, t)
        if m.qk_norm:  # a softmax of ordinary entropy
            s.q.kn = r.randn(m.d, std=0.1, mean=1.0)
        s.a = _attn_inputs(case, r, m)
        s.rope = _rope(case["model"])
        s.att = CascadeAttention(m.hq, m.d, m.d ** -0.5, m.hkv, PAGE, rotary_emb=s.rope)
        s.levels = s.att.create_cascade_levels(s.a.chunks)
        s.append = PagedKVAppend(s.a.kv, s.a.table, s.a.cpos, PAGE)
        s.o = r.randn(m.h, m.hq * m.d, std=0.02)
        s.norm = _norm(r.randn(m.h, std=0.1, mean=1.0), m.eps)
        s.gate_up, s.down = r.randn(2 * m.inter, m.h, std=0.02), r.randn(m.h, m.inter, std=0.02)
        s.graph = None
        if case["graph"]:
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                for _ in range(2):
                    _layer(s)
            torch.cuda.current_stream().wait_stream(side)
            s.graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(s.graph):
                s.outputs = _layer(s)
    return s


# -------------------------------------------------------------------- passes


def _attention_input(s, x, positions):
    m, q, cs = s.m, s.q, s.rope.cos_sin_cache
    if m.qk_norm:
        return qwen3_attention_input(x, q.ln, q.w, None, m.hq, m.hkv, m.eps, positions, cs, q.qn, q.kn,
                                     paged_kv=s.append)
    return llama_attention_input(x, q.ln, q.w, m.hq, m.hkv, m.eps, positions, cs, paged_kv=s.append)


def _mlp(s, x, residual):
    y, res = s.norm(x, residual)
    return linear_add_residual(gate_up_silu_and_mul(y, s.gate_up), s.down, res)


def _layer(s):
    q, _, _ = _attention_input(s, s.q.x, s.a.qpos)
    att = s.att.forward(q, s.a.qpos, s.a.kv, s.levels, 0)
    # o_proj and down_proj join the residual stream in their own epilogues
    x = linear_add_residual(att, s.o, s.q.x)
    y = s.norm(x)
    return linear_add_residual(gate_up_silu_and_mul(y, s.gate_up), s.down, x), s.a.kv


def run(s):
    if s.kind == "qkv":
        out = _attention_input(s, s.q.x, s.pos)
        return (out, s.cache) if s.append is not None else out
    if s.kind == "mlp":
        return _mlp(s, s.x, s.res)
    if s.kind == "attn":
        return s.att.forward(s.query, s.a.qpos, s.a.kv, s.levels, 0, k_norm=s.k_norm)
    if s.kind == "rows":
        m, t = s.m, s.case["tokens"]
        e = s.embed(s.ids)
        y, res = s.norm(s.x, e)
        qw, kw = m.hq * m.d, m.hkv * m.d
        q, k = s.rope(s.pos, s.packed[:, :qw], s.packed[:, qw:qw + kw])
        append_to_paged_kv_cache_custom(k.view(t, m.hkv, m.d), s.packed[:, qw + kw:].view(t, m.hkv, m.d), s.cache,
                                        s.table, s.cpos, PAGE)
        return e, y, res, q, k, s.cache, silu_and_mul(s.gate_up)
    if s.graph is not None:
        s.graph.replay()
        return s.outputs
    return _layer(s)


# --------------------------------------------------------- work, tolerance


def _qkv_work(m, t, append):
    n = (m.hq + 2 * m.hkv) * m.d
    b = 2 * (t * m.h + m.h + n * m.h + t * n) + 8 * t + 4 * t * m.d
    if append:
        b += 2 * 2 * t * m.hkv * m.d + 12 * t
    return b, 2.0 * t * n * m.h


def _attn_work(m, t, context):
    keys = context + t
    pairs = t * context + t * (t + 1) // 2
    return 2 * (2 * keys * m.hkv * m.d + 2 * t * m.hq * m.d), 4.0 * pairs * m.hq * m.d


def work(case):
    m, t, kind = MODELS[case["model"]], case["tokens"], case["kind"]
    if kind == "qkv":
        b, f = _qkv_work(m, t, case["append"])
    elif kind == "mlp":
        b, f = 2 * (3 * t * m.h + m.h + 3 * m.inter * m.h), 6.0 * t * m.h * m.inter
    elif kind == "attn":
        b, f = _attn_work(m, t, case["context"])
    elif kind == "rows":
        # gather; add+norm (reads x and the gathered rows, writes two); rope of q and k; append of k and v; silu*mul
        b = 2 * (2 * t * m.h + 4 * t * m.h + 2 * t * (m.hq + m.hkv) * m.d + 4 * t * m.hkv * m.d + 3 * t * m.inter)
        b, f = b + t * (8 + 8 + 8 + 4 * m.d), 0.0
    else:
        b, f = _qkv_work(m, t, True)
        ab, af = _attn_work(m, t, case["context"])
        b += ab + 2 * (m.h * m.hq * m.d + 3 * m.inter * m.h + t * m.h)
        f += af + 2.0 * t * m.h * m.hq * m.d + 6.0 * t * m.h * m.inter
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    # about four times the relative error against 64 bits that the operation shows (measured: rows 0.0024,
    # llama qkv 0.0023, qwen3 qkv with its bf16 roundings 0.0037, mlp 0.0049, attention 0.0064, whole layer
    # 0.0056 in bf16; an eighth of it in fp16, where no step rounds to bf16)
    rel = {"rows": 0.01, "qkv": 0.015 if MODELS[case["model"]].qk_norm else 0.01, "mlp": 0.02, "attn": 0.025,
           "layer": 0.025}[case["kind"]]
    if case["dtype"] == "fp16" and not (MODELS[case["model"]].qk_norm and case["kind"] in ("qkv", "layer")):
        rel /= 8
    return {"rel": rel}


# ----------------------------------------------------------- 64-bit results


def _rms64(x, w, eps):
    x = x.double()
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _rope64(x, positions, table):
    """x [T, heads, D] rotated by the table rows of `positions` (half-split pairs)."""
    d = x.shape[-1]
    cs = table[positions].double()[:, None, :]
    c, s = cs[..., : d // 2], cs[..., d // 2:]
    a, b = x[..., : d // 2], x[..., d // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _qkv64(m, q, x, positions, table):
    t = x.shape[0]
    y = _rms64(x, q.ln, m.eps) @ q.w.double().t()
    qh, kh, vh = (v.reshape(t, -1, m.d) for v in y.split([m.hq * m.d, m.hkv * m.d, m.hkv * m.d], -1))
    if m.qk_norm:
        qh, kh = _rms64(qh, q.qn, m.eps), _rms64(kh, q.kn, m.eps)
    return _rope64(qh, positions, table), _rope64(kh, positions, table), vh


def _append64(cache, k, v, pages, slots):
    cache = cache.double()
    cache[pages, 0, :, slots] = k
    cache[pages, 1, :, slots] = v
    return cache


def _attn64(m, a, query, kv, table, k_norm):
    """Attention of query [T, Hq, D] over the chunks' keys in walk order, causal by walk position."""
    ks, vs = [], []
    for c in a.chunks:
        pt = torch.tensor(c.page_table, device=kv.device)
        k, v = (kv[pt, i].double().transpose(1, 2).reshape(-1, m.hkv, m.d)[: c.kv_length] for i in (0, 1))
        delta = c.global_position_start - c.cached_position_start
        if delta:
            k = _rope64(k, torch.full((k.shape[0],), delta, device=kv.device), table)
        ks.append(k)
        vs.append(v)
    k, v = torch.cat(ks).transpose(0, 1), torch.cat(vs).transpose(0, 1)  # [Hkv, keys, D]
    if k_norm is not None:
        k = _rms64(k, k_norm, m.eps)
    t, g = query.shape[0], m.hq // m.hkv
    hide = torch.arange(a.keys, device=kv.device)[None, :] > a.qpos[:, None]
    out = torch.empty(t, m.hq, m.d, dtype=torch.float64, device=kv.device)
    for h in range(m.hq):
        sc = query[:, h].double() @ k[h // g].t() * m.d ** -0.5
        out[:, h] = torch.softmax(sc.masked_fill(hide, float("-inf")), -1) @ v[h // g]
    return out.reshape(t, m.hq * m.d)


def _mlp64(s, y, residual):
    gu = y @ s.gate_up.double().t()
    act = torch.nn.functional.silu(gu[:, : s.m.inter]) * gu[:, s.m.inter:]
    return residual + act @ s.down.double().t()


def exact(case, seed):
    s = prepare(dict(case, graph=False) if "graph" in case else case, seed)
    m, t, table = s.m, case["tokens"], _table(case["model"])
    if s.kind == "qkv":
        q, k, v = _qkv64(m, s.q, s.q.x, s.pos, table)
        out = (q.reshape(t, -1), k.reshape(t, -1), v.reshape(t, -1))
        if s.append is None:
            return out
        p, at = s.append, s.append.positions
        base = p.kv_indptr[:-1].long() if p.kv_indptr is not None else 0
        return out, _append64(s.cache, k, v, p.kv_indices[base + at // PAGE].long(), at % PAGE)
    if s.kind == "mlp":
        res = s.x.double() + s.res.double()
        return _mlp64(s, _rms64(res, s.norm.weight, m.eps), res)
    if s.kind == "attn":
        return _attn64(m, s.a, s.query, s.a.kv, table, s.k_norm.weight if s.k_norm is not None else None)
    if s.kind == "rows":
        e = s.embed.weight[s.ids].double()
        res = s.x.double() + e
        qw, kw = m.hq * m.d, m.hkv * m.d
        p = s.packed.double().split([qw, kw, kw], -1)
        q, k = (_rope64(v.reshape(t, -1, m.d), s.pos, table) for v in p[:2])
        gate, up = s.gate_up.double().chunk(2, -1)
        cache = _append64(s.cache, k, p[2].reshape(t, m.hkv, m.d), s.table[s.cpos // PAGE].long(), s.cpos % PAGE)
        return (e, _rms64(res, s.norm.weight, m.eps), res, q.reshape(t, -1), k.reshape(t, -1), cache,
                torch.nn.functional.silu(gate) * up)
    x = s.q.x
    q, k, v = _qkv64(m, s.q, x, s.a.qpos, table)
    kv = _append64(s.a.kv, k, v, s.a.table[s.a.cpos // PAGE].long(), s.a.cpos % PAGE)
    att = _attn64(m, s.a, q, kv, table, None)
    stream = x.double() + att @ s.o.double().t()
    return _mlp64(s, _rms64(stream, s.norm.weight, m.eps), stream), kv
