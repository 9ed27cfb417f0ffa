"""Performance cases of the paged-KV path, through its public entry points.

A case's "kind" says which call it stands for:

- "reference": one call of the reference-shaped attention over one sequence's
  block table with an uncommitted tail (paged_attention_with_tail_out): what a
  program moved over from the reference issues per layer, with one tail row
  per decoded token or a chunk of rows per prompt piece, any head size and
  page size; the softmax probabilities stay in the caller's score workspace.
- "decode": one layer of a batched decode step (DecodeBatch.attention_layer),
  every sequence at its own length over scattered pages of a cache of fp32,
  bf16 or fp8 pages; with "prefix" > 0 every sequence is a copy-on-write fork
  of one root prompt of that many tokens.
- "prefill": one layer of a chunked-prefill step (DecodeBatch.prefill_layer):
  a chunk of prompt tokens per sequence over that sequence's history.
- "prompt": a prompt's K/V rows committed to a new sequence in every layer and
  gathered back (append_layer_major, copy_layer_out, release_sequence): the
  append and gather directions, bit for bit.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import helix_runtime_amd as hx

DEV = "cuda:0"
K_SCALE, V_SCALE = 0.03, 0.015  # fp8 scales of a calibrated cache (448 * scale covers the rows)


# ------------------------------------------------------------------ cases ----
def listed():
    return [
        # The smallest call: the reference's tiny decode (4 heads of 16 dims
        # over a 64-token history); launch and host latency.
        dict(name="ref_tiny", kind="reference", q_heads=4, kv_heads=4, head_dim=16,
             block_tokens=16, history=64, tail=1),
        # The reference's own attention benchmark shape (8 heads of 64 dims,
        # 128 query rows, 1024 keys): a prompt piece at head_dim 64.
        dict(name="ref_d64_chunk", kind="reference", q_heads=8, kv_heads=8, head_dim=64,
             block_tokens=16, history=896, tail=128),
        # One layer of the reference model's one-token decode, 32/8 heads of
        # 128 dims at an ordinary context.
        dict(name="ref_decode", kind="reference", q_heads=32, kv_heads=8, head_dim=128,
             block_tokens=16, history=2680, tail=1),
        # One layer of a 512-token prompt piece through the same entry.
        dict(name="ref_chunk", kind="reference", q_heads=32, kv_heads=8, head_dim=128,
             block_tokens=16, history=2170, tail=512),
        # Batched decode of 8 sequences without head grouping (32/32 heads).
        dict(name="decode_mha", kind="decode", batch=8, q_heads=32, kv_heads=32, low=128,
             high=2048, prefix=0, dtype="f32"),
        # Batched decode of 64 sequences, 32/8 heads, contexts log-uniform in
        # [512, 8192], on each page type.
        dict(name="decode_f32", kind="decode", batch=64, q_heads=32, kv_heads=8, low=512,
             high=8192, prefix=0, dtype="f32"),
        dict(name="decode_bf16", kind="decode", batch=64, q_heads=32, kv_heads=8, low=512,
             high=8192, prefix=0, dtype="bf16"),
        dict(name="decode_fp8", kind="decode", batch=64, q_heads=32, kv_heads=8, low=512,
             high=8192, prefix=0, dtype="fp8"),
        # 128 forks of one 1032-token prompt with their own suffixes.
        dict(name="decode_shared", kind="decode", batch=128, q_heads=32, kv_heads=8, low=64,
             high=512, prefix=1032, dtype="f32"),
        # Chunked prefill, 16 sequences of 512 rows over histories up to 4096.
        dict(name="prefill_f32", kind="prefill", batch=16, q_heads=32, kv_heads=8, tokens=512,
             low=0, high=4096, dtype="f32"),
        dict(name="prefill_bf16", kind="prefill", batch=16, q_heads=32, kv_heads=8, tokens=512,
             low=0, high=4096, dtype="bf16"),
        # A prompt of ordinary length committed and gathered back, 4 layers.
        dict(name="prompt_f32", kind="prompt", layers=4, kv_heads=8, head_dim=128,
             block_tokens=16, tokens=2048, dtype="f32"),
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["reference", "reference", "reference128", "decode", "decode", "decode",
                       "shared", "prefill", "prefill", "prompt"])
    dtype = rng.choice(["f32", "bf16", "fp8"])
    if kind == "reference":  # any head and page size
        kv_heads, group = rng.choice([(3, 1), (4, 1), (8, 1), (12, 1), (4, 2), (2, 4)])
        dim = rng.choice([16, 32, 37, 64, 64, 80, 96])
        tail = 1 if rng.random() < 0.4 else _log_int(rng, 2, 160)
        return dict(kind="reference", q_heads=kv_heads * group, kv_heads=kv_heads, head_dim=dim,
                    block_tokens=rng.choice([4, 7, 16, 16, 32]),
                    history=_log_int(rng, 1, 2048), tail=tail)
    if kind == "reference128":
        kv_heads, group = rng.choice([(8, 4), (8, 1), (32, 1), (4, 8), (5, 2)])
        tail = 1 if rng.random() < 0.5 else _log_int(rng, 2, 512)
        return dict(kind="reference", q_heads=kv_heads * group, kv_heads=kv_heads, head_dim=128,
                    block_tokens=16, history=_log_int(rng, 16, 4096), tail=tail)
    if kind == "decode":
        kv_heads, group = rng.choice([(8, 4), (8, 4), (32, 1), (4, 8), (16, 2)])
        batch = _log_int(rng, 1, 64)
        high = _log_int(rng, 64, 8192 if kv_heads <= 8 else 2048)
        return dict(kind="decode", batch=batch, q_heads=kv_heads * group, kv_heads=kv_heads,
                    low=max(1, high // rng.choice([1, 4, 16])), high=high, prefix=0, dtype=dtype)
    if kind == "shared":
        kv_heads, group = rng.choice([(8, 4), (8, 4), (16, 1), (4, 8)])
        return dict(kind="decode", batch=_log_int(rng, 4, 128), q_heads=kv_heads * group,
                    kv_heads=kv_heads, low=_log_int(rng, 1, 64), high=_log_int(rng, 64, 512),
                    prefix=_log_int(rng, 100, 2048), dtype=dtype)
    if kind == "prefill":
        kv_heads, group = rng.choice([(8, 4), (8, 4), (32, 1), (4, 8), (16, 2)])
        tokens = _log_int(rng, 16, 512)
        return dict(kind="prefill", batch=_log_int(rng, 1, 12), q_heads=kv_heads * group,
                    kv_heads=kv_heads, tokens=tokens, low=0, high=_log_int(rng, 16, 4096),
                    dtype=dtype)
    return dict(kind="prompt", layers=rng.choice([1, 2, 4, 8]), kv_heads=rng.choice([3, 8, 16]),
                head_dim=rng.choice([64, 80, 128, 128]), block_tokens=rng.choice([7, 16, 16, 32]),
                tokens=_log_int(rng, 16, 4096), dtype=dtype)


# ----------------------------------------------------------------- inputs ----
def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, device=DEV, generator=g)


def _lengths(case):
    """The batch's context lengths: part of the case, the same for every seed."""
    low, high, n = case["low"], case["high"], case["batch"]
    rng = np.random.default_rng([n, low, high])
    if low > 0 and high > 4 * low:  # contexts of a batch spread over their logarithm
        v = np.exp(rng.uniform(math.log(low), math.log(high + 1), size=n)).astype(np.int64)
        return [int(min(high, max(low, x))) for x in v]
    return [int(x) for x in rng.integers(min(low, high), high + 1, size=n)]


def _rows(g, heads, tokens, dim, channel):
    """K and V rows [heads, tokens, dim]: keys with per-channel magnitudes, as
    projections give them, values N(0, 1)."""
    return _randn(g, heads, tokens, dim) * channel, _randn(g, heads, tokens, dim)


def _channel(g, heads, dim):
    return torch.exp(0.4 * _randn(g, heads, 1, dim))


def _batch_inputs(case, seed):
    """Every tensor of a decode or prefill case, from the seed alone."""
    g = _generator(seed)
    hq, hkv, b, d = case["q_heads"], case["kv_heads"], case["batch"], 128
    channel = _channel(g, hkv, d)
    lengths = _lengths(case)
    prefix = case.get("prefix", 0)
    root = _rows(g, hkv, prefix, d, channel) if prefix else None
    own = [_rows(g, hkv, n, d, channel) for n in lengths]
    t = case.get("tokens")
    if t is None:
        q = _randn(g, b, hq, d)
        k, v = _randn(g, b, hkv, d) * channel[:, 0], _randn(g, b, hkv, d)
    else:
        q = _randn(g, b, hq, t, d)
        k, v = _randn(g, b, hkv, t, d) * channel, _randn(g, b, hkv, t, d)
    return lengths, root, own, q, k.contiguous(), v.contiguous()


def _reference_inputs(case, seed):
    g = _generator(seed)
    hq, hkv, d, p = case["q_heads"], case["kv_heads"], case["head_dim"], case["block_tokens"]
    hist, t = case["history"], case["tail"]
    logical = (hist + p - 1) // p
    physical = logical + logical // 4 + 2
    channel = _channel(g, hkv, d)
    kp = _randn(g, physical, hkv, p, d) * channel
    vp = _randn(g, physical, hkv, p, d)
    table = np.random.default_rng(int(seed) + 5).permutation(physical)[:logical]
    q = _randn(g, hq, t, d)
    tk, tv = _randn(g, hkv, t, d) * channel, _randn(g, hkv, t, d)
    return q, kp, vp, [int(x) for x in table], physical, tk.contiguous(), tv.contiguous()


def _cache(case, layers, head_dim, block_tokens, blocks):
    more = dict(k_scale=K_SCALE, v_scale=V_SCALE) if case["dtype"] == "fp8" else {}
    return hx.PagedKvCache(layers, case["kv_heads"], head_dim, block_tokens, blocks,
                           page_dtype=case["dtype"], **more)


def _fill(cache, seqs, rows, seed):
    """Appends each sequence's rows in pieces of 64 tokens, the sequences in
    random turn, so their pages scatter over the pool as in a server whose
    sequences grow side by side."""
    order = [i for i, (k, _) in enumerate(rows) for _ in range((k.shape[1] + 63) // 64)]
    np.random.default_rng(int(seed) + 9).shuffle(order)
    at = [0] * len(seqs)
    for i in order:
        a, (k, v) = at[i], rows[i]
        at[i] = z = min(a + 64, k.shape[1])
        cache.append_layer_major(seqs[i], [k[:, a:z].contiguous()], [v[:, a:z].contiguous()])


def _prompt_inputs(case, seed):
    g = _generator(seed)
    shape = (case["kv_heads"], case["tokens"], case["head_dim"])
    return ([_randn(g, *shape) for _ in range(case["layers"])],
            [_randn(g, *shape) for _ in range(case["layers"])])


def prepare(case, seed):
    kind = case["kind"]
    if kind == "reference":
        q, kp, vp, ids, physical, tk, tv = _reference_inputs(case, seed)
        hq, t, d = q.shape
        return dict(kind=kind, q=q, kp=kp, vp=vp, tk=tk, tv=tv, history=case["history"],
                    table=hx.PagedBlockTable(ids, physical), out=torch.empty(hq, t, d, device=DEV),
                    work=torch.empty(hq, t, case["history"] + t, device=DEV))
    if kind == "prompt":
        keys, values = _prompt_inputs(case, seed)
        p = case["block_tokens"]
        cache = _cache(case, case["layers"], case["head_dim"], p, 2 * (case["tokens"] // p + 2))
        return dict(kind=kind, cache=cache, keys=keys, values=values,
                    out=[(torch.empty_like(k), torch.empty_like(v)) for k, v in zip(keys, values)])
    lengths, root, own, q, k, v = _batch_inputs(case, seed)
    t, prefix = case.get("tokens", 1), case.get("prefix", 0)
    blocks = sum((n + t) // 16 + 2 for n in lengths) + prefix // 16 + 8
    cache = _cache(case, 1, 128, 16, blocks)
    if prefix:
        first = cache.create_sequence()
        cache.append_layer_major(first, [root[0]], [root[1]])
        seqs = [cache.fork_sequence(first, prefix, allow_cow=True) for _ in lengths]
        cache.release_sequence(first)
    else:
        seqs = [cache.create_sequence() for _ in lengths]
    _fill(cache, seqs, own, seed)
    batch = hx.DecodeBatch(cache, seqs, case["q_heads"], max_tokens=prefix + max(lengths) + t + 1)
    if kind == "decode":
        batch.prepare()
    else:
        batch.prepare_chunk(t)
    return dict(kind=kind, cache=cache, batch=batch, q=q, k=k, v=v, out=torch.empty_like(q))


# -------------------------------------------------------------------- run ----
def run(state):
    kind, s = state["kind"], state
    if kind == "reference":
        hx.paged_attention_with_tail_out(s["q"], s["kp"], s["vp"], s["table"].data(), s["history"],
                                         s["tk"], s["tv"], s["out"], s["work"])
        return {"out": s["out"], "probabilities": s["work"]}
    if kind == "decode":
        s["batch"].attention_layer(0, s["q"], s["k"], s["v"], s["out"])
        return s["out"]
    if kind == "prefill":
        s["batch"].prefill_layer(0, s["q"], s["k"], s["v"], s["out"])
        return s["out"]
    cache = s["cache"]
    seq = cache.create_sequence()
    cache.append_layer_major(seq, s["keys"], s["values"])
    for layer, (k, v) in enumerate(s["out"]):
        cache.copy_layer_out(seq, layer, k, v)
    cache.release_sequence(seq)
    return s["out"]


# ------------------------------------------------------------------- work ----
def work(case):
    kind = case["kind"]
    if kind == "reference":
        hq, hkv, d, t = case["q_heads"], case["kv_heads"], case["head_dim"], case["tail"]
        hist = case["history"]
        pairs = t * hist + t * (t + 1) // 2
        return {"bytes": 4 * (2 * hkv * (hist + t) * d + 2 * hq * t * d + hq * t * (hist + t)),
                "flops": 4 * hq * d * pairs}
    size = {"f32": 4, "bf16": 2, "fp8": 1}[case["dtype"]]
    if kind == "prompt":
        rows = 2 * case["layers"] * case["kv_heads"] * case["tokens"] * case["head_dim"]
        return {"bytes": 2 * rows * (4 + size), "flops": 0}
    hq, hkv, d, b = case["q_heads"], case["kv_heads"], 128, case["batch"]
    lengths, t, prefix = _lengths(case), case.get("tokens", 1), case.get("prefix", 0)
    hist = sum(lengths)
    shared = prefix // 16 * 16  # full pages of the root; the partial one is each fork's own
    pages = shared + hist + (prefix - shared) * b
    pairs = sum(t * (prefix + n) + t * (t + 1) // 2 for n in lengths)
    return {"bytes": 2 * hkv * pages * d * size + 4 * (2 * hkv * b * t * d + 2 * hq * b * t * d),
            "flops": 4 * hq * d * pairs}


# -------------------------------------------------------------- tolerance ----
def tolerance(case):
    """About four times what the path shows against exact(): fp32 products and
    sums throughout, whatever the page type (both sides read the same page
    values)."""
    if case["kind"] == "prompt":
        return "exact"
    return {"rel": 3e-6, "max": 6e-5}


# ------------------------------------------------------------------ exact ----
def _page_values(case, x, scale):
    """fp32 rows as their pages hold them."""
    if case["dtype"] == "bf16":
        return x.to(torch.bfloat16).to(torch.float32)
    if case["dtype"] == "fp8":
        by = torch.full((), scale, device=x.device)  # a tensor: a true fp32 division
        codes = (x / by).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
        return codes.to(torch.float32) * by
    return x


def _attend(q, k, v, hist):
    """q [hq, t, d], k and v [hkv, hist + t, d] in 64 bits: row i sees keys up
    to hist + i.  Returns (out, probabilities)."""
    hq, t, d = q.shape
    hkv, n, _ = k.shape
    s = torch.matmul(q.reshape(hkv, hq // hkv * t, d), k.transpose(1, 2).contiguous())
    s = s.reshape(hkv, hq // hkv, t, n) / math.sqrt(d)
    seen = torch.arange(n, device=DEV) <= hist + torch.arange(t, device=DEV)[:, None]
    p = torch.softmax(s.masked_fill(~seen, -math.inf), dim=-1)
    out = torch.matmul(p.reshape(hkv, hq // hkv * t, n), v)
    return out.reshape(hq, t, d), p.reshape(hq, t, n)


def exact(case, seed):
    kind = case["kind"]
    if kind == "reference":
        q, kp, vp, ids, _, tk, tv = _reference_inputs(case, seed)
        hkv, d, hist = case["kv_heads"], case["head_dim"], case["history"]

        def rows(pool, tail):
            x = pool[ids].transpose(0, 1).reshape(hkv, -1, d)[:, :hist]
            return torch.cat([x, tail], dim=1).double()

        out, p = _attend(q.double(), rows(kp, tk), rows(vp, tv), hist)
        return {"out": out, "probabilities": p}
    if kind == "prompt":
        keys, values = _prompt_inputs(case, seed)
        return [(_page_values(case, k, K_SCALE), _page_values(case, v, V_SCALE))
                for k, v in zip(keys, values)]
    lengths, root, own, q, k, v = _batch_inputs(case, seed)
    got = []
    for b in range(case["batch"]):
        parts = ([root] if root else []) + [own[b]]
        qb, kb, vb = q[b], k[b], v[b]
        if kind == "decode":
            qb, kb, vb = qb[:, None], kb[:, None], vb[:, None]
        keys = _page_values(case, torch.cat([x for x, _ in parts] + [kb], dim=1), K_SCALE)
        vals = _page_values(case, torch.cat([x for _, x in parts] + [vb], dim=1), V_SCALE)
        hist = keys.shape[1] - qb.shape[1]
        out, _ = _attend(qb.double(), keys.double(), vals.double(), hist)
        got.append(out[:, 0] if kind == "decode" else out)
    return torch.stack(got)
