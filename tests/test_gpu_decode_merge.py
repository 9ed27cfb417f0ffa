"""The merge of a stream decode's partials in every launch shape: one, two, 4,
8 and 16 half-wavefronts a row, by the row count, and by the bound on a unit's
partials where the batch knows its lengths; units with one partial, a few and
hundreds; a unit whose page lies outside the pool.

Reference: the split decode kernel, whose merge is another kernel, and the
oracle.  Tolerance: max-abs 2e-5 plus rel 1e-4, the fp32 contract; both sides
sum exact products in fp32 in another order."""

import numpy as np
import pytest
import torch

import helix_runtime_amd as hx
import oracle

pytestmark = pytest.mark.gpu

D, P = 128, 16
ATOL, RTOL = 2e-5, 1e-4


# Rows: 64, 480, 512 and 1536, 2048, 4096 (and one head per unit at 192, 4128).
@pytest.mark.parametrize("hkv,group,batch", [(4, 8, 2), (8, 2, 30), (8, 4, 16), (12, 8, 16),
                                             (16, 4, 32), (8, 8, 64), (64, 1, 3), (32, 1, 129)])
@pytest.mark.parametrize("long", [100, 2500, 40000])
def test_ragged_batch_matches_split_kernel(device, hkv, group, batch, long):
    gen = torch.Generator(device=device)
    gen.manual_seed(hkv * batch + long)
    rng = np.random.default_rng(long + batch)
    hq, blocks = hkv * group, 64
    lengths = rng.integers(0, 260, batch).astype(np.int32)
    lengths[batch // 2] = long
    cols = int(lengths.max()) // P + 2
    tables = rng.integers(0, blocks, (batch, cols)).astype(np.int32)
    tables[0, 0], lengths[0] = blocks, 120  # outside the pool: a NaN sequence
    r = lambda *s: torch.randn(*s, device=device, generator=gen)  # noqa: E731
    kp, vp = r(blocks, hkv, P, D), r(blocks, hkv, P, D)
    q, tk, tv = r(batch, hq, D), r(batch, hkv, D), r(batch, hkv, D)
    results = []
    for split in (0, 16):
        ws = hx.decode_workspace(batch, hq, hkv, cols, split)
        out = torch.full_like(q, 7.0)
        hx.paged_decode_attention(q, kp, vp, torch.from_numpy(tables).to(device),
                                  torch.from_numpy(lengths).to(device), tk, tv, out, ws, split)
        torch.cuda.synchronize()
        results.append(out.cpu().numpy())
    assert np.isnan(results[0][0]).all() and np.isfinite(results[0][1:]).all()
    np.testing.assert_allclose(results[0], results[1], atol=ATOL, rtol=RTOL)


@pytest.mark.parametrize("hkv,group,batch,tokens,short", [
    (8, 4, 1, 60, 60), (8, 4, 40, 98, 98), (4, 8, 64, 300, 300), (32, 1, 4, 98, 98),
    (32, 1, 40, 60, 60), (16, 2, 9, 2000, 2000), (8, 4, 70, 700, 700), (8, 4, 130, 4000, 50),
    (32, 1, 130, 1500, 20)])
def test_known_lengths_match_oracle(device, hkv, group, batch, tokens, short):
    """A batch whose table is far wider than its sequences: one of `tokens`,
    the others of about `short`."""
    rng = np.random.default_rng(tokens + batch)
    hq, phys = hkv * group, tokens // P + 2 + batch * (short // P + 2)
    cache = hx.PagedKvCache(1, hkv, D, P, phys)
    rows = rng.standard_normal((2, hkv, tokens, D), dtype=np.float32)
    seqs, lengths = [], []
    for b in range(batch):  # the rows' first tokens, a few fewer each
        n = tokens if b == batch // 2 else short - b % 7
        s = cache.create_sequence()
        cache.append_layer_major(s, *([torch.from_numpy(x[:, :n].copy()).to(device)] for x in rows))
        seqs.append(s)
        lengths.append(n)
    batch_ = hx.DecodeBatch(cache, seqs, hq, max_tokens=20000)
    batch_.prepare()
    q = rng.standard_normal((batch, hq, D), dtype=np.float32)
    tail = rng.standard_normal((2, batch, hkv, D), dtype=np.float32)
    out = torch.empty(batch, hq, D, device=device)
    dev = lambda a: torch.from_numpy(a).to(device)  # noqa: E731
    batch_.attention_layer(0, dev(q), dev(tail[0]), dev(tail[1]), out)
    torch.cuda.synchronize()
    cols = (tokens + P - 1) // P
    pool = np.zeros((2, cols, hkv, P, D), np.float32)
    for i in range(cols):
        part = rows[:, :, i * P:(i + 1) * P]
        pool[:, i, :, :part.shape[2]] = part
    ref = oracle.batched_decode(q, pool[0], pool[1],
                                np.tile(np.arange(cols, dtype=np.uint32), (batch, 1)),
                                np.array(lengths, np.int32), tail[0], tail[1], threads=8)
    np.testing.assert_allclose(out.cpu().numpy(), ref, atol=ATOL, rtol=RTOL)
    batch_.close()
    cache.close()


@pytest.mark.parametrize("dtype", ["f32", "fp8"])
@pytest.mark.parametrize("hkv,group", [(8, 4), (32, 1)])
def test_captured_layer_replays_at_grown_lengths(device, dtype, hkv, group):
    """A layer captured where every unit has few partials, replayed after one
    sequence has grown to hundreds: the launch shape stays, the result follows."""
    gen = torch.Generator(device=device)
    gen.manual_seed(hkv)
    r = lambda *s: torch.randn(*s, device=device, generator=gen)  # noqa: E731
    more = dict(k_scale=0.03, v_scale=0.015) if dtype == "fp8" else {}
    cache = hx.PagedKvCache(1, hkv, D, P, 700, page_dtype=dtype, **more)
    seqs = [cache.create_sequence() for _ in range(4)]
    for s in seqs:
        cache.append_layer_major(s, [r(hkv, 98, D)], [r(hkv, 98, D)])
    batch = hx.DecodeBatch(cache, seqs, hkv * group, max_tokens=9000)
    q, tk, tv = r(4, hkv * group, D), r(4, hkv, D), r(4, hkv, D)
    got, want = torch.empty_like(q), torch.empty_like(q)
    stream = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        batch.prepare()
        batch.attention_layer(0, q, tk, tv, want)
        stream.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            batch.attention_layer(0, q, tk, tv, got)
        for grown in (0, 1, 2500, 5000):
            if grown:
                batch.append_layer(0, tk, tv)
                k, v = r(hkv, grown, D), r(hkv, grown, D)
                stream.synchronize()
                cache.append_layer_major(seqs[1], [k], [v])
                batch.prepare()
            for _ in range(2):
                got.fill_(7.0)
                graph.replay()
                batch.attention_layer(0, q, tk, tv, want)
                stream.synchronize()
                np.testing.assert_allclose(got.cpu().numpy(), want.cpu().numpy(), atol=ATOL, rtol=RTOL)
    assert torch.isfinite(want).all()
    batch.close()
    cache.close()
