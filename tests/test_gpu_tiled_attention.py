"""Reference-shaped attention on the fp32 matrix cores (head sizes other than
128, other page sizes): edges of the 16-row and 16-key tiles, as many key
tiles as wavefronts and one more, head sizes around the 16-, 64-, 128- and
256-dim groups and not multiples of 4, grouped heads, key and value sizes that
differ, both entry points, unaligned tensors, special values.

Reference: 64-bit numpy for finite inputs (max-abs 2e-5 plus rel 1e-4 on
outputs, 2e-6 on probabilities, the contract of the reference-shaped entry),
and the scalar kernel of the probability entry, which follows the
reference's loop order, for infinities, NaN and pages outside the pool."""

import numpy as np
import pytest
import torch

import helix_runtime_amd as hx

pytestmark = pytest.mark.gpu


def inputs(hkv, group, kd, vd, p, hist, t, seed, shift=0):
    rng = np.random.default_rng(seed)
    logical = (hist + p - 1) // p
    n = logical + 3
    f = lambda *s: rng.standard_normal(s, dtype=np.float32)  # noqa: E731
    arrays = [f(hkv * group, t, kd), f(n, hkv, p, kd), f(n, hkv, p, vd), f(hkv, t, kd), f(hkv, t, vd)]
    table = rng.permutation(n)[:logical].astype(np.int32)

    def dev(a):
        flat = torch.zeros(a.size + 4, device="cuda:0")
        flat[shift:shift + a.size] = torch.from_numpy(a.reshape(-1)).cuda()
        return flat[shift:shift + a.size].view(a.shape)

    return arrays, table, [dev(a) for a in arrays], torch.from_numpy(table).cuda()


def reference(q, keys, values, offset):
    hkv, group = keys.shape[0], q.shape[0] // keys.shape[0]
    k = np.repeat(keys.astype(np.float64), group, axis=0)
    v = np.repeat(values.astype(np.float64), group, axis=0)
    s = q.astype(np.float64) @ k.transpose(0, 2, 1) / np.sqrt(q.shape[2])
    seen = np.arange(k.shape[1])[None, :] <= offset + np.arange(q.shape[1])[:, None]
    s = np.where(seen, s, -np.inf)
    e = np.exp(s - s.max(-1, keepdims=True))
    p = e / e.sum(-1, keepdims=True)
    return p @ v, p


def page_rows(pool, table, hist):
    return np.concatenate([pool[b] for b in table], axis=1)[:, :hist]


@pytest.mark.parametrize("hkv,group,kd,vd,p,hist,t", [
    (1, 1, 1, 1, 1, 1, 1), (4, 1, 16, 16, 16, 64, 1), (3, 1, 37, 37, 7, 12, 17),
    (2, 4, 64, 64, 16, 15, 5), (8, 1, 64, 64, 16, 240, 16), (2, 2, 80, 80, 16, 333, 33),
    (1, 8, 96, 64, 32, 500, 3), (2, 1, 128, 128, 8, 100, 40), (2, 1, 130, 20, 16, 31, 9),
    (1, 1, 12, 256, 16, 65, 18), (1, 2, 256, 256, 4, 129, 20), (2, 3, 65, 63, 5, 47, 31),
    (1, 1, 32, 33, 16, 1999, 1), (2, 1, 64, 64, 16, 0, 50),
    # A wavefront per key tile, and one tile more than wavefronts.
    (2, 1, 64, 64, 16, 255, 1), (2, 1, 64, 64, 16, 256, 1), (1, 2, 16, 16, 1, 237, 20),
    (2, 2, 128, 128, 8, 120, 8), (2, 2, 128, 128, 8, 121, 8), (1, 1, 200, 200, 12, 127, 1),
    (1, 1, 200, 200, 12, 128, 1)])
@pytest.mark.parametrize("shift", [0, 1])
def test_tail_entry_matches_64_bit(device, hkv, group, kd, vd, p, hist, t, shift):
    (q, kp, vp, tk, tv), table, d, dtable = inputs(hkv, group, kd, vd, p, hist, t,
                                                   kd + hist + t, shift)
    out = torch.full((q.shape[0], t, vd), 7.0, device=device)
    ws = torch.full((q.shape[0], t, hist + t), 7.0, device=device)
    hx.paged_attention_with_tail_out(d[0], d[1], d[2], dtable, hist, d[3], d[4], out, ws)
    torch.cuda.synchronize()
    keys = np.concatenate([page_rows(kp, table, hist), tk], 1) if hist else tk
    values = np.concatenate([page_rows(vp, table, hist), tv], 1) if hist else tv
    ref, prob = reference(q, keys, values, hist)
    np.testing.assert_allclose(out.cpu().numpy(), ref, atol=2e-5, rtol=1e-4)
    np.testing.assert_allclose(ws.cpu().numpy(), prob, atol=2e-6, rtol=0)


@pytest.mark.parametrize("kd,p,tokens,t,offset", [(64, 16, 100, 20, 3), (64, 16, 100, 20, 80),
                                                  (40, 7, 33, 33, 0), (128, 32, 70, 1, 40)])
def test_history_entry_matches_64_bit(device, kd, p, tokens, t, offset):
    (q, kp, vp, _, _), table, d, dtable = inputs(2, 2, kd, kd, p, tokens, t, offset + kd)
    out = torch.empty(4, t, kd, device=device)
    ws = torch.full((4, t, tokens), 7.0, device=device)
    hx.paged_attention_out(d[0], d[1], d[2], dtable, tokens, offset, out, ws)
    torch.cuda.synchronize()
    ref, prob = reference(q, page_rows(kp, table, tokens), page_rows(vp, table, tokens), offset)
    np.testing.assert_allclose(out.cpu().numpy(), ref, atol=2e-5, rtol=1e-4)
    np.testing.assert_allclose(ws.cpu().numpy(), prob, atol=2e-6, rtol=0)


@pytest.mark.parametrize("kd,p", [(64, 16), (37, 7), (160, 16)])
@pytest.mark.parametrize("hist", [90, 290])
def test_special_values_match_scalar_kernel(device, kd, p, hist):
    t, hkv = 20, 6
    (_, _, _, _, _), table, d, dtable = inputs(hkv, 2, kd, kd, p, hist, t, 5 + kd)
    q, kp, vp, tk, tv = d
    inf, nan = float("inf"), float("nan")
    kp[int(table[2]), 0, 1, 3] = inf          # infinite history key
    tk[1, 7, 0] = -inf                        # infinite chunk key, masked by the rows before
    tv[2, 9, 5], tv[2, 11, 1] = inf, nan      # value rows that earlier rows mask
    vp[int(table[1]), 3, 2, 2] = -inf         # infinite history value
    tk[4, 5, 2] = nan
    q[10, 3] = 0.0
    dtable[-1] = kp.shape[0]                  # the last page is outside the pool
    results = []
    for use in (slice(0, hist), slice(0, hist - hist % p)):
        n = use.stop
        for scalar in (False, True):
            out = torch.full((2 * hkv, t, kd), 7.0, device=device)
            ws = torch.full((2 * hkv, t, n + t), 7.0, device=device)
            hx.paged_attention_with_tail_out(q, kp, vp, dtable, n, tk, tv, out, ws,
                                             probabilities=scalar)
            torch.cuda.synchronize()
            results.append((out.cpu().numpy(), ws.cpu().numpy()))
    for got, want in (results[:2], results[2:]):
        np.testing.assert_allclose(got[0], want[0], atol=2e-5, rtol=1e-4)
        np.testing.assert_allclose(got[1], want[1], atol=2e-6, rtol=0)
    assert np.isfinite(results[2][0]).any() and np.isnan(results[2][0]).any()
