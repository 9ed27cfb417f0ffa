"""Batched decode of bf16 and fp8 pages on the matrix cores, where it can go
wrong: histories around the 16-token page and across many pages, empty
histories, every query group, rows of a partly filled page that hold NaN,
infinite and NaN page elements (recomputed in fp32), rows that are not
16-byte aligned.

Reference: the fp32-page kernel on the pages' own values (it is checked
against the oracle by the other suites), and the oracle itself on the finite
case.  Tolerance: max-abs 2e-5 plus rel 1e-4, the fp32 contract, since both
sides sum exact products in fp32."""

import numpy as np
import pytest
import torch

import helix_runtime_amd as hx
import oracle

pytestmark = pytest.mark.gpu

D, P = 128, 16
ATOL, RTOL = 2e-5, 1e-4
KS, VS = 0.03, 0.015
LENGTHS = [0, 1, 15, 16, 17, 31, 32, 33, 47, 160, 255, 256, 257, 1000, 3, 700]


def pages(dtype, shape, gen):
    """(raw pool, its fp32 values, unscaled grid) of N(0, 1) page elements."""
    x = torch.randn(shape, device="cuda:0", generator=gen)
    if dtype == "bf16":
        raw = x.to(torch.bfloat16)
        return raw, lambda s: raw.float()
    raw = (x * 20).to(torch.float8_e4m3fn).view(torch.uint8)
    return raw, lambda s: raw.view(torch.float8_e4m3fn).float() * s


def build(dtype, hq, hkv, seed):
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(seed)
    rng = np.random.default_rng(seed)
    need = [(n + P - 1) // P for n in LENGTHS]
    blocks, cols = sum(need) + 3, max(need) + 1
    kraw, kval = pages(dtype, (blocks, hkv, P, D), gen)
    vraw, vval = pages(dtype, (blocks, hkv, P, D), gen)
    perm = rng.permutation(blocks)
    tables = np.zeros((len(LENGTHS), cols), np.int32)
    at = 0
    for b, n in enumerate(need):
        tables[b, :n] = perm[at:at + n]
        at += n
    b = len(LENGTHS)
    q = torch.randn(b, hq, D, device="cuda:0", generator=gen)
    tk = torch.randn(b, hkv, D, device="cuda:0", generator=gen)
    tv = torch.randn(b, hkv, D, device="cuda:0", generator=gen)
    return kraw, kval, vraw, vval, tables, q, tk, tv


def grid(dtype, x, scale):
    if dtype == "bf16":
        return x.to(torch.bfloat16).float()
    return torch.from_numpy(oracle.round_fp8(x.cpu().numpy(), scale)).cuda()


def decode(dtype, kp, vp, tables, q, tk, tv, shape):
    lengths = torch.tensor(LENGTHS, dtype=torch.int32, device="cuda:0")
    t = torch.from_numpy(tables).cuda()
    ws = hx.decode_workspace(q.shape[0], q.shape[1], shape[1], tables.shape[1])
    out = torch.empty_like(q)
    scales = dict(k_scale=KS, v_scale=VS) if dtype == "fp8" else {}
    hx.paged_decode_attention(q, kp.data_ptr(), vp.data_ptr(), t, lengths, tk, tv, out, ws,
                              pool_shape=shape, page_dtype=dtype, **scales)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("dtype", ["bf16", "fp8"])
@pytest.mark.parametrize("hq,hkv", [(3, 3), (4, 2), (8, 2), (16, 2)])
@pytest.mark.parametrize("special", [False, True])
def test_decode_pages_match_fp32_kernel(device, dtype, hq, hkv, special):
    kraw, kval, vraw, vval, tables, q, tk, tv = build(dtype, hq, hkv, 7 * hq + hkv)
    nan = torch.full((), float("nan"), dtype=torch.bfloat16, device="cuda:0")
    for b, n in enumerate(LENGTHS):  # rows past the history hold NaN
        if n % P:
            page = int(tables[b, n // P])
            for raw in (kraw, vraw):
                raw[page, :, n % P:] = nan if dtype == "bf16" else 0x7F
    if special:
        # Query entries whose split has zero terms, against infinite keys and
        # values (bf16) and NaN ones, in the first, a middle and the last page.
        q[:, :, ::2] = torch.round(q[:, :, ::2])
        inf = torch.tensor([float("inf"), -float("inf")], device="cuda:0").to(torch.bfloat16)
        for b, (page, row) in {4: (0, 3), 9: (5, 15), 11: (15, 0), 13: (62, 7)}.items():
            phys = int(tables[b, page])
            if dtype == "bf16":
                kraw[phys, 0, row, 6] = inf[b % 2]
                vraw[phys, -1, (row + 1) % 8, 9] = inf[(b + 1) % 2]
            else:
                kraw[phys, 0, row, 6] = 0x7F
        vraw[int(tables[7, 1]), 0, 2, 40] = nan if dtype == "bf16" else 0xFF
        tv[12, 0, 5] = float("nan")
    shape = tuple(kraw.shape)
    got = decode(dtype, kraw, vraw, tables, q, tk, tv, shape)
    kf, vf = kval(KS), vval(VS)
    tkr, tvr = grid(dtype, tk, KS), grid(dtype, tv, VS)
    want = decode("f32", kf, vf, tables, q, tkr, tvr, shape)
    np.testing.assert_allclose(got.cpu().numpy(), want.cpu().numpy(), atol=ATOL, rtol=RTOL)
    assert bool(torch.isnan(got).any()) == special
    if not special:
        ref = oracle.batched_decode(q.cpu().numpy(), np.nan_to_num(kf.cpu().numpy()),
                                    np.nan_to_num(vf.cpu().numpy()), tables.astype(np.uint32),
                                    np.array(LENGTHS, np.int32), tkr.cpu().numpy(),
                                    tvr.cpu().numpy(), threads=8)
        np.testing.assert_allclose(got.cpu().numpy(), ref, atol=ATOL, rtol=RTOL)


@pytest.mark.parametrize("dtype", ["bf16", "fp8"])
@pytest.mark.parametrize("hq", [2, 8, 16])
def test_unaligned_rows_give_the_same_bits(device, dtype, hq):
    """DecodeBatch takes query and tail rows at any 4-byte address."""
    cache = hx.PagedKvCache(1, 2, D, P, 64, page_dtype=dtype)
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(3)
    seqs = []
    for n in (0, 5, 33, 200):
        s = cache.create_sequence()
        if n:
            cache.append_layer_major(s, [torch.randn(2, n, D, device="cuda:0", generator=gen)],
                                     [torch.randn(2, n, D, device="cuda:0", generator=gen)])
        seqs.append(s)
    batch = hx.DecodeBatch(cache, seqs, hq, max_tokens=256)
    batch.prepare()
    rows = [torch.randn(4, h, D, device="cuda:0", generator=gen) for h in (hq, 2, 2)]
    outs = []
    for shift in (0, 1):
        moved = []
        for r in rows:
            flat = torch.zeros(r.numel() + 4, device="cuda:0")
            flat[shift:shift + r.numel()] = r.reshape(-1)
            moved.append(flat[shift:shift + r.numel()].view(r.shape))
        out = torch.empty(4, hq, D, device="cuda:0")
        batch.attention_layer(0, *moved, out)
        torch.cuda.synchronize()
        outs.append(out)
    assert torch.isfinite(outs[0]).all()
    assert torch.equal(outs[0], outs[1])
    batch.close()
    cache.close()
