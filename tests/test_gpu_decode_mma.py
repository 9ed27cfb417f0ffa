"""Batched decode of bf16 and fp8 pages on the matrix cores, where it can go
wrong: histories around the 16-token page, empty histories, every query
group, rows of a partly filled page that hold NaN, infinite and NaN page
elements, rows that are not 16-byte aligned; ranges of one page, of several
pages over several units and of more than 64 pages a wavefront.

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


def decode(dtype, kp, vp, tables, q, tk, tv, shape, lengths=LENGTHS):
    lengths = torch.tensor(lengths, dtype=torch.int32, device="cuda:0")
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


def unit_query():
    """q whose scaled value is 1.0 exactly: its split into bf16 terms has zeros."""
    scale = np.float32(1.4426950408889634) / np.sqrt(np.float32(D))
    q = np.float32(1) / scale
    near = [q, np.nextafter(q, np.float32(0)), np.nextafter(q, np.float32(100))]
    return float(next(x for x in near if np.float32(x * scale) == 1))


def range_lengths(dtype, group, hkv, pages_per_wave):
    """Lengths of a batch whose wavefronts take exactly `pages_per_wave` pages."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    waves = min(4096, cus * 4 * (2 if dtype == "bf16" or group == 8 else 3))
    per_head = pages_per_wave * waves // hkv  # a tail row counts as a page
    lengths = []
    if pages_per_wave > 64:
        lengths = [((per_head - 40) // n - 1) * P - n for n in (3, 2, 7)]  # 3, 2 and 7 short of a page
    left = per_head - sum((n + P - 1) // P + 1 for n in lengths)
    rng = np.random.default_rng(pages_per_wave)
    while left > 0:
        n = int(rng.choice(LENGTHS))
        n = n if (n + P - 1) // P + 1 <= left else (left - 1) * P
        lengths.append(n)
        left -= (n + P - 1) // P + 1
    total = hkv * sum((n + P - 1) // P + 1 for n in lengths)
    assert -(-total // waves) == pages_per_wave and total > (pages_per_wave - 1) * waves
    return lengths


@pytest.mark.parametrize("dtype", ["bf16", "fp8"])
@pytest.mark.parametrize("group", [1, 2, 4, 8])
@pytest.mark.parametrize("pages_per_wave", [4, 65])
def test_ranges_of_several_pages(device, dtype, group, pages_per_wave):
    """Ranges over several pages and units, and of more pages than one set of
    descriptors holds, special values in the middle of some.  The sequences
    share physical pages, except the ones with special values."""
    hkv, spare = 4, 90
    lengths = range_lengths(dtype, group, hkv, pages_per_wave)
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(group)
    kraw, kval = pages(dtype, (spare + 5, hkv, P, D), gen)
    vraw, vval = pages(dtype, (spare + 5, hkv, P, D), gen)
    rng = np.random.default_rng(group)
    tables = rng.integers(0, spare, (len(lengths), max(lengths) // P + 2)).astype(np.int32)
    b = len(lengths)
    q = torch.randn(b, hkv * group, D, device=device, generator=gen)
    tk = torch.randn(b, hkv, D, device=device, generator=gen)
    tv = torch.randn(b, hkv, D, device=device, generator=gen)
    nan = torch.full((), float("nan"), dtype=torch.bfloat16, device=device)
    inf = float("inf")
    long = sorted(range(b), key=lambda i: -lengths[i])[:5]
    for i, s in enumerate(long):  # one page of its own in the middle
        tables[s, lengths[s] // P // 2] = spare + i
    vraw[spare, 1, 5, 7] = nan if dtype == "bf16" else 0x7F
    kraw[spare + 1, 2, 0, 0] = nan if dtype == "bf16" else 0xFF
    q[long[2], :group, 100] = float("nan")
    if dtype == "bf16":
        # An infinite key that takes all the weight, infinite values of keys
        # that all weigh the same, in a page and in the tail row.
        kraw[spare + 3, 0, 9, 6] = inf
        q[long[3], :, 6] = unit_query()
        vraw[spare + 4, 3, 15, 77] = -inf
        q[long[4]] = 0.0
        tv[long[4], 1, 2] = inf
    shape = tuple(kraw.shape)
    got = decode(dtype, kraw, vraw, tables, q, tk, tv, shape, lengths)
    want = decode("f32", kval(KS), vval(VS), tables, q, grid(dtype, tk, KS), grid(dtype, tv, VS),
                  shape, lengths)
    np.testing.assert_allclose(got.cpu().numpy(), want.cpu().numpy(), atol=ATOL, rtol=RTOL)
    nans = torch.isnan(got).view(b, hkv, group, D)
    assert int(nans[long[0]].sum()) == group and bool(nans[long[1], 2].all())
    assert bool(nans[long[2], 0].all()) and int(nans.sum()) == group * (1 + 2 * D)
    assert int(torch.isinf(got).sum()) == (2 * group if dtype == "bf16" else 0)


@pytest.mark.parametrize("dtype", ["bf16", "fp8"])
def test_special_value_costs_no_multiple_of_the_layer(device, dtype):
    """One NaN or infinite element slows the launch by less than 4 times (1.0
    and 1.7 times measured; 9 to 10 when ranges were recomputed row by row)."""
    hkv, cols = 8, 512
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(1)
    lengths = [cols * P - 40] * 16
    kraw, _ = pages(dtype, (cols, hkv, P, D), gen)
    vraw, _ = pages(dtype, (cols, hkv, P, D), gen)
    q, tk, tv = (torch.randn(16, h, D, device=device, generator=gen) for h in (32, hkv, hkv))
    tables = torch.arange(cols, dtype=torch.int32, device=device).repeat(16, 1)
    tables[9] = tables[9].flip(0)
    lens = torch.tensor(lengths, dtype=torch.int32, device=device)
    ws = hx.decode_workspace(16, 32, hkv, cols)
    out = torch.empty_like(q)
    scales = dict(k_scale=KS, v_scale=VS) if dtype == "fp8" else {}
    special = [float("nan")] + ([float("inf")] if dtype == "bf16" else [])

    def layer_us():
        times = []
        for _ in range(12):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            hx.paged_decode_attention(q, kraw.data_ptr(), vraw.data_ptr(), tables, lens, tk, tv,
                                      out, ws, pool_shape=tuple(kraw.shape), page_dtype=dtype,
                                      **scales)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b) * 1e3)
        return float(np.median(times))

    clean = layer_us()
    for x in special:
        kraw[100, 3, 7, 9] = x if dtype == "bf16" else 0x7F
        assert layer_us() < 4 * clean


@pytest.mark.parametrize("dtype", ["bf16", "fp8"])
@pytest.mark.parametrize("hq", [2, 8, 16])
@pytest.mark.parametrize("special", [False, True])
def test_unaligned_rows_give_the_same_bits(device, dtype, hq, special):
    """DecodeBatch takes query, tail and output rows at any 4-byte address."""
    cache = hx.PagedKvCache(1, 2, D, P, 64, page_dtype=dtype)
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(3)
    seqs = []
    for n in (0, 5, 33, 200):
        s = cache.create_sequence()
        if n:
            k = torch.randn(2, n, D, device="cuda:0", generator=gen)
            v = torch.randn(2, n, D, device="cuda:0", generator=gen)
            if special and n == 33:
                v[0, 20, 5], v[1, 3, 8] = float("nan"), float("inf")
            cache.append_layer_major(s, [k], [v])
        seqs.append(s)
    batch = hx.DecodeBatch(cache, seqs, hq, max_tokens=256)
    batch.prepare()
    rows = [torch.randn(4, h, D, device="cuda:0", generator=gen) for h in (hq, 2, 2)]
    if special:
        rows[0][2] = 0.0  # every key weighs the same: zero terms against infinite values
        rows[2][3, 1, 4], rows[1][1, 0, 3] = float("inf"), float("nan")
    outs = []
    for shift in (0, 1):
        moved = []
        for r in rows:
            flat = torch.zeros(r.numel() + 4, device="cuda:0")
            flat[shift:shift + r.numel()] = r.reshape(-1)
            moved.append(flat[shift:shift + r.numel()].view(r.shape))
        out = torch.empty(4 * hq * D + 4, device="cuda:0")[shift:shift + 4 * hq * D]
        batch.attention_layer(0, *moved, out.view(4, hq, D))
        torch.cuda.synchronize()
        outs.append(out.clone())
    # (The sign of a NaN is not part of the result.)
    bits = [torch.nan_to_num(o, nan=12345.0, posinf=1e30, neginf=-1e30) for o in outs]
    assert torch.equal(bits[0], bits[1])
    assert bool(torch.isnan(outs[0]).any()) == special
    assert bool(torch.isinf(outs[0]).any()) == (special and dtype == "bf16")
    batch.close()
    cache.close()
