"""The paged attention's tiled form (many rows per sequence) and its grouped 16-row form against a dense float64
attention: one and two row tiles per wave, tiles cut by sequences and by prefixes, window and kept-prefix edges, score
modifiers."""
import math

import pytest
import torch

from butterfly_amd import ops

F64 = torch.float64
BS = 32


def dense(q, k, v, pos, scale, window, keep, sink, slopes, chunk, qt, cap=0.0, logs=None):
    """q [n, H, D] at positions pos over k [L, G, D], v [L, G, Dv] of one sequence."""
    H, G = q.shape[1], k.shape[1]
    i, j = pos[:, None], torch.arange(k.shape[0])[None]
    low = i - i % chunk if chunk else i - window + 1
    see = (j <= i) & ((j >= low) | (j < keep))
    out = torch.empty(q.shape[0], H, v.shape[2], dtype=F64)
    for h in range(H):
        g = h // (H // G)
        s = q[:, h] @ k[:, g].T * scale
        if qt:
            s = s * (1 + qt[0] * torch.log(torch.floor((i + 1) / qt[1]) + 1))
        if cap:
            s = cap * torch.tanh(s / cap)
        if logs is not None:
            s = s - slopes[h] * torch.log1p(logs[h] * (i - j).clamp(min=0))
        elif slopes is not None:
            s = s - slopes[h] * (i - j)
        s = s.masked_fill(~see, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[h].expand(len(s), 1)], 1)
        out[:, h] = torch.softmax(s, -1)[:, :k.shape[0]] @ v[:, g]
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,G,D,Dv,window,keep,mods,seqs", [
    (16, 4, 128, 128, 1 << 30, 0, "", [(0, 700), (0, 1501)]),         # two row tiles per wave; a ragged last tile
    (16, 4, 128, 128, 300, 5, "sink", [(0, 2400), (0, 33)]),          # window edges and a kept prefix, pages skipped
    (16, 4, 128, 128, 64, 40, "sink", [(37, 1100), (1000, 1100)]),    # chunks over a cached prefix, a kept prefix of two pages
    (8, 2, 128, 128, 300, 0, "slope temp", [(0, 300), (77, 411)]),    # one row tile per wave; distance bias, temperature
    (16, 16, 64, 64, 100, 0, "chunk", [(0, 640)]),                    # no grouping, chunks instead of a window
    (32, 2, 128, 128, 512, 0, "slope", [(0, 1030), (5, 1000)]),       # sixteen query heads per key head, two tiles per wave
    (16, 4, 128, 128, 40, 3, "sink", [(700, 1), (31, 1), (32, 1), (0, 1)]),   # decoded rows: the 16-row form
    (16, 4, 128, 128, 1 << 30, 0, "cap", [(0, 700), (0, 1501)]),      # capped scores, two row tiles per wave
    (8, 2, 128, 128, 200, 3, "cap slope log sink", [(0, 300), (77, 411)]),    # a cap and the logarithmic distance bias, one row tile
    (16, 16, 64, 64, 1 << 30, 0, "slope log temp", [(3, 640)]),
    (8, 8, 32, 32, 100, 0, "", [(0, 333), (40, 200)]),                # the other head sizes
    (8, 2, 96, 96, 1 << 30, 0, "sink", [(0, 333), (40, 200)]),
    (8, 2, 128, 256, 64, 5, "", [(0, 333), (40, 200)]),
    (4, 2, 192, 192, 1 << 30, 0, "cap", [(0, 333), (40, 200)]),
    (6, 1, 256, 192, 90, 0, "", [(0, 333), (40, 200)]),
    (4, 2, 256, 256, 1 << 30, 0, "slope log", [(0, 333), (40, 200)]),
    (16, 4, 64, 64, 1 << 30, 0, "slope log", [(3, 1100), (0, 900)]),  # bf16: rows enough for the tiled form at these sizes
    (16, 16, 64, 64, 100, 0, "chunk", [(0, 2600)]),
    (16, 4, 32, 32, 500, 3, "", [(0, 4150)]),
    (8, 2, 96, 96, 1 << 30, 0, "sink", [(0, 700), (40, 400)]),
    (8, 2, 128, 256, 64, 5, "", [(0, 700), (40, 400)]),
    (4, 2, 192, 192, 1 << 30, 0, "cap", [(0, 1100), (40, 400)]),
    (6, 1, 256, 192, 90, 0, "", [(0, 700), (40, 300)]),
    (4, 2, 256, 256, 1 << 30, 0, "slope log", [(0, 1100), (40, 400)]),
    (16, 4, 128, 128, 1 << 30, 0, "sink", [(400 + 31 * i, 1) for i in range(17)]),      # decoded rows: grouped tiles, pages split
    (16, 4, 128, 128, 1 << 30, 0, "", [(900, 9), (40, 60), (0, 3)]),                    # tiles of one head
])
def test_paged_tiles_match_dense_attention(dt, H, G, D, Dv, window, keep, mods, seqs):
    g = torch.Generator().manual_seed(H + D + window % 1000)
    bf = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)                  # noqa: E731
    dev, scale = "cuda", 2.0 / math.sqrt(D)
    sink = torch.randn(H, generator=g) if "sink" in mods else None
    slopes = 0.5 ** torch.linspace(2, 9, H) if "slope" in mods else None
    qt = (0.3, 50) if "temp" in mods else None
    chunk = 90 if "chunk" in mods else 0
    cap = 3.0 if "cap" in mods else 0.0
    logs = torch.linspace(0.1, 2, H) if "log" in mods else None
    need = [(s + n + BS - 1) // BS for s, n in seqs]
    order = torch.randperm(sum(need), generator=g)
    kc = torch.zeros(sum(need), G, BS, D, dtype=torch.bfloat16)
    vc = torch.zeros(sum(need), G, Dv, BS, dtype=torch.bfloat16)
    tables = torch.zeros(len(seqs), max(need) + 2, dtype=torch.int32)
    qs, want, at = [], [], 0
    for s, (start, n) in enumerate(seqs):
        pages = order[at:at + need[s]]
        at += need[s]
        tables[s, :need[s]] = pages.int()
        q, k, v = bf(n, H, D), bf(need[s] * BS, G, D), bf(need[s] * BS, G, Dv)      # (pages hold values past the last row)
        kc[pages] = k.view(-1, BS, G, D).transpose(1, 2)
        vc[pages] = v.view(-1, BS, G, Dv).permute(0, 2, 3, 1)
        qs.append(q)
        L = start + n
        want.append(dense(q.to(F64), k[:L].to(F64), v[:L].to(F64), torch.arange(start, L), scale, window, keep, sink,
                          slopes, chunk, qt, cap, logs))
    cu = torch.tensor([sum(n for _, n in seqs[:i]) for i in range(len(seqs) + 1)], dtype=torch.int32, device=dev)
    pos = torch.cat([torch.arange(s, s + n) for s, n in seqs]).int().to(dev)
    got = ops.attn_window_paged(torch.cat(qs).to(dev, dt), kc.to(dev, dt), vc.to(dev, dt), tables.to(dev), cu, pos, scale, window, keep,
                                None if sink is None else sink.to(dev), chunk=chunk, q_temp=qt, softcap=cap,
                                dist_bias=None if slopes is None else (slopes.to(dev), None if logs is None else logs.to(dev)))
    # bf16: weights rounded to bf16 (2^-9 each, together at most 2^-9 of the largest value), the output rounded once more;
    # f32: scores of up to 20 with a few eps (6e-8) of their size, which is the relative error of a weight
    err = (got.cpu().to(F64) - torch.cat(want)).abs().max()
    assert err < (2.0 ** -8 if dt == torch.bfloat16 else 1e-5) * vc.float().abs().max() + (1e-3 if dt == torch.bfloat16 else 0)


@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hkv,seqs", [
    (32, 8, [(2000, 64)]),               # few rows: one row tile per wave, pages split over workgroups
    (32, 8, [(3001, 700)]),              # two row tiles per wave, split
    (64, 8, [(100, 40), (0, 33)]),       # too few keys to split; a chunk without a prefix
    (8, 8, [(31, 130), (1500, 257)]),    # no grouping
    (32, 4, [(640, 15)]),                # fewer than 128 pairs: the 16-row kernels
])
def test_chunks_over_a_cached_prefix(Hq, Hkv, seqs):
    g = torch.Generator().manual_seed(Hq + len(seqs))
    bf = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)                  # noqa: E731
    dev, D, scale = "cuda", 128, 1.5 / math.sqrt(128)
    need = [(s + n + BS - 1) // BS for s, n in seqs]
    order = torch.randperm(sum(need), generator=g)
    kc, vc = bf(sum(need), Hkv, BS, D), bf(sum(need), Hkv, D, BS)
    tables = torch.zeros(len(seqs), max(need) + 3, dtype=torch.int32)
    qs, want, at = [], [], 0
    for s, (start, n) in enumerate(seqs):
        pages = order[at:at + need[s]]
        at += need[s]
        tables[s, :need[s]] = pages.int()
        k = kc[pages].transpose(1, 2).reshape(-1, Hkv, D)[:start + n]
        v = vc[pages].permute(0, 3, 1, 2).reshape(-1, Hkv, D)[:start + n]
        qs.append(bf(n, Hq, D))
        want.append(dense(qs[-1].to(F64), k.to(F64), v.to(F64), torch.arange(start, start + n), scale, 1 << 30, 0, None, None, 0,
                          None))
    cu = torch.tensor([sum(n for _, n in seqs[:i]) for i in range(len(seqs) + 1)], dtype=torch.int32, device=dev)
    pos = torch.cat([torch.arange(s, s + n) for s, n in seqs]).int().to(dev)
    wide = torch.zeros(len(pos), Hq + 2, D, dtype=torch.bfloat16, device=dev)        # strided query and output rows
    wide[:, :Hq] = torch.cat(qs).to(dev)
    out = torch.zeros_like(wide)
    ops.attn_prefill_paged(wide[:, :Hq], kc.to(dev), vc.to(dev), tables.to(dev), cu, pos, max(n for _, n in seqs), scale,
                           out=out[:, :Hq])
    err = (out[:, :Hq].cpu().to(F64) - torch.cat(want)).abs().max()
    assert err < 2.0 ** -8 * vc.float().abs().max() + 1e-3
    assert not out[:, Hq:].any()


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,D,Dv,window,keep,seqs", [
    (16, 4, 128, 128, 512, 4, [(0, 31), (0, 32), (0, 33), (20, 1100), (600, 65)]),      # two pages a step, an odd number of them last
    (16, 4, 128, 128, 1 << 30, 0, [(1000 + i, 8) for i in range(65)]),      # more sequences than lanes, 31 to 33 pages in splits
    (32, 8, 128, 128, 511, 70, [(0, 300), (1000, 200), (3, 40)]),             # one page a step
    (6, 1, 256, 192, 1 << 30, 0, [(0, 140)] * 3 + [(33, 200)]),               # pages of uneven segments
    (16, 4, 128, 128, 700, 4, [(1 + 13 * i, 1) for i in range(130)]),        # decoded rows of 130 sequences
    (8, 2, 128, 128, 512, 40, [(2000, 1)]), (16, 1, 256, 192, 1 << 30, 0, [(300, 1), (5, 1), (0, 1)]),      # most splits without a page
    (16, 4, 128, 128, 1 << 30, 0, [(900, 2), (32, 0), (40, 1), (500, 1)]),    # as many rows as sequences, but not one each
    (48, 2, 128, 128, 1 << 30, 0, [(900, 3), (32, 0), (32, 0), (7, 1)]),      # tiles of 24 rows a token, one of them short
    (16, 4, 64, 256, 1024, 0, [(1000 + 37 * i, 1) for i in range(20)]), (16, 4, 128, 128, 224, 0, [(900, 1), (100, 1)]),
])
def test_extended_tiles_match_dense_attention(H, G, D, Dv, window, keep, seqs):
    g = torch.Generator().manual_seed(H + D + len(seqs))
    bf = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)                  # noqa: E731
    dev, scale = "cuda", 2.0 / math.sqrt(D)
    need = [(s + n + BS - 1) // BS for s, n in seqs]
    order = torch.randperm(sum(need), generator=g)
    kc, vc = bf(sum(need), G, BS, D), bf(sum(need), G, Dv, BS)
    tables = torch.zeros(len(seqs), max(need) + 2, dtype=torch.int32)
    qs, want, at = [], [], 0
    for s, (start, n) in enumerate(seqs):
        pages = order[at:at + need[s]]
        at += need[s]
        tables[s, :need[s]] = pages.int()
        k = kc[pages].transpose(1, 2).reshape(-1, G, D)[:start + n]
        v = vc[pages].permute(0, 3, 1, 2).reshape(-1, G, Dv)[:start + n]
        qs.append(bf(n, H, D))
        want.append(dense(qs[-1].to(F64), k.to(F64), v.to(F64), torch.arange(start, start + n), scale, window, keep, None, None, 0,
                          None))
    cu = torch.tensor([sum(n for _, n in seqs[:i]) for i in range(len(seqs) + 1)], dtype=torch.int32, device=dev)
    pos = torch.cat([torch.arange(s, s + n) for s, n in seqs]).int().to(dev)
    got = ops.attn_window_paged(torch.cat(qs).to(dev), kc.to(dev), vc.to(dev), tables.to(dev), cu, pos, scale, window, keep, None,
                                dv_out=Dv)
    err = (got.cpu().to(F64).view(-1, H, Dv) - torch.cat(want)).abs().max()
    assert err < 2.0 ** -8 * vc.float().abs().max() + 1e-3      # weights and output rounded to bf16


@pytest.mark.gpu
def test_pages_that_no_row_of_a_wave_sees_do_not_count():
    """Rows up to a page's end beside rows behind it in one workgroup, the next page's values no numbers."""
    g = torch.Generator().manual_seed(1)
    H, G, D, start, n, dev = 16, 4, 128, 20, 600, "cuda"
    need = (start + n + BS - 1) // BS
    kc, vc = (torch.randn(need, G, *s, generator=g).bfloat16() for s in ((BS, D), (D, BS)))
    q, cu = torch.randn(n, H, D, generator=g).bfloat16().to(dev), torch.tensor([0, n], dtype=torch.int32, device=dev)
    tables, pos = torch.arange(need, dtype=torch.int32, device=dev)[None], torch.arange(start, start + n).int().to(dev)
    run = lambda v: ops.attn_window_paged(q, kc.to(dev), v.to(dev), tables, cu, pos, 0.1, 1 << 30, 0, None, dv_out=D)      # noqa: E731
    clean = run(vc)
    bad = vc.clone()
    bad[1] = float("nan")
    got = run(bad)
    first = 8 * ((BS - start) // 8)      # (a wave has 32 rows: 8 tokens of 4 heads)
    assert first and torch.equal(got[:first], clean[:first]) and got[BS - start:].isnan().all()


@pytest.mark.gpu
@pytest.mark.parametrize("start,n,rest", [(2000, 64, 5), (5000, 300, 40), (100, 40, 3)])      # pages split over workgroups, and not
def test_rows_of_no_sequence_stay(start, n, rest):
    """Rows before the first and after the last sequence keep what the output held, also where partial results are merged."""
    g = torch.Generator().manual_seed(n)
    H, G, D, dev = 32, 8, 128, "cuda"
    need = (start + n + BS - 1) // BS
    kc, vc = (torch.randn(need, G, *s, generator=g).bfloat16().to(dev) for s in ((BS, D), (D, BS)))
    q = torch.randn(2 + n + rest, H, D, generator=g).bfloat16().to(dev)
    tables = torch.arange(need, dtype=torch.int32, device=dev)[None]
    pos = torch.cat([torch.zeros(2), torch.arange(start, start + n), torch.zeros(rest)]).int().to(dev)
    cu = torch.tensor([2, 2 + n], dtype=torch.int32, device=dev)
    out = torch.full_like(q, 3.0)
    ops.attn_prefill_paged(q, kc, vc, tables, cu, pos, n, 0.1, out=out)
    assert (out[:2] == 3).all() and (out[2 + n:] == 3).all()
    alone = ops.attn_prefill_paged(q[2:2 + n], kc, vc, tables, cu - 2, pos[2:2 + n], n, 0.1)
    # (weights and outputs rounded to bf16, the sums of another number of splits)
    assert (out[2:2 + n].float() - alone.float()).abs().max() < 2.0 ** -7 * vc.float().abs().max()


@pytest.mark.gpu
@pytest.mark.parametrize("start,n,nseq", [(32, 60, 5), (0, 100, 1), (196, 60, 3), (197, 60, 3)])      # to 256 positions, and one more
def test_a_known_context_changes_no_result(start, n, nseq):
    g = torch.Generator().manual_seed(start + n)
    H, G, D, dev = 32, 8, 128, "cuda"
    per = (start + n + BS - 1) // BS
    kc, vc = (torch.randn(nseq * per, G, *s, generator=g).bfloat16().to(dev) for s in ((BS, D), (D, BS)))
    tables = torch.randperm(nseq * per, generator=g).int().view(nseq, per).to(dev)
    q = torch.randn(nseq * n, H, D, generator=g).bfloat16().to(dev)
    cu = torch.arange(0, nseq * n + 1, n, dtype=torch.int32, device=dev)
    pos = torch.arange(start, start + n).int().repeat(nseq).to(dev)
    plain, known = (ops.attn_prefill_paged(q, kc, vc, tables, cu, pos, n, 0.1, max_ctx=c).float() for c in (0, start + n))
    assert (plain - known).abs().max() < 2.0 ** -7 * vc.float().abs().max()      # (weights and outputs rounded to bf16 in both)


@pytest.mark.skipif(not ops.load_library(), reason="kernel library not built")
def test_scratch_of_split_pages():
    """Scratch only where workgroups share a tile's pages: few tiles, enough pages; 64 MB at most."""
    need = lambda *a, ctx=0: torch.ops.bfly.attn_prefill_paged_scratch(*a, ctx)        # noqa: E731
    row = 32 * 130
    assert need(64, 1, 32, 8, 128, 250) == 8 * 64 * row          # a chunk over a long prefix
    assert need(64, 1, 32, 8, 128, 20) == 0                      # too few pages to share
    assert need(4000, 1, 32, 8, 128, 250) == 0                   # tiles enough
    assert need(15, 1, 32, 4, 128, 250) == 0 and need(0, 1, 32, 8, 128, 250) == 0      # not on the tiled kernel
    assert need(64, 1, 32, 8, 128, 250, ctx=256) == 0 and need(64, 1, 32, 8, 128, 250, ctx=257) > 0      # nor short contexts
    for rows in (16, 100, 500, 900, 2000, 8000):
        for nseq in (1, 3, 16):
            for Hq, Hkv in ((32, 8), (64, 8), (8, 8), (64, 64)):
                n = need(rows, nseq, Hq, Hkv, 128, 4096)
                assert n <= 1 << 24 and n % (rows * Hq * 130) == 0 and n // (rows * Hq * 130) in (0, *range(2, 9))


@pytest.mark.gpu
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("Hq,Hkv,ctx,max_ctx", [
    (32, 8, [1, 31, 32, 33, 257, 700], 1024),      # split contexts, eight waves; most waves without a page
    (8, 1, [40, 3000], 3008),                      # eight rows, split
    (16, 8, list(range(5, 200, 8)), 256),          # 200 pairs: whole contexts, eight waves
    (64, 8, [100 + i for i in range(48)], 160),    # 384 pairs: four waves
    (16, 1, [65, 1], 96),                          # sixteen query heads on one
])
def test_decode_waves_and_splits(fp8, Hq, Hkv, ctx, max_ctx):
    g = torch.Generator().manual_seed(Hq + len(ctx))
    D, B, scale = 128, len(ctx), 1.5 / math.sqrt(128)
    dt = torch.float8_e4m3fn if fp8 else torch.bfloat16
    need = [(c + BS - 1) // BS for c in ctx]
    kc, vc = torch.randn(sum(need), Hkv, BS, D, generator=g).to(dt), torch.randn(sum(need), Hkv, D, BS, generator=g).to(dt)
    q = torch.randn(B, Hq, D, generator=g).bfloat16()
    tables = torch.zeros(B, (max_ctx + BS - 1) // BS, dtype=torch.int32)
    order, at, want = torch.randperm(sum(need), generator=g), 0, []
    for b, c in enumerate(ctx):
        pages = order[at:at + need[b]]
        at += need[b]
        tables[b, :need[b]] = pages.int()
        k = kc.float()[pages].transpose(1, 2).reshape(-1, Hkv, D)[:c].to(F64)
        v = vc.float()[pages].permute(0, 3, 1, 2).reshape(-1, Hkv, D)[:c].to(F64)
        want.append(dense(q[b:b + 1].to(F64), k, v, torch.tensor([c - 1]), scale, 1 << 30, 0, None, None, 0, None))
    got = ops.attn_decode(q.cuda(), kc.cuda(), vc.cuda(), tables.cuda(), torch.tensor(ctx, dtype=torch.int32).cuda(), scale, max_ctx)
    err = (got.cpu().to(F64) - torch.cat(want)).abs().max()
    assert err < 2.0 ** -8 * vc.float().abs().max() + 1e-3      # weights and output rounded to bf16


@pytest.mark.gpu
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("Hq,Hkv,ctx,max_ctx", [
    (8, 8, [0, 1, 0, 31, 32, 33, 4096, 0], 4096),              # empty sequences, one of many pieces
    (32, 8, [2047, 5, 5, 5, 5, 5, 5, 5, 5, 5, 5, 2048, 700, 1, 256, 257], 2048),     # more segments in a piece than wait in LDS
    (16, 1, [3000], 1 << 18),                                   # sixteen query heads on one, a single sequence far below its bound
    (16, 8, [30 + 11 * i for i in range(64)], 1536),            # the most sequences of one register
    (4, 4, [1 + 23 * i % 1500 for i in range(65)], 1536),       # one more than that
    (4, 4, [0] * 200 + [1600] + [0] * 54 + [9], 2048),          # the most there are
    (24, 3, [0] * 90, 1536),                                    # nothing at all
])
def test_decode_pages_end_to_end(fp8, Hq, Hkv, ctx, max_ctx):
    g = torch.Generator().manual_seed(Hq + len(ctx))
    D, B, scale = 128, len(ctx), 1.5 / math.sqrt(128)
    assert torch.ops.bfly.attn_decode_part_rows(B, Hq, Hkv, max_ctx, 0) == (256 // Hkv + B) * Hq
    dt = torch.float8_e4m3fn if fp8 else torch.bfloat16
    need = [(c + BS - 1) // BS for c in ctx]
    n = sum(need)
    kc, vc = torch.randn(n + 1, Hkv, BS, D, generator=g).to(dt), torch.randn(n + 1, Hkv, D, BS, generator=g).to(dt)
    q = torch.randn(B, Hq, D, generator=g).bfloat16()
    tables = torch.full((B, (max_ctx + BS - 1) // BS), n, dtype=torch.int32)
    order, at, want = torch.randperm(n, generator=g), 0, []
    for b, c in enumerate(ctx):
        pages = order[at:at + need[b]]
        at += need[b]
        tables[b, :need[b]] = pages.int()
        if not c:
            want.append(torch.zeros(1, Hq, D, dtype=F64))
            continue
        k = kc.float()[pages].transpose(1, 2).reshape(-1, Hkv, D)[:c].to(F64)
        v = vc.float()[pages].permute(0, 3, 1, 2).reshape(-1, Hkv, D)[:c].to(F64)
        want.append(dense(q[b:b + 1].to(F64), k, v, torch.tensor([c - 1]), scale, 1 << 30, 0, None, None, 0, None))
    run = lambda kk, vv, part=0: ops.attn_decode(q.cuda(), kk.cuda(), vv.cuda(), tables.cuda(),  # noqa: E731
                                                 torch.tensor(ctx, dtype=torch.int32).cuda(), scale, max_ctx, part)
    got = run(kc, vc)
    err = (got.cpu().to(F64) - torch.cat(want)).abs().max()
    assert err < 2.0 ** -8 * vc.float().abs().max() + 1e-3      # weights and output rounded to bf16
    if n > 1 and not fp8:                                       # values that are no numbers stay in their sequence
        longest = max(range(B), key=lambda b: ctx[b])
        rest = [b for b in range(B) if b != longest]
        page = tables[longest, 0].item()
        bad = vc.clone()
        bad[page] = float("nan")
        poisoned = run(kc, bad)
        assert poisoned[longest].isnan().all()
        assert torch.equal(poisoned[rest], got[rest])
        bad = kc.clone()                                        # and keys: a page that is all of a wave's share has no maximum
        bad[page] = float("nan")
        for part in (0, max_ctx // 8, max_ctx):                 # (and with a workgroup per split, eight and one)
            poisoned, clean = run(bad, vc, part), run(kc, vc, part)
            assert poisoned[longest].isnan().all(), part
            some = [b for b in rest if ctx[b] or not part]      # (a workgroup per split leaves the rows of empty sequences)
            assert torch.equal(poisoned[some], clean[some])


@pytest.mark.gpu
@pytest.mark.parametrize("B,Hkv", [(128, 8), (16, 8), (1, 8), (3, 128)])
def test_decode_with_buffers_of_a_workgroup_per_split(B, Hkv):
    """The operator takes the buffers that its split sizes ask for, none at all for one split, also where pages would run end to end."""
    max_ctx, D, G = 2048 if B > 1 else 1 << 18, 128, 4
    g = torch.Generator(device="cuda").manual_seed(B)
    ctx = torch.randint(1, 300, (B,), generator=g, device="cuda").int()
    kc, vc = (torch.randn(40, Hkv, *s, generator=g, device="cuda").bfloat16() for s in ((BS, D), (D, BS)))
    q = torch.randn(B, Hkv * G, D, generator=g, device="cuda").bfloat16()
    tables = torch.randint(0, 40, (B, max_ctx // BS), generator=g, device="cuda").int()
    op = torch.ops.bfly
    assert op.attn_decode_part_rows(B, Hkv * G, Hkv, max_ctx, 0) == (max(1, 256 // Hkv) + B) * Hkv * G
    part = op.attn_decode_part_tokens(B, Hkv, max_ctx)
    ns = op.attn_decode_splits(max_ctx, part)
    bufs = [torch.empty(B * Hkv * ns * 16 * n, device="cuda") for n in (D, 2)] if ns > 1 else [None, None]
    out = torch.empty_like(q)
    op.attn_decode(q, kc, vc, tables, ctx, 0.1, max_ctx, 0, out, *bufs)
    want = ops.attn_decode(q, kc, vc, tables, ctx, 0.1, max_ctx, part)
    assert torch.equal(out, want) if ns == 1 else torch.allclose(out.float(), want.float(), atol=2e-2)      # (larger ones may do for both)


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("H,G,D,Dv,window,keep,start,n", [
    (8, 2, 128, 128, 1 << 30, 0, 0, 40),      # one tile, the last page partly used
    (4, 4, 64, 64, 40, 3, 50, 200),           # a kept prefix, several tiles
    (6, 1, 256, 192, 64, 0, 7, 90),
])
def test_keys_that_no_row_sees_do_not_count_in_f32(H, G, D, Dv, window, keep, start, n, bad):
    """f32 prompts: what an earlier owner left in the unused rows of a page, and a value outside a row's window or after it,
    reach no output; the rows that see such a value are no numbers."""
    g = torch.Generator().manual_seed(H * D)
    r = lambda *s: torch.randn(*s, generator=g)                                     # noqa: E731
    L, scale = start + n, 1.0 / math.sqrt(D)
    need = (L + BS - 1) // BS
    order = torch.randperm(need, generator=g)
    q, k, v = r(n, H, D), r(need * BS, G, D), r(need * BS, G, Dv)
    pos = torch.arange(start, L)
    k[L:], v[L:] = bad, bad
    odd = start + n // 2
    for hit in (False, True):
        if hit:
            v[odd] = bad
        kc, vc = torch.empty(need, G, BS, D), torch.empty(need, G, Dv, BS)
        kc[order], vc[order] = k.view(-1, BS, G, D).transpose(1, 2), v.view(-1, BS, G, Dv).permute(0, 2, 3, 1)
        cu = torch.tensor([0, n], dtype=torch.int32)
        got = ops.attn_window_paged(q.cuda(), kc.cuda(), vc.cuda(), order.int()[None].cuda(), cu.cuda(), pos.int().cuda(), scale,
                                    window, keep, None).cpu()
        sees = (pos >= odd) & (pos - odd < window) if hit else torch.zeros(n, dtype=torch.bool)
        want = dense(q.to(F64), k[:L].to(F64), v[:L].nan_to_num(0, 0, 0).to(F64), pos, scale, window, keep, None, None, 0, None)
        assert (got[~sees].to(F64) - want[~sees]).abs().max() < 1e-5 * 5
        assert not got[sees].isfinite().any()
