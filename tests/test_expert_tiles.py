"""Score-routed experts over large row groups (the 256-row LDS-DMA tiles and the smaller ones beside them) against float64."""
import math

import pytest
import torch

from butterfly_amd import ops

F64 = torch.float64


def reference(x, ids, w, gu, dn, limit, alpha, offset, scaled, plain):
    T, K = ids.shape
    F = dn.shape[2]
    y = torch.zeros(T, x.shape[1], dtype=F64)
    for e in range(gu.shape[0]):
        t, j = (ids == e).nonzero(as_tuple=True)
        if not t.numel():
            continue
        s = w[t, j][:, None]
        h = (x[t] * s if scaled else x[t]) @ gu[e].T
        if plain:
            a = torch.relu(h) ** 2
        else:
            g = torch.clamp(h[:, :F], max=limit)
            a = g * torch.sigmoid(alpha * g) * (torch.clamp(h[:, F:], -limit, limit) + offset)
        o = a @ dn[e].T
        y.index_add_(0, t, o if scaled else s * o)
    return y


@pytest.mark.gpu
@pytest.mark.parametrize("counts,Hd,F,plain,scaled,limit", [
    ([512, 769, 255, 1], 256, 128, False, True, 7.0),        # tile edges; the smallest panel; one row in a tile
    ([700, 0, 600], 512, 384, False, False, math.inf),       # an expert without rows; weighted outputs
    ([200, 220], 2048, 128, False, True, 7.0),               # a wide model's smaller groups
    ([513, 756, 40, 300], 768, 256, True, False, math.inf),  # plain experts
    ([600, 500], 256, 192, False, True, 7.0),                # F not a multiple of 128: the 128-row tiles
    ([300, 290], 320, 128, True, True, math.inf),            # Hd not a multiple of 256; scores on plain experts
    ([60, 50, 70], 256, 256, False, True, 7.0),              # small groups: the 64-row tiles
])
@pytest.mark.parametrize("stride", [0, 8])
def test_experts_over_row_groups(counts, Hd, F, plain, scaled, limit, stride):
    g = torch.Generator().manual_seed(sum(counts) + F)
    E, TK = len(counts), sum(counts)
    K = 2 if TK % 2 == 0 else 1
    flat = torch.cat([torch.full((c,), e) for e, c in enumerate(counts)])[torch.randperm(TK, generator=g)]
    ids = flat.view(-1, K)
    T = ids.shape[0]
    bf = lambda *s, k=1.0: (k * torch.randn(*s, generator=g)).to(torch.bfloat16)            # noqa: E731
    x = bf(T, Hd + stride)[:, :Hd]
    w = torch.rand(T, K, generator=g) + 0.2
    gu, dn = bf(E, F if plain else 2 * F, Hd, k=2 * Hd ** -0.5), bf(E, Hd, F, k=F ** -0.5)
    d = lambda t: t.to("cuda")                                                           # noqa: E731
    xd = torch.empty(T, Hd + stride, dtype=torch.bfloat16, device="cuda")[:, :Hd].copy_(x)
    got = ops.moe_glu_ffn(xd, d(ids.int()), d(w), d(gu), d(dn), limit, 1.702, 1.0, scaled, "relu2" if plain else None)
    want = reference(x.to(F64), ids, w.to(F64), gu.to(F64), dn.to(F64), limit, 1.702, 1.0, scaled, plain)
    # bf16 hidden rows and output (2^-9 each); the smaller tiles also round the scaled input rows, whose error the
    # squared activation can double
    err = (got.cpu().to(F64) - want).norm() / want.norm()
    assert err < 2.0 ** -7


@pytest.mark.gpu
@pytest.mark.parametrize("counts,Hd,F,plain,scaled", [
    ([1, 0, 0, 0], 64, 64, False, True),                 # one row, one K step
    ([16, 17, 1, 0], 320, 64, False, True),              # edges of the row tiles; fewer K steps than a wave keeps in flight
    ([32, 33, 0, 3], 1088, 192, False, False),           # two and four row tiles; a remainder of the K steps
    ([64, 5, 2, 1], 256, 320, True, False),              # a whole tile; plain experts
    ([65, 4, 1, 1], 512, 64, True, True),                # one row in a second tile
])
def test_experts_over_few_rows(counts, Hd, F, plain, scaled):
    """Weights streamed past the rows; rows of x with a stride, an addend."""
    g = torch.Generator().manual_seed(sum(counts) + F)
    E, TK = len(counts), sum(counts)
    flat = torch.cat([torch.full((c,), e) for e, c in enumerate(counts)])[torch.randperm(TK, generator=g)]
    ids = flat.view(-1, 1)
    bf = lambda *s, k=1.0: (k * torch.randn(*s, generator=g)).to(torch.bfloat16)            # noqa: E731
    x, add, w = bf(TK, Hd + 8)[:, :Hd], bf(TK, Hd), torch.rand(TK, 1, generator=g) + 0.2
    gu, dn = bf(E, F if plain else 2 * F, Hd, k=2 * Hd ** -0.5), bf(E, Hd, F, k=F ** -0.5)
    d = lambda t: t.to("cuda")                                                           # noqa: E731
    xd = torch.empty(TK, Hd + 8, dtype=torch.bfloat16, device="cuda")[:, :Hd].copy_(x)
    got = ops.moe_glu_ffn(xd, d(ids.int()), d(w), d(gu), d(dn), 7.0, 1.702, 1.0, scaled, "relu2" if plain else None,
                          addend=d(add))
    want = reference(x.to(F64), ids, w.to(F64), gu.to(F64), dn.to(F64), 7.0, 1.702, 1.0, scaled, plain) + add.to(F64)
    # bf16 input rows times their score, hidden rows and output (2^-9 each); the squared activation doubles the first
    err = (got.cpu().to(F64) - want).norm() / want.norm()
    assert err < 6e-3


@pytest.mark.gpu
@pytest.mark.parametrize("TK,E", [(1, 1), (2, 33), (63, 32), (64, 1), (64, 31), (64, 65), (64, 200), (17, 1024), (65, 33)])
@pytest.mark.parametrize("beyond", [0, 5])
def test_rows_found_among_the_choices(TK, E, beyond):
    """Up to 64 pairs the streams find an expert's rows themselves; ids from E on belong to no expert."""
    g = torch.Generator().manual_seed(TK + E)
    ids = torch.randint(0, E + beyond, (TK, 1), generator=g)
    bf = lambda *s, k=1.0: (k * torch.randn(*s, generator=g)).to(torch.bfloat16)            # noqa: E731
    x, w = bf(TK, 128), torch.rand(TK, 1, generator=g) + 0.2
    gu, dn = bf(E, 128, 128, k=2 * 128 ** -0.5), bf(E, 128, 64, k=0.125)
    got = ops.moe_glu_ffn(x.cuda(), ids.int().cuda(), w.cuda(), gu.cuda(), dn.cuda(), 7.0, 1.702, 1.0, False, identity=True)
    want = reference(x.to(F64), ids, w.to(F64), gu.to(F64), dn.to(F64), 7.0, 1.702, 1.0, False, False)
    want += (w.to(F64) * (ids >= E)) * x.to(F64)
    # bf16 hidden rows and output, 2^-9 each
    assert (got.cpu().to(F64) - want).norm() / want.norm() < 6e-3


@pytest.mark.gpu
@pytest.mark.parametrize("counts,rest,Hd,F,plain", [
    ([5, 0, 16, 3], 20, 320, 128, False),        # weights streamed past the rows
    ([40, 64, 1, 70], 40, 512, 128, False),      # the 64-row tiles
    ([512, 769, 0, 500], 333, 256, 128, False),  # the 256-row tiles
    ([500, 700], 111, 512, 256, True),
    ([0, 0, 0], 9, 256, 256, False),             # no row for any expert
])
@pytest.mark.parametrize("beyond", [0, 3])
def test_ids_that_name_no_expert(counts, rest, Hd, F, plain, beyond):
    """ids from E on: they return the token's row itself (fewer grouped rows than pairs: the tail of the row groups and the pairs'
    outputs stay unwritten and count nowhere)."""
    g = torch.Generator().manual_seed(sum(counts) + F)
    E = len(counts)
    flat = torch.cat([torch.full((c,), e) for e, c in enumerate(counts)] + [torch.full((rest,), E + beyond)])
    flat = flat[torch.randperm(len(flat), generator=g)]
    ids = flat[:len(flat) // 2 * 2].view(-1, 2)
    T = len(ids)
    bf = lambda *s, k=1.0: (k * torch.randn(*s, generator=g)).to(torch.bfloat16)            # noqa: E731
    x, w = bf(T, Hd), torch.rand(T, 2, generator=g) + 0.2
    gu, dn = bf(E, F if plain else 2 * F, Hd, k=2 * Hd ** -0.5), bf(E, Hd, F, k=F ** -0.5)
    ops.moe_glu_ffn(*(t.cuda() for t in (torch.full_like(x, 1e30), torch.zeros_like(ids).int(), w, gu, dn)), 7.0, 1.702, 1.0, False,
                    "relu2" if plain else None)      # (leaves large values and infinities in the scratch)
    got = ops.moe_glu_ffn(x.cuda(), ids.int().cuda(), w.cuda(), gu.cuda(), dn.cuda(), 7.0, 1.702, 1.0, False,
                          "relu2" if plain else None, identity=True)
    want = reference(x.to(F64), ids, w.to(F64), gu.to(F64), dn.to(F64), 7.0, 1.702, 1.0, False, plain)
    want += (w.to(F64) * (ids >= E)).sum(1, keepdim=True) * x.to(F64)
    # bf16 hidden rows and output, 2^-9 each
    assert (got.cpu().to(F64) - want).norm() / want.norm() < 6e-3


def test_sparse_tile_rows():
    """64-row tiles for a few rows per expert, 256-row tiles as soon as their workgroups pay; 128-row tiles for other sizes."""
    rows = lambda n, E, H, F: ops.moe_sparse_tile_rows(n, E, H, F)                       # noqa: E731
    assert [rows(n, 8, 4096, 14336) for n in (191, 192, 4096)] == [64, 256, 256]
    assert [rows(n, 4, 4096, 14336) for n in (223, 224)] == [64, 256]      # (40 rows each: 302 us and 365, 50: 444 and 373)
    assert [rows(n, 32, 2048, 1024) for n in (1791, 1792)] == [64, 256]
    lines = lambda E, H, F: next(n for n in range(1, 200) if ops.moe_sparse_tile_rows(n * E, E, H, F, True) == 256)      # noqa: E731
    assert [lines(8, 4096, 14336), lines(4, 4096, 4096), lines(8, 1024, 4096)] == [56, 72, 150]      # rows 32 KB apart
    assert [rows(n, 2, 4096, 14336) for n in (191, 192)] == [64, 256]
    assert rows(10 ** 6, 8, 4096 + 128, 14336) == 128 and rows(10 ** 6, 8, 4096, 64) == 128


@pytest.mark.gpu
@pytest.mark.parametrize("counts", [[64] * 8, [1, 0, 257, 70, 100, 2, 255, 80], [256, 0, 0, 0, 128, 0, 129, 65]])
def test_sparse_experts_few_rows_per_big_tile(counts):
    """The sparse SwiGLU experts on 256-row tiles that are mostly empty: one row, none, a row past a tile and past a half; the down
    projection's rows a multiple of 32 KB apart, and 128 bytes more."""
    E, K, H, F = 8, 1, 3072, 2048
    g = torch.Generator().manual_seed(sum(counts))
    ids = torch.cat([torch.full((c,), e) for e, c in enumerate(counts)])[torch.randperm(sum(counts), generator=g)].view(-1, K)
    assert ops.moe_sparse_tile_rows(ids.numel(), E, H, F) == 256
    bf = lambda *s, k=1.0: (k * torch.randn(*s, generator=g)).to(torch.bfloat16)            # noqa: E731
    x, w = bf(ids.shape[0], H), torch.rand(ids.shape[0], K, generator=g) + 0.2
    gu, dn = bf(E * 2 * F, H, k=H ** -0.5), bf(H, E * F, k=F ** -0.5)
    got = ops.moe_sparse_ffn(x.cuda(), ids.int().cuda(), w.cuda(), gu.cuda(), dn.cuda(), 0, E, F)
    wide = torch.empty(H, E * F + 64, dtype=torch.bfloat16, device="cuda")[:, :E * F].copy_(dn)
    same = ops.moe_sparse_ffn(x.cuda(), ids.int().cuda(), w.cuda(), gu.cuda(), wide, 0, E, F)
    assert (same.float() - got.float()).norm() < 2.0 ** -8 * got.float().norm()
    want = ops.reference.moe_sparse_ffn(x.float(), ids, w, gu.float(), dn.float(), 0, E, F)
    # bf16 hidden rows, expert rows and output: 2^-9 each
    assert (got.cpu().float() - want).norm() < 2.0 ** -7 * want.norm()


@pytest.mark.skipif(not ops.load_library(), reason="kernel library not built")
def test_grouped_rows_beyond_32_bit_offsets():
    """Gathered rows that 32-bit byte offsets do not reach go to the tile with 64-bit addresses, and so do slots whose single tile has
    such rows; any number of slots stays, and so do down weights of rows 32 KB apart on the other tile."""
    big4 = torch.ops.bfly.moe_grouped_on_big4                 # x rows, their stride, the weights', gate/up, gathered
    wide, pad = 8 * 14336, 8 * 14336 + 2048
    assert [big4(n, 4096, 4096, True, True) for n in (262143, 262144, 10 ** 6)] == [True, False, False]
    assert [big4(n, 14336, pad, False, False) for n in (74897, 74899, 10 ** 6)] == [True] * 3
    assert [big4(10 ** 6, ld, pad, False, False) for ld in (1 << 22, (1 << 22) - 8)] == [False, True]
    assert not big4(300, 14336, wide, False, False)


@pytest.mark.gpu
@pytest.mark.parametrize("gathered", [False, True])
def test_grouped_rows_of_far_strides(gathered):
    """600 rows 4 MB apart: the last ones lie 2.5 GB behind the first, past 32-bit byte offsets."""
    M, K, N, E, ld = 600, 256, 512, 2, 1 << 21
    g = torch.Generator(device="cuda").manual_seed(M)
    bf = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)            # noqa: E731
    x = torch.empty(M * ld, dtype=torch.bfloat16, device="cuda").view(M, ld)[:, :K].copy_(bf(M, K))
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")                         # noqa: E731
    tiles, rows = [(0, 0, 256, 0), (0, 256, 330, 0), (1, 330, 586, 0), (1, 586, 600, 0)], torch.randperm(M, generator=g, device="cuda")
    if not gathered:
        rows = torch.arange(M, device="cuda")
    w = bf(E, N, K) * K ** -0.5
    want = torch.cat([x[rows[:330]].float() @ w[0].float().T, x[rows[330:]].float() @ w[1].float().T])
    if gathered:      # gate and up rows interleaved in groups of 16
        v = want.view(M, N // 32, 2, 16)
        want = (torch.nn.functional.silu(v[:, :, 0]) * v[:, :, 1]).reshape(M, N // 2)
    out = torch.full_like(want, float("nan"), dtype=torch.bfloat16)
    torch.ops.bfly.moe_grouped_gemm(x, w.view(E * N, K), out, rows.int() if gathered else None, i32(tiles), i32([4]), N * K, N, K, E,
                                    ops.EPILOGUES["silu" if gathered else "none"], 256)
    # one rounding to bf16 (2^-9), f32 sums of 256 products beside it
    assert (out.float() - want).norm() < 2.0 ** -8 * want.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("counts", [[2100, 3000, 129, 0, 2500, 391], [256] * 34, [128, 8400, 1]])
@pytest.mark.parametrize("Hd,F,plain,scaled", [(256, 2048, False, True), (512, 4096, True, False), (4096, 256, False, False)])
def test_workgroups_that_walk_expert_tiles(counts, Hd, F, plain, scaled):
    """More tiles than compute units: whole, short and half ones in turn, four and more steps of K."""
    g = torch.Generator(device="cuda").manual_seed(sum(counts) + F)
    E, TK = len(counts), sum(counts) // 2 * 2
    flat = torch.cat([torch.full((c,), e, device="cuda") for e, c in enumerate(counts)])
    ids = flat[torch.randperm(len(flat), generator=g, device="cuda")][:TK].view(-1, 2)
    bf = lambda *s, k=1.0: (k * torch.randn(*s, generator=g, device="cuda")).to(torch.bfloat16)            # noqa: E731
    x, w = bf(TK // 2, Hd), torch.rand(TK // 2, 2, generator=g, device="cuda") + 0.2
    gu, dn = bf(E, F if plain else 2 * F, Hd, k=2 * Hd ** -0.5), bf(E, Hd, F, k=F ** -0.5)
    got = ops.moe_glu_ffn(x, ids.int(), w, gu, dn, 7.0, 1.702, 1.0, scaled, "relu2" if plain else None).double()
    with torch.device("cuda"):
        want = reference(x.double(), ids, w.double(), gu.double(), dn.double(), 7.0, 1.702, 1.0, scaled, plain)
    # bf16 hidden rows and output (2^-9 each), in every row
    assert ((got - want).norm(dim=1) < 2.0 ** -7 * want.norm(dim=1)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("epi", ["none", "silu"])
@pytest.mark.parametrize("gathered", [False, True])
@pytest.mark.parametrize("K", [128, 256, 1024])
def test_workgroups_that_walk_grouped_tiles(epi, gathered, K):
    """Groups of 2600, 70, 1800 and 4000 rows over 20 column tiles."""
    counts, N = [2600, 70, 1800, 4000], 5120
    M, E = sum(counts), len(counts)
    g = torch.Generator(device="cuda").manual_seed(K)
    x, w = (torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16) for s in ((M, K), (E, N, K)))
    w = w * K ** -0.5
    rows = torch.randperm(M, generator=g, device="cuda") if gathered else torch.arange(M, device="cuda")
    tiles, start, want = [], 0, []
    for e, c in enumerate(counts):
        tiles += [(e, r, start + c, 0) for r in range(start, start + c, 256)]
        want.append(x[rows[start:start + c]].float() @ w[e].float().T)
        start += c
    want = torch.cat(want)
    if epi == "silu":
        v = want.view(M, N // 32, 2, 16)
        want = (torch.nn.functional.silu(v[:, :, 0]) * v[:, :, 1]).reshape(M, N // 2)
    out = torch.full_like(want, float("nan"), dtype=torch.bfloat16)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")                         # noqa: E731
    torch.ops.bfly.moe_grouped_gemm(x, w.view(E * N, K), out, rows.int() if gathered else None, i32(tiles), i32([len(tiles)]), N * K,
                                    N, K, E, ops.EPILOGUES[epi], 256)
    # one rounding to bf16 (2^-9), f32 sums of K products beside it, in every row
    assert ((out.float() - want).norm(dim=1) < 2.0 ** -8 * want.norm(dim=1)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("T", [40, 1000])
def test_sparse_experts_of_padded_rows(T):
    """Gate/up and down rows further apart than they are wide, as models lay out rows of a multiple of 32 KB, on both tiles."""
    E, K, H, F = 4, 2, 512, 256
    g = torch.Generator().manual_seed(T)
    bf = lambda *s, k=1.0: (k * torch.randn(*s, generator=g)).to(torch.bfloat16)            # noqa: E731
    x, ids, w = bf(T, H), torch.rand(T, E, generator=g).topk(K, -1).indices, torch.rand(T, K, generator=g)
    gu, dn = bf(E * 2 * F, H, k=H ** -0.5), bf(H, E * F, k=F ** -0.5)
    d = [t.cuda() for t in (x, ids.int(), w)]
    apart = lambda t: torch.zeros(t.shape[0], t.shape[1] + 64, dtype=t.dtype, device="cuda")[:, :t.shape[1]].copy_(t)      # noqa: E731
    want = ops.moe_sparse_ffn(*d, gu.cuda(), dn.cuda(), 0, E, F)
    ref = ops.reference.moe_sparse_ffn(x.float(), ids, w, gu.float(), dn.float(), 0, E, F)
    # bf16 hidden rows, expert rows and output: 2^-9 each
    assert (want.cpu().float() - ref).norm() < 2.0 ** -7 * ref.norm()
    for a, b in ((apart(gu), dn.cuda()), (gu.cuda(), apart(dn)), (apart(gu), apart(dn))):
        got = ops.moe_sparse_ffn(*d, a, b, 0, E, F)
        assert (got.float() - want.float()).norm() < 2.0 ** -8 * want.float().norm()
