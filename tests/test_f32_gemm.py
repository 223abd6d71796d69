"""True-f32 products (f32 tiles, and three bf16 parts per value): plain GEMM, router logits and grouped experts against float64."""
import pytest
import torch

from butterfly_amd import ops

F64 = torch.float64


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (63, 65, 31), (64, 64, 32), (65, 130, 33), (3, 300, 257), (129, 127, 100),
                                   (2100, 2050, 70)])      # the last one: the 128 x 128 tile
@pytest.mark.parametrize("pad", [0, 3])
def test_gemm_matches_float64(M, N, K, pad):
    g = torch.Generator().manual_seed(M * N + K)
    x, w, b = (torch.randn(*s, generator=g) for s in ((M, K + pad), (N, K + pad), (N,)))
    xd, wd = x.cuda()[:, :K], w.cuda()[:, :K].contiguous()
    got = ops.linear_act(xd, wd, bias=b.cuda(), act="relu2").cpu().to(F64)
    acc = x[:, :K].to(F64) @ w[:, :K].to(F64).T + b.to(F64)
    want = torch.relu(acc) ** 2
    # K products of N(0, 1) values summed in f32: K eps / 2 of sqrt(K) at most, doubled by the square
    tol = 2 * K * 6e-8 * max(1.0, K ** 0.5) * (acc.abs().max() + 1)
    assert (got - want).abs().max() < tol


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(65, 66, 16), (65, 66, 32), (64, 64, 64), (70, 64, 96), (70, 64, 160), (2048, 1792, 64), (2048, 1792, 96),
                                   (2048, 1792, 45), (70, 64, 192), (65, 130, 320), (2048, 1792, 192)])      # one K step, few, and the 128 x 128 tile
def test_sums_that_bf16_parts_cannot_hold(M, N, K):
    g = torch.Generator().manual_seed(M + K)
    x, w = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g)
    x[1] *= 2.0 ** -120                # parts below the smallest bf16
    x[2] = 0
    x[3, 5] = float("inf")
    x[4, K - 1] = float("nan")
    x[5, 0] = 3.4e38                   # rounds to infinity in bf16
    w[1, 5], w[2] = 0, w[2].abs()
    w[:, 0] *= 2.0 ** -20
    got, want = ops.linear_act(x.cuda(), w.cuda()).cpu().to(F64), x.to(F64) @ w.to(F64).T
    assert got[3, 1].isnan() and got[3, 2] == float("inf") and got[4].isnan().all() and (got[2] == 0).all()
    keep = torch.tensor([r for r in range(M) if r not in (3, 4)])
    size = x[keep].to(F64).abs() @ w.to(F64).abs().T
    # K additions in f32, and 2^-24 of each product left out
    assert ((got - want)[keep].abs() <= (K + 2) * 6e-8 * size + 1e-43).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(65, 66, 20), (66, 64, 32), (70, 64, 192), (33, 130, 257), (130, 70, 160), (2048, 1792, 160),
                                   (2048, 1792, 45)])
@pytest.mark.parametrize("small,large", [(-126, 100), (-124, 60), (-115, 60), (-120, 20), (-140, 0), (-135, 100), (-75, -70), (-60, -45)])
def test_small_operands_of_large_ones(M, N, K, small, large):
    """Values whose last bits no bf16 part holds, denormal ones and products that underflow: as exact as sums in f32, alone, among
    ordinary terms and on either side; the rows beside them keep their sums bit for bit."""
    g = torch.Generator().manual_seed(M + K)
    x, w = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g)
    plain = ops.linear_act(x.cuda(), w.cuda()).cpu()
    x[1], x[2, ::3] = x[1] * 2.0 ** small, x[2, ::3] * 2.0 ** small      # a whole row, and some channels of one
    w[5], w[6, ::3] = w[5] * 2.0 ** large, w[6, ::3] * 2.0 ** large
    x[7], w[8] = x[7] * 2.0 ** min(large, 20), w[8] * 2.0 ** small
    got, want = ops.linear_act(x.cuda(), w.cuda()).cpu(), x.to(F64) @ w.to(F64).T
    size = x.to(F64).abs() @ w.to(F64).abs().T
    # K additions in f32, 2^-24 of each product left out; below 2^-126 one denormal (2^-149) per addition
    assert ((got.to(F64) - want).abs() <= (K + 2) * 6e-8 * size + K * 2.0 ** -149).all()
    rows, cols = [r for r in range(M) if r not in (1, 2, 7)], [c for c in range(N) if c not in (5, 6, 8)]
    assert torch.equal(got[rows][:, cols], plain[rows][:, cols])


@pytest.mark.gpu
@pytest.mark.parametrize("N", [64, 70])
@pytest.mark.parametrize("K,units", [(1, 1), (4, 1), (32, 1), (128, 1), (200, 1), (160, 3), (256, 3)])
def test_single_products(N, K, units):
    """One channel that is not zero. On f32 tiles (up to four steps of 32 channels, or rows without whole steps): one rounding (2^-24). As
    products of parts: less than 2^-24 of it is left out, and the last addition cuts to 24 bits (2^-23)."""
    g = torch.Generator().manual_seed(N)
    x, w = torch.zeros(4096, K), torch.zeros(N, K)
    x[:, K - 1], w[:, K - 1] = torch.randn(4096, generator=g), torch.randn(N, generator=g)
    x[0, K - 1] = w[0, K - 1] = 1 + 2.0 ** -8 - 2.0 ** -17 - 2.0 ** -23
    want = x.to(F64) @ w.to(F64).T
    assert ((ops.linear_act(x.cuda(), w.cuda()).cpu().to(F64) - want).abs() <= units * 2.0 ** -24 * want.abs()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("T,H,N,K", [(70, 3, 64, 16), (130, 2, 66, 40), (5, 4, 7, 33)])
@pytest.mark.parametrize("pad,shift", [(0, 0), (4, 0), (3, 0), (4, 1)])      # row strides and starts that allow 16-byte stores or not
def test_outputs_in_views(T, H, N, K, pad, shift):
    g = torch.Generator().manual_seed(T + N)
    x, w = torch.randn(T, H, K, generator=g), torch.randn(H, N, K, generator=g)
    wide = torch.full((T, H * N + pad + shift), 7.0, device="cuda")
    out = wide.as_strided((T, H, N), (H * N + pad + shift, N, 1), shift)
    ops.linear_heads(x.cuda(), w.cuda(), out)
    want = torch.matmul(x.to(F64).transpose(0, 1), w.to(F64).transpose(1, 2)).transpose(0, 1)
    assert (out.cpu().to(F64) - want).abs().max() < K * 6e-8 * K ** 0.5 * (want.abs().max() + 1)
    keep = torch.ones(wide.shape[1], dtype=torch.bool)
    keep[shift:shift + H * N] = False
    assert (wide.cpu()[:, keep] == 7.0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,E,W", [(600, 8, 256), (1025, 5, 512), (700, 64, 264), (41, 100, 64), (515, 9, 130)])
def test_router_choice(dt, T, E, W):
    g = torch.Generator().manual_seed(T + E)
    x, wr = torch.randn(T, W, generator=g).to(dt), (torch.randn(E, W, generator=g) * W ** -0.5).to(dt)
    ids, w = ops.moe_route_scores(x.cuda(), wr.cuda(), 2, scoring="sigmoid", renorm=False)
    s = torch.sigmoid(x.to(F64) @ wr.to(F64).T)
    got = s.gather(1, ids.cpu().long())
    top = s.topk(2, -1).values
    assert (got - top).abs().max() < 1e-5 and (w.cpu().to(F64) - got).abs().max() < 1e-5      # (ties within rounding may swap)


@pytest.mark.gpu
@pytest.mark.parametrize("T,E,Hd,F,plain", [(70, 3, 64, 96, False), (130, 4, 100, 65, False), (200, 2, 96, 64, True)])
def test_experts(T, E, Hd, F, plain):
    g = torch.Generator().manual_seed(T)
    x, ids = torch.randn(T, Hd, generator=g), torch.rand(T, E, generator=g).topk(2, -1).indices
    w = torch.rand(T, 2, generator=g)
    gu, dn = torch.randn(E, F if plain else 2 * F, Hd, generator=g) * Hd ** -0.5, torch.randn(E, Hd, F, generator=g) * F ** -0.5
    got = ops.moe_glu_ffn(x.cuda(), ids.int().cuda(), w.cuda(), gu.cuda(), dn.cuda(), 7.0, 1.702, 1.0, True,
                          "relu2" if plain else None).cpu().to(F64)
    want = torch.zeros(T, Hd, dtype=F64)
    for e in range(E):
        t, j = (ids == e).nonzero(as_tuple=True)
        h = (x[t].to(F64) * w[t, j].to(F64)[:, None]) @ gu[e].to(F64).T
        c = torch.clamp(h[:, :F], max=7.0)
        a = torch.relu(h) ** 2 if plain else c * torch.sigmoid(1.702 * c) * (torch.clamp(h[:, F:], -7.0, 7.0) + 1)
        want.index_add_(0, t, a @ dn[e].to(F64).T)
    assert (got - want).abs().max() < 1e-5 * (1 + want.abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("H,F", [(64, 96), (100, 65)])
def test_experts_of_small_operands(H, F):
    """An expert's inputs of 2^-105 under weights of 2^105, and output columns of 2^-110: as exact as the others."""
    g = torch.Generator().manual_seed(F)
    T, E = 90, 3
    x, ids, w = torch.randn(T, H, generator=g), (torch.arange(T) % E)[:, None], torch.rand(T, 1, generator=g) + 0.2
    gu, dn = torch.randn(E, 2 * F, H, generator=g) * H ** -0.5, torch.randn(E, H, F, generator=g) * F ** -0.5
    x[ids[:, 0] == 1] *= 2.0 ** -105
    gu[1] *= 2.0 ** 105
    dn[:, :8] *= 2.0 ** -110
    got = ops.moe_glu_ffn(x.cuda(), ids.int().cuda(), w.cuda(), gu.cuda(), dn.cuda(), 7.0, 1.702).cpu().to(F64)
    want = torch.zeros(T, H, dtype=F64)
    for e in range(E):
        t = (ids[:, 0] == e).nonzero()[:, 0]
        h = (x[t].to(F64) * w[t].to(F64)) @ gu[e].to(F64).T
        c = torch.clamp(h[:, :F], max=7.0)
        want[t] = (c * torch.sigmoid(1.702 * c) * (torch.clamp(h[:, F:], -7.0, 7.0) + 1)) @ dn[e].to(F64).T
    for part in (slice(0, 8), slice(8, H)):
        assert (got - want)[:, part].abs().max() < 1e-5 * want[:, part].abs().max()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(257, 1152, 64 * 4), (300, 1408, 128), (1000, 1152, 1024), (512, 8320, 256), (513, 1024 + 128, 64 * 9),
                                   (300, 1152, 64), (700, 2048, 64), (520, 1024, 256), (300, 1152, 1024)])      # (one K step: the 128-row tiles)
@pytest.mark.parametrize("bias", [False, True])
def test_prefill_tile_with_half_a_column_tile(M, N, K, bias):
    g = torch.Generator().manual_seed(M + N)
    x, w = torch.randn(M, K, generator=g).bfloat16(), torch.randn(N, K, generator=g).bfloat16()
    b = torch.randn(N, generator=g).bfloat16() if bias else None
    out = torch.full((M, N + 8), 7.0, dtype=torch.bfloat16, device="cuda")
    ops.linear(x.cuda(), w.cuda(), bias=None if b is None else b.cuda(), out=out[:, :N])
    want = x.to(F64) @ w.to(F64).T + (0 if b is None else b.to(F64))
    # one rounding to bf16 (2^-9) of f32 sums
    assert ((out[:, :N].cpu().to(F64) - want).abs() < 2.0 ** -8 * want.abs() + 1e-3 * K ** 0.5).all()
    assert (out[:, N:] == 7.0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 128, 128), (40, 256, 512), (300, 512, 2048), (2100, 1152, 256)])      # skinny, tile + split K, prefill
def test_squared_relu_epilogue(M, N, K):
    g = torch.Generator().manual_seed(M + N)
    x, w = torch.randn(M, K, generator=g).bfloat16(), torch.randn(N, K, generator=g).bfloat16()
    got = ops.linear_act(x.cuda(), w.cuda(), act="relu2").cpu().to(F64)
    want = torch.relu(x.to(F64) @ w.to(F64).T) ** 2
    assert ((got - want).abs() < 2.0 ** -8 * want + 1e-2).all()      # one rounding to bf16 of the squared f32 sum


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,S,W", [(3, 1, 4), (5, 2, 1024), (2, 3, 1028), (4, 4, 4096), (2, 2, 8192), (3, 2, 2050), (2, 5, 64)])
def test_stream_passes(dt, T, S, W):
    g = torch.Generator().manual_seed(S * W)
    r = lambda *s: torch.randn(*s, generator=g)                                     # noqa: E731
    xs, y, mix, wo, wi, nw = r(T, S, W), r(T, W).to(dt), r(S, S), r(S), r(S), r(W)
    unit = lambda u: u / torch.sqrt((u * u).mean(-1, keepdim=True) + 1e-6) * (nw.to(F64) + 1)          # noqa: E731
    new = torch.einsum("tsw,sr->trw", xs.to(F64), mix.to(F64)) + wo.to(F64)[None, :, None] * y.to(F64)[:, None]
    tol = 2e-5 if dt == torch.float32 else 2.0 ** -7
    c = lambda t: t.cuda()                                                         # noqa: E731

    def same(got, want, tol=tol):
        assert (got.cpu().to(F64) - want).abs().max() < tol * (1 + want.abs().max())

    a = c(xs).clone()
    h = ops.hc_post_pre_(a, c(y), c(mix), c(wo), c(wi), c(nw), 1e-6, 1.0, dt)
    same(a, new, 2e-6)
    same(h, unit(torch.einsum("s,tsw->tw", wi.to(F64), new)))
    b = c(xs).clone()
    ops.hc_post_(b, c(y), c(mix), c(wo))
    assert torch.equal(a, b)
    same(ops.hc_pre(c(xs), c(wi), c(nw), 1e-6, 1.0, dt), unit(torch.einsum("s,tsw->tw", wi.to(F64), xs.to(F64))))
    rows = torch.tensor([T - 1, 0])
    same(ops.hc_final(c(xs), c(nw), 1e-6, 1.0, c(rows), dt), unit(xs.to(F64).sum(1))[rows])
    table, ids = r(9, W).to(dt), torch.tensor([8, 0, 3], dtype=torch.int32)
    e = ops.embed_norm_streams(c(ids), c(table), c(nw), 1e-6, 1.0, S)
    for s in range(S):
        same(e[:, s], unit(table.to(F64)[ids.long()]), 2e-6)
