"""Plans of the prefill GEMM: splits of the 256 x 256 tile, half column tiles, row scales."""
import pytest
import torch

from butterfly_amd import ops

pytestmark = pytest.mark.skipif(not ops.load_library(), reason="kernel library not built")


@pytest.mark.parametrize("K", [64, 512, 1024, 4096, 14336])
@pytest.mark.parametrize("N", [256, 1280, 2048, 8192])
def test_splits_pay_for_their_sums(K, N):
    for M in (257, 600, 1500, 3000, 6184, 8192):
        p = ops.gemm_plan(M, N, K)
        if p["kind"] != "big4" or p["bm"] != 256:
            continue
        tiles, sk = -(-M // 256) * -(-N // 256), p["splitk"]
        assert sk == 1 or K // 64 >= 8 * sk, (M, N, K, sk)          # eight K steps per split at least
        # a split has to shorten the rounds of 256 workgroups (each takes its share of K)
        assert sk == 1 or -(-tiles * sk // 256) < sk * -(-tiles // 256), (M, N, K, sk)


@pytest.mark.parametrize("K", [64, 128, 192, 1024, 4096])
@pytest.mark.parametrize("N", [128, 256, 1024, 1152, 1408, 2048, 8320])
def test_every_row_count_has_a_plan_that_runs(K, N):
    """One K step, whole and half column tiles: the plan chosen is one that its kernel takes."""
    for M in (1, 16, 64, 200, 256, 257, 300, 512, 1000, 5000):
        for epi in ("none", "bias", "silu", "relu2"):
            assert torch.ops.bfly.gemm_check(M, N, K, ops.EPILOGUES[epi]) == 0, (M, N, K, epi)


LLAMA = [(6144, 4096), (4096, 4096), (28672, 4096), (4096, 14336), (10240, 8192), (8192, 8192), (57344, 8192), (8192, 28672),
         (2560, 28672), (1152, 4096), (8320, 2048)]


def test_partial_sums_are_bounded_and_reserved(monkeypatch):
    """No plan of a prefill step needs more than 256 MB of partial sums, and none more than what is reserved before serving
    (an outgrown workspace is kept, a captured graph may still use it)."""
    monkeypatch.setattr(ops, "_arena", ops._Arena())
    ops.reserve_workspace(torch.device("cpu"), 8192, *LLAMA[0], shapes=LLAMA)
    have = 4 * next(b for k, b in ops._arena.bufs.items() if k[1] == "gemm").numel()
    rows = sorted({1, 7, 64, 200, 256, 512, 8192, *range(257, 8192, 61), *range(256, 8192, 256)})
    for N, K in LLAMA:
        for M in rows:
            need = torch.ops.bfly.gemm_workspace_size(M, N, K)
            assert need <= have, (M, N, K, need, have)
            assert need <= (256 << 20) + 4 * torch.ops.bfly.gemm_slab_offset(), (M, N, K, need)


# us of one step with 1, 2, 4 and 8 splits (measured once; whatever a plan's clock or unit, the order is what counts)
TIMED = {(2300, 8192, 8192): (314, 340, 395, 551), (2300, 10240, 8192): (320, 372, 461), (2300, 8192, 28672): (1096, 948, 913, 1029),
         (520, 4096, 4096): (75, 53, 42, 57), (1100, 4096, 14336): (235, 148, 168, 174), (2300, 4096, 14336): (256, 304, 298, 353),
         (1800, 4096, 14336): (246, 177, 209, 272), (3300, 2560, 28672): (505, 587, 490, 502), (2300, 2560, 28672): (492, 319, 336, 329)}


@pytest.mark.parametrize("shape", TIMED)
def test_split_is_near_the_fastest(shape):
    t = TIMED[shape]
    sk = ops.gemm_plan(*shape)["splitk"]
    assert t[(1, 2, 4, 8).index(sk)] < 1.08 * min(t), (shape, sk)


# us of one step on 128 x 128 tiles and on 256 x 256 tiles
TIMED_HALF = {(300, 1408, 1024): (15, 24), (520, 1152, 128): (7, 14), (4000, 1152, 128): (10, 15), (1838, 4224, 1024): (24, 31),
              (1838, 8320, 4096): (139, 164), (520, 6272, 2048): (35, 46), (8192, 8320, 2048): (348, 253),
              (6200, 6272, 2048): (200, 153), (1000, 4224, 1024): (37, 30), (4000, 1408, 1024): (43, 30), (6200, 1152, 4096): (98, 79)}


@pytest.mark.parametrize("shape", TIMED_HALF)
def test_half_column_tiles_go_to_the_faster_tile(shape):
    t = TIMED_HALF[shape]
    big = ops.gemm_plan(*shape)["kind"] == "big4"
    assert t[big] < 1.1 * min(t), (shape, big)


HALF = [(300, 1152, 1024), (512, 1152, 1024), (1000, 1408, 4096), (5000, 8320, 256)]


@pytest.mark.parametrize("M,N,K", HALF + [(257, 1152, 64)])
def test_half_column_tiles_take_a_row_scale(M, N, K):
    for epi in ("none", "bias", "silu"):
        assert torch.ops.bfly.gemm_rowscale_check(M, N, K, ops.EPILOGUES[epi]) == 0, epi
    assert torch.ops.bfly.gemm_rowscale_check(512, 2048, K, 0) != 0 or K == 64      # whole column tiles: as ever


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", HALF)
@pytest.mark.parametrize("how", ["bias", "silu", "defer"])
def test_row_scaled_product_with_a_half_column_tile(M, N, K, how):
    g = torch.Generator().manual_seed(M + N)
    x, w = torch.randn(M, K, generator=g).bfloat16().cuda(), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16().cuda()
    b = torch.randn(N, generator=g).bfloat16().cuda() if how == "bias" else None
    ssp = torch.rand(M, 3, generator=g).cuda() * K
    y = ops.linear(ops.RowNormed(x, ssp, 1e-5), w, bias=b, epilogue="silu" if how == "silu" else "none", defer=how == "defer")
    got = ops.materialize(y).cpu().double()
    want = (x.double() @ w.double().T * torch.rsqrt(ssp.double().sum(1, keepdim=True) / K + 1e-5)).cpu()
    if b is not None:
        want += b.cpu().double()
    if how == "silu":
        u = want.view(M, N // 32, 2, 16)
        want = (torch.nn.functional.silu(u[:, :, 0]) * u[:, :, 1]).reshape(M, N // 2)
    # one rounding to bf16 (2^-9) of f32 sums of unit-sized products
    assert ((got - want).abs() < 2.0 ** -8 * want.abs() + 1e-4).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(4100, 1024, 512), (4225, 4224, 1024), (2300, 2560, 192), (1100, 4096, 14336),
                                   (8200, 5120, 128), (8200, 5120, 256), (8192, 8320, 2048)])
@pytest.mark.parametrize("epi", ["none", "bias", "silu", "relu2", "glu"])
def test_results_of_the_large_tile_into_any_rows(M, N, K, epi):
    """A short last row tile, a half column tile, half tiles, split K, workgroups that walk several tiles: rows of any stride and
    alignment take the same values and nothing beside them is written."""
    assert ops.gemm_plan(M, N, K)["kind"] == "big4"
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x, w, b = (torch.randn(*s, device="cuda", generator=g).to(torch.bfloat16) for s in ((M, K), (N, K), (N,)))
    w = w * K ** -0.5
    bias = {"bias": b, "glu": ops.glu_bias_block(b, 7.0, 1.702, 1.0)}.get(epi)
    name = "none" if epi == "bias" else epi
    n = N // 2 if epi in ("silu", "glu") else N
    want = ops.linear(x, w, bias=bias, epilogue=name)
    for first, ld in ((0, n + 8), (8, n + 24), (4, n + 4), (1, n + 1), (3, n + 16)):
        buf = torch.full((M, ld), 77.0, device="cuda", dtype=torch.bfloat16)
        ops.linear(x, w, bias=bias, epilogue=name, out=buf[:, first:first + n])
        assert torch.equal(buf[:, first:first + n], want), (first, ld)
        assert (buf[:, :first] == 77).all() and (buf[:, first + n:] == 77).all(), (first, ld)
    s = x.float() @ w.float().t()
    size = x.float().abs() @ w.float().abs().t()          # sums of K products: 2^-24 of it a step, at most, in any order
    if epi in ("none", "bias"):
        s = s + (b.float() if epi == "bias" else 0)
        assert ((want.float() - s).abs() <= 2.0 ** -8 * s.abs() + K * 2.0 ** -24 * size).all()
    elif epi == "relu2":
        r, d = s.clamp_min(0), K * 2.0 ** -24 * size
        assert ((want.float() - r * r).abs() <= 2.0 ** -8 * (r + d) ** 2 + 2 * r * d + d * d).all()
    else:                                                 # blocks of 16 gate and 16 up columns in turn
        part = lambda t: t.view(-1, N // 32, 2, 16).unbind(2)                                             # noqa: E731
        (gate, up), (dg, du), (bg, bu) = part(s), part(K * 2.0 ** -24 * size), part(b.float())
        if epi == "glu":
            gate, up = (gate + bg).clamp_max(7.0), (up + bu).clamp(-7.0, 7.0) + 1.0
        act = gate * torch.sigmoid((1.702 if epi == "glu" else 1.0) * gate)      # (its slope is below 1.1 in either form)
        bound = 2.0 ** -8 * (act * up).abs() + 1.1 * dg * (up.abs() + du) + act.abs() * du + 1e-6
        assert ((want.float().view_as(act) - act * up).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("epi", ["none", "silu"])
def test_results_of_the_large_tile_into_far_rows(epi):
    """Rows 2 MB apart and more leave by 64-bit addresses (the values of rows side by side, which the test above has)."""
    M, N, K = 2300, 2560, 192
    g = torch.Generator(device="cuda").manual_seed(N)
    x, w = (torch.randn(*s, device="cuda", generator=g).to(torch.bfloat16) for s in ((M, K), (N, K)))
    want = ops.linear(x, w, epilogue=epi)
    far = torch.empty(M * (1 << 20), device="cuda", dtype=torch.bfloat16).view(M, 1 << 20)[:, 3:3 + want.shape[1]]
    ops.linear(x, w, epilogue=epi, out=far)
    assert torch.equal(far, want)


BOUNDED = [(2048, 1024), (2048, 8192), (1024, 1024), (28672, 4096), (8192, 4160), (3584, 4096), (4096, 7168), (4096, 4096), (6144, 4096),
           (10240, 8192), (8192, 28672), (128, 512), (1152, 4096), (8320, 2048), (4224, 1024), (128256, 4096)]


@pytest.mark.parametrize("shape", BOUNDED, ids=str)
@pytest.mark.parametrize("most", [1, 64, 128, 200, 512, 1000, 8192])
def test_no_number_of_rows_asks_for_more_than_the_bound(shape, most):
    """Each shape by itself, every number of rows: fewer may split K more, so none stands for the others."""
    have = torch.ops.bfly.gemm_workspace_bound(most, *shape)
    need = [torch.ops.bfly.gemm_workspace_size(m, *shape) for m in range(1, most + 1)]
    assert max(need) == have


@pytest.mark.parametrize("N", [128, 384, 2048, 10240])
def test_nothing_is_split_behind_the_rows_that_the_bound_looks_at(N):
    for K in (1024, 8192, 28672):
        last = 256 * (512 // -(-N // 256))
        for M in (*range(last + 1, last + 600, 7), 2 * last, 3 * last + 5):
            assert torch.ops.bfly.gemm_workspace_size(M, N, K) == 0, (M, K)


@pytest.mark.parametrize("M", [2, 3, 4, 5])
@pytest.mark.parametrize("N,K", [(8192, 4160), (8192, 4096), (16384, 4160), (10240, 8192)])
def test_few_rows_have_room_for_every_plan(M, N, K):
    """Row-major weights run the plan of their own rows, packed ones of many columns that of five."""
    room = torch.ops.bfly.gemm_workspace_size(M, N, K)
    for rows in (M, 5 if N % 256 == 0 else M):
        sk = ops.gemm_plan(rows, N, K)["splitk"]
        assert sk == 1 or room >= 4 * (torch.ops.bfly.gemm_slab_offset() + sk * M * N)
