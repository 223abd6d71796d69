"""Products whose rows stand far apart, overlap or are one and the same: tiles with 32-bit row offsets leave them to one without."""
import pytest
import torch

from butterfly_amd import ops

pytestmark = pytest.mark.skipif(not ops.load_library(), reason="kernel library not built")


@pytest.mark.parametrize("M,N,K,tile", [(65, 2048, 2048, 128), (256, 6272, 2048, 128), (1000, 2048, 2048, 128), (2100, 2048, 2048, 256),
                                        (256, 28672, 8192, 256)])
@pytest.mark.parametrize("epi", ["none", "bias", "silu"])
def test_where_the_lines_are(M, N, K, tile, epi):
    """A tile's rows times their distance stay below 2^31 bytes, and rows do not overlap."""
    own = ops.gemm_plan(M, N, K, epi)
    assert own["kind"] in ("mid4", "mid8", "big4") and max(own["bm"], own["bn"]) == tile
    far = lambda t: ((1 << 30) - 1) // t                                                             # noqa: E731
    for kw in ({"ldx": K}, {"ldx": far(own["bm"])}, {"ldw": far(own["bn"])}):
        assert ops.gemm_plan(M, N, K, epi, **kw) == own, kw
    for kw in ({"ldx": 0}, {"ldx": K - 8}, {"ldx": far(own["bm"]) + 1}, {"ldx": 1 << 33}, {"ldw": 0}, {"ldw": K - 8},
               {"ldw": far(own["bn"]) + 1}, {"ldw": 1 << 33}):
        p = ops.gemm_plan(M, N, K, epi, **kw)
        assert p["kind"] == "tile" and p["bm"] == 128, kw


def test_few_rows_know_no_line():
    for M in (1, 7, 16, 48, 64):
        assert ops.gemm_plan(M, 2048, 2048, "none", ldx=1 << 33, ldw=0) == ops.gemm_plan(M, 2048, 2048, "none")


def _near(got, want):
    assert (got.double() - want).norm() < 2.0 ** -8 * want.norm()      # one rounding to bf16 (2^-9 of an element) of f32 sums


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,far_x", [(65, 256, 256, True), (200, 2048, 2048, True), (300, 1024, 2048, True), (128, 256, 256, False),
                                         (300, 512, 256, False)])
def test_rows_far_apart(M, N, K, far_x):
    """Rows of one operand just past the line, the others close together."""
    own = ops.gemm_plan(M, N, K, "none")
    rows, tile = (M, own["bm"]) if far_x else (N, own["bn"])
    ld = ((1 << 30) - 1) // tile // 8 * 8 + 8
    assert own["kind"] != "tile" and ops.gemm_plan(M, N, K, "none", **{"ldx" if far_x else "ldw": ld})["kind"] == "tile"
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x, w = (torch.randn(r, K, generator=g, device="cuda").bfloat16() for r in (M, N))
    w = (w * K ** -0.5).bfloat16()
    buf = torch.empty((rows - 1) * ld + K, dtype=torch.bfloat16, device="cuda")
    wide = buf.as_strided((rows, K), (ld, 1)).copy_(x if far_x else w)
    a, b = (wide, w) if far_x else (x, wide)
    want = x.double() @ w.double().T
    _near(ops.linear(a, b), want)
    _near(ops.linear_act(a, b, act="relu2"), torch.relu(want) ** 2)
    _near(ops.materialize(ops.linear(a, b, defer=True)), want)
    if far_x:      # a packed copy of the weight has no tile for such rows: the weight itself
        _near(ops.linear(a, b, packed=ops.pack_w256(b)), want)
    ssp = torch.rand(M, 3, generator=g, device="cuda") * K
    scaled = want * torch.rsqrt(ssp.double().sum(1, keepdim=True) / K + 1e-5)
    if ops.rowscale_ok(M, N, K):
        _near(ops.materialize(ops.linear(ops.RowNormed(a, ssp, 1e-5), b, defer=True)), scaled)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [65, 200, 300, 1000])
def test_rows_that_overlap(M):
    """One row for all, and windows of a sequence, as either operand."""
    g = torch.Generator(device="cuda").manual_seed(M)
    K, N = 512, 1024
    r = torch.randn(8 * max(M, N) + K, generator=g, device="cuda").bfloat16()
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    for x in (r[:K].expand(M, K), r.as_strided((M, K), (8, 1))):
        _near(ops.linear(x, w), x.double() @ w.double().T)
    x, v = r[:K * 2].view(2, K)[:1].expand(M, K).contiguous(), (r * K ** -0.5).bfloat16()
    for y in (v[:K].expand(N, K), v.as_strided((N, K), (8, 1))):
        _near(ops.linear(x, y), x.double() @ y.double().T)
