"""Residual step with a norm on both sides, rows held in registers (and the widths beside them) against float64."""
import pytest
import torch

from butterfly_amd import ops

F64 = torch.float64


def norm(x, w, b, eps):
    if b is None:
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps) * w + b


@pytest.mark.gpu
@pytest.mark.parametrize("dt,tol", [(torch.float32, 4e-6), (torch.bfloat16, 2.0 ** -8)])
@pytest.mark.parametrize("rms", [False, True])
@pytest.mark.parametrize("W", [4, 252, 256, 260, 1020, 1024, 1028, 2048, 2052, 4096, 4100])      # edges of a thread's share
def test_step_over_row_widths(dt, tol, rms, W):
    g = torch.Generator().manual_seed(W)
    T, eps, m = 3, 1e-5, 0.7
    rnd = lambda *s: torch.randn(*s, generator=g)            # noqa: E731
    x, y, extra = 3 * rnd(T, W) + 2, rnd(T, W).to(dt), rnd(T, W)
    w1, w2 = 1 + 0.2 * rnd(2, W)
    b1, b2 = (None, None) if rms else 0.2 * rnd(2, W)
    D = lambda t: None if t is None else t.to(F64)            # noqa: E731
    d = lambda t: None if t is None else t.to("cuda")         # noqa: E731
    for e in (None, extra):
        want = D(x) + m * norm(D(y), D(w1), D(b1), eps) + (0 if e is None else D(e))
        xg = d(x)
        h = ops.post_norm_add_norm(xg, d(y), d(w1), d(b1), eps, m, d(e), d(w2), d(b2), dt, rms=rms)
        wh = norm(want, D(w2), D(b2), eps)
        # f32 sums of up to 4100 terms, rounded a few times (6e-8 each); h in bf16: 2^-9 of its value
        assert (xg.cpu().to(F64) - want).abs().max() < 4e-6 * want.abs().max()
        assert (h.cpu().to(F64) - wh).abs().max() < tol * wh.abs().max()
    xg = d(x)
    assert ops.post_norm_add_norm(xg, d(y), d(w1), d(b1), eps, m, None, None, None, dt, rms=rms) is None
    want = D(x) + m * norm(D(y), D(w1), D(b1), eps)
    assert (xg.cpu().to(F64) - want).abs().max() < 4e-6 * want.abs().max()


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,W,K,scaled", [(1, 260, 1, True), (3, 1028, 2, False), (2, 2048, 3, True), (5, 4096, 4, False), (70, 1024, 2, True),
                                          (3, 256, 2, False), (2, 4100, 2, True)])      # the last two: the sum in a launch
def test_experts_summed_by_the_row_kernels(dt, T, W, K, scaled):
    """The sum over the choices inside the row kernels is that of its own launch, bit for bit."""
    g = torch.Generator().manual_seed(W + K)
    d = lambda *s, k=1.0: (k * torch.randn(*s, generator=g)).cuda()            # noqa: E731
    E, F = 5, 64
    x, gu, dn = d(T, W).to(dt), d(E, 2 * F, W, k=W ** -0.5).to(dt), d(E, W, F, k=F ** -0.5).to(dt)
    ids, w = torch.rand(T, E, generator=g).topk(K, -1).indices.int().cuda(), torch.rand(T, K, generator=g).cuda()
    args = (x, ids, w, gu, dn, 7.0, 1.702, 1.0, scaled)
    r, w1, w2, b1, b2, e = d(T, W), d(W), d(W), d(W), d(W), d(T, W)
    for rms in (False, True):
        got, want = r.clone(), r.clone()
        bias = (None, None) if rms else (b1, b2)
        y = ops.moe_glu_rows(*args)
        assert isinstance(y, ops.ExpertRows) == (256 < W <= 4096)
        h = ops.post_norm_add_norm(got, y, w1, bias[0], 1e-5, 0.7, e, w2, bias[1], dt, rms=rms)
        h2 = ops.post_norm_add_norm(want, ops.moe_glu_ffn(*args), w1, bias[0], 1e-5, 0.7, e, w2, bias[1], dt, rms=rms)
        assert torch.equal(got, want) and torch.equal(h, h2)
    for S in (1, 2, 4):
        xs, mix, wo, wi = d(T, S, W), d(S, S), d(S), d(S)
        got, want = xs.clone(), xs.clone()
        h = ops.hc_post_pre_(got, ops.moe_glu_rows(*args), mix, wo, wi, w1, 1e-5, 1.0, dt)
        h2 = ops.hc_post_pre_(want, ops.moe_glu_ffn(*args), mix, wo, wi, w1, 1e-5, 1.0, dt)
        assert torch.equal(got, want) and torch.equal(h, h2)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 5, 16, 33, 64, 200])
@pytest.mark.parametrize("N,K", [(256, 2048), (384, 4096), (1024, 2048), (2048, 1024), (4096, 6144), (4224, 4096)])
def test_slabs_summed_by_the_row_kernels(M, N, K):
    """The slabs of a product with K split are summed inside the row kernels as by the reduce launch, bit for bit."""
    slabs(M, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,kind,splits", [
    (257, 4096, 8192, "big4", 8), (1025, 2048, 4096, "big4", 4), (513, 4096, 4096, "big4", 4),      # a row past a tile, short last tiles
    (555, 2048, 8192, "big4", 8), (777, 4096, 6144, "big4", 4), (257, 4096, 4096, "mid8", 4), (100, 1152, 8192, "tile", 16),
    (257, 2048, 2048, "mid4", 4), (300, 1024, 2048, "mid4", 4), (300, 4096, 6144, "big4", 8), (300, 1152, 4096, "mid4", 8),
])
def test_slabs_of_prompts(M, N, K, kind, splits):
    """The same behind the tiles that prompts run on."""
    plan = ops.gemm_plan(M, N, K)
    assert (plan["kind"], plan["splitk"]) == (kind, splits)
    slabs(M, N, K)


def slabs(M, N, K):
    g = torch.Generator().manual_seed(M + N)
    d = lambda *s, k=1.0: (k * torch.randn(*s, generator=g)).cuda()            # noqa: E731
    dt = torch.bfloat16
    x, w = d(M, K).to(dt), d(N, K, k=K ** -0.5).to(dt)
    r, w1, w2, b1, b2 = d(M, N), d(N), d(N), d(N), d(N)
    got, want = r.clone(), r.clone()
    h = ops.post_norm_add_norm(got, ops.linear_rows(x, w), w1, b1, 1e-5, 0.7, None, w2, b2, dt)
    h2 = ops.post_norm_add_norm(want, ops.linear_act(x, w), w1, b1, 1e-5, 0.7, None, w2, b2, dt)
    assert torch.equal(got, want) and torch.equal(h, h2)
    for S in (2, 4, 5):
        xs, mix, wo, wi = d(M, S, N), d(S, S), d(S), d(S)
        got, want = xs.clone(), xs.clone()
        h = ops.hc_post_pre_(got, ops.linear_rows(x, w), mix, wo, wi, w1, 1e-5, 1.0, dt)
        h2 = ops.hc_post_pre_(want, ops.linear_act(x, w), mix, wo, wi, w1, 1e-5, 1.0, dt)
        assert torch.equal(got, want) and torch.equal(h, h2)
        ops.hc_post_(got, ops.linear_rows(x, w), mix, wo)
        ops.hc_post_(want, ops.linear_act(x, w), mix, wo)
        assert torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("W,scaled", [(512, True), (1028, False), (4096, False)])
def test_experts_summed_where_the_row_kernel_cannot(dt, W, scaled):
    """Outputs of experts in front of kernels that take whole rows only (no norm on them, five streams, the last update, streams off
    a 16-byte line) are summed first, bit for bit as by moe_glu_ffn; rows of another type stay refused."""
    g = torch.Generator().manual_seed(W)
    d = lambda *s, k=1.0: (k * torch.randn(*s, generator=g)).cuda()            # noqa: E731
    T, E, F = 6, 5, 64
    x, gu, dn = d(T, W).to(dt), d(E, 2 * F, W, k=W ** -0.5).to(dt), d(E, W, F, k=F ** -0.5).to(dt)
    ids, w = torch.rand(T, E, generator=g).topk(2, -1).indices.int().cuda(), torch.rand(T, 2, generator=g).cuda()
    args = (x, ids, w, gu, dn, 7.0, 1.702, 1.0, scaled)
    want_y = ops.moe_glu_ffn(*args)
    rows = ops.moe_glu_rows(*args)
    assert isinstance(rows, ops.ExpertRows) and torch.equal(ops.materialize(rows), want_y)
    r, w1 = d(T, W), d(W)
    got, want = r.clone(), r.clone()
    h = ops.post_norm_add_norm(got, ops.moe_glu_rows(*args), None, None, 1e-5, 0.7, None, w1, None, dt, rms=True)
    h2 = ops.post_norm_add_norm(want, want_y, None, None, 1e-5, 0.7, None, w1, None, dt, rms=True)
    assert torch.equal(got, want) and torch.equal(h, h2)
    for S, off in ((5, 0), (2, 1)):
        xs, mix, wo, wi = d(T * S * W + 1)[off:][:T * S * W].view(T, S, W), d(S, S), d(S), d(S)
        got, want = torch.empty(T * S * W + 1, device="cuda")[off:][:T * S * W].view(T, S, W).copy_(xs), xs.clone()
        h = ops.hc_post_pre_(got, ops.moe_glu_rows(*args), mix, wo, wi, w1, 1e-5, 1.0, dt)
        h2 = ops.hc_post_pre_(want if off == 0 else xs, want_y, mix, wo, wi, w1, 1e-5, 1.0, dt)
        assert torch.equal(got, want if off == 0 else xs) and torch.equal(h, h2)
        ops.hc_post_(got, ops.moe_glu_rows(*args), mix, wo)
        ops.hc_post_(want if off == 0 else xs, want_y, mix, wo)
        assert torch.equal(got, want if off == 0 else xs)
        with pytest.raises(RuntimeError):
            ops.hc_post_pre_(got, ops.moe_glu_rows(*args), mix, wo, wi, w1, 1e-5, 1.0,
                             torch.float32 if dt == torch.bfloat16 else torch.bfloat16)
