"""f32 products of bf16 parts on each of their tiles: remainders of rows, columns and steps, sums that parts cannot hold, experts."""
import pytest
import torch

from butterfly_amd import ops

F64 = torch.float64


# 64 x 64, 64 x 128, 128 x 128 and 128 x 256 (parts_tile: the fewest rounds of 256 tiles by what a round takes)
@pytest.mark.gpu
@pytest.mark.parametrize("M,N", [(70, 200), (1838, 1000), (1838, 2010), (1900, 4150)])
@pytest.mark.parametrize("K", [160, 416])      # five and thirteen steps: a last one of the pair left over
def test_every_tile(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + K)
    x, w = (torch.randn(*s, generator=g, device="cuda") for s in ((M, K), (N, K)))
    b = torch.randn(N, generator=g, device="cuda")
    plain = ops.linear_act(x, w)
    r = slice(M - 70, M)
    assert torch.equal(plain[r], ops.linear_act(x[r], w))      # a row's sums do not depend on the tile it falls on
    assert torch.equal(ops.linear_act(x, w, bias=b, act="relu2"), torch.relu(plain + b) ** 2)
    x[1], x[2, ::3], x[M - 1] = x[1] * 2.0 ** -126, x[2, ::3] * 2.0 ** -120, x[M - 1] * 2.0 ** 20
    w[5], w[N - 1, ::3], w[8] = w[5] * 2.0 ** 100, w[N - 1, ::3] * 2.0 ** 60, w[8] * 2.0 ** -124
    got, want, size = ops.linear_act(x, w), x.to(F64) @ w.to(F64).T, x.to(F64).abs() @ w.to(F64).abs().T
    # K additions in f32, 2^-24 of each product left out; below 2^-126 one denormal (2^-149) per addition
    assert ((got.to(F64) - want).abs() <= (K + 2) * 6e-8 * size + K * 2.0 ** -149).all()
    rows, cols = [i for i in range(M) if i not in (1, 2, M - 1)], [i for i in range(N) if i not in (5, 8, N - 1)]
    assert torch.equal(got[rows][:, cols], plain[rows][:, cols])
    x[3, 5], x[M - 2, K - 1] = float("inf"), float("nan")
    w[1, 5], w[2] = 0, w[2].abs()
    got = ops.linear_act(x, w)
    assert got[3, 1].isnan() and got[3, 2] == float("inf") and got[M - 2].isnan().all()
    rows, cols = list(range(4, M - 2)), [i for i in cols if i not in (1, 2)]
    assert torch.equal(got[rows][:, cols], plain[rows][:, cols])


# groups on 64-row tiles, on 128-row ones of 128 and of 256 columns for both products, and ones that mix them
@pytest.mark.gpu
@pytest.mark.parametrize("T,E,Hd,F,plain", [(150, 8, 192, 160, False), (150, 8, 192, 160, True), (1500, 3, 1024, 1120, False),
                                            (1500, 3, 1024, 1120, True), (1900, 8, 192, 1056, False), (1900, 8, 2080, 160, True)])
def test_experts(T, E, Hd, F, plain):
    g = torch.Generator(device="cuda").manual_seed(T + F)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")                                     # noqa: E731
    x, ids, w = r(T, Hd + 4)[:, :Hd], torch.rand(T, E, generator=g, device="cuda").topk(2, -1).indices, r(T, 2).abs()
    gu, dn = r(E, F if plain else 2 * F, Hd) * Hd ** -0.5, r(E, Hd, F) * F ** -0.5
    x[3] *= 2.0 ** -110      # (its tiles are formed again; many hidden values to a row, so that no cancelled one is its norm)
    got = ops.moe_glu_ffn(x, ids.int(), w, gu, dn, 7.0, 1.702, 1.0, True, "relu2" if plain else None).to(F64)
    want = torch.zeros(T, Hd, dtype=F64, device="cuda")
    for e in range(E):
        t, j = (ids == e).nonzero(as_tuple=True)
        h = (x[t].to(F64) * w[t, j].to(F64)[:, None]) @ gu[e].to(F64).T
        c = torch.clamp(h[:, :F], max=7.0)
        a = torch.relu(h) ** 2 if plain else c * torch.sigmoid(1.702 * c) * (torch.clamp(h[:, F:], -7.0, 7.0) + 1)
        want.index_add_(0, t, a @ dn[e].to(F64).T)
    # rows of f32 sums, K additions of 2^-24 in each of two products, doubled by the square
    assert ((got - want).norm(dim=1) <= 4 * (Hd + F) ** 0.5 * 6e-8 * want.norm(dim=1) + 1e-30).all()
