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
