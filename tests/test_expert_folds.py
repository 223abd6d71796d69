"""Experts over a few rows, their weights streamed 16 rows a workgroup (moe_up_fold_kernel, moe_down_fold_kernel)."""
import pytest
import torch

from butterfly_amd import ops
from tests.test_expert_tiles import reference


@pytest.mark.gpu
@pytest.mark.parametrize("counts,Hd,F,plain,scaled", [
    ([1, 0, 0, 0, 0, 0, 0, 0], 128, 128, False, True),           # one row, one K step
    ([8, 9, 1, 0, 2, 0, 0, 0], 384, 128, False, True),           # both sides of the fold; steps for some waves only
    ([16, 9, 0, 3, 0, 0, 0, 0], 1152, 640, False, False),       # a whole pass; a remainder of the K steps
    ([17, 5, 2, 1, 0, 0, 0, 0], 256, 320, True, False),          # two passes (the down product does not fold: 320 channels)
    ([25, 0, 7, 0, 0, 0, 0, 0], 640, 2176, True, True),
    ([60, 2, 3, 1] + [1] * 60, 2048, 128, False, False),         # rows found through the sorted list
    ([3, 0, 1, 7, 9, 2, 1, 17], 2048, 1024, False, True),         # loaded past the caches
    ([3, 0, 1, 7, 9, 2, 1, 17, 10], 2048, 1024, True, False),
    # sixteen pairs, of which no group can be crowded, and one more
    ([16, 0, 0, 0, 0, 0, 0, 0], 2048, 640, False, True),
    ([9, 0, 7, 0, 0, 0, 0, 0], 2304, 384, True, False),
    ([16, 0, 0, 1, 0, 0, 0, 0], 2048, 2048, False, False),
    # crowded groups: 17 to 64 rows at once, pieces that do not fill their eights, groups whose pieces alternate, both products
    ([17, 31, 0, 0, 0, 0, 0, 0], 2048, 128, False, True),
    ([32, 16, 0, 0, 0, 0, 0, 0], 2176, 640, True, False),
    ([0, 33, 15, 0, 0, 0, 0, 0], 2048, 384, False, False),
    ([48, 0, 0, 0, 0, 0, 0, 0], 2112, 1024, False, True),
    ([64] + [0] * 15, 2048, 256, True, True),
    ([20, 0, 24, 0, 20] + [0] * 11, 2048, 2048, False, True),
    ([80, 64, 129, 1] + [0] * 60, 2048, 192, False, True),       # through the list: whole tiles of 64 rows and what is left of them
    ([18, 21, 40, 2] + [0] * 60, 2048, 128, True, False),
])
def test_few_rows(counts, Hd, F, plain, scaled):
    g = torch.Generator().manual_seed(sum(counts) + F)
    counts = counts if Hd >= 2048 else counts + [0] * 56
    E, TK = len(counts), sum(counts)
    ids = torch.cat([torch.full((c,), e) for e, c in enumerate(counts)])[torch.randperm(TK, generator=g)].view(-1, 1)
    bf = lambda *s, k=1.0: (k * torch.randn(*s, generator=g)).to(torch.bfloat16)            # noqa: E731
    x, w = bf(TK, Hd), torch.rand(TK, 1, generator=g) + 0.2
    gu, dn = bf(E, F if plain else 2 * F, Hd, k=2 * Hd ** -0.5), bf(E, Hd, F, k=F ** -0.5)
    f64 = lambda *t: [v.to(torch.float64) for v in t]                                          # noqa: E731
    xd = torch.empty(TK, Hd + 8, dtype=torch.bfloat16, device="cuda")[:, :Hd].copy_(x)          # rows with a stride
    assert 2 * TK <= (12 if Hd >= 2048 else 1) * E      # (else the streams of 32 rows)
    got = ops.moe_glu_ffn(xd, ids.int().cuda(), w.cuda(), gu.cuda(), dn.cuda(), 7.0, 1.702, 1.0, scaled, "relu2" if plain else None)
    want = reference(*f64(x), ids, *f64(w, gu, dn), 7.0, 1.702, 1.0, scaled, plain)
    # bf16 input rows times their score, hidden rows and output (2^-9 each); the squared activation doubles the first
    assert (got.cpu().to(torch.float64) - want).norm() / want.norm() < 6e-3


@pytest.mark.gpu
@pytest.mark.parametrize("Hd,F,plain", [(2048, 640, False), (2304, 128, True)])
def test_a_row_beside_many_others(Hd, F, plain):
    """Up to eight rows fold K; from nine on a row's sums do not depend on how many others share its expert."""
    g = torch.Generator(device="cuda").manual_seed(F)
    bf = lambda *s, k=1.0: (k * torch.randn(*s, generator=g, device="cuda")).to(torch.bfloat16)            # noqa: E731
    E, x = 32, bf(64, Hd)
    w = torch.rand(64, 1, generator=g, device="cuda") + 0.2
    gu, dn = bf(E, F if plain else 2 * F, Hd, k=2 * Hd ** -0.5), bf(E, Hd, F, k=F ** -0.5)
    run = lambda T: ops.moe_glu_ffn(x[:T], torch.full((T, 1), 3, device="cuda", dtype=torch.int32), w[:T], gu, dn, 7.0, 1.702, 1.0, True,  # noqa: E731
                                    "relu2" if plain else None)
    want = run(9)
    for T in (16, 17, 32, 33, 48, 64):
        got = run(T)
        assert torch.equal(got[:9], want), T
