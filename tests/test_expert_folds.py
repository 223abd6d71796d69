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
