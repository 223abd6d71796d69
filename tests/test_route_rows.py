"""Router logits and choice of a few rows in one launch against the two launches of larger steps (the same sums)."""
import pytest
import torch

from butterfly_amd import ops


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,E,Hd,top,stride", [
    (1, 1, 64, 1, 0), (1, 8, 1024, 2, 0), (16, 8, 2048, 2, 8), (5, 12, 100, 3, 1), (3, 17, 512, 4, 0), (256, 32, 72, 6, 0),
])
def test_one_launch_routes_like_two(dt, T, E, Hd, top, stride):
    g = torch.Generator().manual_seed(T + E)
    x = torch.empty(T, Hd + stride, device="cuda", dtype=dt)[:, :Hd].copy_(torch.randn(T, Hd, generator=g))
    if T > 2:
        x[1] = float("nan")                                   # selects nothing: id -1, weight 0
    wr = torch.randn(E, Hd, generator=g).to("cuda", dt)
    bias, sel = torch.randn(2, E, generator=g).cuda()
    for scoring, sc in (("softmax", 0), ("sigmoid", 1)):
        for b, s, groups in ((None, None, (1, 1)), (bias, sel, (1, 1)), (bias, None, (4, 2))):
            if E % groups[0] or top > E // groups[0] * groups[1]:
                continue
            for renorm in (True, False):
                ids, w = ops.moe_route_scores(x, wr, top, scoring, renorm, b, s, groups, 1e-6, 1.5)
                logits = torch.empty(T, E, device="cuda")
                torch.ops.bfly.router_logits(x[:128], wr, logits[:128])      # (per token and expert: the same sums)
                torch.ops.bfly.router_logits(x[128:].contiguous(), wr, logits[128:])
                ids2, w2 = torch.empty_like(ids), torch.empty_like(w)
                torch.ops.bfly.moe_topk_scores(logits, b, top, sc, renorm, ids2, w2, s, *groups, 1e-6, 1.5)
                assert torch.equal(ids, ids2) and torch.equal(w, w2)
