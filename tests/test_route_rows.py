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


# us with one launch, with waves, with the GEMM (both with a choice launch) for (tokens, experts, width, f32)
TIMED = {(16, 8, 2048, False): (6.4, 8.4, None), (16, 32, 4096, False): (14.0, 13.0, None), (64, 16, 7168, True): (13.4, 10.8, None),
         (16, 32, 7168, False): (16.7, 13.9, None), (256, 32, 4096, False): (15, 34, 62), (8192, 32, 2048, False): (None, 77, 58),
         (4096, 32, 2048, False): (None, 44, 48), (512, 48, 1024, False): (None, 26, 23), (512, 48, 4096, False): (None, 41, 60),
         (2048, 8, 2048, False): (None, 12, 33), (16384, 16, 2048, False): (None, 76, 62), (8192, 64, 1024, False): (None, 79, 42),
         (8192, 32, 2048, True): (None, 151, 246), (16384, 32, 2048, True): (None, 293, 271), (8192, 64, 4096, True): (None, 531, 477)}


@pytest.mark.parametrize("step", TIMED)
def test_the_form_is_near_the_fastest(step):
    t = TIMED[step][("one launch", "waves", "gemm").index(ops.route_form(*step))]
    assert t < 1.05 * min(v for v in TIMED[step] if v), step


@pytest.mark.gpu
@pytest.mark.parametrize("T,E", [(300, 16), (200, 32), (300, 64), (70, 65)])
def test_router_rows_with_a_stride(T, E):
    """More than 4096 logits take a router whose rows are a view into wider ones."""
    g = torch.Generator().manual_seed(E)
    x, wide = torch.randn(T, 64, generator=g).cuda(), torch.randn(E, 80, generator=g).cuda()
    ids, w = ops.moe_route_scores(x, wide[:, :64], 2)
    ids2, w2 = ops.moe_route_scores(x, wide[:, :64].contiguous(), 2)
    assert torch.equal(ids, ids2) and (w - w2).abs().max() < 1e-5      # (sums of 64 f32 products in another order)
