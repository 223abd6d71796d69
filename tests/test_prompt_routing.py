"""Routing of prompt steps: router and choice on tiles, the choice among few experts, pairs sorted in parts."""
import pytest
import torch

from butterfly_amd import ops

F64 = torch.float64
pytestmark = pytest.mark.skipif(not ops.load_library(), reason="kernel library not built")


def _choice(logits, top, scoring, renorm, bias, sel):
    """ids, weights in 64 bits"""
    z = logits + (0 if bias is None else bias.to(F64))
    s = torch.softmax(z, -1) if scoring == "softmax" else torch.sigmoid(z)
    ids = (s if sel is None else s + sel.to(F64)).topk(top, -1).indices
    w = s.gather(1, ids)
    return s, ids, (w / (w.sum(-1, keepdim=True) + 1e-6) if renorm else w) * 1.5


@pytest.mark.gpu
@pytest.mark.parametrize("T,E,Hd,top", [(512, 8, 1024, 2), (1037, 16, 2048, 6), (2000, 1, 1024, 1), (700, 5, 3072, 5)])
@pytest.mark.parametrize("scoring", ["softmax", "sigmoid"])
def test_router_on_tiles(T, E, Hd, top, scoring):
    g = torch.Generator().manual_seed(T + E)
    x = torch.empty(T, Hd + 8, device="cuda", dtype=torch.bfloat16)[:, :Hd].copy_(torch.randn(T, Hd, generator=g))
    wr = (torch.randn(E, Hd, generator=g) * Hd ** -0.5).to("cuda", torch.bfloat16)
    bias, sel = 0.3 * torch.randn(2, E, generator=g).cuda()
    assert torch.ops.bfly.moe_route_tiles(x, wr, top, 1, 1) and not torch.ops.bfly.moe_route_tiles(x[:511], wr, top, 1, 1)
    for b, s in ((None, None), (bias, sel)):
        ids, w = ops.moe_route_scores(x, wr, top, scoring, True, b, s, (1, 1), 1e-6, 1.5)
        scores, want, ww = _choice(x.to(F64) @ wr.to(F64).T, top, scoring, True, b, s)
        near = scores if s is None else scores + s.to(F64)
        got, best = near.gather(1, ids.long()), near.gather(1, want)
        assert (got - best).abs().max() < 1e-5      # f32 sums of Hd products: near ties may swap
        assert all(len(set(r)) == top for r in ids[:64].tolist())
        same = (ids == want).all(-1)
        assert same.float().mean() > 0.99 and (w.to(F64) - ww)[same].abs().max() < 1e-5
    x[3] = float("nan")
    ids2, w2 = ops.moe_route_scores(x, wr, top, scoring, True, bias, sel, (1, 1), 1e-6, 1.5)
    assert (ids2[3] == -1).all() and torch.equal(ids2[4:], ids[4:]) and torch.equal(w2[:3], w[:3])


@pytest.mark.gpu
@pytest.mark.parametrize("E", [1, 8, 9, 16, 17, 32])
@pytest.mark.parametrize("scoring,code", [("softmax", 0), ("sigmoid", 1)])
@pytest.mark.parametrize("renorm", [False, True])
def test_choice_among_few(E, scoring, code, renorm):
    g = torch.Generator().manual_seed(E)
    T, top = 77, min(E, 5)
    logits, (bias, sel) = torch.randn(T, E, generator=g).cuda(), torch.randn(2, E, generator=g).cuda()
    logits[5], logits[6, 0], logits[7], logits[8] = float("nan"), -float("inf"), 2.0, -float("inf")
    for b, s in ((None, None), (bias, sel)):
        ids, w = torch.empty(T, top, dtype=torch.int32, device="cuda"), torch.empty(T, top, device="cuda")
        torch.ops.bfly.moe_topk_scores(logits, b, top, code, renorm, ids, w, s, 1, 1, 1e-6, 1.5)
        _, want, ww = _choice(logits.to(F64), top, scoring, renorm, b, s)
        keep = torch.tensor([t for t in range(T) if t not in (5, 7, 8) and (t != 6 or E > 1)], device="cuda")
        assert torch.equal(ids[keep].long(), want[keep]) and (w.to(F64) - ww)[keep].abs().max() < 1e-5
        assert (ids[5] == -1).all()
        if s is None and b is None:
            assert ids[7].tolist() == list(range(top))      # ties to the lowest


@pytest.mark.gpu
@pytest.mark.parametrize("T,E,skew", [(4096, 1, 0), (4097, 8, 0), (9000, 8, 3), (5000, 64, 0), (6001, 64, 60), (5000, 65, 0)])      # the last one in one workgroup
def test_pairs_sorted_in_parts(T, E, skew):
    """Every pair reaches its expert: experts that add their own number to a row."""
    g = torch.Generator().manual_seed(T)
    ids = torch.randint(skew, E, (T, 1), generator=g)
    ids[7], ids[T - 1] = E, -1                    # no expert: nothing is written for them
    Hd = F = 64
    x = torch.randn(T, Hd, generator=g).bfloat16()
    gu = torch.eye(Hd).bfloat16().repeat(E, 1, 1)
    dn = torch.eye(Hd).repeat(E, 1, 1) * torch.arange(1, E + 1)[:, None, None]
    got = ops.moe_glu_ffn(x.cuda(), ids.int().cuda(), torch.ones(T, 1).cuda(), gu.cuda(), dn.bfloat16().cuda(), 7.0, 1.0, 0.0, False, "relu2")
    want = torch.relu(x.float()) ** 2
    want = want.bfloat16().float() * (ids + 1)
    keep = [t for t in range(T) if t not in (7, T - 1)]
    assert ((got.cpu().float() - want)[keep].abs() <= 2.0 ** -8 * want[keep]).all()      # one rounding to bf16
