"""Steps that mix decoded rows, short and long prompts: the recurrent scans take each sequence row by row or in chunks."""
import pytest
import torch

from butterfly_amd import ops

STEPS = {
    "single rows": [(9, 1)] * 20,
    "short prompts": [(0, 2), (5, 11), (0, 3), (7, 10)],                                   # none reaches the chunks
    "one short prompt": [(0, 8)],
    "one prompt": [(3, 45)],
    "prompts alone": [(0, 70), (5, 33), (0, 40)],                                          # one launch of chunks
    "mixed": [(9, 1)] * 30 + [(0, 16), (4, 15), (0, 12), (8, 11), (20, 61), (0, 32), (3, 31)],
    "a chunk and a little": [(9, 1)] * 20 + [(0, 17), (3, 20), (0, 24), (7, 28), (0, 33)],   # whether a padded chunk pays
    "empty and padded": [(9, 1)] * 9 + [(0, 0), (0, 50), (0, 0), (6, 14)] + [(1, 1)] * 3,      # (the last two: no slot)
}


def place(seqs):
    n = len(seqs)
    slots = torch.arange(n - 1, -1, -1, dtype=torch.int32)
    if any(m == 0 for _, m in seqs):
        slots[-2:] = -1
    cu = torch.tensor([sum(m for _, m in seqs[:i]) for i in range(n + 1)], dtype=torch.int32)
    return slots, cu, torch.cat([torch.arange(s, s + m) for s, m in seqs]).int()


def same(op, x, rows, **kw):
    got, ref = {k: t.cuda() for k, t in x.items()}, {k: t.clone() for k, t in x.items()}
    o, w = op(**got, **kw), op(**ref, **kw)
    # two f32 evaluations: sums over up to 96 channels in another order, products of up to 16 decays
    assert (o.cpu() - w)[rows].abs().max() < 1e-5 * w[rows].abs().max()
    assert (got["state"].cpu() - ref["state"]).abs().max() < 1e-5 * ref["state"].abs().max()


@pytest.mark.gpu
@pytest.mark.parametrize("H", [2, 24])      # (few workgroups: a single launch; many: one for either form)
@pytest.mark.parametrize("name", STEPS)
@pytest.mark.parametrize("which", ["gla", "gla bf16", "delta"])
def test_every_sequence_of_a_mixed_step(which, name, H):
    g = torch.Generator().manual_seed(H + len(name))
    rnd = lambda *s: torch.randn(*s, generator=g)            # noqa: E731
    slots, cu, pos = place(STEPS[name])
    T, n, D, Dv = len(pos), len(slots), 48, 96
    rows = torch.cat([torch.arange(int(a), int(b)) for a, b, s in zip(cu, cu[1:], slots) if s >= 0])
    idx = dict(state_slots=slots, row_cu=cu, positions=pos)
    hint = {"max_rows": max(m for _, m in STEPS[name])} if H == 2 else {}
    if which == "delta":
        same(ops.delta_scan, dict(q=rnd(T, H // 2, D), k=rnd(T, H // 2, D), v=rnd(T, H, Dv), b=rnd(T, H), a=rnd(T, H), a_log=rnd(H) - 1,
                                  dt_bias=rnd(H), state=rnd(n, H, Dv, D), **idx), rows, q_scale=D ** -0.5, **hint)
        return
    dt = torch.bfloat16 if "bf16" in which else torch.float32
    x = dict(q=rnd(T, H, D).to(dt), k=rnd(T, H, D).to(dt), v=rnd(T, H, Dv).to(dt), z=(2 + rnd(T, H * D)).to(dt),
             state=rnd(n, H, D, Dv), **idx)
    same(ops.gla_scan, x, rows, tau=16.0, q_scale=D ** -0.5, **hint)
