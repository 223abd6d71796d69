"""Gated linear attention over prompt rows (chunks of 16 on the f32 matrix cores) against a float64 token loop."""
import pytest
import torch

from butterfly_amd import ops

F64 = torch.float64


@pytest.mark.gpu
@pytest.mark.parametrize("dt,tol", [(torch.float32, 3e-6), (torch.bfloat16, 3e-5)])
@pytest.mark.parametrize("H,D,Dv,seqs", [
    (2, 128, 128, [(0, 17), (5, 16), (0, 1), (3, 2)]),       # chunk edges; fresh and continued sequences; one row beside prompts
    (3, 24, 40, [(0, 33)]), (1, 96, 64, [(7, 15), (0, 48)]),   # sizes between the channel tiles
    (1, 200, 70, [(0, 31)]), (2, 256, 128, [(1, 100)]), (2, 64, 256, [(0, 300), (0, 3)]),
])
def test_prompt_chunks_match_the_token_loop(dt, tol, H, D, Dv, seqs):
    token_loop(dt, tol, H, D, Dv, seqs)


@pytest.mark.gpu
@pytest.mark.parametrize("dt,tol", [(torch.float32, 3e-6), (torch.bfloat16, 3e-5)])
@pytest.mark.parametrize("H,D,Dv,seqs", [      # whole chunks, one row over, one short; all channel tiles
    (2, 128, 128, [(0, 64)]), (2, 128, 128, [(5, 65), (0, 111), (0, 1), (3, 2)]), (3, 128, 72, [(0, 79), (7, 33)]),
    (3, 24, 40, [(0, 127)]), (2, 32, 64, [(4, 97), (0, 160)]), (1, 96, 64, [(7, 81), (0, 48)]), (2, 80, 100, [(0, 144)]),
    (1, 192, 128, [(0, 49), (2, 64)]), (2, 64, 64, [(0, 113), (6, 64)]), (1, 250, 30, [(0, 35)]),
])
def test_long_prompts_match_the_token_loop(dt, tol, H, D, Dv, seqs):
    """Steps whose every sequence runs in chunks, in two launches."""
    assert torch.ops.bfly.gla_scan_forms(sum(n for _, n in seqs), len(seqs), H, D, Dv, dt == torch.float32, 0) == [0, 2, 0]
    token_loop(dt, tol, H, D, Dv, seqs)


def token_loop(dt, tol, H, D, Dv, seqs):
    g = torch.Generator().manual_seed(D + Dv)
    T, nslots, tau = sum(n for _, n in seqs), len(seqs) + 1, 16.0
    rnd = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(dt)            # noqa: E731
    q, k, v, z = rnd(T, H, D), rnd(T, H, D), rnd(T, H, Dv), 2 + 2 * rnd(T, H * D)
    z[:, ::7] -= 40.0                                       # channels that forget at once, and others that never do
    z[:, 3::11] += 60.0
    st = torch.randn(nslots, H, D, Dv, generator=g)
    slots = torch.randperm(nslots, generator=g)[:len(seqs)].int()
    cu = torch.tensor([sum(n for _, n in seqs[:i]) for i in range(len(seqs) + 1)], dtype=torch.int32)
    pos = torch.cat([torch.arange(s, s + n) for s, n in seqs]).int()
    a = torch.sigmoid(z.to(F64)).view(T, H, D) ** (1 / tau)
    want, state = torch.empty(T, H, Dv, dtype=F64), st.to(F64).clone()
    for s, (start, n) in enumerate(seqs):
        m = state[slots[s]] if start else torch.zeros(H, D, Dv, dtype=F64)
        for t in range(int(cu[s]), int(cu[s]) + n):
            m = a[t][:, :, None] * m + k[t].to(F64)[:, :, None] * v[t].to(F64)[:, None]
            want[t] = ((q[t].to(F64) * D ** -0.5)[:, None] @ m)[:, 0]
        state[slots[s]] = m
    d = lambda t: t.to("cuda")                             # noqa: E731
    sd = d(st)
    o = ops.gla_scan(d(q), d(k), d(v), d(z), sd, d(slots), d(cu), d(pos), tau, D ** -0.5)
    # f32 sums of up to 256 channels and products of 16 decays (f32 eps 6e-8 each); hardware exp / log for bf16 inputs
    for got, ref in ((o, want), (sd, state)):
        assert (got.cpu().to(F64) - ref).abs().max() < tol * ref.abs().max()


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("where", ["q", "k", "v", "z"])
@pytest.mark.parametrize("row", [0, 7, 11, 16, 31, 33])      # of three chunks: first row, both blocks, the last rows
def test_values_that_are_no_numbers_reach_later_rows_only(row, where, bad):
    """As in a loop over the rows: from their row on (q: in it), in their column (v) or state row (k, z), and not another
    sequence."""
    g = torch.Generator().manual_seed(row)
    seqs, H, D, Dv = [(3, 35), (0, 40)], 2, 64, 80
    T, rnd = 75, lambda *s: torch.randn(*s, generator=g)            # noqa: E731
    x = dict(q=rnd(T, H, D), k=rnd(T, H, D), v=rnd(T, H, Dv), z=2 + rnd(T, H * D), state=rnd(2, H, D, Dv),
             state_slots=torch.tensor([1, 0], dtype=torch.int32), row_cu=torch.tensor([0, 35, 75], dtype=torch.int32),
             positions=torch.cat([torch.arange(s, s + n) for s, n in seqs]).int())
    x[where].view(T, H, -1)[row, 1, 5] = bad
    got, ref = {k: t.cuda() for k, t in x.items()}, {k: t.clone() for k, t in x.items()}
    o, w = (ops.gla_scan(**a, tau=16.0, q_scale=D ** -0.5) for a in (got, ref))
    for a, b in ((o.cpu(), w), (got["state"].cpu(), ref["state"])):
        assert torch.equal(a.isfinite(), b.isfinite())
        ok = b.isfinite()
        assert (a - b)[ok].abs().max() < 1e-5 * b[ok].abs().max()


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("where", ["q", "k", "v", "z"])
@pytest.mark.parametrize("row", [0, 7, 11, 16, 47, 69])
@pytest.mark.parametrize("D", [64, 128])
def test_values_that_are_no_numbers_in_long_prompts(D, row, where, bad):
    """The same where both sequences are long enough for chunks in two launches; the first ends in a chunk of six rows."""
    g = torch.Generator().manual_seed(row)
    seqs, H, Dv = [(3, 70), (0, 100)], 2, 80
    T, rnd = 170, lambda *s: torch.randn(*s, generator=g)            # noqa: E731
    assert torch.ops.bfly.gla_scan_forms(T, 2, H, D, Dv, True, 0) == [0, 2, 0]
    x = dict(q=rnd(T, H, D), k=rnd(T, H, D), v=rnd(T, H, Dv), z=2 + rnd(T, H * D), state=rnd(2, H, D, Dv),
             state_slots=torch.tensor([1, 0], dtype=torch.int32), row_cu=torch.tensor([0, 70, T], dtype=torch.int32),
             positions=torch.cat([torch.arange(s, s + n) for s, n in seqs]).int())
    x[where].view(T, H, -1)[row, 1, 5] = bad
    got, ref = {k: t.cuda() for k, t in x.items()}, {k: t.clone() for k, t in x.items()}
    o, w = (ops.gla_scan(**a, tau=16.0, q_scale=D ** -0.5) for a in (got, ref))
    for a, b in ((o.cpu(), w), (got["state"].cpu(), ref["state"])):
        assert torch.equal(a.isfinite(), b.isfinite())
        ok = b.isfinite()
        assert (a - b)[ok].abs().max() < 1e-5 * b[ok].abs().max()


@pytest.mark.gpu
def test_records_of_a_long_step_come_in_parts():
    """More chunks than are prepared at once (256 MB of records: 222 chunks of 64 heads of 128): sequences that end, begin and go
    on from one part to the next give what each gives in a step of its own, bit for bit."""
    g = torch.Generator().manual_seed(1)
    seqs, H, D, Dv = [(0, 1203), (7, 1777), (0, 20), (2, 2600)], 64, 128, 24
    T = sum(n for _, n in seqs)
    rnd = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).cuda()            # noqa: E731
    q, k, v, z = rnd(T, H, D), rnd(T, H, D), rnd(T, H, Dv), 2 + rnd(T, H * D)
    state = torch.randn(4, H, D, Dv, generator=g).cuda()
    cu = [sum(n for _, n in seqs[:i]) for i in range(5)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")                  # noqa: E731
    pos = [torch.arange(s, s + n).int().cuda() for s, n in seqs]
    got = state.clone()
    o = ops.gla_scan(q, k, v, z, got, i32([2, 0, 3, 1]), i32(cu), torch.cat(pos), 16.0, D ** -0.5)
    for i, slot in enumerate([2, 0, 3, 1]):
        r = slice(cu[i], cu[i + 1])
        one = state.clone()
        w = ops.gla_scan(q[r], k[r], v[r], z[r], one, i32([slot]), i32([0, seqs[i][1]]), pos[i], 16.0, D ** -0.5)
        assert torch.equal(o[r], w) and torch.equal(got[slot], one[slot])
