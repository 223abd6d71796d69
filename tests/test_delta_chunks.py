"""The gated delta rule over prompt rows (chunks of 16 on the f32 matrix cores) against a float64 token loop."""
import pytest
import torch

from butterfly_amd import ops

F64 = torch.float64


def step(seqs, H, G, D, Dv, seed, dt=torch.float32):
    """Inputs of one step over sequences (first position, rows): delta_scan's arguments up to the positions, on the CPU."""
    g = torch.Generator().manual_seed(seed)
    T, n = sum(n for _, n in seqs), len(seqs)
    rnd = lambda *s: torch.randn(*s, generator=g)            # noqa: E731
    return dict(q=rnd(T, G, D), k=rnd(T, G, D), v=rnd(T, H, Dv), b=(1 + rnd(T, H)).to(dt), a=rnd(T, H).to(dt), a_log=rnd(H) - 1,
                dt_bias=rnd(H), state=rnd(n, H, Dv, D), state_slots=torch.arange(n, dtype=torch.int32),
                row_cu=torch.tensor([sum(m for _, m in seqs[:i]) for i in range(n + 1)], dtype=torch.int32),
                positions=torch.cat([torch.arange(s, s + m) for s, m in seqs]).int())


def both(x, D, eps):
    """(outputs, state) of the kernel and of the f32 reference loop."""
    got, ref = {k: t.cuda() for k, t in x.items()}, {k: t.clone() for k, t in x.items()}
    o = ops.delta_scan(**got, q_scale=D ** -0.5, unit_eps=eps)
    w = ops.delta_scan(**ref, q_scale=D ** -0.5, unit_eps=eps)
    return (o.cpu(), got["state"].cpu()), (w, ref["state"])


@pytest.mark.gpu
@pytest.mark.parametrize("D,seqs", [(64, [(0, 17)]), (128, [(5, 20), (0, 39)]), (40, [(0, 30)])])
def test_unit_vectors_without_an_epsilon(D, seqs):
    """unit_eps 0: a last chunk that is partly empty has no vector of length zero."""
    for got, want in zip(*both(step(seqs, 2, 1, D, 48, D), D, 0.0)):
        assert (got - want).abs().max() < 1e-5 * want.abs().max()      # two f32 evaluations


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])      # (of the logits)
@pytest.mark.parametrize("H,G,D,Dv,seqs", [
    (4, 2, 128, 128, [(0, 17), (5, 16), (0, 1), (3, 2)]),       # chunk edges; fresh and continued sequences; one row beside prompts
    (3, 1, 24, 40, [(0, 33)]), (2, 2, 64, 64, [(7, 15), (0, 48)]),
    (2, 1, 70, 70, [(0, 31), (9, 32)]),                           # rows that are not a multiple of four elements
    (1, 1, 150, 96, [(0, 40)]), (2, 1, 256, 128, [(1, 100)]), (1, 1, 96, 256, [(0, 300), (0, 3)]),
])
def test_prompt_chunks_match_the_token_loop(dt, H, G, D, Dv, seqs):
    g = torch.Generator().manual_seed(D + Dv)
    T, nslots = sum(n for _, n in seqs), len(seqs) + 1
    rnd = lambda *s: torch.randn(*s, generator=g)            # noqa: E731
    q, k, v = rnd(T, G, D), rnd(T, G, D), rnd(T, H, Dv)
    k[1::5] = k[0::5][:len(k[1::5])]                        # the same key again at once: the strongest coupling inside a chunk
    k[2::7] *= 1e-3
    b, a = (1 + 3 * rnd(T, H)).to(dt), rnd(T, H).to(dt)
    a[3::9] += 40.0                                         # rows that forget everything, and rows that forget nothing
    a[4::3] -= 40.0
    a_log, dt_bias = rnd(H) - 1, rnd(H)
    st = rnd(nslots, H, Dv, D)
    slots = torch.randperm(nslots, generator=g)[:len(seqs)].int()
    cu = torch.tensor([sum(n for _, n in seqs[:i]) for i in range(len(seqs) + 1)], dtype=torch.int32)
    pos = torch.cat([torch.arange(s, s + n) for s, n in seqs]).int()
    unit = lambda x: (x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, 1)      # noqa: E731
    qu, ku = unit(q.to(F64)) * D ** -0.5, unit(k.to(F64))
    beta = torch.sigmoid(b.to(F64))
    decay = torch.exp(-torch.exp(a_log.to(F64)) * torch.nn.functional.softplus(a.to(F64) + dt_bias.to(F64)))
    want, state = torch.empty(T, H, Dv, dtype=F64), st.to(F64).clone()
    for s, (start, n) in enumerate(seqs):
        m = state[slots[s]] if start else torch.zeros(H, Dv, D, dtype=F64)
        for t in range(int(cu[s]), int(cu[s]) + n):
            m = decay[t][:, None, None] * m
            u = beta[t][:, None] * (v[t].to(F64) - (m @ ku[t][:, :, None])[:, :, 0])
            m = m + u[:, :, None] * ku[t][:, None]
            want[t] = (m @ qu[t][:, :, None])[:, :, 0]
        state[slots[s]] = m
    d = lambda t: t.to("cuda")                             # noqa: E731
    sd = d(st)
    o = ops.delta_scan(d(q), d(k), d(v), d(b), d(a), d(a_log), d(dt_bias), sd, d(slots), d(cu), d(pos), D ** -0.5, 1e-6)
    # f32 sums of up to 256 channels, a solve of up to 16 coupled rows, products of 16 decays (f32 eps 6e-8 each)
    for got, ref in ((o, want), (sd, state)):
        assert (got.cpu().to(F64) - ref).abs().max() < 5e-6 * ref.abs().max()


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("where", ["q", "k", "v", "a", "b"])
@pytest.mark.parametrize("row", [0, 7, 11, 16, 18])      # of two chunks: first row, both blocks, the last rows
def test_values_that_are_no_numbers_reach_later_rows_only(row, where, bad):
    """As in a loop over the rows: from their row on (q: in it), in their column (v) or all of them, and not another sequence."""
    D, Dv = 64, 80
    x = step([(3, 19), (0, 20)], 2, 2, D, Dv, row)
    x[where][row, 1, ...] = bad if where in "ab" else x[where][row, 1]
    if where not in "ab":
        x[where][row, 1, 5] = bad
    for got, want in zip(*both(x, D, 1e-6)):
        assert torch.equal(got.isfinite(), want.isfinite())
        ok = want.isfinite()
        assert (got - want)[ok].abs().max() < 1e-5 * want[ok].abs().max()


def loop64(x, D, eps):
    """The token loop in float64 on the GPU: outputs [T, H, Dv] and the state pool."""
    x = {k: t.cuda() for k, t in x.items()}
    H, G, cu = x["v"].shape[1], x["q"].shape[1], x["row_cu"].tolist()
    unit = lambda t: (t.to(F64) / torch.sqrt((t.to(F64) ** 2).sum(-1, keepdim=True) + eps)).repeat_interleave(H // G, 1)      # noqa: E731
    q, k, v, beta = unit(x["q"]) * D ** -0.5, unit(x["k"]), x["v"].to(F64), torch.sigmoid(x["b"].to(F64))
    decay = torch.exp(-torch.exp(x["a_log"].to(F64)) * torch.nn.functional.softplus(x["a"].to(F64) + x["dt_bias"].to(F64)))
    o, state = torch.zeros(v.shape, dtype=F64, device="cuda"), x["state"].to(F64).clone()
    for s, slot in enumerate(x["state_slots"].tolist()):
        if slot < 0 or cu[s] == cu[s + 1]:
            continue
        m = state[slot] if int(x["positions"][cu[s]]) else torch.zeros_like(state[slot])
        for t in range(cu[s], cu[s + 1]):
            m = decay[t][:, None, None] * m
            u = beta[t][:, None] * (v[t] - (m @ k[t][:, :, None])[:, :, 0])
            m = m + u[:, :, None] * k[t][:, None]
            o[t] = (m @ q[t][:, :, None])[:, :, 0]
        state[slot] = m
    return o.cpu(), state.cpu()


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,D,Dv,seqs,no_slot", [
    (8, 2, 128, 128, [(0, 300), (5, 161), (0, 2), (9, 0), (0, 17)], 3),       # an empty sequence; one without a slot
    (3, 3, 40, 33, [(7, 200), (0, 176)], None),                                 # one head to a key head, rows not a multiple of four
    (6, 1, 64, 80, [(0, 143), (3, 144), (0, 145)], 1),                          # last chunks of 15, 16 and 1 rows
    (10, 2, 96, 64, [(1, 257)], None), (4, 2, 150, 64, [(0, 250)], None), (8, 1, 256, 48, [(2, 400)], None),
    (64, 32, 128, 16, [(0, 6000)], None),                                       # more records than a launch holds
])
def test_chunks_in_two_launches_match_the_token_loop(H, G, D, Dv, seqs, no_slot):
    x = step(seqs, H, G, D, Dv, D + H, torch.bfloat16)
    if no_slot is not None:
        x["state_slots"][no_slot] = -1
    T, most = len(x["q"]), max(n for _, n in seqs)
    assert torch.ops.bfly.delta_record_floats(T, len(seqs), H, G, D, Dv, H * Dv, most) > 0
    got = {k: t.cuda() for k, t in x.items()}
    o = ops.delta_scan(**got, q_scale=D ** -0.5, unit_eps=1e-6, max_rows=most)
    want, state = loop64(x, D, 1e-6)
    # f32 sums of up to 256 channels, a solve of up to 16 coupled rows, products of 16 decays (f32 eps 6e-8 each)
    for a, b in ((o, want), (got["state"], state)):
        assert (a.cpu().to(F64) - b).abs().max() < 5e-6 * b.abs().max()


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("where", ["q", "k", "v", "a", "b"])
@pytest.mark.parametrize("row", [0, 23, 31, 149])      # of ten chunks: first row, both blocks, the last row
def test_two_launches_values_that_are_no_numbers_reach_later_rows_only(row, where, bad):
    D, Dv = 64, 80
    x = step([(3, 150), (0, 160)], 4, 2, D, Dv, row)
    assert torch.ops.bfly.delta_record_floats(310, 2, 4, 2, D, Dv, 4 * Dv, 160) > 0
    x[where][row, 1, ...] = bad if where in "ab" else x[where][row, 1]
    if where not in "ab":
        x[where][row, 1, 5] = bad
    got, ref = {k: t.cuda() for k, t in x.items()}, {k: t.clone() for k, t in x.items()}
    o = ops.delta_scan(**got, q_scale=D ** -0.5, unit_eps=1e-6, max_rows=160)
    w = ops.delta_scan(**ref, q_scale=D ** -0.5, unit_eps=1e-6)
    for a, b in ((o.cpu(), w), (got["state"].cpu(), ref["state"])):
        assert torch.equal(a.isfinite(), b.isfinite())
        ok = b.isfinite()
        assert (a - b)[ok].abs().max() < 1e-5 * b[ok].abs().max()      # two f32 evaluations


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,D,Dv,rows,one,two", [
    (16, 4, 128, 128, [64], 64, 128), (16, 4, 192, 192, [150] * 4, 150, 300), (8, 2, 256, 256, [100], 100, 500),
    (32, 8, 64, 64, [100] * 20, 100, 500), (6, 3, 200, 70, [90, 46, 33], 90, 450), (16, 4, 128, 100, [61], 61, 128),
])
def test_one_and_two_launches_agree_to_the_bit(H, G, D, Dv, rows, one, two):
    """Which form runs follows the bound that the caller gives; the values do not."""
    x = {k: t.cuda() for k, t in step([(3 * (i % 2), n) for i, n in enumerate(rows)], H, G, D, Dv, D + len(rows)).items()}
    floats = lambda m: torch.ops.bfly.delta_record_floats(sum(rows), len(rows), H, G, D, Dv, H * Dv, m)      # noqa: E731
    assert floats(one) == 0 < floats(two)
    outs = []
    for m in (one, two):
        state = x["state"].clone()
        outs.append((ops.delta_scan(**dict(x, state=state), q_scale=D ** -0.5, max_rows=m), state))
    for a, b in zip(*outs):
        assert torch.equal(a, b)
