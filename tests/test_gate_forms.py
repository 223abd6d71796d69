"""Chunks of gated linear attention and of the forget gate in one launch (short sequences) and in two (records, then a chain): the
line between them, and that both give what a loop over the rows gives."""
import pytest
import torch

from butterfly_amd import ops

built = pytest.mark.skipif(not ops.load_library(), reason="kernel library not built")


@built
def test_which_steps_take_one_launch():
    forget, gla = torch.ops.bfly.forget_scan_launches, torch.ops.bfly.gla_scan_forms      # T, sequences, H, D, Dv, f32, max_rows
    assert [forget(n, 1, 16, 128, 128, False, 0) for n in (1, 16, 17, 1000)] == [1, 1, 2, 2]
    assert [forget(8 * n, 8, 16, 128, 128, False, n) for n in (32, 33)] == [1, 2]
    assert [forget(n, 1, 16, 128, 128, True, 0) for n in (16, 17)] == [1, 2]
    assert [forget(n, 1, 8, 64, 64, False, 0) for n in (32, 33)] == [1, 2]
    assert [forget(8 * 16, 8, 16, 128, 128, False, m) for m in (16, 0, 100)] == [1, 2, 2]      # (0: one might have them all)
    assert [forget(64 * 16, 64, 16, 128, 128, False, 16), forget(64 * 64, 64, 8, 64, 64, False, 64)] == [2, 1]
    assert forget(300, 1, 4, 512, 64, False, 0) == 1                                          # row by row
    # rows?, chunks (0 none, 1 in one launch, 2 in two), the fewest rows of a sequence in chunks
    assert [gla(n, 1, 16, 128, 128, False, 0) for n in (8, 16, 64)] == [[1, 0, -1], [0, 1, 0], [0, 2, 0]]
    assert [gla(8 * n, 8, 16, 128, 128, False, n)[1] for n in (16, 20, 32, 33)] == [1, 2, 1, 2]
    assert gla(16 + 256, 17, 32, 32, 32, False, 256) == [1, 2, 44]
    assert gla(16 + 64, 17, 16, 128, 128, False, 64) == [1, 0, -1]


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["gla", "forget"])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D,Dv", [(24, 40), (64, 64), (96, 130), (128, 64), (192, 60), (256, 128)])
@pytest.mark.parametrize("bad", [0.0, float("inf")])
def test_one_launch_and_two(kind, dt, D, Dv, bad):
    """Whole and padded chunks, an empty sequence and one without a slot; a value that is no number in a chunk's middle."""
    seqs = [(0, 16), (5, 17), (0, 32), (9, 15), (3, 0), (0, 31), (4, 9), (2, 12)]
    g = torch.Generator().manual_seed(D)
    n, H, T = len(seqs), 2 if D > 64 else 5, sum(m for _, m in seqs)
    rnd = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(dt)            # noqa: E731
    x = dict(q=rnd(T, H, D), v=rnd(T, H, Dv), state=torch.randn(n, H, D, Dv, generator=g))
    x["v"][20, 1, 3] += bad                                   # row 4 of the second sequence
    x["state_slots"] = torch.tensor([7, 6, 5, 4, 3, 2, -1, 0], dtype=torch.int32)
    x["row_cu"] = torch.tensor([sum(m for _, m in seqs[:i]) for i in range(n + 1)], dtype=torch.int32)
    x["positions"] = torch.cat([torch.arange(s, s + m) for s, m in seqs]).int()
    z = 2 + 2 * rnd(T, H * D)
    if kind == "gla":
        op, kw = ops.gla_scan, dict(tau=16.0, q_scale=D ** -0.5)
        x.update(k=rnd(T, H, D), z=z)
    else:
        op, kw = ops.forget_scan, dict(act="silu")
        x.update(z=z.view(T, H, D), f_bias=torch.randn(H * D, generator=g), lower=0.9 * torch.rand(H * D, generator=g))
    ref = {k: t.clone() for k, t in x.items()}
    want = op(**ref, **kw)
    rows = torch.ones(T, dtype=torch.bool)
    rows[16 + 17 + 32 + 15 + 31:][:9] = False                 # (no slot)
    for m in (32, 1000):                                      # as many rows are said to be the most: one launch, and two
        got = {k: t.clone().cuda() for k, t in x.items()}
        o = op(**got, **kw, max_rows=m).cpu()
        assert (o[~rows] == 0).all()
        for a, b in ((o[rows], want[rows]), (got["state"].cpu(), ref["state"])):
            ok = b.isfinite()
            assert torch.equal(a.isfinite(), ok)
            # f32 sums over up to 256 channels in another order, products of up to 16 decays; hardware exp / log for bf16 inputs
            assert (a - b)[ok].abs().max() < (3e-5 if dt == torch.bfloat16 else 1e-5) * b[ok].abs().max()


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("where", ["q", "k", "v", "z"])
@pytest.mark.parametrize("row", [0, 7, 11, 16, 30])      # of a whole chunk and one of 15 rows: both blocks, the last row
def test_values_that_are_no_numbers_in_one_launch(row, where, bad):
    g = torch.Generator().manual_seed(row)
    n, H, D, Dv = 31, 2, 32, 80
    assert torch.ops.bfly.gla_scan_forms(n, 1, H, D, Dv, False, 0) == [0, 1, 0]
    rnd = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)            # noqa: E731
    x = dict(q=rnd(n, H, D), k=rnd(n, H, D), v=rnd(n, H, Dv), z=2 + rnd(n, H * D), state=torch.randn(1, H, D, Dv, generator=g),
             state_slots=torch.tensor([0], dtype=torch.int32), row_cu=torch.tensor([0, n], dtype=torch.int32),
             positions=torch.arange(3, 3 + n).int())
    x[where].view(n, H, -1)[row, 1, 5] = bad
    got, ref = {k: t.cuda() for k, t in x.items()}, {k: t.clone() for k, t in x.items()}
    o, w = (ops.gla_scan(**a, tau=16.0, q_scale=D ** -0.5) for a in (got, ref))
    for a, b in ((o.cpu(), w), (got["state"].cpu(), ref["state"])):
        ok = b.isfinite()
        assert torch.equal(a.isfinite(), ok)
        # f32 sums in another order, products of up to 16 decays; hardware exp / log
        assert (a - b)[ok].abs().max() < 3e-5 * b[ok].abs().max()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["gla", "forget"])
@pytest.mark.parametrize("far,ld", [("qkz", (1 << 21) + 8), ("v", 1 << 26)])
def test_rows_far_apart(kind, far, ld):
    """Row strides that the 24-bit offsets of one launch and the 32-bit ones of two do not hold give what dense rows give."""
    n, H, D, Dv = 40, 2, 64, 64
    g = torch.Generator().manual_seed(1)
    rnd = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).cuda()            # noqa: E731
    q, k, v, z = rnd(n, H, D), rnd(n, H, D), rnd(n, H, Dv), rnd(n, H, D) + 2
    idx = [torch.tensor(t, dtype=torch.int32, device="cuda") for t in ([0], [0, n], list(range(n)))]
    apart = lambda t: torch.empty(n, ld, dtype=t.dtype, device="cuda")[:, :t[0].numel()].view(t.shape).copy_(t)      # noqa: E731
    fb, lo = torch.randn(H * D, generator=g).cuda(), (0.9 * torch.rand(H * D, generator=g)).cuda()

    def run(q, k, v, z):
        state = torch.zeros(1, H, D, Dv, device="cuda")
        if kind == "gla":
            return ops.gla_scan(q, k, v, z.view(n, H * D), state, *idx, 16.0, D ** -0.5), state
        return ops.forget_scan(q, z, v, fb, lo, state, *idx, "silu"), state

    want = run(q, k, v, z)
    got = run(apart(q), apart(k), v, apart(z)) if far == "qkz" else run(q, k, apart(v), z)
    # the same sums in f32, in another order
    for a, b in zip(got, want):
        assert (a - b).abs().max() < 3e-5 * b.abs().max()


@pytest.mark.gpu
@pytest.mark.parametrize("T,H", [(40, 0), (0, 2)])
def test_nothing_to_scan(T, H):
    D, Dv, z = 32, 64, lambda *s: torch.zeros(*s, device="cuda")            # noqa: E731
    idx = [torch.tensor(t, dtype=torch.int32, device="cuda") for t in ([0], [0, T], list(range(T)))]
    assert ops.gla_scan(z(T, H, D), z(T, H, D), z(T, H, Dv), z(T, H * D), z(1, H, D, Dv), *idx, 16.0, 1.0).shape == (T, H, Dv)
    assert ops.forget_scan(z(T, H, D), z(T, H, D), z(T, H, Dv), z(H * D), z(H * D), z(1, H, D, Dv), *idx).shape == (T, H, Dv)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["gla", "forget", "delta"])
@pytest.mark.parametrize("H,n", [(16, 8), (16, 9), (16, 16), (16, 17), (16, 40), (16, 41), (8, 63), (8, 64), (8, 65)])
def test_ragged_sequences_in_any_order(kind, H, n):
    """Sequences of the same, of no and of very different lengths (up to five rounds of 256 workgroups and 64 sequences take their places by length):
    each has the same result wherever it stands in the step."""
    g = torch.Generator(device="cuda").manual_seed(n)
    D = 128
    lens = [(0, 300, 300, 1, 17, 190, 64, 33)[i % 8] + 5 * (i // 8) * (i % 3) for i in range(n)]
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")            # noqa: E731
    heads = {k: [rnd(m, h, D) for m in lens] for k, h in (("q", H), ("k", H), ("v", H), ("z", H))}
    logits = {k: [rnd(m, H).to(torch.bfloat16) for m in lens] for k in "ab"}
    states = [rnd(H, D, D) for _ in lens]
    const = dict(a_log=0.5 * rnd(H) - 1, dt_bias=rnd(H), f_bias=rnd(H * D), lower=0.9 * torch.rand(H * D, generator=g, device="cuda"))

    def run(order):
        pick = lambda v: torch.cat([v[i] for i in order])                   # noqa: E731
        q, k, v, z = (pick(heads[x]) for x in "qkvz")
        cu = torch.tensor([sum(lens[i] for i in order[:j]) for j in range(n + 1)], dtype=torch.int32, device="cuda")
        pos = torch.cat([torch.arange(lens[i]) + 7 * (i % 2) for i in order]).int().cuda()
        st, slots = torch.stack([states[i] for i in order]), torch.arange(n, dtype=torch.int32, device="cuda")
        if kind == "delta":
            o = ops.delta_scan(q, k, v, pick(logits["b"]), pick(logits["a"]), const["a_log"], const["dt_bias"], st, slots, cu, pos,
                               D ** -0.5, 1e-6, max_rows=max(lens))
        elif kind == "gla":
            b = lambda t: t.to(torch.bfloat16)                              # noqa: E731
            o = ops.gla_scan(b(q), b(k), b(v), b(2 + z).view(-1, H * D), st, slots, cu, pos, 16.0, D ** -0.5, max_rows=max(lens))
        else:
            o = ops.forget_scan(q, z, v, const["f_bias"], const["lower"], st, slots, cu, pos, max_rows=max(lens))
        at = cu.tolist()
        return {i: (o[at[j]:at[j + 1]], st[j]) for j, i in enumerate(order)}

    a, b = run(list(range(n))), run([(5 * i + 3) % n if n % 5 else n - 1 - i for i in range(n)])
    for i in range(n):
        assert torch.equal(a[i][0], b[i][0]) and torch.equal(a[i][1], b[i][1]), (i, lens[i])
