"""Rotation and cache writes of several rows per workgroup against one row each (the same values)."""
import pytest
import torch

from butterfly_amd import ops


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T", [1024, 1027, 1792, 1795, 4096, 4099])
@pytest.mark.parametrize("H,G,D,Dv,nrot,bs", [(4, 2, 128, 64, 32, 32), (3, 1, 36, 40, 5, 12), (2, 2, 20, 17, 10, 16), (1, 1, 300, 8, 140, 8)])
def test_rows_together_and_alone(dt, T, H, G, D, Dv, nrot, bs):
    g = torch.Generator(device="cuda").manual_seed(T + D)
    wide = torch.randn(T, H * D + G * D + G * Dv + 1, generator=g, device="cuda").to(dt)
    slots, at, free = [], 0, 2 * bs
    for n in (1, 7, 8, 130, 64, 333, T):              # sequences that begin anywhere, each on pages of its own; rows without a place
        n = min(n, T - at)
        slots += [-1] * min(3, n) + list(range(free, free + n))[min(3, n):]
        at, free = at + n, free + -(-n // bs) * bs + bs * (n % 2)
    slots = torch.tensor(slots, dtype=torch.int32, device="cuda")
    pos = torch.randint(0, 5000, (T,), generator=g, device="cuda").int()
    inv = 10000.0 ** (-torch.arange(nrot, device="cuda") / nrot)
    pages = free // bs + 2

    def run(step):
        x = wide.clone()
        q, k = x[:, :H * D].unflatten(1, (H, D)), x[:, H * D:(H + G) * D].unflatten(1, (G, D))
        v = x[:, (H + G) * D:(H + G) * D + G * Dv].unflatten(1, (G, Dv))
        kc, vc = torch.full((pages, G, bs, D), 7.0, device="cuda", dtype=dt), torch.full((pages, G, Dv, bs), 7.0, device="cuda", dtype=dt)
        for i in range(0, T, step):
            ops.rope_partial_kv(q[i:i + step], k[i:i + step], v[i:i + step], pos[i:i + step].contiguous(), inv,
                                slots[i:i + step].contiguous(), kc, vc)
        return x, kc, vc

    for a, b in zip(run(T), run(512)):
        assert torch.equal(a, b)


def _turned(x, pos, inv):
    """Pairs (2 i, 2 i + 1) of the last dimension: u c - (w s), w c + (u s), the products in brackets rounded to f32, then the sums."""
    a = (pos.float()[:, None] * inv).double()[:, None]
    c, s = a.cos().float(), a.sin().float()
    u, w = x[..., 0::2].float(), x[..., 1::2].float()
    y = torch.stack([u.double() * c.double() - (w * s).double(), w.double() * c.double() + (u * s).double()], -1)
    return y.float().flatten(-2)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T", [5, 1792, 4096])
@pytest.mark.parametrize("D", [64, 66])               # accesses of 16 bytes and single pairs
def test_every_form_rounds_alike(dt, T, D):
    """The rotation's two products are rounded in one order everywhere, so that a row's values depend neither on the rows beside it
    nor on which kernel turned it (a float64 sum is off by a second rounding in fewer than one of 2^28 values)."""
    g = torch.Generator(device="cuda").manual_seed(T + D)
    x = torch.randn(T, 4, D, generator=g, device="cuda").to(dt)
    pos = torch.randint(0, 5000, (T,), generator=g, device="cuda").int()
    inv = 10000.0 ** (-torch.arange(D // 2, device="cuda") / (D // 2))
    want = _turned(x, pos, inv).to(dt)
    out = torch.empty_like(x)
    ops.rope_heads_copy(x, out, pos, inv)
    assert torch.equal(out, want)
    ops.rope_partial_kv(x, None, None, pos, inv)
    assert torch.equal(x, want)
