"""Results of the generic product and expert tiles that leave through LDS: short tiles, rows of any stride and alignment."""
import pytest
import torch

from butterfly_amd import ops
from tests.test_expert_tiles import reference

F64 = torch.float64


def draw(seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return lambda *s, k=1.0: k * torch.randn(*s, generator=g, device="cuda")


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(512, 128, 16), (513, 129, 72), (700, 200, 128), (600, 331, 40), (2000, 1000, 192), (511, 127, 24), (4200, 1001, 16)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("first,pad", [(0, 0), (8, 16), (3, 5), (1, 8)])
def test_products_into_any_rows(M, N, K, dtype, first, pad):
    r = draw(M + N)
    x, w, b = r(M, K).to(torch.bfloat16), r(N, K).to(torch.bfloat16), r(N).to(torch.bfloat16)
    buf = torch.full((M, N + first + pad), 77.0, device="cuda", dtype=dtype)
    out = buf[:, first:first + N]
    torch.ops.bfly.gemm_any(x, w, b, 1, 0.0, 0.0, out)
    acc = x.to(F64) @ w.to(F64).T + b.to(F64)
    want = torch.relu(acc) ** 2
    size = x.to(F64).abs() @ w.to(F64).abs().T + b.to(F64).abs()      # sums of K products: 2^-24 of it a step, twice of that squared
    tol = 2 * (K + 2) * 2.0 ** -24 * size * (acc.abs() + 1) + (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -22) * want
    assert ((out.to(F64) - want).abs() <= tol).all()
    assert (buf[:, :first] == 77).all() and (buf[:, first + N:] == 77).all()


@pytest.mark.gpu
@pytest.mark.parametrize("T,H,N,K,cols", [(600, 3, 192, 128, 192), (513, 2, 130, 64, 131), (700, 2, 128, 192, 144)])
def test_products_per_head_into_any_rows(T, H, N, K, cols):
    r = draw(T)
    x, w = r(T, H, K).to(torch.bfloat16), r(H, N, K, k=K ** -0.5).to(torch.bfloat16)
    buf = torch.full((T, H, cols), 77.0, device="cuda", dtype=torch.bfloat16)
    ops.linear_heads(x, w, buf[:, :, :N])
    want = torch.stack([x[:, h].to(F64) @ w[h].to(F64).T for h in range(H)], 1)
    assert ((buf[:, :, :N].to(F64) - want).abs() <= 2.0 ** -8 * want.abs() + K * 2.0 ** -18).all()      # (sums of |x w| below 64)
    assert (buf[:, :, N:] == 77).all()


@pytest.mark.gpu
@pytest.mark.parametrize("counts", [[300, 41, 0, 1], [20, 30], [700, 500]])
@pytest.mark.parametrize("Hd,F", [(250, 130), (132, 65), (320, 200), (256, 192)])
@pytest.mark.parametrize("plain", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_experts_of_any_width(counts, Hd, F, plain, dtype):
    r, E = draw(sum(counts) + F), len(counts)
    flat = torch.cat([torch.full((c,), e, device="cuda") for e, c in enumerate(counts)])
    ids = flat[torch.randperm(len(flat), device="cuda")].view(-1, 1)
    x, w = r(len(ids), Hd).to(dtype), r(len(ids), 1).abs() + 0.2
    gu, dn = r(E, F if plain else 2 * F, Hd, k=2 * Hd ** -0.5).to(dtype), r(E, Hd, F, k=F ** -0.5).to(dtype)
    got = ops.moe_glu_ffn(x, ids.int(), w, gu, dn, 7.0, 1.702, 1.0, False, "relu2" if plain else None).to(F64)
    with torch.device("cuda"):
        want = reference(x.to(F64), ids, w.to(F64), gu.to(F64), dn.to(F64), 7.0, 1.702, 1.0, False, plain)
    # bf16 hidden rows and output (2^-9 each), or f32 sums of up to 250 products, in every row
    tol = 2.0 ** -7 if dtype == torch.bfloat16 else 1e-5
    assert ((got - want).norm(dim=1) <= tol * want.norm(dim=1) + 1e-30).all()
