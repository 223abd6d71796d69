"""Products of few rows as weight streams (gemm_stream_kernel): every tile, the rules' edges, the epilogues, deferred sums."""
import pytest
import torch

from butterfly_amd import ops
from butterfly_amd.ops import reference as ref

pytestmark = pytest.mark.skipif(not ops.load_library(), reason="kernel library not built")

DEV = "cuda"
# [kind, row tiles, column tiles, waves, chunks in flight, fold, 1] and the rows it takes
PLANS = [([8, 1, 1, 4, 4, 4, 1], 4), ([8, 1, 1, 4, 4, 2, 1], 8), ([8, 1, 1, 8, 4, 2, 1], 8), ([8, 1, 2, 8, 4, 2, 1], 8),
         ([8, 1, 1, 4, 4, 1, 1], 16), ([8, 1, 1, 8, 4, 1, 1], 16), ([8, 1, 2, 8, 4, 1, 1], 16), ([8, 2, 1, 8, 4, 1, 1], 32)]


def _operands(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(M + 7 * N + K)
    x, w = (torch.randn(*s, generator=g, device=DEV).to(torch.bfloat16) for s in ((M, K), (N, K)))
    return x, (w * K ** -0.5).to(torch.bfloat16)


def _near(out, want):
    # one rounding to bf16 (at most 2^-9 of an element) beside f32 sums
    assert (out.double() - want).norm() < 2.0 ** -8 * want.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("plan,rows", PLANS)
@pytest.mark.parametrize("chunks", [1, 3, 17, 37])      # fewer chunks than waves, a last step of some waves only, a last step of fewer
def test_every_tile(plan, rows, chunks):
    K, N = 64 * plan[5] * chunks, 160
    for M in (1, rows - 1, rows):
        x, w = _operands(M, N, K)
        want = x.double() @ w.double().T
        for epi in ("none", "silu"):
            out = torch.full((M, N // 2 if epi == "silu" else N), float("nan"), device=DEV, dtype=torch.bfloat16)
            torch.ops.bfly.gemm_with_plan(x, w, out, plan, ops.EPILOGUES[epi], None, None)
            if epi == "silu":
                v = want.view(M, N // 32, 2, 16)
                want = (torch.nn.functional.silu(v[:, :, 0]) * v[:, :, 1]).reshape(M, N // 2)
            _near(out, want)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 4, 5, 8, 9, 16, 17, 32, 33])
@pytest.mark.parametrize("N,K", [(128, 128), (1024, 1024), (2688, 1152), (4224, 1024), (2048, 2048), (5248, 2048), (4096, 4224), (2048, 8192), (10368, 4096)])
def test_rules(M, N, K):
    """Whatever form the rules choose on both sides of their lines, with rows that stand apart in memory."""
    xs, ws = _operands(M, N, K + 64)
    x, w = xs[:, :K], ws[:, 64:]
    want = x.double() @ w.double().T
    g = torch.Generator(device=DEV).manual_seed(K)
    bias = torch.randn(N, generator=g, device=DEV).to(torch.bfloat16)
    _near(ops.linear(x, w), want)
    _near(ops.linear(x, w, bias=bias), want + bias.double())
    _near(ops.linear(x, w, epilogue="relu2"), torch.relu(want) ** 2)
    glu = ops.glu_bias_block(bias, 1.5, 1.702, 1.0)
    _near(ops.linear(x, w, bias=glu, epilogue="glu"), ref.linear(x.double(), w.double(), glu, "glu").double())
    # a reader that takes the sums gets the same rows
    assert torch.equal(ops.materialize(ops.linear(x, w, defer=True)), ops.linear(x, w))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,epi", [(1, 10240, 8192, "none"), (1, 1024, 1024, "none"), (1, 57344, 8192, "silu"), (4, 2048, 2048, "silu"), (8, 4096, 4096, "none"),
                                       (16, 3072, 2048, "none"), (30, 2560, 1024, "none"), (3, 28672, 4096, "none"), (4, 24576, 4096, "silu")])
def test_packed_copies_of_few_rows(M, N, K, epi):
    """The operator over a packed copy, which `linear` leaves for the weight where rows stream: the same streams, bit for bit, or (two to four rows
    of many columns) the tiles of five."""
    x, w = _operands(M, N, K)
    want = ops.linear(x, w, epilogue=epi)
    assert ops.gemm_plan(M, N, K, epi)["kind"] == "stream" and torch.ops.bfly.gemm_packed_check(M, N, K, ops.EPILOGUES[epi]) == 0
    out = torch.full_like(want, float("nan"))
    ws = torch.zeros(torch.ops.bfly.gemm_workspace_size(M, N, K) // 4 + 1, dtype=torch.float32, device=DEV)
    assert torch.ops.bfly.gemm_packed(x, ops.pack_w256(w), out, ops.EPILOGUES[epi], None, 0.0, None, 0, 1, ws) == 1
    if torch.ops.bfly.gemm_streams(M, N, K, ops.EPILOGUES[epi]):
        assert torch.equal(out, want)
    exact = x.double() @ w.double().T
    if epi == "silu":
        v = exact.view(M, N // 32, 2, 16)
        exact = (torch.nn.functional.silu(v[:, :, 0]) * v[:, :, 1]).reshape(M, N // 2)
    _near(out, exact)
