"""Products of 65 to some 2000 rows on mid-M tiles: where they run, and their results with every epilogue."""
import pytest
import torch

from butterfly_amd import ops
from butterfly_amd.ops import reference as ref

pytestmark = pytest.mark.skipif(not ops.load_library(), reason="kernel library not built")


@pytest.mark.parametrize("M,N,K,kind", [(64, 2048, 2048, "tile"), (65, 2048, 2048, "mid4"), (256, 6272, 2048, "mid4"), (100, 2048, 192, "tile"),
                                        (100, 2048, 8192, "tile"), (200, 2048, 8192, "mid4"), (257, 2048, 2048, "mid4"), (300, 1024, 1024, "mid4"),
                                        (320, 2688, 1024, "mid4"), (320, 4096, 2048, "mid4"), (300, 4096, 8192, "big4"),
                                        (937, 4096, 4096, "mid4"), (1000, 2048, 2048, "mid4"),
                                        (2100, 2048, 2048, "big4"), (1000, 8192, 8192, "big4"), (1000, 4224, 1024, "big4"), (8192, 8192, 8192, "big4")])
def test_where_they_run(M, N, K, kind):
    assert ops.gemm_plan(M, N, K)["kind"] == kind


# one and two row tiles with remainders, half column tiles, the shortest K, steps that no split divides evenly, two rounds of tiles
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(65, 128, 256), (129, 256, 320), (200, 1152, 448), (256, 2048, 2048), (130, 4224, 1088), (330, 1408, 1024),
                                   (777, 2048, 2048), (385, 1024, 4160), (255, 12416, 256)])
def test_results(M, N, K):
    assert ops.gemm_plan(M, N, K)["kind"] == "mid4"
    g = torch.Generator(device="cuda").manual_seed(M + N)
    xs, ws = (torch.randn(r, K + 8, generator=g, device="cuda").bfloat16() for r in (M, N))
    x, w = xs[:, :K], (ws * K ** -0.5)[:, 8:]      # rows that stand apart
    b = torch.randn(N, generator=g, device="cuda").bfloat16()
    glu = ops.glu_bias_block(b, 1.5, 1.702, 1.0)
    want = x.double() @ w.double().T
    v = want.view(M, N // 32, 2, 16)
    near = lambda got, want: bool((got.double() - want).norm() < 2.0 ** -8 * want.norm())           # one rounding to bf16  # noqa: E731
    out = torch.full((M, N + 8), 7.0, dtype=torch.bfloat16, device="cuda")
    assert near(ops.linear(x, w, out=out[:, :N]), want) and (out[:, N:] == 7).all()
    assert near(ops.linear(x, w, bias=b), want + b.double())
    assert near(ops.linear(x, w, epilogue="relu2"), torch.relu(want) ** 2)
    assert near(ops.linear(x, w, epilogue="silu"), (torch.nn.functional.silu(v[:, :, 0]) * v[:, :, 1]).reshape(M, N // 2))
    assert near(ops.linear(x, w, bias=glu, epilogue="glu"), ref.linear(x.double(), w.double(), glu, "glu").double())
    assert near(ops.materialize(ops.linear(x, w, defer=True)), want)
    if N % 256 == 0:
        wc = w.contiguous()
        assert near(ops.linear(x, wc, packed=ops.pack_w256(wc)), want)
