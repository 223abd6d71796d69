"""Tiles of few rows that do not split K: packed weights with a column tile for each compute unit, short K under wide results."""
import pytest
import torch

from butterfly_amd import ops

pytestmark = pytest.mark.skipif(not ops.load_library(), reason="kernel library not built")


@pytest.mark.parametrize("M,N,kind", [(16, 16384, "skinny"), (16, 16512, "tile"), (17, 8192, "skinny"), (17, 8320, "tile"), (64, 32000, "tile"), (4, 32000, "stream")])
def test_short_products_under_wide_results(M, N, kind):
    p = ops.gemm_plan(M, N, 1024, "none")
    assert (p["kind"], p["splitk"]) == (kind, 1)


def _check(M, N, K, packed):
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16)
    wp = ops.pack_w256(w) if packed else None
    want = x.double() @ w.double().T
    # one rounding to bf16 (at most 2^-9 of an element) beside f32 sums
    assert (ops.linear(x, w, packed=wp).double() - want).norm() < 2.0 ** -8 * want.norm()
    if packed:
        d = ops.linear(x, w, packed=wp, defer=True)
        assert (ops.materialize(d).double() - want).norm() < 2.0 ** -8 * want.norm()
        v = want.view(M, N // 32, 2, 16)
        want = (torch.nn.functional.silu(v[:, :, 0]) * v[:, :, 1]).reshape(M, N // 2)
        assert (ops.linear(x, w, packed=wp, epilogue="silu").double() - want).norm() < 2.0 ** -8 * want.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("M", [5, 16, 17, 32, 33, 64, 65])
@pytest.mark.parametrize("N,K", [(20224, 256), (20480, 192), (20480, 1088), (32768, 256), (33024, 512)])
def test_packed(M, N, K):
    """Both sides of the rule's lines: 158, 160, 256 and 258 column tiles, three and four K steps."""
    _check(M, N, K, True)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [5, 16, 17, 33, 64])
@pytest.mark.parametrize("N,K", [(8320, 1024), (16512, 64), (16512, 960), (32000, 1024)])
def test_short(M, N, K):
    _check(M, N, K, False)


@pytest.mark.parametrize("M,N,K,sk", [(16, 8320, 2048, 3), (64, 8320, 2048, 3), (32, 16384, 2048, 2), (32, 2048, 2048, 8), (16, 1024, 1536, 4),
                                       (6, 15360, 4096, 4), (32, 16384, 4096, 4), (12, 65536, 2048, 1)])
def test_splits_of_streams(M, N, K, sk):
    p = ops.gemm_plan(M, N, K)
    assert (p["kind"], p["splitk"]) == ("tile", sk)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(16, 8320, 2048), (17, 12416, 1280), (33, 8448, 1088), (64, 16640, 320), (48, 12416, 4096)])
def test_splits_that_divide_nothing(M, N, K):
    _check(M, N, K, N % 256 == 0)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [5, 16, 32, 33, 64])
@pytest.mark.parametrize("N,K", [(14336, 4096), (16384, 2048), (9216, 4096)])
def test_packed_weights_split_by_their_own_estimate(M, N, K):
    """Fewer splits than of the row-major weight, or more; the sums have room in either."""
    _check(M, N, K, True)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("N,K", [(7936, 4096), (8192, 4096), (8448, 8192), (28672, 4096), (8192, 4032)])
def test_packed_weights_of_many_columns(M, N, K):
    """Two to four rows run the tiles of five; both sides of the rule's lines."""
    _check(M, N, K, True)
