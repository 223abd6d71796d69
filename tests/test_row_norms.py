"""Layer norms with the row in registers or in LDS, scaled embeddings."""
import pytest
import torch

from butterfly_amd import ops

F64 = torch.float64
pytestmark = pytest.mark.skipif(not ops.load_library(), reason="kernel library not built")


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("W", [4, 252, 260, 1024, 1028, 2048, 4096, 8192, 8196, 130])
def test_layer_norm_rows(dt, W):
    g = torch.Generator().manual_seed(W)
    x, w, b = torch.randn(9, W, generator=g) * 3 + 5, torch.randn(W, generator=g), torch.randn(W, generator=g)
    for idx in (None, torch.tensor([8, 0, 3, 3])):
        got = ops.layer_norm_rows(x.cuda(), w.cuda(), b.cuda(), 1e-6, None if idx is None else idx.cuda(), dt).cpu().to(F64)
        want = torch.nn.functional.layer_norm((x if idx is None else x[idx]).to(F64), (W,), w.to(F64), b.to(F64), 1e-6)
        assert (got - want).abs().max() < (1e-5 if dt == torch.float32 else 2.0 ** -8) * (1 + want.abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,W", [(1, 4), (3, 1028), (5000, 1024), (7, 130)])
def test_scaled_embedding(dt, T, W):
    g = torch.Generator().manual_seed(W)
    table, ids = torch.randn(50, W, generator=g).to(dt), torch.randint(0, 50, (T,), generator=g).int()
    got = ops.embed_scaled(ids.cuda(), table.cuda(), 0.37)
    assert torch.equal(got.cpu(), table[ids.long()].float() * torch.tensor(0.37))
