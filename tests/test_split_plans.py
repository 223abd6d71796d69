"""Split-K choice of the 256 x 256 prefill tile."""
import pytest

from butterfly_amd import ops

pytestmark = pytest.mark.skipif(not ops.load_library(), reason="kernel library not built")


@pytest.mark.parametrize("K", [64, 512, 1024, 4096, 14336])
@pytest.mark.parametrize("N", [256, 1280, 2048, 8192])
def test_splits_pay_for_their_sums(K, N):
    for M in (257, 600, 1500, 3000, 6184, 8192):
        p = ops.gemm_plan(M, N, K)
        if p["kind"] != "big4" or p["bm"] != 256:
            continue
        tiles, sk = -(-M // 256) * -(-N // 256), p["splitk"]
        assert sk == 1 or K // 64 >= 8 * sk, (M, N, K, sk)          # eight K steps per split at least
        # a split has to shorten the rounds of 256 workgroups (each takes its share of K)
        assert sk == 1 or -(-tiles * sk // 256) < sk * -(-tiles // 256), (M, N, K, sk)


@pytest.mark.parametrize("K", [64, 128, 192, 1024, 4096])
@pytest.mark.parametrize("N", [128, 256, 1024, 1152, 1408, 2048, 8320])
def test_every_row_count_has_a_plan_that_runs(K, N):
    """One K step, whole and half column tiles: the plan chosen is one that its kernel takes."""
    import torch

    for M in (1, 16, 64, 200, 256, 257, 300, 512, 1000, 5000):
        for epi in ("none", "bias", "silu", "relu2"):
            assert torch.ops.bfly.gemm_check(M, N, K, ops.EPILOGUES[epi]) == 0, (M, N, K, epi)
