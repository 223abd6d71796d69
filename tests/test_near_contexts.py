"""Decode steps whose contexts lie far below max_seq_len: the bound that decode attention is told follows the contexts."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from butterfly_amd import ops
from butterfly_amd.config import EngineConfig, ModelConfig
from butterfly_amd.engine.engine import LLMEngine
from butterfly_amd.models import build_model


def _engine(device, rows, **kw):
    cfg = ModelConfig(name="small", arch="llama", hidden_size=256, num_layers=2, num_heads=4, num_kv_heads=1, head_dim=128, intermediate_size=512,
                      vocab_size=512)
    model = build_model(cfg, device=torch.device(device), dtype=torch.bfloat16 if device == "cuda" else torch.float32)
    model.init_random(seed=3)
    ecfg = EngineConfig(max_batch=rows, max_seq_len=4096, kv_cache_tokens=8192, graph_batch_sizes=[rows],
                        dtype="bf16" if device == "cuda" else "fp32", **kw)
    return LLMEngine(cfg, engine_cfg=ecfg, device=torch.device(device), model=model)


def _step(runner, ctx, pages=250):
    B = len(ctx)
    tables = np.array([[(37 * b + 11 * j) % pages for j in range(runner.max_blocks)] for b in range(B)], dtype=np.int32)
    c = np.array(ctx, dtype=np.int32)
    return dict(ids=np.arange(1, B + 1, dtype=np.int32), pos=c - 1, ctx=c, tables=tables, slots=np.full(B, -1, dtype=np.int32))


@pytest.mark.parametrize("ctx", [[1], [60, 17], [5, 4096]])
def test_eager_steps_tell_their_longest_context(ctx):
    r = _engine("cpu", 4, use_graphs=False).runner
    inp = _step(r, ctx)
    assert r.decode_batch(inp).max_ctx == max(ctx)
    assert r.decode_batch(dict(inp, ctx=torch.from_numpy(inp["ctx"]))).max_ctx == max(ctx)
    n = len(ctx)
    man = SimpleNamespace(fill_decode_tables=lambda sids, t, c: c.__setitem__(slice(None), ctx), block_table=lambda s: [0, 1])
    real, r.kv = r.kv, SimpleNamespace(manager=man)
    plan = SimpleNamespace(num_decode=n, seq_ids=list(range(n + 1)), decode_positions=inp["pos"].tolist(), decode_slots=[0] * n,
                           prefill_starts=[0], prefill_lens=[3], prefill_slots=[[1, 2, 3]], prefill_final=[True])
    fb, _ = r.mixed_batch(plan, lambda s: [7] * 3)
    r.kv = real
    assert fb.num_decode == n and fb.max_ctx == max(ctx)


@pytest.mark.parametrize("B,hkv,bound", [(1, 8, 1 << 18), (24, 8, 8000), (64, 1, 4096), (200, 8, 4096), (256, 1, 1536), (5, 3, 70000)])
def test_buffers_hold_every_nearer_bound(B, hkv, bound):
    """(a workspace sized for max_seq_len is frozen when a step with a nearer bound comes)"""
    if not ops.load_library():
        pytest.skip("kernel library not built")
    op = torch.ops.bfly
    most = op.attn_decode_part_rows_up_to(B, 16 * hkv, hkv, bound)
    assert max(op.attn_decode_part_rows(B, 16 * hkv, hkv, m, 0) for m in range(1, bound + 1, 7 if bound < 10000 else 97)) <= most
    near = op.attn_decode_near(B, hkv, bound)
    flat = op.attn_decode_part_rows(B, hkv, hkv, bound, 0) == (max(1, 256 // hkv) + B) * hkv
    assert (near > 0) == flat and near < bound
    if near:                      # a workgroup per split under it: 16 rows for every split there is
        assert op.attn_decode_part_rows(B, hkv, hkv, near, 0) % 16 == 0
        assert op.attn_decode_near(B, hkv, near) == 0


@pytest.mark.gpu
def test_captured_steps_follow_their_contexts():
    """A bucket of pages end to end under max_seq_len is captured under the nearer bound too; the longest context picks the form, in
    any order of steps, with the eager step's results (replays between which the program computes and waits)."""
    rows = 64
    eng = _engine("cuda", rows)
    r = eng.runner
    for k, v in eng.kv.layers:
        k.normal_(generator=torch.Generator(device="cuda").manual_seed(1))
        v.normal_(generator=torch.Generator(device="cuda").manual_seed(2))
    assert eng.precapture_decode(rows)
    g = r.graphs[rows]
    assert g.near == 768 and len(g.forms) == 2
    for longest, form in ((40, 1), (4096, 0), (768, 1), (769, 0), (3, 1), (769, 0)):
        ctx = [longest] + [1 + (7 * i) % min(longest, 50) for i in range(rows - 2)]      # (one row of padding)
        inp = _step(r, ctx)
        out = r.run_decode(inp)
        assert out.data_ptr() == g.forms[form][1].data_ptr(), longest
        want = r.run(r.decode_batch(inp))
        torch.cuda.synchronize()
        assert torch.allclose(out.float(), want.float(), atol=5e-2, rtol=5e-2), longest
