"""Residual step with a norm on both sides, rows held in registers (and the widths beside them) against float64."""
import pytest
import torch

from butterfly_amd import ops

F64 = torch.float64


def norm(x, w, b, eps):
    if b is None:
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps) * w + b


@pytest.mark.gpu
@pytest.mark.parametrize("dt,tol", [(torch.float32, 4e-6), (torch.bfloat16, 2.0 ** -8)])
@pytest.mark.parametrize("rms", [False, True])
@pytest.mark.parametrize("W", [4, 252, 256, 260, 1020, 1024, 1028, 2048, 2052, 4096, 4100])      # edges of a thread's share
def test_step_over_row_widths(dt, tol, rms, W):
    g = torch.Generator().manual_seed(W)
    T, eps, m = 3, 1e-5, 0.7
    rnd = lambda *s: torch.randn(*s, generator=g)            # noqa: E731
    x, y, extra = 3 * rnd(T, W) + 2, rnd(T, W).to(dt), rnd(T, W)
    w1, w2 = 1 + 0.2 * rnd(2, W)
    b1, b2 = (None, None) if rms else 0.2 * rnd(2, W)
    D = lambda t: None if t is None else t.to(F64)            # noqa: E731
    d = lambda t: None if t is None else t.to("cuda")         # noqa: E731
    for e in (None, extra):
        want = D(x) + m * norm(D(y), D(w1), D(b1), eps) + (0 if e is None else D(e))
        xg = d(x)
        h = ops.post_norm_add_norm(xg, d(y), d(w1), d(b1), eps, m, d(e), d(w2), d(b2), dt, rms=rms)
        wh = norm(want, D(w2), D(b2), eps)
        # f32 sums of up to 4100 terms, rounded a few times (6e-8 each); h in bf16: 2^-9 of its value
        assert (xg.cpu().to(F64) - want).abs().max() < 4e-6 * want.abs().max()
        assert (h.cpu().to(F64) - wh).abs().max() < tol * wh.abs().max()
    xg = d(x)
    assert ops.post_norm_add_norm(xg, d(y), d(w1), d(b1), eps, m, None, None, None, dt, rms=rms) is None
    want = D(x) + m * norm(D(y), D(w1), D(b1), eps)
    assert (xg.cpu().to(F64) - want).abs().max() < 4e-6 * want.abs().max()
