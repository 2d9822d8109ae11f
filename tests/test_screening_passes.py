"""The screening module's fused passes (screen_fused.hip) against float64 torch
at sizes around their tiles: one row, a wave's and a block's rows, row groups
with and without a remainder, columns below, at and past 64.  Tolerances: fp32
1e-5 of the largest magnitude (sums of up to 300 terms, 2^-24 each), bf16
outputs 2^-8 (one rounding, 2^-9, and its input's)."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 1e-5, torch.bfloat16: 2.0 ** -8}
SIZES = [(1, 1), (3, 64), (4, 65), (70, 130), (4100, 33)]


def _close(name, got, want):
    scale = float(want.abs().max()) or 1.0
    err = float((got.double().cpu() - want).abs().max()) / scale
    assert got.shape == want.shape and err <= TOL[got.dtype], (name, err)


def _rand(*shape, dtype=torch.float32):
    return torch.randn(*shape).to(dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,C", SIZES)
def test_row_passes(hip_lib, rows, C, dtype):
    from rwkv7m_amd.kernels import screening_hip as sh
    torch.manual_seed(rows + C)
    print("case: screening passes", rows, C, dtype, flush=True)
    x, read, hb, g = (_rand(rows, C, dtype=dtype) for _ in range(4))
    bias, lam = _rand(C), torch.tensor(0.3)
    leaves = [t.double().requires_grad_() for t in (x, read, hb, bias, lam)]
    X, R, HB, B, L = leaves
    xd, rd, hd, bd, ld, gd = (t.cuda() for t in (x, read, hb, bias, lam, g))
    # the unit norm
    want = X / torch.sqrt((X * X).sum(-1, keepdim=True) + 1e-12)
    _close("unit", sh.unit(xd, 1e-6), want.detach())
    dx, = torch.autograd.grad(want, X, g.double())
    if C > 1:  # (a single column's norm has no derivative but rounding)
        _close("unit dx", sh.unit_backward(xd, 1e-6, gd.float()), dx)
    # the gated residual: x as the gate's pre-activation
    want = HB + L * torch.sigmoid(X + B) * R
    _close("residual", sh.residual(xd, bd, ld, rd, hd), want.detach())
    grads = torch.autograd.grad(want, (X, B, L, R), g.double())
    for n, a, b in zip(("d_pre", "d_bias", "d_lam", "d_read"),
                       sh.residual_backward(xd, bd, ld, rd, gd), grads):
        _close("residual " + n, a, b)


@pytest.mark.parametrize("B,T,M", [(1, 1, 1), (3, 37, 5), (8, 260, 16),
                                   (2, 3, 300)])
@pytest.mark.parametrize("write", [False, True])
def test_statistics(hip_lib, B, T, M, write):
    from rwkv7m_amd.kernels import screening_hip as sh
    torch.manual_seed(B * T + M)
    print("case: screening statistics", B, T, M, write, flush=True)
    rel = torch.rand(B, T, M).pow(4)
    rel_w = torch.rand(B, T, M).pow(4) if write else None
    zn, un, u0 = torch.rand(B, T), torch.rand(B, T), torch.rand(B, M)
    upd2 = torch.rand(B, T, M, 2)
    floor, d = 0.01, 0.97
    usage, stats = sh.stats(rel.cuda(), None if rel_w is None else
                            rel_w.cuda(), zn.cuda(), un.cuda(), upd2.cuda(),
                            u0.cuda(), floor, d)
    r = rel.double()
    rw = r * 0 if rel_w is None else rel_w.double()
    act = torch.maximum(r, rw) if write else r
    u, means = u0.double(), []
    for t in range(T):
        u = d * u + (1 - d) * act[:, t]
        means.append(u.mean())
    want = torch.stack([
        r.mean(), r.amax((0, 2)).mean(), (rel > 1e-3).sum(-1).double().mean(),
        rw.mean(), rw.clamp(min=floor).mean() if write else rw.mean(),
        act.mean(), upd2.double().sum(-1).sqrt().mean(), zn.double().mean(),
        un.double().mean(), torch.stack(means).mean()])
    _close("usage", usage, u)
    assert torch.allclose(stats.double().cpu(), want, rtol=1e-5, atol=0)
