"""The screening module's fused passes (screen_fused.hip): the gated residual
against the torch expression it stands for, bit for bit, around a workgroup's
256 elements and past its largest grid, and the statistics against float64
torch (fp32, 1e-5 of the largest magnitude: sums of up to 300 terms, 2^-24
each)."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 1e-5}


def _close(name, got, want):
    scale = float(want.abs().max()) or 1.0
    err = float((got.double().cpu() - want).abs().max()) / scale
    assert got.shape == want.shape and err <= TOL[got.dtype], (name, err)


@pytest.mark.parametrize("pre_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("h_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(1, 1, 1), (1, 5, 51), (2, 2, 64),
                                   (1, 1, 257), (5, 683, 309)])
def test_residual_equals_torch(hip_lib, shape, h_dtype, pre_dtype):
    from rwkv7m_amd.screening import _Residual
    print("case: screening residual", shape, h_dtype, pre_dtype, flush=True)
    g = torch.Generator("cuda").manual_seed(sum(shape))

    def rand(dtype):
        x = torch.randn(shape, generator=g, device="cuda")
        return (3.0 * x).to(dtype)

    leaves = [rand(pre_dtype), torch.tensor(0.3, device="cuda"),
              rand(h_dtype), rand(h_dtype)]
    leaves = [t.requires_grad_() for t in leaves]
    pre, lam, read, hb = leaves
    dh = rand(h_dtype)
    want = (hb.float() + lam * torch.sigmoid(pre.float()) * read.float()).to(
        h_dtype)
    got = _Residual.apply(*leaves)
    for n, a, b in zip(("h", "d_pre", "d_lam", "d_read", "d_h_base"),
                       (got, *torch.autograd.grad(got, leaves, dh)),
                       (want, *torch.autograd.grad(want, leaves, dh))):
        assert a.dtype == b.dtype and torch.equal(a, b), n


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_residual_second_derivatives(hip_lib, dtype):
    """Against torch's, to the rounding of sums in another order (fp32: 25
    terms of 2^-24; bf16 gradients round once more, 2^-8)."""
    from rwkv7m_amd.screening import _Residual
    print("case: screening residual, second derivatives", dtype, flush=True)
    torch.manual_seed(3)
    leaves = [torch.randn(2, 3, 25).to(dtype).cuda(),
              torch.tensor(0.3).cuda(), *(torch.randn(2, 3, 25).to(dtype)
                                          .cuda() for _ in range(2))]
    pre, lam, read, hb = leaves = [t.requires_grad_() for t in leaves]
    dh = torch.randn(2, 3, 25).to(dtype).cuda().requires_grad_()
    out = []
    for h in (_Residual.apply(*leaves),
              (hb.float() + lam * torch.sigmoid(pre.float()) * read.float())
              .to(dtype)):
        g = torch.autograd.grad(h, leaves[:3], dh, create_graph=True)
        out.append(torch.autograd.grad([t.float().pow(2).sum() for t in g],
                                       [*leaves[:3], dh]))
    tol = 1e-5 if dtype == torch.float32 else 2.0 ** -7
    for n, a, b in zip(("pre", "lam", "read", "dh"), *out):
        err = float((a - b).abs().max() / b.abs().max())
        assert float(b.abs().max()) > 0 and err <= tol, (n, err)


@pytest.mark.parametrize("write", [False, True])
def test_an_empty_call_has_zero_gradients(hip_lib, write):
    from rwkv7m_amd.screening import (ScreeningConfig, StateLevelScreening,
                                      init_screen_state)
    print("case: screening, no tokens", write, flush=True)
    cfg = ScreeningConfig(d_model=96, d_slot=32, d_k=16, d_v=16, n_slots=3,
                          bank_ids=(0, 1, 2), use_write_screening=write)
    mod = StateLevelScreening(cfg, device="cuda")
    x = torch.zeros(2, 0, 96, device="cuda")
    # (what an uninitialised gradient would show: freed blocks of NaN)
    junk = [torch.full((n,), float("nan"), device="cuda")
            for n in (1, 16, 96, 192, 32 * 16) for _ in range(4)]
    del junk
    h, new, _ = mod(x, x, init_screen_state(2, cfg, "cuda"),
                    phase="read_write" if write else "read_screening_only")
    (h.sum() + new.slots.sum()).backward()
    torch.cuda.synchronize()
    assert h.shape == (2, 0, 96)
    for n, p in mod.named_parameters():
        assert p.grad is None or not p.grad.any(), n


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
