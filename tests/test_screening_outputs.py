"""The screening module's outputs where the compute dtype rounds: against the
same module written with plain torch operations around the recurrence and
read kernels, in which every intermediate is rounded where torch rounds it.
A sum taken in another order turns some of the roundings of a bf16
intermediate, and through the thresholds behind it every gradient moves by
1e-3; so the states, the output and every gradient are compared exactly, at the
0.185B preset's sizes (of 4096 rows of 768 values some always lie at a
rounding's edge).
"""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _inputs(dtype, B=8, T=512, C=768, write=False, seed=3):
    from rwkv7m_amd.screening import (ScreeningConfig, ScreenState,
                                      StateLevelScreening)
    cfg = ScreeningConfig(d_model=C, d_slot=128, d_k=64, d_v=64, n_slots=6,
                          bank_ids=(0, 0, 1, 1, 2, 2),
                          use_write_screening=write)
    mod = StateLevelScreening(cfg, compute_dtype=dtype, device="cuda",
                              seed=seed)
    g = torch.Generator("cuda").manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device="cuda")

    with torch.no_grad():
        mod.gate_bias.copy_(0.5 * normal(C))
        mod.screen_ln_scale.add_(0.1 * normal(C))
        mod.screen_ln_bias.add_(0.1 * normal(C))
    x, h, dh = (normal(B, T, C).to(dtype) for _ in range(3))
    state = ScreenState(0.3 * normal(B, 6, 128),
                        torch.zeros(B, 6, device="cuda"),
                        torch.rand(B, 6, generator=g, device="cuda"))
    return mod, x.requires_grad_(), h.requires_grad_(), dh, state


def _read_phase(mod, x, h, state):
    """The read-only phase of nnx_model.py:1015-1160 without the usage EMA:
    (h, slots)."""
    from rwkv7m_amd import screening as sc
    cfg, cd, eps, C = mod.config, mod.compute_dtype, mod.config.eps, x.size(-1)
    x_ln = F.layer_norm(x.float(), (C,), mod.screen_ln_scale.float(),
                        mod.screen_ln_bias.float(), eps=1e-6).to(cd)
    q = (x_ln @ mod.q_proj_r.to(cd)).float()
    q = q / torch.sqrt((q * q).sum(-1, keepdim=True) + eps * eps)
    gate = torch.sigmoid((x_ln @ mod.gate_kernel.to(cd)
                          + mod.gate_bias.to(cd)).float())
    dker = mod.delta_kernel.to(cd)
    base = (x_ln @ dker[:C] + h.to(cd) @ dker[C:2 * C]
            + mod.delta_bias.to(cd))
    term = (mod.slot_embed.to(cd) @ dker[2 * C:]).float()
    seq, slots, _ = sc._SlotScan.apply(base, term, mod.compute_mu(),
                                       state.slots.float())
    kv = torch.cat([mod.k_proj_r, mod.v_proj], dim=1).to(cd)
    u, _, _, _ = sc._ScreenRead.apply(
        q, sc._SlotProjection.apply(seq, kv),
        2.0 * torch.sigmoid(mod.tau_r_raw.float()) - 1.0, None, cfg, cfg.d_v)
    read = (u @ mod.out_proj.to(cd)).to(h.dtype)
    lam = F.softplus(mod.lambda_raw.float())
    return (h.float() + lam * gate * read.float()).to(h.dtype), slots


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_read_phase_equals_torch(hip_lib, dtype):
    print("case: screening read phase, outputs and gradients", dtype,
          flush=True)
    mod, x, h, dh, state = _inputs(dtype)
    leaves = [x, h, *mod.parameters()]
    names = ["x", "h_base", *(n for n, _ in mod.named_parameters())]
    out, new, _ = mod(x, h, state)
    want, slots = _read_phase(mod, x, h, state)
    torch.cuda.synchronize()
    assert torch.equal(out, want) and torch.equal(new.slots, slots)
    for n, a, b in zip(names, torch.autograd.grad(out, leaves, dh),
                       torch.autograd.grad(want, leaves, dh)):
        assert torch.equal(a, b), n


def test_inputs_broadcast_over_the_batch(hip_lib):
    """h_base_seq, and the usage EMA over the batch and (with one sequence)
    over more rows, as the torch expressions take them."""
    print("case: screening, broadcast inputs", flush=True)
    mod, x, h, _, state = _inputs(torch.float32, B=3, T=20, C=96)
    one, wide = h.detach()[:1], h.detach()[:1].expand(3, -1, -1).contiguous()
    outs, grads = [], []
    for hb in (one, wide):
        hb = hb.clone().requires_grad_()
        out, new, _ = mod(x, hb, state)
        outs.append([out, *new])
        g, = torch.autograd.grad(out.square().sum(), hb)
        grads.append(g.sum(0))
    # (the projection of one batch row's h_base may sum in another order than
    # three rows': 192 terms of 2^-24)
    for a, b in zip(*outs):
        assert torch.allclose(a, b, rtol=1e-5, atol=1e-5)
    assert torch.allclose(*grads, rtol=1e-5, atol=1e-5)

    def usage(rows, u):
        u = u.clone().requires_grad_()
        sub = state._replace(slots=state.slots[:rows], ages=state.ages[:rows],
                             usage_ema=u)
        _, new, stats = mod(x[:rows], h[:rows], sub)
        g, = torch.autograd.grad(new.usage_ema.sum(), u)
        return new.usage_ema, stats["slot_usage_ema_mean"], g

    u = state.usage_ema
    got, mean, g = usage(3, u[:1])
    want, wmean, wg = usage(3, u[:1].expand(3, -1).contiguous())
    assert got.shape == (3, 6) and torch.allclose(got, want, atol=1e-6)
    assert torch.allclose(mean, wmean, rtol=1e-5)
    assert torch.allclose(g, wg.sum(0, keepdim=True), rtol=1e-5)
    got, mean, g = usage(1, u)
    assert got.shape == (3, 6)
    rows = [usage(1, u[i:i + 1]) for i in range(3)]
    assert torch.allclose(got, torch.cat([r[0] for r in rows]), atol=1e-6)
    assert torch.allclose(mean, sum(r[1] for r in rows) / 3, rtol=1e-5)
    assert torch.allclose(g, torch.cat([r[2] for r in rows]), rtol=1e-5)


def test_an_empty_batch_is_refused(hip_lib):
    print("case: screening, no batch rows", flush=True)
    mod, x, h, _, state = _inputs(torch.float32, B=3, T=4, C=96)
    with pytest.raises(IndexError):
        mod(x[:0], h[:0], type(state)(*(t[:0] for t in state)))


def _write_args(dtype, B=2, T=96, M=3, ds=80, dk=32, seed=4):
    g = torch.Generator().manual_seed(seed)

    def n(*shape):
        return torch.randn(*shape, generator=g)

    q = n(B, T, dk)
    kw = (n(ds, dk) / ds ** 0.5).to(dtype)
    return [t.cuda() for t in (
        n(B, T, ds).to(dtype), 0.3 * n(M, ds), 0.5 * n(M, ds), kw,
        q / q.norm(dim=-1, keepdim=True), torch.tensor(-0.6),
        torch.full((M,), 0.02), 0.3 * n(B, M, ds),
        torch.zeros(B, M))], 0.05, 1e-6


def test_bf16_write_keys_are_rounded_projections(hip_lib):
    """rel_w against the recurrence in float64 with the roundings of a bf16
    projection, round(round(S + e) W): a rounding turned by the sums' order
    moves single values, all others agree to fp32 (without the roundings all
    are about 2^-9 off)."""
    from rwkv7m_amd.screening import _WriteScan
    print("case: screening write phase, bf16 keys", flush=True)
    args, floor, eps = _write_args(torch.bfloat16)
    _, _, rel_w, _, s_t, _ = _WriteScan.apply(*args, floor, eps)
    torch.cuda.synchronize()
    base, st, se, kw, q, tau, mu, S, _ = (t.double().cpu() for t in args)

    def rnd(x):
        return x.bfloat16().double()

    want = []
    for t in range(base.shape[1]):
        k = rnd(rnd(S + se) @ kw)
        sim = (k * q[:, t, None]).sum(-1) / torch.sqrt(
            (k * k).sum(-1) + eps * eps)
        rel = torch.clamp((sim - tau) / (1.0 - tau + eps), min=0.0) ** 2
        want.append(rel)
        rate = mu * torch.clamp(rel, min=floor)
        S = S + rate[..., None] * (rnd(torch.tanh(base[:, t, None] + st)) - S)
    want = torch.stack(want, 1)
    err = (rel_w.double().cpu() - want).abs()
    assert float(want.max()) > 0.1
    assert float((err > 1e-5).double().mean()) < 0.05
    assert float(err.max()) < 2.0 ** -7


def test_write_phase_under_autocast(hip_lib):
    """The keys are the kernels' own fp32 products: an autocast region does
    not turn them into bf16 ones."""
    from rwkv7m_amd.screening import _WriteScan
    print("case: screening write phase under autocast", flush=True)
    args, floor, eps = _write_args(torch.float32)
    res = []
    for on in (False, True):
        leaves = [t.clone().requires_grad_() for t in args]
        with torch.autocast("cuda", torch.bfloat16, enabled=on):
            out = _WriteScan.apply(*leaves, floor, eps)
            diff = [out[0], out[2], out[4]]
            grads = torch.autograd.grad(
                [t.float().square().sum() for t in diff],
                leaves[:3] + leaves[4:8])
        res.append([*out, *grads])
    torch.cuda.synchronize()
    for i, (a, b) in enumerate(zip(*res)):
        assert torch.isfinite(a).all() and torch.equal(a, b), i


@pytest.mark.parametrize("B,T,M,ds,dk", [(1, 1, 1, 1, 1), (1, 5, 3, 17, 15),
                                         (2, 8, 4, 16, 16), (1, 13, 5, 33, 64),
                                         (1, 3, 7, 130, 65),
                                         (2, 9, 2, 300, 128)])
def test_write_products(hip_lib, B, T, M, ds, dk):
    """delta_keys and wp at the edges of their 16-row, 16-column tiles, against
    float64: one rounding and tanh's few ulps, 1e-6 of the terms' size."""
    from rwkv7m_amd.kernels import screening_hip as sh
    from rwkv7m_amd.kernels import wkv_hip
    print("case: screening write products", B, T, M, ds, dk, flush=True)
    g = torch.Generator("cuda").manual_seed(ds + dk)

    def n(*shape):
        return torch.randn(*shape, generator=g, device="cuda")

    base, st, se, kw = n(B, T, ds), n(M, ds), n(M, ds), n(ds, dk)
    keys, q = n(B, T, M, dk), n(B, T, dk)
    dkeys, p, wp = (torch.full((B, T, M, k), float("nan"), device="cuda")
                    for k in (dk, dk, ds))
    sim = torch.empty(B, T, M, device="cuda")
    P, strm = wkv_hip._p, wkv_hip._stream(base.device)
    sh._call("rwkv7m_screen_write_delta_keys", B, T, M, ds, dk, P(base), P(st),
             P(se), P(kw), P(dkeys), strm)
    sh._call("rwkv7m_screen_write_keys", B, T, M, ds, dk, P(keys), P(q), P(kw),
             1e-6, P(p), P(sim), P(wp), strm)
    x = torch.tanh(base.double()[:, :, None] + st.double()) + se.double()
    for got, a, w in ((dkeys, x, kw.double()), (wp, p.double(),
                                                kw.double().t())):
        a, w = a.cpu(), w.cpu()
        err = (got.double().cpu() - a @ w).abs()
        assert (err <= 1e-6 * (a.abs() @ w.abs()) + 1e-30).all(), \
            float(err.max())


@pytest.mark.parametrize("T,M,ds,dk", [(70, 3, 128, 64), (30, 2, 300, 30),
                                       (20, 2, 260, 72), (20, 3, 256, 64)])
def test_projecting_and_carried_write_keys_agree(hip_lib, T, M, ds, dk):
    """rwkv7m_screen_write (the key projected at every step) in fp32, for
    callers of the C interface, against the carried key's kernels: forward and
    every cotangent, to 1e-5 of the largest (sums of up to 300 terms and T
    steps of 2^-24 each)."""
    from rwkv7m_amd.kernels import screening_hip as sh
    print("case: screening write keys", T, M, ds, dk, flush=True)
    (base, st, se, kw, q, tau, mu, s0, a0), floor, eps = _write_args(
        torch.float32, T=T, M=M, ds=ds, dk=dk)
    args = (base, st, se, kw, q, tau, mu, floor, eps)
    want = sh.write(*args, s0, a0)
    *got, keys = sh.write_scan(*args, s0, a0)
    g = torch.Generator("cuda").manual_seed(6)
    cots = [torch.randn(t.shape, generator=g, device="cuda")
            for t in (want[0], want[5], want[3], want[2], want[6])]
    wb = list(sh.write_backward(*args, want[1], *cots))
    gb = list(sh.write_scan_backward(*args, got[1], keys, *cots))
    wb[6] = wb[6].sum(2)
    torch.cuda.synchronize()
    assert torch.equal(got[2], want[2])  # ages
    assert float(want[3].max()) > floor  # the relevance is in play
    for n, a, b in zip(("seq", "s32", "ages", "rel_w", "upd2", "s_t", "a_t",
                        "d_pre", "d_slots0", "d_ages0", "d_embed", "d_mu",
                        "d_keys", "dq_w", "d_tau"), (*got, *gb),
                       (*want, *wb)):
        err = float((a - b).abs().max()) / (float(b.abs().max()) or 1.0)
        assert err <= 1e-5, (n, err)
