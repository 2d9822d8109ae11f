"""The work a program built on rwkv7m_amd has it do, as cases to be timed.

WKV-7 training steps (``wkv7`` / ``wkv7_batch_major``, forward and backward)
from the reference's own microbenchmark shape to the long carry-state
segments, inference prefill, single-token decode, the time mix's fused
section and the screening module in both training phases.  Sizes are those of
``rwkv7m_amd.synthetic.CONFIGS``, ``bench.py`` and the tests, or generic.

``exact`` restates each path in float64 torch, without this package's code.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

import rwkv7m_amd
from rwkv7m_amd.kernels import wkv_hip
from rwkv7m_amd.screening import (ScreeningConfig, ScreenState,
                                  StateLevelScreening)
from rwkv7m_amd.synthetic import make_inputs

VEC = ("r", "w", "k", "v", "neg_kk", "kka")
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
DEV = "cuda"


def listed():
    return [
        # the reference's WKV microbenchmark: one sequence of one model
        # chunk, where launches and host work count
        dict(name="train_small", kind="train", dtype="bf16", layout="tbhn",
             B=1, T=128, H=12, N=64, carry=False),
        # the WKV call of a 0.185B model's training step
        dict(name="train_0185b", kind="train", dtype="bf16", layout="tbhn",
             B=8, T=512, H=12, N=64, carry=False),
        # the same of a 1B model at its full context (the headline)
        dict(name="train_1b", kind="train", dtype="bf16", layout="tbhn",
             B=8, T=4096, H=32, N=64, carry=False),
        # streaming training at 7B width: slow decays, the state of the
        # segment before and its cotangent, the model's batch-major layout
        dict(name="train_7b_carry", kind="train", dtype="bf16",
             layout="bthn", B=4, T=8192, H=64, N=64, carry=True),
        # training in float32 (the module default; parity and debugging runs)
        dict(name="train_f32", kind="train", dtype="f32", layout="tbhn",
             B=8, T=512, H=12, N=64, carry=False),
        # a model with heads of 128
        dict(name="train_n128", kind="train", dtype="bf16", layout="tbhn",
             B=4, T=1024, H=16, N=128, carry=False),
        # prompts of odd length read into the state before decoding
        dict(name="prefill", kind="prefill", dtype="bf16", layout="bthn",
             B=2, T=1999, H=32, N=64, carry=True),
        # one sequence decoding: a single launch
        dict(name="decode_one", kind="decode", dtype="bf16", B=1, H=12, N=64),
        # a full serving batch decoding at 7B width
        dict(name="decode_7b", kind="decode", dtype="bf16", B=256, H=64,
             N=64),
        # the time mix's WKV section in the 1B model's training step
        dict(name="time_mix_1b", kind="timemix", dtype="bf16", B=8, T=4096,
             H=32, N=64),
        # the screening module of the 0.185B preset in the phase the
        # training loop runs
        dict(name="screen_read", kind="screen", dtype="bf16", B=8, T=512,
             C=768, ds=128, dk=64, dv=64, M=16, write=False, age=False),
        # the same with writes, in the module's default float32 (in bf16 a
        # rounding turns some of the age counters' threshold decisions, so
        # that two correct runs' ages cannot be compared)
        dict(name="screen_write", kind="screen", dtype="f32", B=8, T=512,
             C=768, ds=128, dk=64, dv=64, M=16, write=True, age=False),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo),
                                                      math.log(hi))))))


def draw(rng):
    kind = rng.choice(("train", "train", "train_seq", "prefill", "decode",
                       "timemix", "screen"))
    H = rng.choice((8, 12, 16, 25, 32, 40, 64))
    if kind in ("train", "prefill"):
        B = rng.randint(1, 8)
        T = _log(rng, 32, min(8192, (1 << 21) // (B * H)))
        return dict(kind=kind, dtype="bf16",
                    layout=rng.choice(("tbhn", "bthn")), B=B, T=T, H=H, N=64,
                    carry=rng.random() < 0.5)
    if kind == "train_seq":  # float32 vectors, and other head sizes
        dtype, N = rng.choice((("f32", 64), ("f32", 64), ("f32", 32),
                               ("bf16", 128), ("bf16", 32), ("f32", 16)))
        B = rng.randint(1, 8)
        H = rng.choice((4, 8, 12, 16))
        T = _log(rng, 32, min(1024, (1 << 16) // (B * H)))
        return dict(kind="train", dtype=dtype,
                    layout=rng.choice(("tbhn", "bthn")), B=B, T=T, H=H, N=N,
                    carry=rng.random() < 0.5)
    if kind == "decode":
        return dict(kind=kind, dtype=rng.choice(("bf16", "bf16", "f32")),
                    B=_log(rng, 1, 256), H=H, N=64)
    if kind == "timemix":
        B = rng.randint(1, 8)
        T = _log(rng, 32, min(4096, (1 << 20) // (B * H)))
        return dict(kind=kind, dtype="bf16", B=B, T=T, H=H, N=64)
    C, ds, dv = rng.choice(((768, 128, 64), (1024, 256, 128)))
    write = rng.random() < 0.5
    return dict(kind="screen", dtype="f32" if write else "bf16",
                B=rng.randint(1, 8), T=_log(rng, 32, 512 if ds == 128 else 256),
                C=C, ds=ds, dk=64, dv=dv, M=16, write=write,
                age=rng.random() < 0.5)


# --- inputs ---------------------------------------------------------------

def _time_mix_inputs(c, seed):
    dt, C = DTYPES[c["dtype"]], c["H"] * c["N"]
    g = torch.Generator(DEV).manual_seed(seed)

    def act(scale=1.0, shift=0.0):
        x = torch.randn(c["B"], c["T"], C, generator=g, device=DEV)
        return (x * scale + shift).to(dt)

    x = {"r": act(), "w_raw": act(0.5, -0.5), "k": act(), "v": act(),
         "a": torch.sigmoid(act().float()).to(dt), "g": act()}
    for n, scale, shift in (("k_k", 0.1, 0.7), ("k_a", 0.1, 1.0),
                            ("r_k", 0.1, -0.04), ("ln_scale", 0.1, 0.8),
                            ("ln_bias", 0.1, 0.0)):
        x[n] = torch.randn(C, generator=g, device=DEV) * scale + shift
    # the state of the segment before (from a zero state the first tokens' y
    # is a multiple of v, and the norm divides by next to nothing)
    x["s0"] = 0.1 * torch.randn(c["B"], c["H"], c["N"], c["N"], generator=g,
                                device=DEV)
    return x, act()


def _screen_inputs(c, seed):
    dt = DTYPES[c["dtype"]]
    cfg = ScreeningConfig(
        d_model=c["C"], d_slot=c["ds"], d_k=c["dk"], d_v=c["dv"],
        n_slots=c["M"],
        bank_ids=tuple(min(2, 4 * i // c["M"] - 1 if 2 * i >= c["M"] else 0)
                       for i in range(c["M"])),
        use_write_screening=c["write"], use_age_mask=c["age"])
    mod = StateLevelScreening(cfg, compute_dtype=dt, device=DEV, seed=seed)
    g = torch.Generator(DEV).manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device=DEV)

    B, T, C, M, ds = c["B"], c["T"], c["C"], c["M"], c["ds"]
    # the residual stream and its cotangent have a mean, and slots that have
    # followed one sequence resemble each other: without these the scalar
    # parameters' gradients would be sums of nothing but noise
    x = normal(B, T, C).to(dt)
    h, dh = ((normal(B, T, C) + 0.5 * normal(C)).to(dt) for _ in range(2))
    state = ScreenState(0.1 * normal(B, M, ds) + 0.2 * normal(B, 1, ds),
                        torch.randint(0, 64, (B, M), generator=g,
                                      device=DEV).float(),
                        torch.rand(B, M, generator=g, device=DEV) * 0.2)
    return mod, x, h, dh, state


def prepare(case, seed):
    """The tensors, module and registration a program holds before the call."""
    c, kind = case, case["kind"]
    rwkv7m_amd.register_hip_backend(replace=True)
    s = {"case": c}
    if kind == "screen":
        mod, x, h, dh, state = _screen_inputs(c, seed)
        s.update(mod=mod, x=x.requires_grad_(), h=h.requires_grad_(), dh=dh,
                 state=state, params=list(mod.parameters()))
        return s
    if kind == "timemix":
        x, dout = _time_mix_inputs(c, seed)
        s.update(x=[t.requires_grad_() for t in x.values()], dout=dout)
        return s
    T = c.get("T", 1)
    std = 0.1 if kind == "decode" or c["carry"] else 0.0
    inp = make_inputs(T, c["B"], c["H"], c["N"], dtype=DTYPES[c["dtype"]],
                      seed=seed, slow_decay=c.get("carry", False),
                      state_std=std, dstate_std=std, device=DEV,
                      generator="torch")
    if c.get("layout") == "bthn":
        for n in (*VEC, "dy"):
            inp[n] = inp[n].transpose(0, 1).contiguous()
    if kind == "train":
        for n in (*VEC, "s0") if c["carry"] else VEC:
            inp[n].requires_grad_()
    s["x"] = [inp[n] for n in (*VEC, "s0")]
    s["dy"], s["ds_t"] = inp["dy"], inp["ds_t"]
    return s


def run(state):
    """One pass, as a program calls it."""
    s = state
    c, kind = s["case"], s["case"]["kind"]
    if kind == "decode":
        *vecs, st = s["x"]
        return [wkv_hip.decode_inplace(*vecs, st), st]
    if kind == "timemix":
        out, s_t = rwkv7m_amd.time_mix_wkv(*s["x"], n_heads=c["H"])
        return [out, s_t, *torch.autograd.grad(out, s["x"], s["dout"])]
    if kind == "screen":
        h, new, stats = s["mod"](
            s["x"], s["h"], s["state"],
            phase="read_write" if c["write"] else "read_screening_only")
        grads = torch.autograd.grad(h, [s["x"], s["h"], *s["params"]],
                                    s["dh"])
        return [h, list(new), list(grads), stats]
    call = rwkv7m_amd.wkv7 if c["layout"] == "tbhn" else \
        rwkv7m_amd.wkv7_batch_major
    if kind == "prefill":
        with torch.no_grad():
            return list(call(*s["x"], "ffi"))
    y, s_t = call(*s["x"], "ffi")
    if c["carry"]:
        g = torch.autograd.grad((y, s_t), s["x"], (s["dy"], s["ds_t"]))
    else:
        g = torch.autograd.grad(y, s["x"][:6], s["dy"])
    return [y, s_t, *g]


# --- what a pass cannot do without ---------------------------------------

def work(case):
    """Bytes: each input read and each output written once by the forward
    and once by the backward (two calls; the cotangent arrives in between).
    Operations: the recurrence's products as the step states them, and the
    projections of the screening module."""
    c, kind = case, case["kind"]
    eb = 2 if c["dtype"] == "bf16" else 4
    if kind == "screen":
        R, C, ds, kv = c["B"] * c["T"], c["C"], c["ds"], c["dk"] + c["dv"]
        par = C * c["dk"] + ds * kv + c["dv"] * C + C * C + (2 * C + ds) * ds
        proj = R * (C * c["dk"] + C * C + 2 * C * ds + c["dv"] * C
                    + c["M"] * ds * kv)
        if c["write"]:
            par += (2 * C + ds) * c["dk"]
            proj += R * (2 * C + c["M"] * ds) * c["dk"]
        # x, h, and in the backward dh, in; h and the gradients of x and h
        # out; the parameters in twice and their gradients out (fp32)
        return {"bytes": R * C * eb * 8 + par * 4 * 3,
                "flops": 3 * 2 * proj + 12 * R * c["M"] * ds}
    B, T, H, N = c["B"], c.get("T", 1), c["H"], c["N"]
    V, S, step = B * T * H * N * eb, B * H * N * N * 4, B * T * H * N * N
    if kind in ("decode", "prefill"):
        return {"bytes": 7 * V + 2 * S, "flops": 9 * step}
    if kind == "timemix":
        # forward: r, w_raw, k, v, a, g in, out out; backward: those and
        # dout in, six gradients out
        return {"bytes": 20 * V + 4 * S, "flops": 29 * step}
    return {"bytes": 20 * V + (5 if c["carry"] else 2) * S,
            "flops": 29 * step}


def tolerance(case):
    c = case
    if c["dtype"] == "f32":
        return {"rel": 1e-4 if c["kind"] == "screen" else 2e-6}
    return {"rel": 3e-2 if c["kind"] in ("screen", "timemix") else 2e-2}


# --- float64 restatement --------------------------------------------------

class _Scan64(torch.autograd.Function):
    """WKV-7 over [T, B, H, N] float64 vectors; the backward recomputes the
    states of 64 tokens at a time from kept ones."""

    KEEP = 64

    @staticmethod
    def step(S, d, k, v, a, b):
        sa = (S * a[..., None, :]).sum(-1)
        return (S * d[..., None, :] + sa[..., None] * b[..., None, :]
                + v[..., None] * k[..., None, :]), sa

    @staticmethod
    def forward(ctx, r, w, k, v, a, b, s0):
        d = torch.exp(-torch.exp(w))
        S, y, kept = s0, torch.empty_like(r), []
        for t in range(r.shape[0]):
            if t % _Scan64.KEEP == 0:
                kept.append(S)
            S, _ = _Scan64.step(S, d[t], k[t], v[t], a[t], b[t])
            y[t] = (S * r[t][..., None, :]).sum(-1)
        ctx.save_for_backward(r, w, k, v, a, b)
        ctx.kept = kept
        return y, S

    @staticmethod
    def backward(ctx, dy, ds_t):
        r, w, k, v, a, b = ctx.saved_tensors
        d = torch.exp(-torch.exp(w))
        g = [torch.empty_like(r) for _ in range(6)]
        G = ds_t
        for c in range(len(ctx.kept) - 1, -1, -1):
            S, before = ctx.kept[c], []
            ts = range(c * _Scan64.KEEP,
                       min(r.shape[0], (c + 1) * _Scan64.KEEP))
            for t in ts:
                before.append(S)
                S, _ = _Scan64.step(S, d[t], k[t], v[t], a[t], b[t])
            for t in reversed(ts):
                P = before.pop()
                _, sa = P, (P * a[t][..., None, :]).sum(-1)
                g[0][t] = (S * dy[t][..., None]).sum(-2)
                G = G + dy[t][..., None] * r[t][..., None, :]
                g[1][t] = -(G * P).sum(-2) * d[t] * torch.exp(w[t])
                g[2][t] = (G * v[t][..., None]).sum(-2)
                g[3][t] = (G * k[t][..., None, :]).sum(-1)
                g[5][t] = (G * sa[..., None]).sum(-2)
                dsa = (G * b[t][..., None, :]).sum(-1)
                g[4][t] = (P * dsa[..., None]).sum(-2)
                G = G * d[t][..., None, :] + dsa[..., None] * a[t][..., None, :]
                S = P
        return (*g, G)


def _leaves64(tensors, grad):
    return [t.detach().double().requires_grad_(grad) for t in tensors]


def _time_mix64(c, x, dout):
    r, w_raw, k, v, a, g, k_k, k_a, r_k, sc, bi, s0 = L = _leaves64(x, True)
    B, T, H, N = c["B"], c["T"], c["H"], c["N"]

    def heads(t):
        return t.reshape(B, T, H, N)

    w = -F.softplus(-w_raw) - 0.5
    kk = F.normalize(heads(k * k_k), dim=-1, eps=1e-12)
    kp = k * (1.0 + (a - 1.0) * k_a)
    vecs = [heads(t).transpose(0, 1)
            for t in (r, w, kp, v, -kk, kk * heads(a))]
    y, s_t = _Scan64.apply(*vecs, s0)
    y = y.transpose(0, 1)
    dev = y - y.mean(-1, keepdim=True)
    y = dev / torch.sqrt((dev * dev).mean(-1, keepdim=True) + 64e-5)
    y = y * sc.view(H, N) + bi.view(H, N)
    bonus = (heads(r) * heads(kp) * r_k.view(H, N)).sum(-1, keepdim=True)
    out = (y + bonus * heads(v)).reshape(B, T, H * N) * g
    return [out, s_t, *torch.autograd.grad(out, L, dout.double())]


def _screen64(c, mod, x, h, dh, state):
    cfg, eps = mod.config, mod.config.eps
    names = [n for n, _ in mod.named_parameters()]
    x, h, *ps = L = _leaves64([x, h, *mod.parameters()], True)
    P = dict(zip(names, ps))
    slots, ages, usage = (t.double() for t in state)
    C, T = c["C"], c["T"]

    def un(t):
        return t / torch.sqrt((t * t).sum(-1, keepdim=True) + eps * eps)

    def trim(sim, tau):
        return torch.clamp((sim - tau) / (1.0 - tau + eps), min=0.0) ** 2

    x_ln = F.layer_norm(x, (C,), P["screen_ln_scale"], P["screen_ln_bias"],
                        1e-6)
    q = un(x_ln @ P["q_proj_r"])
    tau = 2.0 * torch.sigmoid(P["tau_r_raw"]) - 1.0
    mu = (mod._mu_max.double() * torch.sigmoid(P["mu_by_bank_raw"]))[
        mod._bank_ids]
    gate = torch.sigmoid(x_ln @ P["gate_kernel"] + P["gate_bias"])
    dker = P["delta_kernel"]
    base = x_ln @ dker[:C] + h @ dker[C:2 * C] + P["delta_bias"]
    pre = base[:, :, None] + P["slot_embed"] @ dker[2 * C:]
    if c["write"]:
        q_w = un(torch.cat([x_ln, h], -1) @ P["q_proj_w"])
        tau_w = 2.0 * torch.sigmoid(P["tau_w_raw"]) - 1.0
    us = []
    for t in range(T):
        sim = (q[:, t, None] * un(slots @ P["k_proj_r"])).sum(-1)
        rel = trim(sim, tau)
        if c["age"]:
            rel = rel * torch.sigmoid((cfg.age_ref - ages)
                                      / (cfg.age_sigma + eps))
        z = (rel[..., None] * un(slots @ P["v_proj"])).sum(1)
        n = torch.sqrt((z * z).sum(-1, keepdim=True) + eps * eps)
        us.append(torch.tanh(n) / n * z)
        rate, act = mu.expand(c["B"], -1), rel
        if c["write"]:
            kw = un((slots + P["slot_embed"]) @ P["k_proj_w"])
            rel_w = trim((q_w[:, t, None] * kw).sum(-1), tau_w)
            rate = mu * torch.clamp(rel_w, min=cfg.write_rel_floor)
            ages = torch.where(rel_w > 1e-3, 0.0, ages + 1.0)
            act = torch.maximum(rel, rel_w)
        slots = slots + rate[..., None] * (torch.tanh(pre[:, t]) - slots)
        usage = cfg.usage_ema_decay * usage + (1 - cfg.usage_ema_decay) * act
    read = torch.stack(us, 1) @ P["out_proj"]
    out = h + F.softplus(P["lambda_raw"]) * gate * read
    return [out, [slots, ages, usage],
            list(torch.autograd.grad(out, L, dh.double())), None]


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "screen":
        return _screen64(c, *_screen_inputs(c, seed))
    if kind == "timemix":
        x, dout = _time_mix_inputs(c, seed)
        return _time_mix64(c, list(x.values()), dout)
    s = prepare(c, seed)
    x = s["x"]
    if c.get("layout") == "bthn":
        x = [t.transpose(0, 1) for t in x[:6]] + x[6:]
    L = _leaves64(x, kind == "train")
    with torch.set_grad_enabled(kind == "train"):
        y, s_t = _Scan64.apply(*L)
    if kind == "decode":
        return [y, s_t]
    bt = c["layout"] == "bthn"
    out = [y.transpose(0, 1) if bt else y, s_t]
    if kind == "train":
        dy = s["dy"].double()
        g = torch.autograd.grad(
            (y, s_t), L if c["carry"] else L[:6],
            (dy.transpose(0, 1) if bt else dy, s["ds_t"].double()))
        out += [t.transpose(0, 1) if bt and i < 6 else t
                for i, t in enumerate(g)]
    return out
