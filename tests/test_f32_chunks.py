"""The chunked fp32 kernels (wkv7_f32.hip) against the float64 oracle: every
head size, both vector types and layouts, whole and partial last chunks,
intervals other than the chunk, absent cotangents, added cotangents, and heads
whose chunks leave the factored form's range (served by the sequential
kernels).  Tolerances are the repository's: 1e-4 (fp32) and 2e-2 (bf16) of the
oracle's largest magnitude; the kernels' own error is 2e-7 (fp32) or the bf16
rounding of the outputs (4e-3).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from rwkv7m_amd.synthetic import make_inputs

pytestmark = pytest.mark.gpu

NAMES = ("r", "w", "k", "v", "neg_kk", "kka")
GRADS = ("dr", "dw", "dk", "dv", "dneg_kk", "dkka", "ds0")
TOL = {torch.float32: 1e-4, torch.bfloat16: 2e-2}


@pytest.fixture(scope="module")
def hip(hip_lib):
    from rwkv7m_amd.kernels import wkv_hip
    return wkv_hip


def _np(t):
    return t.detach().float().cpu().numpy().astype(np.float64)


def _close(name, got, want, tol, tag):
    err = oracle.normalized_max_error(_np(got), want)
    assert err <= tol, f"{tag} {name}: {err:.3e} > {tol}"


def _dev(inp, layout):
    t = {n: x.cuda() for n, x in inp.items()}
    if layout == "bthn":
        for n in (*NAMES, "dy"):
            t[n] = t[n].transpose(0, 1).contiguous()
    return t


CASES = [
    # T, B, H, N, dtype, layout
    (256, 1, 2, 16, torch.float32, "tbhn"),
    (273, 2, 1, 16, torch.bfloat16, "bthn"),
    (192, 1, 3, 32, torch.float32, "bthn"),
    (207, 1, 2, 32, torch.bfloat16, "tbhn"),
    (128, 1, 2, 64, torch.float32, "tbhn"),
    (145, 2, 2, 64, torch.float32, "bthn"),
    (64, 1, 1, 128, torch.float32, "tbhn"),
    (97, 1, 3, 128, torch.bfloat16, "bthn"),
]


@pytest.mark.parametrize("T,B,H,N,dtype,layout", CASES)
def test_matches_oracle(hip, T, B, H, N, dtype, layout):
    tag = f"T{T} B{B} H{H} N{N} {dtype} {layout}"
    print("case: chunked fp32", tag, flush=True)
    inp = make_inputs(T, B, H, N, dtype=dtype, seed=T + N, state_std=0.1,
                      dstate_std=0.1)
    host = [_np(inp[n]) for n in NAMES]
    ey, es, eck = oracle.forward(*host, _np(inp["s0"]),
                                 checkpoint_interval=16)
    eg = oracle.backward(*host, _np(inp["s0"]), _np(inp["dy"]),
                         _np(inp["ds_t"]))
    if layout == "bthn":
        ey = ey.swapaxes(0, 1)
        eg = [g.swapaxes(0, 1) for g in eg[:6]] + [eg[6]]
    d = _dev(inp, layout)
    vecs = [d[n] for n in (*NAMES, "s0")]
    (y, s_t), aux = hip.forward_with_aux(*vecs, layout=layout)
    assert hip.last_path() == "f32_forward", tag
    call = dict(layout=layout)
    grads = hip.backward(*vecs, d["dy"], d["ds_t"], *aux, **call)
    assert hip.last_path() == "f32_backward", tag
    y2, s2 = hip.forward(*vecs, layout=layout)
    again = hip.backward(*vecs, d["dy"], d["ds_t"], *aux, **call)
    torch.cuda.synchronize()
    _close("y", y, ey, TOL[dtype], tag)
    _close("s_t", s_t, es, 1e-4, tag)
    _close("checkpoints", aux[0], eck, 1e-4, tag)
    for n, g, e in zip(GRADS, grads, eg):
        _close(n, g, e, 1e-4 if n == "ds0" else TOL[dtype], tag)
    assert torch.equal(y, y2) and torch.equal(s_t, s2)
    assert all(torch.equal(a, b) for a, b in zip(grads, again))
    # an interval of three chunks: the same kernels, fewer checkpoints
    (y3, s3), aux3 = hip.forward_with_aux(*vecs, checkpoint_interval=48,
                                          layout=layout)
    assert hip.last_path() == "f32_forward"
    torch.cuda.synchronize()
    assert torch.equal(y, y3) and torch.equal(s_t, s3)
    assert torch.equal(aux3[0][:-1], aux[0][:-1:3])
    assert torch.equal(aux3[0][-1], s_t)
    # absent cotangents are zeros
    z = hip.backward(*vecs, torch.zeros_like(d["dy"]), d["ds_t"], *aux, **call)
    n = hip.backward(*vecs, None, d["ds_t"], *aux, **call)
    assert all(torch.equal(a, b) for a, b in zip(z, n))
    if layout == "bthn":  # cotangents of r, k, v from other uses
        adds = [torch.randn(y.shape, device="cuda").to(dtype) for _ in range(3)]
        summed = hip.backward(*vecs, d["dy"], d["ds_t"], *aux, layout=layout,
                              add=adds)
        assert hip.last_path() == "f32_backward"
        torch.cuda.synchronize()
        for i, a in zip((0, 2, 3), adds):
            _close(f"{GRADS[i]} + added", summed[i], eg[i] + _np(a),
                   TOL[dtype], tag)
        for i in (1, 4, 5, 6):
            assert torch.equal(summed[i], grads[i])


def _similar_keys(T, H, N, noise, decay, a, seed=1):
    """Tokens whose keys share a direction (noise 0: one key, repeated): kk of
    unit norm, a near sigmoid(a), decays of exp(-exp(-softplus(-decay)))."""
    g = torch.Generator().manual_seed(seed)

    def n(*shape):
        return torch.randn(*shape, generator=g, dtype=torch.float64)

    z = n(1, 1, H, N) + noise * n(T, 1, H, N)
    kk = z / z.norm(dim=-1, keepdim=True)
    w = -torch.nn.functional.softplus(-(n(T, 1, H, N) + decay)) - 0.5
    vals = (n(T, 1, H, N), w, 3.0 * z, n(T, 1, H, N), -kk,
            kk * torch.sigmoid(n(T, 1, H, N) + a), 0.1 * n(1, H, N, N),
            n(T, 1, H, N), 0.1 * n(1, H, N, N))
    return {k: v.float() for k, v in zip((*NAMES, "s0", "dy", "ds_t"), vals)}


@pytest.mark.parametrize("noise,decay,a", [(0.0, -2.0, 3.0), (0.1, -2.0, 3.0),
                                           (0.5, -2.0, 3.0), (0.0, -6.0, 5.0)])
@pytest.mark.parametrize("N", [16, 32, 64, 128])
def test_similar_keys(hip, N, noise, decay, a):
    """The chunk's triangular system where it is far from the identity, to
    2e-6 in the 2-norm: the token-by-token recurrence in float32 is 1.2e-6 off
    at most on these inputs (slowest decay), 2.7e-7 on the others, and the
    chunked kernels may take twice its roundings."""
    T, tag = 512, f"N{N} noise {noise} decay {decay} a {a}"
    print("case: chunked fp32, similar keys", tag, flush=True)
    inp = _similar_keys(T, 2, N, noise, decay, a)
    host = [_np(inp[n]) for n in (*NAMES, "s0")]
    want = [*oracle.forward(*host),
            *oracle.backward(*host, _np(inp["dy"]), _np(inp["ds_t"]))]
    d = _dev(inp, "tbhn")
    vecs = [d[n] for n in (*NAMES, "s0")]
    (y, s_t), aux = hip.forward_with_aux(*vecs)
    assert hip.last_path() == "f32_forward"
    grads = hip.backward(*vecs, d["dy"], d["ds_t"], *aux)
    assert hip.last_path() == "f32_backward"
    for n, got, e in zip(("y", "s_t", *GRADS), (y, s_t, *grads), want):
        err = np.linalg.norm(_np(got) - e) / np.linalg.norm(e)
        assert err <= 2e-6, f"{tag} {n}: {err:.2e}"


@pytest.mark.parametrize("N,dtype", [(64, torch.float32),
                                     (128, torch.bfloat16)])
def test_heads_out_of_range_take_the_sequential_kernels(hip, N, dtype):
    T, H = 150, 3
    print("case: chunked fp32, heads out of range, N", N, flush=True)
    inp = make_inputs(T, 1, H, N, dtype=dtype, seed=5, state_std=0.1,
                      dstate_std=0.1)
    plain = {n: x.clone() for n, x in inp.items()}
    inp["w"][40:44, :, 1] = 4.0  # decays of exp(-55) in one chunk of head 1
    outs = []
    for x in (plain, inp):
        d = _dev(x, "tbhn")
        vecs = [d[n] for n in (*NAMES, "s0")]
        (y, s_t), aux = hip.forward_with_aux(*vecs)
        assert hip.last_path() == "f32_forward"
        g = hip.backward(*vecs, d["dy"], d["ds_t"], *aux)
        assert hip.last_path() == "f32_backward"
        outs.append([y, *g[:6], s_t[None], g[6][None]])
    torch.cuda.synchronize()
    for a, b in zip(*outs):  # the other heads do not change
        assert torch.equal(a[:, :, ::2], b[:, :, ::2])
    host = [_np(inp[n]) for n in NAMES]
    ey, es = oracle.forward(*host, _np(inp["s0"]))
    eg = oracle.backward(*host, _np(inp["s0"]), _np(inp["dy"]),
                         _np(inp["ds_t"]))
    for n, got, e in zip(("y", *GRADS[:6], "s_t", "ds0"), outs[1],
                         (ey, *eg[:6], es[None], eg[6][None])):
        _close(n, got, e, TOL[dtype], f"N{N} strong decay")


def test_a_value_out_of_range_does_not_reach_earlier_tokens(hip):
    print("case: chunked fp32, an infinite v", flush=True)
    inp = make_inputs(130, 1, 2, 64, dtype=torch.float32, seed=6)
    inp["v"][70, 0, 0, 3] = float("inf")
    d = _dev(inp, "tbhn")
    y, _ = hip.forward(*[d[n] for n in (*NAMES, "s0")])
    assert hip.last_path() == "f32_forward"
    torch.cuda.synchronize()
    assert torch.isfinite(y[:70]).all() and torch.isfinite(y[:, :, 1]).all()
    rows = torch.arange(64) != 3  # state rows are independent
    assert torch.isfinite(y[:, 0, 0, rows.cuda()]).all()


def test_segment_of_one_partial_chunk(hip):
    """From 915 heads of 128 on the backward's time segments hold one chunk,
    the last one here one token: the cotangents equal those of the same heads
    in a call of a few (one segment)."""
    T, B, H, N, M = 33, 23, 40, 128, 6
    print("case: chunked fp32 backward, segments of one chunk", flush=True)
    inp = make_inputs(T, B, H, N, seed=8, state_std=0.1, dstate_std=0.1,
                      device="cuda", generator="torch")
    outs = []
    for bs, hs in ((slice(None), slice(None)), (slice(-1, None),
                                                slice(-M, None))):
        x = {n: (t[bs, hs] if n in ("s0", "ds_t") else t[:, bs, hs])
             .contiguous() for n, t in inp.items()}
        vecs = [x[n] for n in (*NAMES, "s0")]
        _, aux = hip.forward_with_aux(*vecs)
        g = hip.backward(*vecs, x["dy"], x["ds_t"], *aux)
        assert hip.last_path() == "f32_backward"
        outs.append([t[-1:, -M:] if n == "ds0" else t[:, -1:, -M:]
                     for n, t in zip(GRADS, g)])
    torch.cuda.synchronize()
    for n, a, b in zip(GRADS, *outs):
        assert torch.equal(a, b), n


@pytest.mark.parametrize("N,dtype,B,H,T", [(128, torch.bfloat16, 32, 32, 181),
                                           (64, torch.float32, 8, 32, 1366)])
def test_time_segments(hip, N, dtype, B, H, T):
    """Many heads: the workspace holds five chunks of 16 tokens forward (four at
    interval 32) and one backward at N = 128, 39 (38) and 19 at N = 64, so the
    state, its cotangent and the checkpoints pass from segment to segment,
    three times and more.  Heads equal
    the same heads in a call of few (one segment) bit for bit; three heads have
    a chunk out of range, in the first, a middle and the last segment."""
    tag = f"T{T} B{B} H{H} N{N} {dtype}"
    print("case: chunked fp32, time segments", tag, flush=True)
    x = make_inputs(T, B, H, N, dtype=dtype, seed=9, state_std=0.1,
                    dstate_std=0.1, device="cuda", generator="torch")
    nch = (T + 15) // 16
    for h, ch in ((-1, 0), (-2, nch // 2), (-3, nch - 1)):
        x["w"][16 * ch + 1:16 * ch + 4, -1, h] = 4.0
    x["add"] = torch.randn(T, B, H, N, device="cuda").to(dtype)
    states = ("s0", "ds_t", "s_t", "ds0")
    x = {n: t if n in states else t.transpose(0, 1).contiguous()
         for n, t in x.items()}

    def last8(n, t):  # of the last batch row
        return t[-1:, -8:] if n in states else t[:, -1:, -8:] if n == "ckpt" \
            else t[-1:, :, -8:]

    def in_range(n, t):
        return t.narrow(1 if n in states else 2, 0, 5)

    def run(x, ci):
        vecs = [x[n] for n in (*NAMES, "s0")]
        (y, s_t), aux = hip.forward_with_aux(*vecs, checkpoint_interval=ci,
                                             layout="bthn")
        assert hip.last_path() == "f32_forward"
        out = {"y": y, "s_t": s_t, "ckpt": aux[0]}
        if ci == 16:
            g = hip.backward(*vecs, x["dy"], x["ds_t"], *aux, layout="bthn",
                             add=(x["add"], None, x["add"]))
            assert hip.last_path() == "f32_backward"
            out.update(zip(GRADS, g))
        return out

    few = {n: last8(n, t).contiguous() for n, t in x.items()}
    big = {}
    for ci in (16, 32):
        small = run(few, ci)
        big[ci] = {n: last8(n, t).clone() for n, t in run(x, ci).items()}
        torch.cuda.synchronize()
        for n, t in big[ci].items():
            assert torch.equal(in_range(n, t), in_range(n, small[n])), \
                (tag, ci, n)
    host = [_np(few[n]).swapaxes(0, 1) for n in NAMES]
    host.append(_np(few["s0"]))
    ey, es, eck = oracle.forward(*host, checkpoint_interval=16)
    eg = list(oracle.backward(*host, _np(few["dy"]).swapaxes(0, 1),
                              _np(few["ds_t"])))
    want = {"s_t": es, "ckpt": eck, "ds0": eg[6]}
    for n, e in (("y", ey), *zip(GRADS, eg[:6])):
        want[n] = e.swapaxes(0, 1) + (_np(few["add"]) if n in ("dr", "dv")
                                      else 0.0)
    for n, e in want.items():
        tol = 1e-4 if n in (*states, "ckpt") else TOL[dtype]
        _close(n, big[16][n], e, tol, tag)
    _close("y", big[32]["y"], want["y"], TOL[dtype], tag + " interval 32")
    _close("s_t", big[32]["s_t"], es, 1e-4, tag + " interval 32")
    # (the last entry is the final state)
    eck = np.concatenate([eck[:-1:2], eck[-1:]])
    _close("ckpt", big[32]["ckpt"], eck, 1e-4, tag + " interval 32")


@pytest.mark.parametrize("N,dtype", [(16, torch.bfloat16), (32, torch.float32),
                                     (64, torch.float32)])
def test_forward_of_more_heads_than_cus(hip, N, dtype):
    """Up to a head a CU the chunked forward, past that the sequential one;
    the backward is chunked either way, from either's checkpoints."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    T = 336
    for H, path in ((cus, "f32_forward"), (cus + 1, "seq_forward")):
        print("case: fp32 dispatch by heads", N, H, flush=True)
        inp = make_inputs(T, 1, H, N, dtype=dtype, seed=4, state_std=0.1,
                          dstate_std=0.1)
        d = _dev(inp, "tbhn")
        vecs = [d[n] for n in (*NAMES, "s0")]
        hip.forward(*vecs)
        assert hip.last_path() == path
        (y, s_t), aux = hip.forward_with_aux(*vecs)
        assert hip.last_path() == path
        g = hip.backward(*vecs, d["dy"], d["ds_t"], *aux)
        assert hip.last_path() == "f32_backward"
        pick = slice(H - 2, H)
        host = [_np(inp[n][:, :, pick]) for n in NAMES]
        host.append(_np(inp["s0"][:, pick]))
        ey, es = oracle.forward(*host)
        eg = oracle.backward(*host, _np(inp["dy"][:, :, pick]),
                             _np(inp["ds_t"][:, pick]))
        _close("y", y[:, :, pick], ey, TOL[dtype], path)
        _close("s_t", s_t[:, pick], es, 1e-4, path)
        for n, a, e in zip(GRADS, g, eg):
            a = a[:, pick] if n == "ds0" else a[:, :, pick]
            _close(n, a, e, 1e-4 if n == "ds0" else TOL[dtype], path)


@pytest.mark.parametrize("N,few,many", [(16, 256, 320), (32, 192, 320),
                                        (64, 128, 192), (128, 64, 96)])
def test_forward_dispatch_by_tokens(hip, N, few, many):
    """The forward's shortest chunked calls, to a quarter of the CUs in heads
    and past it; both kernels give the same heads the same results."""
    q = torch.cuda.get_device_properties(0).multi_processor_count // 4
    print("case: fp32 dispatch by tokens", N, flush=True)
    for T in (few - 1, few, many - 1, many):
        inp = make_inputs(T, 1, q + 1, N, dtype=torch.float32, seed=T,
                          state_std=0.1, device="cuda", generator="torch")
        vecs = [inp[n] for n in (*NAMES, "s0")]
        outs = []
        for H, line in ((q, few), (q + 1, many)):
            y, s_t = hip.forward(*(x[:, :, :H].contiguous()
                                   for x in vecs[:6]),
                                 vecs[6][:, :H].contiguous())
            assert hip.last_path() == ("f32_forward" if T >= line else
                                       "seq_forward"), (T, H)
            outs.append((y[:, :, :q], s_t[:, :q]))
        torch.cuda.synchronize()
        for a, b in zip(*outs):  # (2e-6: the kernels' own errors, twice)
            assert float((a - b).norm() / b.norm()) <= 2e-6
