"""The chunked fp32 form of the outer-product recurrences (csrc/mixers/chunk_scan.hip) against the token loop in fp64.

Tolerance: a term of the state has one rounding of its factor and at most one of each sum that it is part of, as in the token
loop, so an entry errs by some 2^-24 of its terms' sizes per token that it remembers; with gates close to one and k = 1 - f the
rounding of the gate itself is 2^-24 / (1 - f) of a term. 2e-5 of the output's root mean square covers both for the sizes here.
How the errors compare with the token loop's own is tested apart."""
import math

import pytest
import torch

from xgserve.ops import seqmix as sq

from _seq_util import record_native, seq_meta

F64 = torch.float64
TOL = 2e-5

pytestmark = pytest.mark.gpu


def scan(q, f, k, v, S):
    """q, f, k [T, H, dk], v [T, H, dv], S [H, dk, dv], fp64."""
    out = []
    for t in range(q.shape[0]):
        S = f[t][:, :, None] * S + k[t][:, :, None] * v[t][:, None, :]
        out.append(torch.einsum("hkd,hk->hd", S, q[t]))
    return torch.stack(out), S


def close(got, ref):
    got = got.detach().cpu().to(F64)
    bad = ~torch.isfinite(ref)
    assert torch.equal(torch.isnan(got), torch.isnan(ref)) and torch.equal(got[bad & ~torch.isnan(ref)], ref[bad & ~torch.isnan(ref)])
    ok = ~bad
    if ok.any():
        scale = ref[ok].pow(2).mean().sqrt() + 1e-30
        assert float((got[ok] - ref[ok]).abs().max() / torch.maximum(scale, ref[ok].abs().max() * 1e-2)) < TOL


def layout(portions):
    """[(context, tokens)] -> SeqMeta on slots 1, 2, ... of a 16-token paged layout."""
    tables, at = [], 0
    for ctx, n in portions:
        m = (ctx + n + 15) // 16
        tables.append(list(range(at, at + m)))
        at += m
    return seq_meta("cuda", [(i + 1, ctx, n) for i, (ctx, n) in enumerate(portions)], 16, tables)


PORTIONS = [[(0, 16)], [(5, 15), (0, 16), (3, 1)], [(0, 17), (9, 33)], [(0, 300), (40, 31), (7, 64)],
            [(2, 1700), (0, 9)]]


@pytest.mark.parametrize("portions", PORTIONS, ids=str)
@pytest.mark.parametrize("H,dk,dv", [(3, 6, 1), (2, 32, 16), (2, 33, 70), (2, 64, 128), (1, 96, 130), (2, 128, 64)])
@pytest.mark.parametrize("form", ["raw", "complement", "given"])
@pytest.mark.parametrize("decay", ["mild", "steep", "zero"])
def test_gates(portions, H, dk, dv, form, decay, monkeypatch):
    calls = record_native(monkeypatch, sq)
    monkeypatch.setattr(sq, "CHUNK_SCAN_MIN_SEG", 16)     # the long portion in segments, the short ones whole
    g = torch.Generator().manual_seed(dk * dv + len(portions))
    T, n = sum(p[1] for p in portions), H * dk
    sm = layout(portions)
    bias = {"mild": 1.0, "steep": -9.0, "zero": 0.0}[decay]
    z = torch.randn(T, n, generator=g) + bias              # steep: about 2^-13 a token, past the scaled form's range
    if decay == "zero":
        z[torch.rand(T, n, generator=g) < 0.05] = -200.0   # a gate that shuts altogether
    zq, v = torch.randn(T, n, generator=g), torch.randn(T, H * dv, generator=g).bfloat16()
    state = torch.randn(len(portions) + 1, H, dk, dv, generator=g)
    st = state.cuda()
    if form == "raw":
        low = torch.zeros(n) if decay != "mild" else torch.rand(n, generator=g) * 0.9
        z, zq = z.bfloat16(), zq.bfloat16()
        proj = torch.cat([torch.zeros(T, 3).bfloat16(), zq, z, v], 1).cuda()
        got = sq.lower_bound_recurrence(proj, 3, 3 + n, 3 + 2 * n, None, low.cuda(), st, H, dk, dv, sm)
        f = low.to(F64) + (1 - low.to(F64)) * torch.sigmoid(z.to(F64))
        q, k = torch.nn.functional.silu(zq.to(F64)), 1 - f
    else:
        f32 = torch.sigmoid(z)
        k32 = torch.randn(T, n, generator=g) if form == "given" else None
        got = sq.gated_linear_scan(zq.cuda(), f32.cuda(), None if k32 is None else k32.cuda(), v.cuda(), st, H, dk, dv, sm)
        q, f = zq.to(F64), f32.to(F64)
        k = 1 - f if k32 is None else k32.to(F64)
    assert "chunk_scan_gates" in calls
    at = 0
    for i, (ctx, m) in enumerate(portions):
        S0 = state[i + 1].to(F64) * (ctx > 0)
        r = slice(at, at + m)
        o, S = scan(*(t[r].view(m, H, -1) for t in (q, f, k, v.to(F64))), S0)
        close(got[r].view(m, H, dv), o)
        close(st[i + 1], S)
        at += m
    assert torch.equal(st[0].cpu(), state[0])


@pytest.mark.parametrize("portions", PORTIONS, ids=str)
@pytest.mark.parametrize("H,G,N,P", [(4, 2, 8, 16), (2, 1, 64, 24), (8, 2, 128, 64), (3, 3, 40, 70)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("rate", [0.0, 4.0])               # 4: e^4 of decay per unit of dt, past the chunk form's range
def test_ssm(portions, H, G, N, P, dtype, rate, monkeypatch):
    monkeypatch.setattr(sq, "CHUNK_SCAN_MIN_SEG", 16)
    calls = record_native(monkeypatch, sq)
    g = torch.Generator().manual_seed(N * P + len(portions))
    T = sum(p[1] for p in portions)
    sm = layout(portions)
    W = H * P + 2 * G * N
    xbc = torch.randn(T, (W + 7) // 8 * 8, generator=g).to(dtype)
    dt = torch.randn(T, H, generator=g).to(dtype)
    bias, A, D = torch.randn(H, generator=g) * 0.5 - 1, torch.randn(H, generator=g) * 0.5 + rate, torch.randn(H, generator=g)
    state = torch.randn(len(portions) + 1, H, N, P, generator=g)
    st = state.cuda()
    got = sq.ssm_scan(xbc.cuda()[:, :W], dt.cuda(), bias.cuda(), A.cuda(), D.cuda(), st, H, G, N, P, sm)
    # (B and C that do not lie on 16 bytes keep the token loop)
    assert ("chunk_scan_ssm" in calls) == (H * P * xbc.element_size() % 16 == 0) and ("ssm_scan" in calls) != ("chunk_scan_ssm" in calls)
    d = torch.nn.functional.softplus(dt.to(F64) + bias.to(F64))
    f = torch.exp(-torch.exp(A.to(F64)) * d)[..., None].expand(T, H, N)
    x = xbc.to(F64)[:, :H * P].view(T, H, P)
    B, C = (xbc.to(F64)[:, H * P + i * G * N:H * P + (i + 1) * G * N].view(T, G, N).repeat_interleave(H // G, 1) for i in (0, 1))
    at = 0
    for i, (ctx, m) in enumerate(portions):
        r = slice(at, at + m)
        o, S = scan(C[r], f[r], d[r][..., None] * B[r], x[r], state[i + 1].to(F64) * (ctx > 0))
        close(got[r].view(m, H, P), o + D.to(F64)[:, None] * x[r])
        close(st[i + 1], S)
        at += m


@pytest.mark.parametrize("where", ["v", "k", "q", "f"])
@pytest.mark.parametrize("value", [math.inf, math.nan, 3e38])
def test_values_out_of_range_reach_what_the_token_loop_lets_them_reach(where, value):
    """One bad input at token 21 of 48: the tokens before it (of the same chunk too) stay what they are."""
    g = torch.Generator().manual_seed(3)
    H, dk, dv, T, bad = 1, 64, 128, 48, 21
    t = {n: torch.rand(T, H * dk, generator=g) for n in "qfk"}
    t["v"] = torch.rand(T, H * dv, generator=g)
    t[where][bad, 5] = value
    st = torch.zeros(1, H, dk, dv).cuda()
    sm = seq_meta("cuda", [(0, 0, T)], 16, [[0, 1, 2]])
    got = sq.gated_linear_scan(t["q"].cuda(), t["f"].cuda(), t["k"].cuda(), t["v"].cuda(), st, H, dk, dv, sm).cpu()
    ref, _ = scan(*(t[n].to(F64).view(T, H, -1) for n in "qfkv"), torch.zeros(H, dk, dv, dtype=F64))
    close(got[:bad], ref[:bad].reshape(bad, -1))
    ref = ref.reshape(T, -1).float()   # (what fp32 holds of it)
    assert torch.equal(torch.isfinite(got[bad:]), torch.isfinite(ref[bad:]))


def error(got, ref):
    return float((got.detach().cpu().to(F64) - ref).norm() / ref.norm())


@pytest.mark.parametrize("form", ["raw", "given", "ssm"])
@pytest.mark.parametrize("level", [0, 1, 2, 3])
@pytest.mark.parametrize("dk,dv,portion", [(64, 128, (3, 400)), (128, 64, (3, 400)), (32, 32, (3, 1500))])
def test_errors_are_those_of_the_token_loop(form, level, dk, dv, portion, monkeypatch):
    """The error against fp64 of outputs and of the carried state, beside the token loop's on the same inputs, from decays of
    about 0.1 a token to 0.999. The chunks have as many roundings of a term as the loop; their order differs, so that either
    may come out ahead: a tenth is allowed for it, and for an error below 2^-24 what its own rounding makes."""
    g = torch.Generator().manual_seed(level + dk)
    H, T = 4, portion[1]
    sm = layout([portion])
    state = torch.randn(2, H, dk, dv, generator=g)
    if form == "ssm":
        xbc = torch.randn(T, H * dv + 2 * dk, generator=g)
        dt, bias, D = torch.randn(T, H, generator=g), torch.randn(H, generator=g) * 0.5 - 1, torch.randn(H, generator=g)
        A = torch.randn(H, generator=g) * 0.3 + (1.0, 0.0, -2.0, -5.0)[level]
        d = torch.nn.functional.softplus(dt.to(F64) + bias.to(F64))
        f = torch.exp(-torch.exp(A.to(F64)) * d)[..., None].expand(T, H, dk)
        x = xbc.to(F64)[:, :H * dv].view(T, H, dv)
        B, C = (xbc.to(F64)[:, None, H * dv + i * dk:H * dv + (i + 1) * dk].expand(T, H, dk) for i in (0, 1))
        ref, S = scan(C, f, d[..., None] * B, x, state[1].to(F64))
        ref = ref + D.to(F64)[:, None] * x

        def run(st):
            return sq.ssm_scan(xbc.cuda(), dt.cuda(), bias.cuda(), A.cuda(), D.cuda(), st, H, 1, dk, dv, sm)
    else:
        n = H * dk
        z, zq, v = (torch.randn(T, m, generator=g).bfloat16() for m in (n, n, H * dv))
        z = (z.float() + (-2.0, 0.0, 3.0, 7.0)[level]).bfloat16()
        f = torch.sigmoid(z.to(F64))
        if form == "raw":
            q, k, proj, low = torch.nn.functional.silu(zq.to(F64)), 1 - f, torch.cat([zq, z, v], 1).cuda(), torch.zeros(n).cuda()

            def run(st):
                return sq.lower_bound_recurrence(proj, 0, n, 2 * n, None, low, st, H, dk, dv, sm)
        else:
            f32, q32, k32 = f.float(), zq.float(), torch.randn(T, n, generator=g)
            f, q, k = f32.to(F64), q32.to(F64), k32.to(F64)

            def run(st):
                return sq.gated_linear_scan(q32.cuda(), f32.cuda(), k32.cuda(), v.cuda(), st, H, dk, dv, sm)
        ref, S = scan(*(t.view(T, H, -1) for t in (q, f, k, v.to(F64))), state[1].to(F64))
    errs = []
    for chunks in (True, False):
        with monkeypatch.context() as m:
            if not chunks:
                m.setattr(sq, "_chunk_scan_ok", lambda *a: False)
            calls, st = record_native(m, sq), state.cuda()
            o = run(st)
            assert any(c.startswith("chunk_scan_") for c in calls) == chunks
        errs.append((error(o.view(T, H, dv), ref), error(st[1], S)))
    (o, s), (o0, s0) = errs
    assert o <= 1.1 * o0 + 2.0 ** -27 and s <= 1.1 * s0 + 2.0 ** -28, errs


@pytest.mark.parametrize("segments", [False, True], ids=["one", "segments"])
def test_negative_and_growing_decays(segments, monkeypatch):
    """gated_linear_scan takes any f: signs alternate, factors above one, zeros; whole and in segments."""
    g = torch.Generator().manual_seed(9)
    H, dk, dv, T, ctx = 2, 64, 64, 700, 4
    q, k = torch.randn(T, H * dk, generator=g), torch.randn(T, H * dk, generator=g)
    f = torch.rand(T, H * dk, generator=g) * 0.9
    f[torch.rand(T, H * dk, generator=g) < 0.05] *= -1.0
    f[torch.rand(T, H * dk, generator=g) < 0.02] = 1.5
    f[torch.rand(T, H * dk, generator=g) < 0.01] = 0.0
    v, state = torch.randn(T, H * dv, generator=g), torch.randn(2, H, dk, dv, generator=g)
    state[:, :, ::3] = 0.0
    sm = layout([(ctx, T)])
    if not segments:
        monkeypatch.setattr(sq, "CHUNK_SCAN_MAX_SEGS", 1)
    assert (sq._chunk_scan_segments(sm, T, H, dk, dv, 64, "cuda")[1] is not None) == segments
    st = state.cuda()
    calls = record_native(monkeypatch, sq)
    got = sq.gated_linear_scan(q.cuda(), f.cuda(), k.cuda(), v.cuda(), st, H, dk, dv, sm)
    assert "chunk_scan_gates" in calls
    ref, S = scan(*(t.to(F64).view(T, H, -1) for t in (q, f, k, v)), state[1].to(F64))
    close(got.view(T, H, dv), ref)
    close(st[1], S)


@pytest.mark.parametrize("where", ["x", "B", "C", "dt"])
@pytest.mark.parametrize("value", [math.inf, math.nan, 1e36])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
def test_state_space_values_out_of_range(where, value, dtype, monkeypatch):
    """One bad input at token 21 of 48: the tokens before it stay what they are, and what is finite in the token loop is finite."""
    g = torch.Generator().manual_seed(4)
    H, N, P, T, bad = 1, 64, 64, 48, 21
    xbc, dt = torch.rand(T, P + 2 * N, generator=g).to(dtype), torch.rand(T, H, generator=g).to(dtype)
    (dt if where == "dt" else xbc)[bad, {"x": 5, "B": P + 7, "C": P + N + 9, "dt": 0}[where]] = value
    zero, st = torch.zeros(H), torch.zeros(1, H, N, P).cuda()
    sm = seq_meta("cuda", [(0, 0, T)], 16, [[0, 1, 2]])
    calls = record_native(monkeypatch, sq)
    got = sq.ssm_scan(xbc.cuda(), dt.cuda(), zero.cuda(), zero.cuda(), zero.cuda(), st, H, 1, N, P, sm).cpu()
    assert "chunk_scan_ssm" in calls
    d, z = torch.nn.functional.softplus(dt.to(F64)), xbc.to(F64)
    ref, _ = scan(z[:, None, P + N:], torch.exp(-d)[..., None].expand(T, H, N), d[..., None] * z[:, None, P:P + N], z[:, None, :P],
                  torch.zeros(H, N, P, dtype=F64))
    ref = ref.reshape(T, -1)
    close(got[:bad], ref[:bad])
    # (+ D x with D = 0: an infinite x is not a number in the sum)
    ref = (ref + 0.0 * z[:, :P]).float()
    assert torch.equal(torch.isfinite(got[bad:]), torch.isfinite(ref[bad:]))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
def test_state_space_products_that_only_x_keeps_in_range(dtype):
    """B and C whose product leaves fp32 beside an x that brings it back, and beside an x of 0."""
    g = torch.Generator().manual_seed(5)
    H, N, P, T = 2, 128, 64, 64
    xbc = torch.rand(T, H * P + 2 * N, generator=g)
    xbc[20:24, H * P:H * P + N] *= 1e30
    xbc[:, H * P + N:] *= 1e15
    xbc[20:24, :H * P] *= 1e-28
    xbc[20:24, :8] = 0.0
    xbc, dt = xbc.to(dtype), torch.rand(T, H, generator=g).to(dtype)
    zero, state = torch.zeros(H), torch.randn(2, H, N, P, generator=g)
    st = state.cuda()
    got = sq.ssm_scan(xbc.cuda(), dt.cuda(), zero.cuda(), zero.cuda(), zero.cuda(), st, H, 1, N, P, layout([(2, T)]))
    d, z = torch.nn.functional.softplus(dt.to(F64)), xbc.to(F64)
    B, C = (z[:, None, H * P + i * N:H * P + (i + 1) * N].expand(T, H, N) for i in (0, 1))
    ref, S = scan(C, torch.exp(-d)[..., None].expand(T, H, N), d[..., None] * B, z[:, :H * P].view(T, H, P), state[1].to(F64))
    assert bool(torch.isfinite(ref).all())
    close(got.view(T, H, P), ref)
    close(st[1], S)
