"""The chunked fp32 form of the outer-product recurrences (csrc/mixers/chunk_scan.hip) against the token loop in fp64.

Tolerance: a chunk's factors are 2^(sum of at most 60 bits of decay); the sum carries 60 x 2^-24 of absolute error, a factor
ln 2 times that, and a weight is the product of two of them: 60 x 2^-24 x 0.69 x 2 = 5e-6 of each term; 4 times that of the
output's root mean square bounds the sums seen here. Chunks beyond 60 bits run token by token (2^-24 per step)."""
import math

import pytest
import torch

from xgserve.ops import seqmix as sq

from _seq_util import seq_meta

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
