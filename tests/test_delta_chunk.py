"""The chunked form of the generalized delta rule (csrc/mixers/delta_chunk.hip) against the token loop in fp64.

Tolerance: a term has one rounding of each factor and one of each sum that it is part of, some 2^-24 of its size per token that the
state remembers; keys that repeat make the terms larger than their sum. 2e-5 of the output's root mean square covers the sizes
here. How the errors compare with the token loop's own is tested apart."""
import math

import pytest
import torch

from xgserve.ops import seqmix as sq

from _seq_util import record_native
from test_chunk_scan import close, error, layout

F64 = torch.float64
pytestmark = pytest.mark.gpu


def reference(t, S):
    """t: fp64 r, k, v, a-logits + bias, decay logits + bias, each [T, H, D]."""
    u = t["k"] / torch.sqrt(t["k"].pow(2).sum(-1, keepdim=True) + 1e-6)
    b = torch.sigmoid(t["a"]) * u
    w = torch.exp(-math.exp(-0.5) * torch.sigmoid(t["w"]))
    out = []
    for i in range(u.shape[0]):
        uS = torch.einsum("hk,hkd->hd", u[i], S)
        S = w[i][:, :, None] * S - b[i][:, :, None] * uS[:, None] + t["k"][i][:, :, None] * t["v"][i][:, None]
        out.append(torch.einsum("hk,hkd->hd", t["r"][i], S))
    return torch.stack(out), S


def case(portions, H, D, dtype, g, tweak=lambda x: None):
    T, n = sum(p[1] for p in portions), H * D
    x = {c: torch.randn(T, n, generator=g) for c in "rkvaw"}
    tweak(x)
    x = {c: v.to(dtype) for c, v in x.items()}
    ab, wb = torch.randn(n, generator=g) * 0.5, torch.randn(n, generator=g)
    proj = torch.cat([torch.zeros(T, 8).to(dtype)] + [x[c] for c in "rkva"], 1).cuda()
    state = torch.randn(len(portions) + 1, H, D, D, generator=g)
    st = state.cuda()
    got = sq.delta_rule_scan(proj, 8, 8 + n, 8 + 2 * n, 8 + 3 * n, x["w"].cuda(), ab.cuda(), wb.cuda(), st, H, D, layout(portions))
    t = {c: v.to(F64).view(T, H, D) for c, v in x.items()}
    t["a"], t["w"] = t["a"] + ab.to(F64).view(H, D), t["w"] + wb.to(F64).view(H, D)
    return got.view(T, H, D), st, state, t


@pytest.mark.parametrize("portions", [[(0, 32)], [(5, 15), (0, 33), (3, 1), (2, 16)], [(9, 47), (0, 48)], [(0, 300), (40, 31), (7, 64)]], ids=str)
@pytest.mark.parametrize("H,D", [(3, 32), (2, 64), (5, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("keys", ["random", "repeated", "none"])
def test_portions(portions, H, D, dtype, keys, monkeypatch):
    """repeated: every token removes what the last one wrote (the triangular system at its fullest); none: zero keys."""
    def tweak(x):
        if keys == "repeated":
            x["k"][:] = x["k"][:1]
            x["a"] += 6.0
        elif keys == "none":
            x["k"][::2] = 0.0
    calls = record_native(monkeypatch, sq)
    got, st, state, t = case(portions, H, D, dtype, torch.Generator().manual_seed(H * D + len(portions)), tweak)
    assert calls.count("delta_chunk") == 1 and "delta_scan" not in calls
    at = 0
    for i, (ctx, m) in enumerate(portions):
        r = slice(at, at + m)
        o, S = reference({c: v[r] for c, v in t.items()}, state[i + 1].to(F64) * (ctx > 0))
        close(got[r], o)
        close(st[i + 1], S)
        at += m
    assert torch.equal(st[0].cpu(), state[0])


@pytest.mark.parametrize("where", list("rkvaw"))
@pytest.mark.parametrize("value", [math.inf, -math.inf, math.nan])
def test_values_out_of_range_reach_what_the_token_loop_lets_them_reach(where, value):
    def tweak(x):
        x[where][21, 5] = value
    got, _, state, t = case([(0, 48)], 1, 64, torch.float32, torch.Generator().manual_seed(3), tweak)
    ref, _ = reference(t, state[1].to(F64) * 0)
    close(got[:21], ref[:21])
    assert torch.equal(torch.isfinite(got[21:].cpu()), torch.isfinite(ref[21:].float()))


@pytest.mark.parametrize("by_token", [[0], [6], [2, 3], [0, 2, 4, 6], [1, 3, 5], list(range(7))], ids=str)
@pytest.mark.parametrize("D", [32, 64])
def test_chunks_run_token_by_token_between_others(by_token, D):
    """A chunk's outputs are stored by the one that follows it: either may be one that runs token by token (an r of 2^29)."""
    large = [min(16 * c + 5 * c % 13, 99) for c in by_token]
    def tweak(x):
        x["r"][large, 3::D] = 2.0 ** 29
    got, st, state, t = case([(7, 100)], 2, D, torch.bfloat16, torch.Generator().manual_seed(D + len(by_token)), tweak)
    o, S = reference(t, state[1].to(F64))
    rest = [i for i in range(100) if i not in large]
    close(got[rest], o[rest])
    close(got[large], o[large])
    close(st[1], S)


@pytest.mark.parametrize("mid", [-4.0, 0.0, 4.0])
@pytest.mark.parametrize("H,D", [(4, 32), (4, 64)])
def test_errors_are_those_of_the_token_loop(mid, H, D, monkeypatch):
    """Errors against fp64 beside the token loop's on the same inputs, decays around 0.97, 0.73 and 0.55. State and outputs have as
    many roundings of their size as in the loop; the order differs, so that either may come out ahead: a tenth is allowed for it."""
    def tweak(x):
        x["w"] += mid
        x["r"] = 0.8 * x["r"] + 0.6 * x["k"]
    errs = []
    for chunks in (True, False):
        with monkeypatch.context() as m:
            if not chunks:
                m.setattr(sq, "DELTA_CHUNK_MIN", 1 << 30)
            calls = record_native(m, sq)
            got, st, state, t = case([(3, 700)], H, D, torch.bfloat16, torch.Generator().manual_seed(D), tweak)
            assert ("delta_chunk" in calls) == chunks
        o, S = reference(t, state[1].to(F64))
        errs.append((error(got, o), error(st[1], S)))
    (o, s), (o0, s0) = errs
    assert o <= 1.1 * o0 and s <= 1.1 * s0, errs
