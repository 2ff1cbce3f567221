"""State-space chunks of 64 tokens (csrc/mixers/ssm_chunk.hip) against the token loop in fp64.

Tolerance: as in test_chunk_scan.py, 2e-5 of the output's root mean square for some 2^-24 of a term's size per token that it
remembers. How the errors compare with the fp32 token loop's own is tested apart, with a tenth for another order of the sums."""
import math

import pytest
import torch

from xgserve.ops import seqmix as sq

from _seq_util import record_native
from test_chunk_scan import F64, close, error, layout, scan

pytestmark = pytest.mark.gpu


def inputs(portions, H, G, N, P, level, seed):
    g = torch.Generator().manual_seed(seed)
    T = sum(n for _, n in portions)
    xbc = torch.nn.functional.silu(torch.randn(T, H * P + 2 * G * N, generator=g)).bfloat16()
    dt = torch.randn(T, H, generator=g).bfloat16()
    return (xbc, dt, torch.randn(H, generator=g) * 0.5 - 1, torch.randn(H, generator=g) * 0.3 + level, torch.randn(H, generator=g),
            torch.randn(len(portions) + 1, H, N, P, generator=g))


def run(args, portions, H, G, N, P):
    xbc, dt, bias, A, D, state = (t.cuda() for t in args)
    out = sq.ssm_scan(xbc, dt, bias, A, D, state, H, G, N, P, layout(portions))
    return out, state


def reference(args, portions, H, G, N, P):
    xbc, dt, bias, A, D, state = args
    T = xbc.shape[0]
    d = torch.nn.functional.softplus(dt.to(F64) + bias.to(F64))
    f = torch.exp(-torch.exp(A.to(F64)) * d)[..., None].expand(T, H, N)
    z = xbc.to(F64)
    x = z[:, :H * P].view(T, H, P)
    B, C = (z[:, H * P + i * G * N:H * P + (i + 1) * G * N].view(T, G, N).repeat_interleave(H // G, 1) for i in (0, 1))
    out, states, at = [], [], 0
    for i, (ctx, n) in enumerate(portions):
        r = slice(at, at + n)
        o, S = scan(C[r], f[r], d[r][..., None] * B[r], x[r], state[i + 1].to(F64) * (ctx > 0))
        out.append(o + D.to(F64)[:, None] * x[r])
        states.append(S)
        at += n
    return torch.cat(out).reshape(T, H * P), states


@pytest.mark.parametrize("portions", [[(0, 16)], [(3, 63), (0, 64)], [(0, 65), (9, 1), (2, 31)], [(5, 127), (0, 129), (1, 17)],
                                      [(0, 700), (40, 300), (7, 64)]], ids=str)
@pytest.mark.parametrize("H,G,N,P", [(8, 2, 128, 64), (3, 3, 64, 16), (4, 1, 64, 80), (2, 2, 128, 128)])
@pytest.mark.parametrize("level", [-0.5, 2.5])   # 2.5: some sub-chunks past 2^-90, which run token by token
@pytest.mark.parametrize("two_pass", [True, False])
def test_chunks(portions, H, G, N, P, level, two_pass, monkeypatch):
    monkeypatch.setattr(sq, "SCAN_TWO_PASS", two_pass)
    calls = record_native(monkeypatch, sq)
    args = inputs(portions, H, G, N, P, level, N + P + len(portions))
    got, state = run(args, portions, H, G, N, P)
    assert "chunk_scan_ssm" in calls and ("ssm_chunk_scratch_floats" in calls) == (two_pass and portions[0][1] == 700)
    want, states = reference(args, portions, H, G, N, P)
    close(got, want)
    for i, S in enumerate(states):
        close(state[i + 1], S)
    assert torch.equal(state[0].cpu(), args[-1][0])


@pytest.mark.parametrize("level", [0.0, -0.5, -2.0, -5.0])
@pytest.mark.parametrize("N,P,T", [(128, 64, 300), (64, 64, 200)])
def test_errors_are_those_of_the_token_loop(level, N, P, T, monkeypatch):
    """The mean of six draws: where decays are strong, a carried state is a few tokens and one draw a few dozen roundings."""
    portions, H, G, errs = [(3, T)], 8, 2, []
    for seed in range(6):
        args = inputs(portions, H, G, N, P, level, seed)
        want, states = reference(args, portions, H, G, N, P)
        for chunks in (True, False):
            with monkeypatch.context() as m:
                if not chunks:
                    m.setattr(sq, "_chunk_scan_ok", lambda *a: False)
                out, state = run(args, portions, H, G, N, P)
            errs += [error(out, want), error(state[1], states[0])]
    o, s, o0, s0 = (sum(errs[i::4]) / 6 for i in range(4))
    assert o <= 1.1 * o0 and s <= 1.1 * s0, (o, s, o0, s0)


@pytest.mark.parametrize("value", [3e37, math.inf, math.nan])
def test_states_that_cannot_be_split(value):
    """One entry of the incoming state: its column goes the way of the token loop, the others do not see it."""
    portions, H, G, N, P = [(3, 150)], 2, 1, 128, 64
    args = inputs(portions, H, G, N, P, -6.0, 5)
    ref, _ = run(args, portions, H, G, N, P)
    args[-1][1, 1, 40, 21] = value
    got, state = run(args, portions, H, G, N, P)
    keep = torch.ones(H * P, dtype=torch.bool)
    keep[P + 21] = False
    torch.testing.assert_close(got[:, keep], ref[:, keep], rtol=1e-4, atol=1e-4)
    want, states = reference(args, portions, H, G, N, P)
    close(got[:, ~keep].float(), want[:, ~keep].float().to(F64))
    close(state[1, 1, :, 21].float(), states[0][1, :, 21].float().to(F64))


@pytest.mark.parametrize("level", [0.6, 1.4])   # a chunk's decay is 2^-86 and 2^-192, no sub-chunk's past 2^-90
@pytest.mark.parametrize("large", [1e28, 1e31, 9e35])
def test_large_states_that_fade_before_large_rows_read_them(level, large):
    """C S of a whole chunk would leave fp32 (or what is left of the state, its decays), where a token's own sum does not. Tokens from 8
    on write nothing, so that every output is what is left of the state; C is 500 from token 24 on."""
    portions, H, G, N, P = [(3, 150)], 2, 1, 128, 64
    xbc, dt, bias, A, D, state = inputs(portions, H, G, N, P, level, 5)
    dt[:], bias[:], A[:], D[:] = -0.4, 0.0, level, 0.0   # steps of 0.513: decays of e^-0.93 and e^-2.08
    xbc[8:, :H * P] = 0
    xbc[24:, H * P + N + 40] = 500.0
    state[1, 1, :, 21] = 0
    state[1, 1, 40, 21] = large
    args = (xbc, dt, bias, A, D, state)
    got, after = run(args, portions, H, G, N, P)
    want, states = reference(args, portions, H, G, N, P)
    assert bool(torch.isfinite(got).all()) and bool(torch.isfinite(after).all())
    col, ref = got[:, P + 21].cpu().to(F64), want[:, P + 21]
    seen = ref.abs() > 1e-30   # (a state's entry is a product of up to 150 roundings of decays, 2^-23 each with the step's own)
    assert int(seen.sum()) > 40 and float(((col - ref).abs() / ref.abs())[seen].max()) < 150 * 2.0 ** -22
    assert float((after[1].cpu().to(F64) - states[0]).abs().max()) <= 150 * 2.0 ** -22 * float(states[0].abs().max()) + 1e-37


@pytest.mark.parametrize("portions", [[(9, 1)] * 5 + [(4, 700)] + [(0, 1), (3, 64), (5, 300), (0, 65)], [(0, 256)] + [(2, 1)] * 70,
                                      [(1, 100), (0, 257), (6, 1), (2, 513), (0, 128), (7, 129)], [(3, 1)] * 67 + [(0, 400), (5, 2)]], ids=len)
@pytest.mark.parametrize("H,G,N,P", [(8, 2, 128, 64), (2, 1, 64, 80)])
def test_sequences_of_one_and_of_several_segments(portions, H, G, N, P, monkeypatch):
    """Their order, single tokens of more than 64 sequences in front, lengths around whole segments; states with and without a past."""
    calls = record_native(monkeypatch, sq)
    args = inputs(portions, H, G, N, P, -0.5, N + len(portions))
    got, state = run(args, portions, H, G, N, P)
    assert "ssm_chunk_scratch_floats" in calls
    want, states = reference(args, portions, H, G, N, P)
    close(got, want)
    for i, S in enumerate(states):
        close(state[i + 1], S)
    assert torch.equal(state[0].cpu(), args[-1][0])


def test_scratch_does_not_grow_with_single_tokens():
    H, N, P = 8, 128, 64
    for singles in (0, 200):
        portions = [(3, 1)] * singles + [(0, 256)]
        seg, scratch = sq._ssm_chunk_segments(layout(portions), 256 + singles, H, N, P, 64, "cuda")
        assert seg < 256 and scratch.numel() <= (2 * ((256 + singles) // seg) + 2) * H * (N * P + 1) + 4


@pytest.mark.parametrize("where", ["x", "B", "C", "dt"])
@pytest.mark.parametrize("value", [2.0 ** 29, math.inf, math.nan])
def test_values_out_of_range_in_a_segment_between_others(where, value):
    """One bad input at token 300 of 700: what lies before it stays what it is, what follows is what the token loop makes of it."""
    portions, H, G, N, P, bad = [(3, 1), (4, 700)], 2, 1, 128, 64, 301
    args = inputs(portions, H, G, N, P, -4.0, 7)
    if where == "dt":
        args[1][bad, 1] = value
    else:
        args[0][bad, {"x": 21, "B": H * P + 40, "C": H * P + N + 40}[where]] = value
    got, state = run(args, portions, H, G, N, P)
    want, states = reference(args, portions, H, G, N, P)
    close(got[:bad], want[:bad])
    finite = torch.isfinite(want[bad:].float())
    assert torch.equal(torch.isfinite(got[bad:].cpu()), finite)
    # (a column's terms are of its largest output's size; 400 tokens' roundings of 2^-24, the step's among them twice)
    err = (torch.where(finite, got[bad:].cpu().to(F64) - want[bad:], 0.0)).abs()
    assert bool((err <= 400 * 2.0 ** -23 * torch.where(finite, want[bad:], 0.0).abs().amax(0) + 1e-5).all())
    assert torch.equal(torch.isfinite(state[2].cpu()), torch.isfinite(states[1].float()))


@pytest.mark.parametrize("two_pass", [True, False])
@pytest.mark.parametrize("H,G,N,P", [(8, 2, 128, 64), (2, 1, 64, 80)])
def test_chunks_of_few_tokens(H, G, N, P, two_pass, monkeypatch):
    """Sequences and remainders of one to six tokens, of which up to four run one by one."""
    monkeypatch.setattr(sq, "SCAN_TWO_PASS", two_pass)
    portions = [(9 * (n % 2), n) for n in range(1, 7)] + [(0, 65), (3, 66), (0, 68), (2, 69), (4, 259), (0, 4), (0, 324)]
    args = inputs(portions, H, G, N, P, -0.5, P)
    got, state = run(args, portions, H, G, N, P)
    want, states = reference(args, portions, H, G, N, P)
    close(got, want)
    for i, S in enumerate(states):
        close(state[i + 1], S)


@pytest.mark.parametrize("portions,chunk", [([(0, 16)] * 12, 16), ([(0, 16)], 16), ([(5, 8)] * 20 + [(0, 16)] * 20, 16), ([(0, 17)] * 12, 64),
                                            ([(5, 1)] * 20 + [(0, 16)] * 20, 64), ([(5, 1)] * 60 + [(0, 16)], 64), ([(0, 16)] * 6 + [(0, 33)], 64)],
                         ids=lambda v: str(v)[:20])
def test_portions_that_fill_a_chunk_of_16_alone_keep_it(portions, chunk, monkeypatch):
    H, G, N, P = 2, 1, 128, 64
    real, split = sq.mixers(), []

    class Recorder:
        def __getattr__(self, name):
            return (lambda *a: (split.append(a[-2]), real.chunk_scan_ssm(*a))) if name == "chunk_scan_ssm" else getattr(real, name)
    monkeypatch.setattr(sq, "mixers", Recorder)
    args = inputs(portions, H, G, N, P, -0.5, len(portions))
    got, state = run(args, portions, H, G, N, P)
    assert split == [chunk == 64]
    want, states = reference(args, portions, H, G, N, P)
    close(got, want)
    close(state[1:], torch.stack(states))


def test_few_heads_run_in_more_segments():
    for T, H, n in ((4001, 4, 32), (4001, 16, 32), (4001, 32, 16), (4001, 64, 8), (4001, 128, 4), (2000, 8, 16), (700, 8, 11)):
        seg, _ = sq._ssm_chunk_segments(layout([(0, T)]), T, H, 128, 64, 64, "cuda")
        assert -(-T // seg) == n, (T, H)
