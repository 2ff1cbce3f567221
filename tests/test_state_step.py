"""Single tokens of the matrix-valued recurrences against fp64.

Tolerance: fp32 products and sums of dk (or D) terms, relative to the sum of their magnitudes; bf16 results rounded once
(2^-8). The state keeps one fused update per element."""
import pytest
import torch

from xgserve.ops import seqmix as sq

from _seq_util import record_native

pytestmark = pytest.mark.gpu


def meta(slots, ctx):
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    T = len(slots)
    return sq.SeqMeta(T, 1, i32(list(range(T + 1))), i32([c + 1 for c in ctx]), i32(slots), i32([[0]] * T), i32(list(range(T))),
                      i32(ctx), i32([0] * T))


SLOTS, CTX = [2, -1, 0, 4], [5, 3, 0, 1]


@pytest.mark.parametrize("H,dk,dv", [(1, 1, 4), (3, 64, 128), (2, 128, 128), (2, 256, 64), (3, 33, 20), (2, 16, 256)])
@pytest.mark.parametrize("mode", ["plain", "complement", "raw", "decay", "bonus"])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_gated_linear(H, dk, dv, mode, dt, monkeypatch):
    calls = record_native(monkeypatch, sq)
    g = torch.Generator().manual_seed(dk + dv)
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    T, n, sm = len(SLOTS), H * dk, meta(SLOTS, CTX)
    state = rnd(5, H, dk, dv)
    pad = -2 * n % 4
    proj = rnd(T, 2 * n + pad + H * dv).to(dt)
    lower, bias = torch.rand(n, generator=g), rnd(n)
    q, f, k = rnd(T, n), torch.rand(T, n, generator=g), rnd(T, n)
    decay, bonus = torch.rand(H, generator=g), rnd(n)
    off_v = 2 * n + pad
    v = proj[:, off_v:]
    c = lambda t: t.cuda()  # noqa: E731
    st, pg = c(state), c(proj)
    assert sq._gla_step_ok(pg[:, off_v:], sm, dk, dv)
    if mode == "raw":
        o = sq.lower_bound_recurrence(pg, 0, n, off_v, c(bias), c(lower), st, H, dk, dv, sm)
        z = proj.double()
        qd = z[:, :n] * torch.sigmoid(z[:, :n])
        fd = lower.double() + (1 - lower.double()) * torch.sigmoid(z[:, n:2 * n] + bias.double())
        kd = 1 - fd
    else:
        kw = dict(decay=c(decay)) if mode == "decay" else dict(bonus=c(bonus)) if mode == "bonus" else {}
        o = sq.gated_linear_scan(c(q), None if mode == "decay" else c(f), None if mode == "complement" else c(k), pg[:, off_v:], st,
                                 H, dk, dv, sm, **kw)
        qd, kd = q.double(), k.double()
        fd = decay.double().repeat_interleave(dk).expand(T, n) if mode == "decay" else f.double()
        if mode == "complement":
            kd = 1 - fd
    assert "gla_step" in calls and "gated_linear_scan" not in calls
    want = state.double().clone()
    for t, s in enumerate(SLOTS):
        if s < 0:
            continue
        S = state[s].double() if CTX[t] else torch.zeros(H, dk, dv, dtype=torch.float64)
        kv = kd[t].view(H, dk, 1) * v[t].double().view(H, 1, dv)
        new = fd[t].view(H, dk, 1) * S + kv
        src = S + bonus.double().view(H, dk, 1) * kv if mode == "bonus" else new
        qt = qd[t].view(H, dk, 1)
        err = (o[t].double().cpu().view(H, dv) - (qt * src).sum(1)).abs()
        mag = (qt.abs() * (S.abs() + kv.abs() * (1 + bonus.double().abs().max()) + v[t].double().abs().max())).sum(1)
        assert bool((err <= (dk + 40) * 2.0 ** -24 * mag + 1e-12).all())
        want[s] = new
    err = (st.double().cpu() - want).abs()
    assert bool((err <= 40 * 2.0 ** -24 * (want.abs() + float(v.double().abs().max()) * 4)).all())


@pytest.mark.parametrize("H,G,N,P", [(1, 1, 1, 4), (4, 2, 128, 64), (6, 2, 33, 20), (2, 1, 256, 64), (2, 2, 16, 256)])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_state_space(H, G, N, P, dt, monkeypatch):
    calls = record_native(monkeypatch, sq)
    g = torch.Generator().manual_seed(N + P)
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    T, sm = len(SLOTS), meta(SLOTS, CTX)
    xbc, raw = rnd(T, -(-(H * P + 2 * G * N) // 4) * 4).to(dt), rnd(T, H + 3).to(dt)
    bias, A, D, state = rnd(H), rnd(H), rnd(H), rnd(5, H, N, P)
    st, xg = state.cuda(), xbc.cuda()
    assert sq._gla_step_ok(xg, sm, N, P)
    y = sq.ssm_scan(xg, raw.cuda()[:, 3:], bias.cuda(), A.cuda(), D.cuda(), st, H, G, N, P, sm)
    assert calls == ["ssm_step"]
    z = xbc.double()
    x = z[:, :H * P].view(T, H, P)
    B, C = (z[:, H * P + i * G * N:H * P + (i + 1) * G * N].view(T, G, N).repeat_interleave(H // G, 1) for i in (0, 1))
    step = torch.nn.functional.softplus(raw[:, 3:].double() + bias.double())
    want = state.double().clone()
    for t, s in enumerate(SLOTS):
        if s < 0:
            continue
        S = state[s].double() if CTX[t] else torch.zeros(H, N, P, dtype=torch.float64)
        dec = torch.exp(-torch.exp(A.double()) * step[t])
        new = dec[:, None, None] * S + (step[t][:, None] * B[t])[:, :, None] * x[t][:, None]
        out = torch.einsum("hnp,hn->hp", new, C[t]) + D.double()[:, None] * x[t]
        mag = torch.einsum("hnp,hn->hp", new.abs(), C[t].abs()) + D.double().abs()[:, None] * x[t].abs()
        assert bool(((y[t].double().cpu().view(H, P) - out).abs() <= (N + 60) * 2.0 ** -24 * (mag + 1) * 4).all())
        want[s] = new
    assert bool(((st.double().cpu() - want).abs() <= 200 * 2.0 ** -24 * (want.abs() + 1) * 4).all())


@pytest.mark.parametrize("H,D,lr", [(2, 32, 8), (3, 64, 32), (2, 128, 64), (1, 64, 256)])
def test_delta_rule(H, D, lr, monkeypatch):
    calls = record_native(monkeypatch, sq)
    g = torch.Generator().manual_seed(D + lr)
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    T, HD, sm = len(SLOTS), H * D, meta(SLOTS, CTX)
    proj = rnd(T, 5 * HD + lr).bfloat16()
    w2 = (rnd(HD, lr) / lr ** 0.5).bfloat16()
    a_bias, w0, norm, state = rnd(HD), rnd(HD), rnd(HD), rnd(5, H, D, D)
    st = state.cuda()
    y = sq.delta_rule_mix(proj.cuda(), w2.cuda(), a_bias.cuda(), w0.cuda(), norm.cuda(), st, 1e-5, H, D, sm, torch.bfloat16)
    assert calls == ["delta_step"]
    p = proj.double()
    r, k, v, gate, za = (p[:, i * HD:(i + 1) * HD].view(T, H, D) for i in range(5))
    wl = torch.tanh(p[:, 5 * HD:]) @ w2.double().T
    w = torch.exp(-sq.DECAY_SCALE * torch.sigmoid(wl + w0.double())).view(T, H, D)
    a = torch.sigmoid(za + a_bias.double().view(H, D))
    u = k / (k.pow(2).sum(-1, keepdim=True) + sq.UNIT_KEY_EPS).sqrt()
    want = state.double().clone()
    for t, s in enumerate(SLOTS):
        if s < 0:
            continue
        S = state[s].double() if CTX[t] else torch.zeros(H, D, D, dtype=torch.float64)
        uS = torch.einsum("hi,hij->hj", u[t], S)
        new = w[t][:, :, None] * S - (a[t] * u[t])[:, :, None] * uS[:, None] + k[t][:, :, None] * v[t][:, None]
        o = torch.einsum("hij,hi->hj", new, r[t])
        yt = (o / (o.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt()).reshape(HD) * norm.double() * torch.sigmoid(gate[t].reshape(HD))
        # a sum of D terms of the state times r, relative to the head's root mean square
        rel = (D + lr + 60) * 2.0 ** -23 * float((new.abs() * r[t].abs()[:, :, None]).sum(1).max()) / float(
            o.pow(2).mean(-1).sqrt().min())
        err = (y[t].double().cpu() - yt).abs()
        assert bool((err <= yt.abs() * 2.0 ** -8 + rel * norm.double().abs().max() * 2).all())
        want[s] = new
    assert bool(((st.double().cpu() - want).abs() <= (D + lr + 60) * 2.0 ** -23 * (want.abs().max() + 8)).all())


def test_odd_states_run_as_scans():
    v = torch.zeros(4, 8, device="cuda")
    sm = meta(SLOTS, CTX)
    assert sq._gla_step_ok(v, sm, 8, 8) and not sq._gla_step_ok(v, sm, 8, 6) and not sq._gla_step_ok(v[:, 1:], sm, 8, 4)
    assert not sq._gla_step_ok(v, sm, 256, 128)
    sm.max_q = 2
    assert not sq._gla_step_ok(v, sm, 8, 8)


@pytest.mark.parametrize("dk,dv", [(88, 176), (168, 96), (120, 136)])
def test_states_with_too_many_rows_per_thread_run_as_scans(dk, dv, monkeypatch):
    """Sizes within 128 x 128 elements whose columns do not divide the workgroup: one token, through the public ops."""
    g = torch.Generator().manual_seed(dk)
    T, H, sm = len(SLOTS), 2, meta(SLOTS, CTX)
    q, f, k = (torch.rand(T, H * dk, generator=g) for _ in range(3))
    v, state = torch.randn(T, H * dv, generator=g), torch.randn(5, H, dk, dv, generator=g)
    xbc = torch.randn(T, H * dv + 2 * dk, generator=g)
    dt, bias, A, D = torch.randn(T, H, generator=g), torch.randn(H, generator=g), torch.randn(H, generator=g), torch.randn(H, generator=g)
    st, st2 = state.cuda(), state.cuda()
    calls = record_native(monkeypatch, sq)
    o = sq.gated_linear_scan(q.cuda(), f.cuda(), k.cuda(), v.cuda(), st, H, dk, dv, sm).cpu().double()
    y = sq.ssm_scan(xbc.cuda(), dt.cuda(), bias.cuda(), A.cuda(), D.cuda(), st2, H, 1, dk, dv, sm).cpu().double()
    assert calls == ["gated_linear_scan", "ssm_scan"]
    step = torch.nn.functional.softplus(dt.double() + bias.double())
    for t, s in enumerate(SLOTS):
        if s < 0:
            continue
        S = state[s].double() if CTX[t] else torch.zeros(H, dk, dv, dtype=torch.float64)
        new = f[t].double().view(H, dk, 1) * S + k[t].double().view(H, dk, 1) * v[t].double().view(H, 1, dv)
        want = (q[t].double().view(H, dk, 1) * new).sum(1).reshape(-1)
        assert bool(((o[t] - want).abs() <= (dk + 40) * 2.0 ** -24 * (q[t].double().view(H, dk, 1) * new.abs()).sum(1).reshape(-1) * 4).all())
        x, B, C = (z.double() for z in xbc[t].split([H * dv, dk, dk]))
        new = torch.exp(-torch.exp(A.double()) * step[t])[:, None, None] * S + step[t][:, None, None] * B[:, None] * x.view(H, 1, dv)
        want = (C[:, None] * new).sum(1) + D.double()[:, None] * x.view(H, dv)
        mag = (C.abs()[:, None] * new.abs()).sum(1) + D.double().abs()[:, None] * x.abs().view(H, dv)
        assert bool(((y[t].view(H, dv) - want).abs() <= (dk + 60) * 2.0 ** -24 * (mag + 1) * 4).all())
