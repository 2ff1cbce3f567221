"""Residual updates that add the parts of a product themselves and form the next convolution (ops.seqmix.norm_conv,
residual_norm_conv, post_norm_residual, linear_parts), against the separate kernels on the added product in fp64.

Tolerance: fp32 arithmetic throughout (a few 2^-24 per term, n 2^-24 relative for a sum of n squares, halved by the root); bf16
results rounded once (2^-8)."""
import pytest
import torch

from xgserve.ops import seqmix as sq

from _seq_util import record_native

pytestmark = pytest.mark.gpu


def meta(T, slots, ctx, max_q=1):
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    return sq.SeqMeta(T, max_q, i32(list(range(T + 1))), i32([c + 1 for c in ctx]), i32(slots), i32([[0]] * T), i32(list(range(T))),
                      i32(ctx), i32([0] * T), parts=True)


def close(got, want, terms, scale):
    bits = 2.0 ** -8 if got.dtype == torch.bfloat16 else 0.0
    assert bool(((got.double().cpu() - want).abs() <= want.abs() * bits + terms * 2.0 ** -23 * scale).all())


def norm(v, eps=1e-5):
    return v / (v.pow(2).mean(-1, keepdim=True) + eps).sqrt()


def source(g, S, T, W):
    """(what the kernel takes, its value in fp64): bf16 rows of a wider tensor, or S slabs."""
    if S == 0:
        y = torch.randn(T, W + 8, generator=g).bfloat16()[:, 4:4 + W]
        return y.cuda(), y.double()
    part = torch.randn(S, T, W, generator=g)
    return sq.Parts(part.cuda()), part.double().sum(0)


def conv(r, w, state, slots, ctx):
    nh, out, new = w.shape[1] - 1, torch.zeros_like(r), state.double().clone()
    for t, s in enumerate(slots):
        if s >= 0:
            hist = state[s].double() * (torch.arange(-nh, 0)[:, None] + ctx[t] >= 0)
            ext = torch.cat([hist, r[t:t + 1]])
            out[t] = r[t] + (w.double().T * ext).sum(0)
            new[s] = ext[1:]
    return out, new


@pytest.mark.parametrize("W,taps", [(4, 4), (2048, 4), (2052, 3), (4100, 2), (8192, 4)])
@pytest.mark.parametrize("S1,S2", [(0, 0), (1, 2), (4, 0), (8, 3)])
@pytest.mark.parametrize("T", [1, 5])
def test_norms_and_convolution(W, taps, S1, S2, T, monkeypatch):
    calls = record_native(monkeypatch, sq)
    g = torch.Generator().manual_seed(W + S1)
    slots, ctx = [3, -1, 0, 4, 2][:T], [7, 0, 0, 1, 2][:T]
    sm = meta(T, slots, ctx)
    x = torch.randn(T, W, generator=g)
    w, b, a1, a2 = (torch.randn(W, generator=g) for _ in range(4))
    cw, state = torch.randn(W, taps, generator=g), torch.randn(5, taps - 1, W, generator=g)
    live = [t for t in range(T) if slots[t] >= 0]
    y, yd = source(g, S1, T, W)
    assert sq.step_rows(sm, x.cuda(), torch.bfloat16, taps)
    # the normed sum becomes the residual
    xg, st = x.cuda(), state.cuda()
    h = sq.norm_conv(xg, y, w.cuda(), 1e-5, 0.7, b.cuda(), (cw.cuda(), st), sm, torch.bfloat16)
    r = norm(0.7 * x.double() + yd + b.double()) * (1 + w.double())
    want_h, want_st = conv(r, cw, state, slots, ctx)
    big = float(r.abs().max())
    close(xg, r, W / 2 + 16, big)
    close(h[live], want_h[live], W / 2 + 40, big * 8)
    close(st, want_st, W / 2 + 16, max(big, 5.0))
    xg = x.cuda()
    assert sq.norm_conv(xg, y, w.cuda(), 1e-5, 0.7, None, None, sm, torch.bfloat16) is None
    r = norm(0.7 * x.double() + yd) * (1 + w.double())
    close(xg, r, W / 2 + 16, float(r.abs().max()))
    # the sum stays the residual, its norm goes on
    z, zd = source(g, S2, T, W)
    y3 = torch.randn(T, W, generator=g)
    for f32, y2, y2d, t3 in ((True, z, zd, y3), (False, z, zd, None), (False, None, 0.0, None)):
        xg, st = x.cuda(), state.cuda()
        n32, n, h = sq.residual_norm_conv(xg, y, a1.cuda(), y2, None if t3 is None else t3.cuda(), a2.cuda(), w.cuda(), 1e-5,
                                          torch.bfloat16, (cw.cuda(), st), f32, sm)
        v = x.double() + a1.double() * yd + a2.double() * (y2d + (0.0 if t3 is None else t3.double()))
        r = norm(v) * w.double()
        want_h, want_st = conv(r, cw, state, slots, ctx)
        big = float(r.abs().max())
        close(xg, v, 24, float(v.abs().max()) + 30)
        close(n, r, W / 2 + 16, big)
        assert (n32 is not None) == f32
        if f32:
            close(n32, r, W / 2 + 16, big)
        close(h[live], want_h[live], W / 2 + 40, big * 8)
        close(st, want_st, W / 2 + 16, max(big, 5.0))
    assert calls == ["row_update"] * 5


@pytest.mark.parametrize("W", [4, 2048, 4096, 4100])
@pytest.mark.parametrize("S1,S2", [(2, None), (8, None), (4, 2), (2, 0), (0, 4)])
def test_post_norm(W, S1, S2):
    g, T = torch.Generator().manual_seed(W), 3
    x, b, pw, nw, p1, p2 = (torch.randn(*s, generator=g) for s in ((T, W), (W,), (W,), (W,), (W,), (W,)))
    y, yd = source(g, S1, T, W)
    y2, y2d = (None, None) if S2 is None else source(g, S2, T, W)
    xg = x.cuda()
    kw = {} if y2 is None else dict(y2=y2, pre_w=(p1.cuda(), p2.cuda()))
    n = sq.post_norm_residual(xg, y, b.cuda() if y2 is None else None, pw.cuda(), 0.5, None, nw.cuda(), 1e-5, torch.bfloat16, **kw)
    if y2 is None:
        u = yd + b.double()
    else:   # (parts beside rows are rounded to the rows' type first)
        rnd = (lambda v: v.bfloat16().double()) if 0 in (S1, S2) else (lambda v: v)
        u = 0.5 * (norm(rnd(yd.float())) * p1.double() + norm(rnd(y2d.float())) * p2.double())
    v = x.double() + 0.5 * norm(u) * (1 + pw.double())
    r = norm(v) * (1 + nw.double())
    close(xg, v, W + 40, float(v.abs().max()))
    close(n, r, W + 40, float(r.abs().max()))


def test_products_stay_in_parts_where_the_step_says_so():
    g = torch.Generator().manual_seed(0)
    x, w = torch.randn(17, 2048, generator=g).bfloat16().cuda(), (torch.randn(2048, 2048, generator=g) / 45).bfloat16().cuda()
    sm = meta(1, [0], [0])
    y = sq.linear_parts(x, w, sm)
    assert isinstance(y, sq.Parts) and y.part.shape == (4, 17, 2048)
    want = (x.double() @ w.double().T).cpu()
    assert bool(((y.part.double().sum(0).cpu() - want).abs() <= 2048 * 2.0 ** -24 * 60).all())
    sm.parts = False
    assert sq.linear_parts(x, w, sm).dtype == torch.bfloat16
    sm.parts = True
    assert sq.linear_parts(torch.cat([x] * 4), w, sm).dtype == torch.bfloat16       # more than 64 rows
    sm.max_q = 2
    assert not sq.step_rows(sm, x.float(), torch.bfloat16, 4) and sq.step_rows(sm, x.float(), torch.bfloat16)
    assert not sq.step_rows(sm, x.float(), torch.float32)


def test_weights_off_16_bytes_take_the_separate_kernels():
    """Parameters and states that are slices of a larger buffer: the same results, by launches that take them."""
    g = torch.Generator().manual_seed(2)
    T, W, taps, slots, ctx = 3, 64, 4, [2, 0, 1], [7, 0, 2]
    sm = meta(T, slots, ctx)
    x, w, a1, a2 = torch.randn(T, W, generator=g), *(torch.randn(W, generator=g) for _ in range(3))
    cw, state = torch.randn(W, taps, generator=g), torch.randn(3, taps - 1, W, generator=g)
    y, z = (sq.Parts(torch.randn(2, T, W, generator=g).cuda()) for _ in range(2))

    def off(t):
        return torch.cat([torch.zeros(1), t.flatten()]).cuda()[1:].view(t.shape)
    outs = []
    for place in (lambda t: t.cuda(), off):
        xg, st = x.cuda(), place(state)
        h = sq.norm_conv(xg, y, place(w), 1e-5, 0.7, None, (place(cw), st), sm, torch.bfloat16)
        x2, st2 = x.cuda(), place(state)
        rest = sq.residual_norm_conv(x2, y, place(a1), z, None, place(a2), place(w), 1e-5, torch.bfloat16, (place(cw), st2), True, sm)
        outs.append([xg, st, h, x2, st2, *rest])
    for a, b in zip(*outs):   # (the product's sum is rounded to bf16 there)
        torch.testing.assert_close(a.float(), b.float(), rtol=2e-2, atol=4e-2)
