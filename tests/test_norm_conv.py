"""The residual sum, its norm and the convolution behind it of prompt rows in one pass (ops.seqmix.norm_conv_rows,
residual_norm_conv_rows), against fp64.

Tolerance: fp32 arithmetic (a few 2^-24 per term, n 2^-24 relative for a sum of n squares, halved by the root); bf16 results
rounded once (2^-8)."""
import pytest
import torch

from xgserve.ops import seqmix as sq

from _seq_util import record_native

pytestmark = pytest.mark.gpu


def meta(lens, ctx, slots):
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    n, first = len(lens), [sum(lens[:i]) for i in range(len(lens) + 1)]
    one = i32([0])
    return sq.SeqMeta(n, max(lens), i32(first), i32([q + c for q, c in zip(lens, ctx)]), i32(slots), one, one, one, one), first


def close(got, want, terms, scale):
    bits = 2.0 ** -8 if got.dtype == torch.bfloat16 else 0.0
    assert bool(((got.double().cpu() - want).abs() <= want.abs() * bits + terms * 2.0 ** -23 * scale).all())


def norm(v, eps=1e-5):
    return v / (v.pow(2).mean(-1, keepdim=True) + eps).sqrt()


def conv(r, w, state, lens, first, ctx, slots):
    """(outputs, rows that have one, carried inputs)"""
    nh, out, live, new = w.shape[1] - 1, r.clone(), torch.zeros(r.shape[0], dtype=torch.bool), state.double().clone()
    for q, a, c, s in zip(lens, first, ctx, slots):
        if s < 0 or q == 0:
            continue
        hist = state[s].double() * (torch.arange(-nh, 0)[:, None] + c >= 0)
        ext = torch.cat([hist, r[a:a + q]])
        for j in range(nh + 1):
            out[a:a + q] += w.double()[:, j] * ext[j:j + q]
        live[a:a + q] = True
        new[s] = ext[-nh:]
    return out, live, new


# strips of 5 rows (4 taps), up to 33 where there are many rows of few columns; sequences that end at a strip, one row before or behind
@pytest.mark.parametrize("W,taps,lens,behind", [
    (4, 4, [1, 2, 3, 4, 5, 6, 0, 9, 10, 11], 0), (2048, 4, [5, 1, 7, 16, 2], 3), (2052, 3, [6, 12, 7, 1, 13], 1), (4096, 2, [7, 1, 8, 14, 15], 0),
    (64, 4, [4001, 1999, 33, 1], 2), (8, 4, [9000, 7000, 2500, 34, 35], 0), (16, 2, [9000, 7000, 2500, 34, 35], 40)])
def test_against_fp64(W, taps, lens, behind, monkeypatch):
    calls = record_native(monkeypatch, sq)
    g = torch.Generator().manual_seed(W + taps)
    n = len(lens)
    ctx, slots = [(0, 7, 1, 2, 0)[i % 5] for i in range(n)], [(-1 if i == 3 else n - 1 - i) for i in range(n)]
    sm, first = meta(lens, ctx, slots)
    T = first[-1] + behind
    x, w, b, a1, a2 = torch.randn(T, W, generator=g), *(torch.randn(W, generator=g) for _ in range(4))
    y, z = (torch.randn(T, W + 8, generator=g).bfloat16()[:, 4:4 + W] for _ in range(2))
    yg, zg = (torch.randn(T, W + 8).bfloat16().cuda()[:, 4:4 + W].copy_(t) for t in (y, z))
    cw, state = torch.randn(W, taps, generator=g), torch.randn(n, taps - 1, W, generator=g)
    for bias in (b, None):
        xg, st = x.cuda(), state.cuda()
        out, h = sq.norm_conv_rows(xg, yg, w.cuda(), 1e-5, 0.7, None if bias is None else bias.cuda(), (cw.cuda(), st), sm, torch.bfloat16)
        r = norm(0.7 * x.double() + y.double() + (0 if bias is None else bias.double())) * (1 + w.double())
        want, live, new = conv(r, cw, state, lens, first, ctx, slots)
        big = float(r.abs().max())
        assert torch.equal(xg.cpu(), x)
        close(out, r, W / 2 + 16, big)
        close(h[live], want[live], W / 2 + 40, big * 8)
        close(st, new, W / 2 + 16, max(big, 5.0))
    for f32, z2, s1, s2 in ((True, zg, a1, a2), (False, zg, None, a2), (False, None, a1, None)):
        xg, st = x.cuda(), state.cuda()
        out, n32, nact, h = sq.residual_norm_conv_rows(xg, yg, None if s1 is None else s1.cuda(), z2, None, None if s2 is None else s2.cuda(),
                                                       w.cuda(), 1e-5, torch.bfloat16, (cw.cuda(), st), f32, sm)
        v = x.double() + (1 if s1 is None else s1.double()) * y.double()
        if z2 is not None:
            v = v + (1 if s2 is None else s2.double()) * z.double()
        r = norm(v) * w.double()
        want, live, new = conv(r, cw, state, lens, first, ctx, slots)
        big = float(r.abs().max())
        close(out, v, 24, float(v.abs().max()) + 30)
        close(nact, r, W / 2 + 16, big)
        assert (n32 is not None) == f32
        if f32:
            close(n32, r, W / 2 + 16, big)
        close(h[live], want[live], W / 2 + 40, big * 8)
        close(st, new, W / 2 + 16, max(big, 5.0))
    assert calls == ["norm_conv"] * 5


@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("W", [8, 1024, 1028, 2052])
@pytest.mark.parametrize("strip", [8, 12, 20, 36])
def test_strips(strip, W, taps, monkeypatch):
    """Strips of every length, which go by the rows and the CUs: sequences that end with one or two of them, a row before and a row behind,
    at a start, behind carried inputs and behind fewer of those than there are taps."""
    rows = strip + 1 - taps
    lens = [n for k in (1, 2) for n in (k * rows - 1, k * rows, k * rows + 1) for _ in range(3)] + [1, 1, 1]
    T = sum(lens)
    # workgroups that strips of this length need, and shorter ones exceed (strips of 8 have one workgroup a CU, as all of wide rows have)
    wgs = -(-T // rows)
    cus = wgs if strip == 8 or W > 2048 else -(-wgs // 2)
    assert strip == 8 or -(-T // (rows - 4)) > (cus if strip == 12 or W > 2048 else 2 * cus)
    monkeypatch.setattr(sq, "cu_count", lambda d: cus)
    g, n = torch.Generator().manual_seed(strip + taps), len(lens)
    ctx, slots = [(0, 7, 1)[i % 3] for i in range(n)], [n - 1 - i for i in range(n)]
    sm, first = meta(lens, ctx, slots)
    x, w, a1 = torch.randn(T, W, generator=g), torch.randn(W, generator=g), torch.randn(W, generator=g)
    y = torch.randn(T, W, generator=g).bfloat16()
    cw, state = torch.randn(W, taps, generator=g), torch.randn(n, taps - 1, W, generator=g)
    for keep in (True, False):
        st = state.cuda()
        if keep:
            out, h = sq.norm_conv_rows(x.cuda(), y.cuda(), w.cuda(), 1e-5, 0.7, a1.cuda(), (cw.cuda(), st), sm, torch.bfloat16)
            r = norm(0.7 * x.double() + y.double() + a1.double()) * (1 + w.double())
            close(out, r, W / 2 + 16, float(r.abs().max()))
        else:
            out, _, nact, h = sq.residual_norm_conv_rows(x.cuda(), y.cuda(), a1.cuda(), None, None, None, w.cuda(), 1e-5, torch.bfloat16,
                                                         (cw.cuda(), st), False, sm)
            v = x.double() + a1.double() * y.double()
            r = norm(v) * w.double()
            close(out, v, 24, float(v.abs().max()) + 30)
            close(nact, r, W / 2 + 16, float(r.abs().max()))
        want, live, new = conv(r, cw, state, lens, first, ctx, slots)
        big = float(r.abs().max())
        assert bool(live.all())
        close(h, want, W / 2 + 40, big * 8)
        close(st, new, W / 2 + 16, max(big, 5.0))


@pytest.mark.parametrize("W", [64, 1024, 1032, 2048, 2056, 3000, 4096])
@pytest.mark.parametrize("lens", [[1, 2, 3, 40], [257, 33], [2599]])
def test_the_bits_of_the_separate_launches(W, lens):
    """A row's sum is formed in one order, whichever launch forms it (rows of whole 16 bytes; others were summed entry by entry)."""
    g, n, T = torch.Generator().manual_seed(W + len(lens)), len(lens), sum(lens)
    sm, _ = meta(lens, [(0, 5)[i % 2] for i in range(n)], list(range(n)))
    x, w, a1, a2, cw = (torch.randn(*s, generator=g).cuda() for s in ((T, W), (W,), (W,), (W,), (W, 4)))
    y, z = (torch.randn(T, W, generator=g).bfloat16().cuda() for _ in range(2))
    state = torch.randn(n, 3, W, generator=g).cuda()

    def both(rows, separate):
        s1, s2, old = state.clone(), state.clone(), x.clone()
        got, want = rows(x, s1), separate(old, s2)
        want = (old, *(want if isinstance(want, tuple) else (want,)), s2)
        for a, b in zip((*got, s1), want):
            assert torch.equal(a, b)
    both(lambda v, s: sq.norm_conv_rows(v, y, w, 1e-5, 0.7, a1, (cw, s), sm, torch.bfloat16),
         lambda v, s: sq.norm_conv(v, y, w, 1e-5, 0.7, a1, (cw, s), sm, torch.bfloat16))
    both(lambda v, s: sq.residual_norm_conv_rows(v, y, a1, z, None, a2, w, 1e-5, torch.bfloat16, (cw, s), True, sm),
         lambda v, s: sq.residual_norm_conv(v, y, a1, z, None, a2, w, 1e-5, torch.bfloat16, (cw, s), True, sm))


def test_others_take_the_separate_kernels(monkeypatch):
    """More than 4096 columns, fp32 rows, a sum over experts, weights off 16 bytes: in place, by the launches they had."""
    calls = record_native(monkeypatch, sq)
    lens, ctx, slots, T = [3, 6], [0, 2], [1, 0], 9
    sm, _ = meta(lens, ctx, slots)

    def ones(*s):
        return torch.ones(*s, device="cuda")
    for W, dtype, off in ((4100, torch.bfloat16, 0), (64, torch.float32, 0), (64, torch.bfloat16, 1)):
        x, w = ones(T, W), ones(W + 4)[off:off + W]
        out, h = sq.norm_conv_rows(x, ones(T, W).to(dtype), w, 1e-5, 1.0, None, (ones(W, 4), ones(2, 3, W)), sm, dtype)
        assert out is x and h.dtype == dtype
    x = ones(T, 64)
    assert sq.residual_norm_conv_rows(x, ones(T, 64).bfloat16(), None, None, ones(T, 64), None, ones(64), 1e-5, torch.bfloat16,
                                      (ones(64, 4), ones(2, 3, 64)), False, sm)[0] is x
    assert "norm_conv" not in calls


@pytest.mark.parametrize("W,lens,one", [(4096, [65], False), (4096, [699], False), (4096, [700], True), (4096, [64], True), (2048, [65], True),
                                        (4096, [1] * 96, True), (2056, [1, 70], False)])
def test_wide_rows_of_some_hundred_tokens(W, lens, one, monkeypatch):
    """One branch: in two launches where one is the slower, with the same bits."""
    calls = record_native(monkeypatch, sq)
    g, n, T = torch.Generator().manual_seed(W), len(lens), sum(lens)
    sm, _ = meta(lens, [0] * n, list(range(n)))
    x, w, cw = (torch.randn(*s, generator=g).cuda() for s in ((T, W), (W,), (W, 4)))
    y, state = torch.randn(T, W, generator=g).bfloat16().cuda(), torch.zeros(n, 3, W, device="cuda")
    got = sq.norm_conv_rows(x.clone(), y, w, 1e-5, 0.7, None, (cw, state), sm, torch.bfloat16)
    assert ("norm_conv" in calls) == one
    monkeypatch.setattr(sq, "NORM_CONV_WIDE_MIN", 1 << 30 if one else 0)
    monkeypatch.setattr(sq, "_conv_rows", lambda *a: not one)
    again = sq.norm_conv_rows(x, y, w, 1e-5, 0.7, None, (cw, torch.zeros_like(state)), sm, torch.bfloat16)
    assert torch.equal(got[0], again[0]) and torch.equal(got[1], again[1])
