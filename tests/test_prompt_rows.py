"""Prompt attention over causal prompts, whose early and late rows share workgroups, against fp64 softmax attention.

Tolerance: scores of bf16 inputs with fp32 sums; weights rounded to bf16 (2^-9 each, independent), the sum of weighted values
relative to the largest value, the result rounded once (2^-8)."""
import pytest
import torch

from xgserve.ops import seqmix as sq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,G,dk,dv", [(4, 1, 64, 64), (2, 1, 64, 64), (3, 3, 64, 128), (8, 1, 128, 128)])
@pytest.mark.parametrize("lens,ctx", [([64], [0]), ([65, 96, 33], [0, 0, 0]), ([300, 1, 257], [0, 7, 40]), ([513], [100])])
@pytest.mark.parametrize("dist", [False, True])
def test_causal_prompts(H, G, dk, dv, lens, ctx, dist):
    g = torch.Generator().manual_seed(H + sum(lens))
    T, S, bs = sum(lens), len(lens), 16
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    q0 = [sum(lens[:i]) for i in range(S + 1)]
    total = [n + c for n, c in zip(lens, ctx)]
    pages = [-(-n // bs) for n in total]
    bt = torch.zeros(S, max(pages), dtype=torch.int32)
    at = 0
    for i, n in enumerate(pages):
        bt[i, :n] = torch.arange(at, at + n).flip(0)
        at += n
    tseq = sum([[i] * n for i, n in enumerate(lens)], [])
    pos = sum([list(range(c, c + n)) for n, c in zip(lens, ctx)], [])
    sm = sq.SeqMeta(S, max(lens), i32(q0), i32(total), i32(list(range(S))), bt.cuda(), i32(tseq), i32(pos), i32([0] * T))
    q, k, v = rnd(T, H * dk).bfloat16(), rnd(at * bs, G * dk).bfloat16(), rnd(at * bs, G * dv).bfloat16()
    r1, r2 = torch.rand(H, generator=g), torch.rand(H, generator=g)
    scale = dk ** -0.5
    kw = dict(dist=(r1.cuda(), r2.cuda())) if dist else {}
    got = sq.masked_attention(q.cuda(), k.cuda(), v.cuda(), H, G, dk, dv, sq.MASK_CAUSAL, 0, scale, None, None, bs, sm, **kw)
    for s in range(S):
        j = torch.arange(total[s])
        rows = bt[s][j // bs].long() * bs + j % bs
        kk, vv = k[rows].double().view(-1, G, dk), v[rows].double().view(-1, G, dv)
        for h in range(H):
            qh = q[q0[s]:q0[s + 1], h * dk:(h + 1) * dk].double()
            sc = qh @ kk[:, h // (H // G)].T * scale
            d = torch.arange(ctx[s], total[s])[:, None] - j[None]
            if dist:
                sc = sc - r1[h].double() * torch.log1p(r2[h].double() * d.clamp(min=0))
            p = torch.softmax(sc.masked_fill(d < 0, float("-inf")), -1)
            want = p @ vv[:, h // (H // G)]
            err = (got[q0[s]:q0[s + 1], h * dv:(h + 1) * dv].double().cpu() - want).abs()
            # independent roundings of the weights: at most 2^-9 of the root of their squares, 6 sigma
            bound = want.abs() * 2.0 ** -8 + 6 * 2.0 ** -9 * p.pow(2).sum(-1, keepdim=True).sqrt() * vv.abs().max() + 1e-5
            assert bool((err <= bound).all()), (s, h, float((err / bound).max()))


@pytest.mark.parametrize("dk,dv", [(64, 64), (128, 128)])
@pytest.mark.parametrize("mask,size", [(sq.MASK_CAUSAL, 0), (sq.MASK_WINDOW, 90), (sq.MASK_CHUNK, 100)])
@pytest.mark.parametrize("sink", [False, True])
def test_scales_of_any_sign_and_growing_scores(dk, dv, mask, size, sink):
    """Scales of either sign, 0 and large (some keys far above all before them, the reference catches up), with and without a sink, on
    pages of 48 keys. Same tolerance; a score errs by 2^-23 of its size and a weight by as much of itself."""
    g = torch.Generator().manual_seed(dk + size)
    H, n, bs = 4, 330, 48
    q, k, v = (torch.randn(n, H * d, generator=g).bfloat16() for d in (dk, dk, dv))
    k[::37] *= 8.0
    temp, sinks = torch.tensor([1.0, -1.3, 0.0, 25.0]), torch.randn(H, generator=g) * 2
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    sm = sq.SeqMeta(1, n, i32([0, n]), i32([n]), i32([0]), i32([list(range(-(-n // bs)))]), i32([0] * n), i32(list(range(n))), i32(list(range(n))))
    cache = [torch.cat([t, torch.zeros(-n % bs, t.shape[1])]).bfloat16().cuda() for t in (k, v)]
    got = sq.masked_attention(q.cuda(), *cache, H, H, dk, dv, mask, size, dk ** -0.5, temp.cuda(), sinks.cuda() if sink else None, bs, sm)
    i, j = torch.arange(n)[:, None], torch.arange(n)[None]
    seen = (j <= i) & (i - j < size if mask == sq.MASK_WINDOW else i // size == j // size if mask == sq.MASK_CHUNK else j <= i)
    for h in range(H):
        sc = (q[:, h * dk:(h + 1) * dk].double() @ k[:, h * dk:(h + 1) * dk].double().T * dk ** -0.5 * temp[h].double()).masked_fill(~seen, float("-inf"))
        full = torch.cat([sc, sinks[h].double().expand(n, 1)], 1) if sink else sc
        p = torch.softmax(full, -1)[:, :n]
        vv = v[:, h * dv:(h + 1) * dv].double()
        want = p @ vv
        err = (got[:, h * dv:(h + 1) * dv].double().cpu() - want).abs()
        big = sc.masked_fill(~seen, 0).abs().amax(-1, keepdim=True)
        bound = want.abs() * 2.0 ** -8 + (6 * 2.0 ** -9 * p.pow(2).sum(-1, keepdim=True).sqrt() + big * 2.0 ** -22) * vv.abs().max() + 1e-5
        assert bool((err <= bound).all()), (h, float((err / bound).max()))


@pytest.mark.parametrize("dk,dv", [(64, 64), (128, 128), (64, 128)])
@pytest.mark.parametrize("sink", [False, True])
def test_penalties_beside_scales_of_any_size(dk, dv, sink):
    """A penalty is taken in units of products, except where those would leave fp32: scales of either sign, 0, 1e-20 and 1e-36, penalties
    that come to nothing, small, so large that a row's own key is all it sees, and negative. Same tolerance."""
    g = torch.Generator().manual_seed(dk + dv)
    H, n, bs = 8, 330, 16
    q, k, v = (torch.randn(n, H * d, generator=g).bfloat16() for d in (dk, dk, dv))
    temp = torch.tensor([1.0, -1.3, 0.0, 1e-20, 1e-36, 4.0, -1e-25, 1.0])
    r1 = torch.tensor([0.7, 1.1, 0.4, 0.9, 0.6, 1e6, 1e12, -0.2])
    r2, sinks = torch.rand(H, generator=g) + 0.1, torch.randn(H, generator=g)
    r2[5] = 0.0   # (a large penalty of nothing)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    sm = sq.SeqMeta(1, n, i32([0, n]), i32([n]), i32([0]), i32([list(range(-(-n // bs)))]), i32([0] * n), i32(list(range(n))), i32(list(range(n))))
    cache = [torch.cat([t, torch.zeros(-n % bs, t.shape[1])]).bfloat16().cuda() for t in (k, v)]
    got = sq.masked_attention(q.cuda(), *cache, H, H, dk, dv, sq.MASK_CAUSAL, 0, dk ** -0.5, temp.cuda(), sinks.cuda() if sink else None, bs, sm,
                              dist=(r1.cuda(), r2.cuda()))
    d = (torch.arange(n)[:, None] - torch.arange(n)[None]).double()
    for h in range(H):
        sc = q[:, h * dk:(h + 1) * dk].double() @ k[:, h * dk:(h + 1) * dk].double().T * dk ** -0.5 * temp[h].double()
        pen = r1[h].double() * torch.log1p(r2[h].double() * d.clamp(min=0))
        sc = (sc - pen).masked_fill(d < 0, float("-inf"))
        full = torch.cat([sc, sinks[h].double().expand(n, 1)], 1) if sink else sc
        p = torch.softmax(full, -1)[:, :n]
        vv = v[:, h * dv:(h + 1) * dv].double()
        want = p @ vv
        err = (got[:, h * dv:(h + 1) * dv].double().cpu() - want).abs()
        # (a score errs by 2^-22 of its own and of the nearest keys' penalty)
        big = torch.where(p > 1e-12, pen.abs(), 0.0).amax(-1, keepdim=True) + sc.masked_fill(p < 1e-12, 0).abs().amax(-1, keepdim=True)
        bound = want.abs() * 2.0 ** -8 + (6 * 2.0 ** -9 * p.pow(2).sum(-1, keepdim=True).sqrt() + big * 2.0 ** -22) * vv.abs().max() + 1e-5
        assert bool((err <= bound).all()), (h, float((err / bound).max()))
