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
