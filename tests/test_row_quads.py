"""Row kernels that take four neighbouring values per thread (short convolutions, group norms, q / k norms), against fp64 and
on both sides of what they accept (sizes and alignments; the other inputs keep the general kernels).

Tolerance: fp32 arithmetic on exact inputs, a few roundings of 2^-24 per term and, for a norm, of its sum of n squares
(n 2^-24 relative, halved by the root); bf16 results are rounded once (2^-8)."""
import pytest
import torch

from xgserve.ops import seqmix as sq

pytestmark = pytest.mark.gpu


def meta(lens, ctx, slots, dev="cuda"):
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)  # noqa: E731
    q = [0]
    for n in lens:
        q.append(q[-1] + n)
    return sq.SeqMeta(len(lens), max(lens), i32(q), i32([n + c for n, c in zip(lens, ctx)]), i32(slots), i32([[0]] * len(lens)),
                      i32(sum([[i] * n for i, n in enumerate(lens)], [])), i32([0] * q[-1]), i32([0] * q[-1]))


def close(got, want, terms, scale):
    bits = 2.0 ** -8 if got.dtype == torch.bfloat16 else 0.0
    assert bool(((got.double().cpu() - want).abs() <= want.abs() * bits + terms * 2.0 ** -23 * scale).all())


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("W,taps,pad", [(4, 4, 0), (260, 4, 4), (1028, 3, 0), (12, 2, 8), (258, 4, 2), (64, 5, 0), (64, 4, 1)])
@pytest.mark.parametrize("lens,ctx", [([1, 1, 1], [0, 1, 40]), ([1, 2, 3, 9], [0, 0, 2, 1]), ([8, 17, 7, 40], [0, 5, 3, 0])])
def test_short_convolution(dt, W, taps, pad, lens, ctx):
    g = torch.Generator().manual_seed(W + taps)
    slots = list(range(len(lens)))[::-1]
    slots[1] = -1                                                       # a sequence without a slot: left alone
    sm, T, nh = meta(lens, ctx, slots), sum(lens), taps - 1
    x = torch.randn(T, W + pad, generator=g).to(dt)
    w, b = torch.randn(W, taps, generator=g), torch.randn(W, generator=g)
    state = torch.randn(len(lens), nh, W, generator=g)
    for residual, silu, bias in ((True, False, None), (False, True, b), (False, False, None)):
        st = state.clone().cuda()
        out = sq.causal_conv(x.cuda()[:, pad:], w.cuda(), None if bias is None else bias.cuda(), st, sm, dt, residual=residual,
                             silu=silu)
        at, want_st = 0, state.clone()
        for s, n in enumerate(lens):
            xs = x[at:at + n, pad:].double()
            if slots[s] >= 0:
                hist = state[slots[s]].double() * (torch.arange(-nh, 0)[:, None] + ctx[s] >= 0)
                ext = torch.cat([hist, xs])
                y = sum(w[:, j].double() * ext[j:j + n] for j in range(taps)) + (xs if residual else 0)
                y = y + (0 if bias is None else bias.double())
                y = y * torch.sigmoid(y) if silu else y
                close(out[at:at + n], y, taps + 8, 40.0)
                want_st[slots[s]] = ext[-nh:].float()
            at += n
        assert torch.equal(st.cpu(), want_st)


@pytest.mark.parametrize("n,groups,wn", [(64, 16, 4), (256, 4, 64), (512, 1, 512), (2048, 2, 2048), (4096, 8, 4096), (96, 2, 48),
                                         (4096, 1, 4096), (128, 2, 64)])
@pytest.mark.parametrize("T", [1, 5])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_group_norm(n, groups, wn, T, dt):
    g = torch.Generator().manual_seed(n)
    y, w = torch.randn(T, n, generator=g), torch.randn(wn, generator=g)
    for off in (0, 4, 1):
        z = torch.randn(T, n + 8, generator=g).to(dt)[:, off:off + n]
        for after in (False, True):
            for zz, ww in ((z, w), (None, w), (z, None)):
                got = sq.gated_group_norm(y.cuda(), None if zz is None else zz.cuda(), None if ww is None else ww.cuda(), 1e-5,
                                          groups, dt, gate_after=after)
                gate = 1.0 if zz is None else zz.double() * torch.sigmoid(zz.double())
                v = y.double() if after else y.double() * gate
                v = v.view(T, groups, -1)
                v = (v / (v.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt()).view(T, n)
                v = v * (1.0 if ww is None else ww.double().repeat(n // wn)) * (gate if after else 1.0)
                close(got, v, n // groups / 2 + 16, float(v.abs().max()))


@pytest.mark.parametrize("H,D", [(1, 4), (3, 32), (5, 64), (2, 256), (3, 12)])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_delta_out(H, D, dt):
    g = torch.Generator().manual_seed(D)
    o, w = torch.randn(7, H, D, generator=g), torch.randn(H * D, generator=g)
    gate = torch.randn(7, H * D + 8, generator=g).to(dt)[:, 4:4 + H * D]
    got = sq.delta_rule_out(o.cuda(), w.cuda(), gate.cuda(), 1e-5, H, D, dt)
    v = o.double() / (o.double().pow(2).mean(-1, keepdim=True) + 1e-5).sqrt()
    v = v.view(7, -1) * w.double() * torch.sigmoid(gate.double())
    close(got, v, D / 2 + 16, float(v.abs().max()))


@pytest.mark.parametrize("nq,nk,nv", [(4, 4, 4), (1024, 512, 1028), (2048, 512, 512), (4096, 1024, 1024), (4100, 4, 4), (6, 2, 2)])
@pytest.mark.parametrize("norm", [(True, True), (True, False), (False, False)])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_qk_norm(nq, nk, nv, norm, dt):
    g = torch.Generator().manual_seed(nq)
    T = 5
    proj = torch.randn(T, nq + nk + nv + 8, generator=g).to(dt)
    wq, wk = (torch.randn(n, generator=g) if on else None for n, on in zip((nq, nk), norm))
    sm = meta([T], [0], [0])
    sm.slot_mapping = torch.tensor([3, -1, 0, 6, 5], dtype=torch.int32, device="cuda")
    k0, v0 = torch.full((7, nk), 9.0, dtype=dt), torch.full((7, nv), 9.0, dtype=dt)
    k, v = k0.cuda(), v0.cuda()
    c = lambda t: None if t is None else t.cuda()  # noqa: E731
    q = sq.qk_norm_cache(proj.cuda(), nq, nk, nv, c(wq), c(wk), 1e-5, sm, k, v)
    p = proj.double()

    def normed(a, w):
        return a if w is None else a / (a.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt() * w.double()
    want_q, want_k = normed(p[:, :nq], wq), normed(p[:, nq:nq + nk], wk)
    close(q, want_q, nq / 2 + 8, float(want_q.abs().max()))
    wk_, wv_ = k0.double(), v0.double()
    for t, s in enumerate(sm.slot_mapping.tolist()):
        if s >= 0:
            wk_[s], wv_[s] = want_k[t], p[t, nq + nk:nq + nk + nv]
    close(k, wk_, nk / 2 + 8, 9.0)
    assert torch.equal(v.double().cpu(), wv_)


@pytest.mark.parametrize("dk,rot_dims,half", [(4, 4, False), (64, 32, False), (64, 32, True), (128, 128, True), (256, 64, False),
                                              (96, 32, False)])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_head_norm(dk, rot_dims, half, dt):
    g = torch.Generator().manual_seed(dk)
    T, H, G = 5, 3, 2
    src = torch.randn(T, (H + 2 * G) * dk, generator=g)
    wq, wk = torch.randn(dk, generator=g), torch.randn(dk, generator=g)
    ang = torch.rand(8, rot_dims // 2, generator=g) * 6
    rot = torch.stack([ang.cos(), ang.sin()], -1)
    sm = meta([T], [0], [0])
    sm.positions = torch.tensor([4, 5, 6, 7, 0], dtype=torch.int32, device="cuda")
    sm.slot_mapping = torch.tensor([3, -1, 0, 6, 5], dtype=torch.int32, device="cuda")
    k, v = (torch.zeros(7, G * dk, dtype=dt, device="cuda") for _ in range(2))
    q = sq.head_norm_rope_cache(src.cuda(), H, G, dk, dk, wq.cuda(), wk.cuda(), 1e-5, rot.cuda(), rot_dims, sm, k, v, dt,
                                half=half)

    def ref(x, w, n):
        x = x.double().view(T, n, dk)
        x = x / (x.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt() * w.double()
        r = rot[sm.positions.cpu().long()].double()[:, None]
        h = rot_dims // 2
        i = torch.arange(h) if half else 2 * torch.arange(h)
        j = i + h if half else i + 1
        y = x.clone()
        y[..., i] = x[..., i] * r[..., 0] - x[..., j] * r[..., 1]
        y[..., j] = x[..., j] * r[..., 0] + x[..., i] * r[..., 1]
        return y.reshape(T, n * dk)
    want = ref(src[:, :H * dk], wq, H)
    close(q, want, dk / 2 + 16, float(want.abs().max()))
    want = ref(src[:, H * dk:(H + G) * dk], wk, G)
    for t, s in enumerate(sm.slot_mapping.tolist()):
        if s >= 0:
            close(k[s], want[t], dk / 2 + 16, float(want.abs().max()))
            assert torch.equal(v[s].cpu(), src[t, (H + G) * dk:].to(dt))


@pytest.mark.parametrize("lo,hi", [(-0.5, 0.0), (-1.0, -0.5), (-2.0, -1.0), (-30.0, -2.0), (0.0, 6.0)])
@pytest.mark.parametrize("F", [4096, 30])
def test_xielu_keeps_fp32_accuracy(lo, hi, F):
    """fp32 in and out: e^z - 1 - z to three roundings of its size, the sum with z / 2 to one (both forms of the kernel)."""
    g = torch.Generator().manual_seed(1)
    sp, cn = torch.tensor(0.7), torch.tensor(1.2)
    z = torch.rand(512, F, generator=g) * (hi - lo) + lo
    got = sq.xielu(z.cuda(), None, float(sp), float(cn)).cpu().double()
    zd = z.double()
    part = torch.where(zd > 0, sp.double() * zd * zd, cn.double() * (torch.expm1(zd.clamp(max=0)) - zd))
    want = part + 0.5 * zd
    assert bool(((got - want).abs() <= 2.0 ** -24 * (3 * part + want.abs()) + 1e-30).all())


def test_xielu_of_extremes():
    z = torch.tensor([[float("inf"), float("-inf"), float("nan"), -3e38, -1e30, 1e30, 0.0, -0.0]])
    got = sq.xielu(z.cuda(), None, 0.7, 0.6).cpu()[0]
    assert got[0] == float("inf") and got[1].isnan() and got[2].isnan() and got[5] == float("inf") and not got[6:].any()
    torch.testing.assert_close(got[3:5].double(), 0.1 * -z[0, 3:5].double(), rtol=1e-5, atol=0)
