"""Row kernels of prompts in quads (latent projections, heads' maps mixed over many rows, group norms over every size of a lane
group), against fp64 and on both sides of what they accept.

Tolerance: fp32 arithmetic on exact inputs, a few roundings of 2^-24 per term and, for a norm, of its sum of n squares
(n 2^-24 relative, halved by the root); bf16 results are rounded once (2^-8)."""
import pytest
import torch

from xgserve.ops import seqmix as sq

pytestmark = pytest.mark.gpu


def close(got, want, terms, scale):
    bits = 2.0 ** -8 if got.dtype == torch.bfloat16 else 0.0
    assert bool(((got.double().cpu() - want).abs() <= want.abs() * bits + terms * 2.0 ** -23 * scale).all())


def normed(a, w):
    return a / (a.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt() * w.double()


@pytest.mark.parametrize("Rq,R,rd,rot_dims,off", [(768, 256, 32, 32, 0), (768, 260, 32, 16, 4), (1536, 512, 64, 64, 0), (4, 4, 4, 2, 0),
                                                  (2048, 2048, 64, 64, 8), (2048, 2052, 64, 64, 0), (768, 254, 32, 32, 0),
                                                  (768, 256, 32, 32, 2), (1000, 24, 36, 32, 0), (1000, 28, 36, 32, 0)])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_latent_rows(Rq, R, rd, rot_dims, off, dt):
    g, T, slots = torch.Generator().manual_seed(Rq + R), 5, [3, -1, 0, 6, 5]
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    one = i32([0])
    sm = sq.SeqMeta(1, T, i32([0, T]), i32([T]), one, one, one, i32([4, 0, 9, 2, 7]), i32(slots))
    proj = torch.randn(T, off + Rq + R + rd + 8, generator=g).to(dt)
    wq, wk = torch.randn(Rq, generator=g), torch.randn(R, generator=g)
    rot = sq.build_rot_table(rot_dims, 10000.0, 16, "cpu")
    p = proj.double()
    want = normed(p[:, off:off + Rq], wq)
    k, r = normed(p[:, off + Rq:off + Rq + R], wk), p[:, off + Rq + R:off + Rq + R + rd].clone()
    cs = rot.double().view(16, -1, 2)[sm.positions.long().cpu()]
    u, v = r[:, 0:rot_dims:2].clone(), r[:, 1:rot_dims:2].clone()
    r[:, 0:rot_dims:2], r[:, 1:rot_dims:2] = u * cs[..., 0] - v * cs[..., 1], v * cs[..., 0] + u * cs[..., 1]
    for own in (True, False):
        cache = torch.full((7, R + rd), 9.0, dtype=dt, device="cuda")
        cq = sq.latent_prep(proj.cuda(), off, Rq, off + Rq if own else -1, R, rd, wq.cuda(), wk.cuda() if own else None, 1e-5, rot.cuda(),
                            rot_dims, sm, cache)
        close(cq, want, Rq / 2 + 8, float(want.abs().max()))
        held = torch.full((7, R + rd), 9.0, dtype=torch.float64)
        for t, s in enumerate(slots):
            if own and s >= 0:
                held[s] = torch.cat([k[t], r[t]])
        close(cache, held, R / 2 + 8, 9.0)


@pytest.mark.parametrize("Rq,R", [(768, 256), (1536, 512), (1024, 512), (100, 12), (4, 4), (1028, 1020), (1000, 28), (2048, 2048), (512, 1536)])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_latent_rows_sum_in_one_order(Rq, R, dt):
    """Rows in quads and rows off their alignment, entry by entry, give the same bits."""
    g, T, rd = torch.Generator().manual_seed(Rq + R), 130, 32
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    one = i32([0])
    sm = sq.SeqMeta(1, T, i32([0, T]), i32([T]), one, one, one, i32([0] * T), i32(list(range(T))))
    row = torch.randn(T, Rq + R + rd, generator=g).to(dt)
    wq, wk, rot = torch.randn(Rq, generator=g).cuda(), torch.randn(R, generator=g).cuda(), sq.build_rot_table(rd, 1e4, 1, "cuda")

    def prep(off):
        proj = torch.zeros(T, Rq + R + rd + 4, dtype=dt)
        proj[:, off:off + row.shape[1]] = row
        cache = torch.zeros(T, R + rd, dtype=dt, device="cuda")
        return sq.latent_prep(proj.cuda(), off, Rq, off + Rq, R, rd, wq, wk, 1e-5, rot, rd, sm, cache), cache
    for got, want in zip(prep(0), prep(1)):
        assert torch.equal(got, want)


@pytest.mark.parametrize("H,G,dv", [(16, 2, 64), (16, 2, 128), (8, 4, 32), (8, 2, 4), (4, 4, 64), (6, 2, 64), (16, 2, 48), (8, 1, 1024)])
@pytest.mark.parametrize("T", [256, 257, 300])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_mixed_maps_of_many_rows(H, G, dv, T, dt):
    g = torch.Generator().manual_seed(H * dv)
    o, talk = torch.randn(T, H * G * dv, generator=g).to(dt), torch.randn(H, H, generator=g)
    gate = torch.randn(T, H + 3, generator=g).to(dt)
    wide = o.double().view(T, H, G, dv)[:, :, torch.arange(H) // (H // G)]
    want = (wide * talk.double().T[None, :, :, None]).sum(1)
    for gt in (gate, None):
        got = sq.talk_mix(o.cuda(), talk.cuda(), H, G, dv, gate=None if gt is None else gt.cuda())
        ref = want if gt is None else want * torch.sigmoid(gt[:, :H].double())[:, :, None]
        close(got, ref.reshape(T, -1), H + 12, 30.0)


@pytest.mark.parametrize("H,G,dv", [(16, 2, 64), (8, 4, 32), (8, 2, 4), (8, 1, 256), (4, 4, 64)])
@pytest.mark.parametrize("T", [1999, 2000, 2049])
def test_mixed_maps_of_few_reads(H, G, dv, T):
    """Up to 31 reads a thread the kernel of many rows begins at 2000; both give the same bits."""
    g = torch.Generator().manual_seed(H * dv)
    o, talk = torch.randn(T, H * G * dv, generator=g).bfloat16().cuda(), torch.randn(H, H, generator=g).cuda()
    gate = torch.randn(T, H, generator=g).bfloat16().cuda()
    few = torch.cat([sq.talk_mix(o[i:i + 1000], talk, H, G, dv, gate=gate[i:i + 1000]) for i in range(0, T, 1000)])
    assert torch.equal(sq.talk_mix(o, talk, H, G, dv, gate=gate), few)


@pytest.mark.parametrize("size", [4, 8, 16, 32, 64, 128, 256, 512, 1024])
@pytest.mark.parametrize("groups", [1, 3, 40])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_group_norms(size, groups, dt):
    g, T, n = torch.Generator().manual_seed(size), 3, size * groups
    y, z = torch.randn(T, n, generator=g), (3 * torch.randn(T, n, generator=g)).to(dt)
    for wn in {size, n}:
        w = torch.randn(wn, generator=g)
        got = sq.gated_group_norm(y.cuda(), z.cuda(), w.cuda(), 1e-5, groups, dt)
        v = (y.double() * z.double() * torch.sigmoid(z.double())).view(T, groups, -1)
        v = (v / (v.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt()).view(T, n) * w.double().repeat(n // wn)
        close(got, v, size / 2 + 16, float(v.abs().max()))


@pytest.mark.parametrize("H,D", [(1, 4), (1, 64), (3, 16), (5, 32), (15, 16), (1, 128), (2, 128), (2, 2), (63, 4), (64, 4)])
@pytest.mark.parametrize("T", [1, 5, 255, 257, 1000])
def test_rows_of_few_lanes(H, D, T):
    """Rows of less than a wave share workgroups: any number of them, the last workgroup's in part."""
    g, n = torch.Generator().manual_seed(H * D + T), H * D
    y, z, w = torch.randn(T, n, generator=g), torch.randn(T, n, generator=g).bfloat16(), torch.randn(n, generator=g)
    heads = y.double().view(T, H, D)
    v = (heads / (heads.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt()).view(T, n) * w.double()
    got = sq.delta_rule_out(y.cuda(), w.cuda(), z.cuda(), 1e-5, H, D, torch.bfloat16)
    close(got, v * torch.sigmoid(z.double()), D / 2 + 16, float(v.abs().max()))
    got = sq.gated_group_norm(y.cuda(), z.cuda(), w.cuda(), 1e-5, H, torch.bfloat16, gate_after=True)
    close(got, v * z.double() * torch.sigmoid(z.double()), D / 2 + 24, 4 * float(v.abs().max()))


def test_gates_behind_which_bf16_follows():
    """Their error against fp64 is that of the rounding: as with expf and a division, to 1 in 10^4."""
    x = torch.linspace(-12, 12, 1 << 16).bfloat16()
    o, w = torch.ones(1, x.numel()), torch.ones(x.numel())
    got = sq.delta_rule_out(o.cuda(), w.cuda(), x[None].cuda(), 0.0, x.numel() // 4, 4, torch.bfloat16).double().cpu()[0]
    want = torch.sigmoid(x.double())
    rounded = torch.sigmoid(x.double()).float().bfloat16().double()
    assert (got - want).norm() <= 1.0001 * (rounded - want).norm()


@pytest.mark.parametrize("T", [3, 300])
def test_bf16_results_are_those_of_fp32_rounded(T):
    """The same arithmetic in fp32 for either type of the rows, gates (spread 3) too: a bf16 result is the fp32 one, rounded once."""
    g = torch.Generator().manual_seed(T)

    def rows(n):
        return (3 * torch.randn(T, n, generator=g)).bfloat16().cuda()

    def weights(*s):
        return torch.randn(*s, generator=g).cuda()
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    one, n = i32(0), 2048
    sm = sq.SeqMeta(1, T, i32(0, T), i32(T), one, one, one, one, one)
    x, y, cw, cb = rows(n), weights(T, n), weights(n, 4), weights(n)
    o, talk, gate = rows(16 * 2 * 64), weights(16, 16), rows(16)

    def results(dt):
        state = torch.zeros(1, 3, n, device="cuda")
        yield sq.causal_conv(x, cw, cb, state, sm, dt, silu=True)
        yield sq.delta_rule_out(y, cb, x.to(dt), 1e-5, n // 64, 64, dt)
        yield sq.gated_group_norm(y, x.to(dt), cb, 1e-5, 8, dt)
        yield sq.gated_group_norm(y, x.to(dt), cb[:128], 1e-5, n // 128, dt, gate_after=True)
        yield sq.talk_mix(o.to(dt), talk, 16, 2, 64, gate=gate.to(dt))
    for got, want in zip(results(torch.bfloat16), results(torch.float32)):
        assert got.dtype == torch.bfloat16 and want.dtype == torch.float32
        assert torch.equal(got, want.bfloat16())
