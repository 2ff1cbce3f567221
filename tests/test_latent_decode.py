"""Latent attention of single tokens in shares of the window, with the heads' value expansion, against fp64.

Tolerance: scores of bf16 inputs with fp32 sums (relative to the largest sum of magnitudes, R 2^-24), weights rounded to bf16
(2^-9), the merged sum rounded to bf16 (2^-9) before the expansion, the result rounded once more (2^-9): the first two move
every row by at most a share of the largest value, the expansion sums R of them as independent errors."""
import pytest
import torch

from xgserve.ops import seqmix as sq

from _seq_util import record_native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,dn,rd,dv,R,rot", [(32, 64, 32, 64, 256, 32), (3, 32, 32, 16, 64, 16), (40, 64, 64, 128, 512, 64),
                                              (16, 16, 64, 80, 128, 0)])
@pytest.mark.parametrize("lens,window,bs", [([1], 8, 16), ([64, 65, 1], 64, 16), ([300, 1, 129, 1000, 7], 512, 16),
                                            ([2100, 40], 4096, 1), ([700] * 9, 333, 32)])
def test_against_fp64(H, dn, rd, dv, R, rot, lens, window, bs, monkeypatch):
    g = torch.Generator().manual_seed(H + len(lens))
    T, dq = len(lens), dn + rd
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    pages = [-(-n // bs) for n in lens]
    order = torch.randperm(sum(pages) + 1, generator=g).to(torch.int32)
    bt, at = torch.zeros(T, max(pages), dtype=torch.int32), 0
    for i, n in enumerate(pages):
        bt[i, :n] = order[at:at + n]
        at += n
    slots = list(range(T))
    if T > 2:
        slots[1] = -1                                                       # a padding row
    sm = sq.SeqMeta(T, 1, i32(list(range(T + 1))), i32(lens), i32(slots), bt.cuda(), i32(list(range(T))),
                    i32([n - 1 for n in lens]), i32([0] * T))
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    cache = rnd((sum(pages) + 1) * bs, R + rd).bfloat16()
    q, gate = rnd(T, H, dq).bfloat16(), rnd(T, H + 8).bfloat16()[:, 8:]
    uk, uv = (rnd(H * dn, R) / R ** 0.5).bfloat16(), (rnd(H * dv, R) / R ** 0.5).bfloat16()
    table = sq.build_rot_table(rot, 1e4, max(lens) + 1, "cpu") if rot else torch.zeros(max(lens) + 1, 1, 2)
    scale = dq ** -0.5
    dev = [t.cuda() for t in (q, gate, cache, uk, uv, table)]
    assert sq._latent_shares(dev[0], dev[4], R, rd, dv, window, bs, sm) > 0
    calls = record_native(monkeypatch, sq)
    got = sq.latent_attention_heads(dev[0], dn, dev[1], dev[2], dev[3], dev[4], dev[5], rot, window, scale, bs, sm)
    assert calls == ["latent_decode"]
    # the queries in latent space as the step rounds them
    qabs = torch.bmm(dev[0][:, :, :dn].transpose(0, 1), dev[3].view(H, dn, R)).cpu().double()
    for t, n in enumerate(lens):
        if slots[t] < 0:
            assert not bool(got[t].any())
            continue
        j = torch.arange(max(0, n - window), n)
        rows = cache[bt[t][j // bs].long() * bs + j % bs].double()
        qr = q[t, :, dn:].double().clone()
        if rot:
            c, s = table[n - 1, :, 0].double(), table[n - 1, :, 1].double()
            a, b = qr[:, 0:rot:2].clone(), qr[:, 1:rot:2].clone()
            qr[:, 0:rot:2], qr[:, 1:rot:2] = a * c - b * s, b * c + a * s
        qr = qr.bfloat16().double()
        p = torch.softmax((qabs[:, t] @ rows[:, :R].T + qr @ rows[:, R:].T) * scale, -1)
        lat = (p @ rows[:, :R]) * torch.sigmoid(gate[t, :H].double())[:, None]
        want = torch.einsum("hr,hdr->hd", lat, uv.view(H, dv, R).double()).reshape(-1)
        mag = (p @ rows[:, :R].abs()).amax()       # what a weight's rounding is relative to
        err = (got[t].double().cpu() - want).abs()
        bound = want.abs() * 2.0 ** -8 + mag * (2.0 ** -9 * 2 + R * 2.0 ** -22) * uv.double().view(H, dv, R).norm(dim=-1).reshape(-1) * 4
        assert bool((err <= bound).all()), (t, float((err / bound).max()))


@pytest.mark.parametrize("T", [8, 9, 16, 17, 32, 33])
def test_tokens_to_a_workgroup(T, monkeypatch):
    """32 heads of 8, 16 and 32 tokens are where the value expansion takes one, two, four and eight tokens to a workgroup."""
    test_against_fp64(32, 64, 32, 64, 256, 32, [20 + 7 * i % 45 for i in range(T)], 64, 16, monkeypatch)


def test_other_steps_keep_the_general_kernels():
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    sm = sq.SeqMeta(2, 1, i32([0, 1, 2]), i32([5, 9]), i32([0, 1]), i32([[0], [1]]), i32([0, 1]), i32([4, 8]), i32([4, 24]))
    q, uv = torch.zeros(2, 4, 96, dtype=torch.bfloat16, device="cuda"), torch.zeros(4 * 64, 256, dtype=torch.bfloat16, device="cuda")
    assert sq._latent_shares(q, uv, 256, 32, 64, 64, 16, sm) == 1
    assert sq._latent_shares(q.float(), uv, 256, 32, 64, 64, 16, sm) == 0
    assert sq._latent_shares(q, uv, 240, 32, 64, 64, 16, sm) == 0 and sq._latent_shares(q, uv, 256, 24, 64, 64, 16, sm) == 0
    sm.block_tables = torch.zeros(2, 1 << 20, dtype=torch.int32, device="cuda")
    assert sq._latent_shares(q, uv, 256, 32, 64, 1 << 20, 1, sm) == 0       # a share's page table would not fit
    sm.max_q = 2
    assert sq._latent_shares(q, uv, 256, 32, 64, 64, 16, sm) == 0


def test_sequences_without_a_token():
    """A sequence that waits (no token in the step) between others, and a row behind the last token: rows follow the sequences."""
    g = torch.Generator().manual_seed(7)
    H, dn, rd, dv, R, bs, window = 4, 64, 32, 64, 256, 16, 64
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    lens, qsl, token_seq = [40, 9, 100, 23], [0, 1, 1, 2, 3], [0, 2, 3, -1]
    bt, at = torch.zeros(4, 7, dtype=torch.int32), 0
    for i, n in enumerate(lens):
        m = -(-n // bs)
        bt[i, :m] = torch.arange(at, at + m)
        at += m
    rnd = lambda *s: torch.randn(*s, generator=g).bfloat16().cuda()  # noqa: E731
    cache, q, gate = rnd(at * bs, R + rd), rnd(4, H, dn + rd), rnd(4, H)
    uk, uv = rnd(H * dn, R) / 16, rnd(H * dv, R) / 16
    rot = sq.build_rot_table(rd, 1e4, 101, "cpu").cuda()

    def attend(rows, seqs):
        """The same sequences, each with its token."""
        k = len(seqs)
        sm = sq.SeqMeta(k, 1, i32(list(range(k + 1))), i32([lens[s] for s in seqs]), i32(list(range(k))), bt[seqs].cuda(),
                        i32(list(range(k))), i32([lens[s] - 1 for s in seqs]), i32([0] * k))
        return sq.latent_attention_heads(q[rows].contiguous(), dn, gate[rows].contiguous(), cache, uk, uv, rot, rd, window, 0.1, bs, sm)
    want = attend([0, 1, 2], [0, 2, 3])
    sm = sq.SeqMeta(4, 1, i32(qsl), i32(lens), i32([0, 1, 2, 3]), bt.cuda(), i32(token_seq), i32([39, 99, 22, 0]), i32([0] * 4))
    assert sq._latent_shares(q, uv, R, rd, dv, window, bs, sm, cache) > 0
    got = sq.latent_attention_heads(q, dn, gate, cache, uk, uv, rot, rd, window, 0.1, bs, sm)
    assert torch.equal(got[:3], want) and not bool(got[3].any())


@pytest.mark.gpu
@pytest.mark.parametrize("dn,rd,R", [(32, 32, 64), (64, 32, 256), (128, 64, 512)])
@pytest.mark.parametrize("T", [1, 16, 17, 33, 64, 65, 130])
def test_queries_in_latent_space(dn, rd, R, T):
    """latent_query: q[t, h, :dn] . uk[h], fp32 sums of dn products (dn 2^-24 of their sizes) rounded once to bf16 (2^-8)."""
    from xgserve.ops._native import mixers, stream_ptr
    g, H = torch.Generator().manual_seed(T + R), 5
    q, uk = torch.randn(T, H, dn + rd, generator=g).bfloat16(), (torch.randn(H, dn, R, generator=g) / dn ** 0.5).bfloat16()
    qd, ud, out = q.cuda(), uk.cuda(), torch.full((H, T, R), 7.0, dtype=torch.bfloat16, device="cuda")
    mixers().latent_query(qd.data_ptr(), dn + rd, dn, ud.data_ptr(), out.data_ptr(), T, H, R, stream_ptr())
    a = q[:, :, :dn].double().transpose(0, 1)
    want, size = a @ uk.double(), a.abs() @ uk.double().abs()
    assert bool(((out.double().cpu() - want).abs() <= 2.0 ** -8 * want.abs() + dn * 2.0 ** -24 * size).all())
    for bad in ((dn, rd, R + 32), (dn + 8, rd, R)):
        with pytest.raises(ValueError):
            mixers().latent_query(qd.data_ptr(), sum(bad[:2]), bad[0], ud.data_ptr(), out.data_ptr(), T, H, bad[2], stream_ptr())


@pytest.mark.parametrize("fold", [True, False])
def test_queries_on_both_sides_of_the_line(fold, monkeypatch):
    """By latent_query up to LATENT_QUERY_MACS multiply-adds of a step's queries, by the library beyond."""
    T, H, dn, R = 9, 32, 64, 256
    monkeypatch.setattr(sq, "LATENT_QUERY_MACS", T * H * dn * R - (not fold))
    real, seen = sq.mixers(), []

    class Spy:
        def __getattr__(self, name):
            f = getattr(real, name)
            return lambda *a: (seen.append(a[-2] != 0) if name == "latent_decode" else None, f(*a))[1]
    monkeypatch.setattr(sq, "mixers", Spy)
    test_against_fp64(H, dn, 32, 64, R, 32, [20 + 7 * i for i in range(T)], 64, 16, monkeypatch)
    assert seen == [fold]


def test_large_steps_leave_the_queries_to_the_library():
    for T, H, dn, R, fold in ((64, 32, 64, 256, True), (64, 32, 128, 512, True), (128, 32, 128, 512, False), (256, 64, 64, 512, False)):
        assert (T * H * dn * R <= sq.LATENT_QUERY_MACS) == fold
