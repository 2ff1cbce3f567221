"""Single tokens' key shares merged and mixed over heads in one launch (masked_attention with `talk`) against fp64."""
import pytest
import torch

from xgserve.ops import seqmix as sq

from _seq_util import record_native

F64 = torch.float64


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,dk,dv", [(16, 2, 64, 64), (16, 2, 128, 128), (6, 3, 32, 16), (64, 1, 64, 80)])
@pytest.mark.parametrize("gated", [False, True])
def test_merged_and_mixed(H, G, dk, dv, gated, monkeypatch):
    g = torch.Generator().manual_seed(H + dv)
    lens, bs = [1, 17, 64, 65, 700, 33], 16      # keys of each sequence with this step's; the last is no sequence of the step
    S, width = len(lens), (max(lens) + bs - 1) // bs
    tables = torch.arange(S * width, dtype=torch.int32).view(S, width)
    slots = torch.arange(S, dtype=torch.int32)
    slots[-1] = -1
    pos = torch.tensor([n - 1 for n in lens], dtype=torch.int32)
    sm = sq.SeqMeta(num_seqs=S, max_q=1, qsl=torch.arange(S + 1, dtype=torch.int32), seq_lens=pos + 1, slots=slots,
                    block_tables=tables, token_seq=torch.arange(S, dtype=torch.int32), positions=pos,
                    slot_mapping=torch.tensor([int(tables[s, (n - 1) // bs]) * bs + (n - 1) % bs for s, n in enumerate(lens)],
                                              dtype=torch.int32))
    for name in ("qsl", "seq_lens", "slots", "block_tables", "token_seq", "positions", "slot_mapping"):
        setattr(sm, name, getattr(sm, name).cuda())
    rnd = lambda *s: torch.randn(*s, generator=g).bfloat16()  # noqa: E731
    q, kc, vc, gate = rnd(S, H * dk), rnd(S * width * bs, G * dk), rnd(S * width * bs, G * dv), rnd(S, H)
    talk, r1, r2 = torch.eye(H) + 0.3 * torch.randn(H, H, generator=g), torch.rand(H, generator=g), torch.rand(H, generator=g) + 0.1
    calls = record_native(monkeypatch, sq)
    got = sq.masked_attention(q.cuda(), kc.cuda(), vc.cuda(), H, G, dk, dv, sq.MASK_CAUSAL, 0, dk ** -0.5, None, None, bs, sm,
                              dist=(r1.cuda(), r2.cuda()), values=sq.V_ALL,
                              talk=(talk.cuda(), gate.cuda() if gated else None)).cpu().to(F64)
    assert calls == ["masked_attention_mfma", "talk_mix_parts"]
    assert (got[-1] == 0).all()
    for s, n in enumerate(lens[:-1]):
        rows = tables[s, torch.arange(n) // bs].long() * bs + torch.arange(n) % bs
        k, v = kc[rows].to(F64).view(n, G, dk), vc[rows].to(F64).view(n, G, dv)
        sc = torch.einsum("hd,nhd->hn", q[s].to(F64).view(H, dk), k.repeat_interleave(H // G, 1)) * dk ** -0.5
        sc = sc - r1.to(F64)[:, None] * torch.log1p(r2.to(F64)[:, None] * (n - 1 - torch.arange(n)).to(F64))
        p = talk.to(F64) @ torch.softmax(sc, -1)
        o = torch.einsum("hn,nhd->hd", p, v.repeat_interleave(H // G, 1))
        if gated:
            o = o * torch.sigmoid(gate[s].to(F64))[:, None]
        # bf16 weights of the shares' products (2^-9 each, signs of talk and values at random) and a bf16 result: 0.01 of the
        # row's root mean square is five times what they give
        d = got[s].view(H, dv) - o
        assert float(d.pow(2).mean().sqrt() / o.pow(2).mean().sqrt()) < 0.01
