"""Latent attention of prompt portions over expanded keys and values (csrc/mixers/prompt_attention.hip, LAT) against fp64.

Tolerance: bf16 keeps 2^-9 of keys, values, rotated queries, weights and results. A score is a sum of dk products of unit
spread, so its error is about 2^-9 sqrt(2) in units of the score's own spread (1 here), a weight's the same relatively; with the
roundings of v and of the result the output is off by about 2.5 x 2^-9 = 0.005 of its root mean square: 0.015 is allowed, and
per entry ten times the spread of that."""
import pytest
import torch

from xgserve.ops import seqmix as sq

from _seq_util import record_native
from test_chunk_scan import layout

F64 = torch.float64
pytestmark = pytest.mark.gpu


def turn(v, pos, dims, base):
    f = base ** (-torch.arange(0, dims, 2, dtype=F64) / dims)
    a = pos.to(F64)[:, None, None] * f
    out = v.clone()
    out[..., 0:dims:2] = v[..., 0:dims:2] * a.cos() - v[..., 1:dims:2] * a.sin()
    out[..., 1:dims:2] = v[..., 1:dims:2] * a.cos() + v[..., 0:dims:2] * a.sin()
    return out


@pytest.mark.parametrize("H,dn,rd,dv,R,rot_dims", [(3, 64, 32, 64, 256, 32), (2, 128, 64, 128, 512, 64), (5, 80, 16, 64, 64, 8)])
@pytest.mark.parametrize("portions", [[(0, 64)], [(200, 130), (0, 300), (31, 1), (5, 33)], [(700, 257)], [(0, 1100), (60, 7)]], ids=str)
@pytest.mark.parametrize("window", [1, 17, 300, 5000])
def test_against_fp64(H, dn, rd, dv, R, rot_dims, portions, window, monkeypatch):
    g = torch.Generator().manual_seed(window + dn + len(portions))
    sm = layout(portions)
    T, bs = sum(n for _, n in portions), 16
    routed = []
    monkeypatch.setattr(sq, "_latent_key_rows", lambda *a, f=sq._latent_key_rows: routed.append(f(*a)) or routed[-1])
    rnd = lambda *s: torch.randn(*s, generator=g).bfloat16()  # noqa: E731
    q, gate = rnd(T, H, dn + rd), rnd(T, H)
    uk, uv = (torch.randn(H * dn, R, generator=g) * R ** -0.5).bfloat16(), (torch.randn(H * dv, R, generator=g) * R ** -0.5).bfloat16()
    cache = rnd((int(sm.block_tables.max()) + 1) * bs, R + rd)
    max_pos = int(sm.seq_lens.max())
    rot = sq.build_rot_table(rot_dims, 100.0, max_pos + 1).cuda()
    scale = (dn + rd) ** -0.5
    calls = record_native(monkeypatch, sq)
    got = sq.latent_attention_heads(q.cuda(), dn, gate.cuda(), cache.cuda(), uk.cuda(), uv.cuda(), rot, rot_dims, window, scale, bs, sm)
    # the expanded form, with every key row counted
    assert calls == ["latent_gather", "latent_prompt_attention"]
    assert routed and 32 * T >= routed[0] >= sum(n + min(c, window - 1) for c, n in portions)
    at, out = 0, []
    for i, (ctx, n) in enumerate(portions):
        p = torch.arange(ctx + n)
        rows = cache[sm.block_tables[i].cpu()[p // bs].long() * bs + p % bs].to(F64)
        k = torch.cat([(rows[:, :R] @ uk.to(F64).T).view(-1, H, dn), rows[:, None, R:].expand(-1, H, -1)], -1)
        v = (rows[:, :R] @ uv.to(F64).T).view(-1, H, dv)
        x = q[at:at + n].to(F64)
        x = torch.cat([x[..., :dn], turn(x[..., dn:], p[ctx:], rot_dims, 100.0)], -1)
        s = torch.einsum("thd,jhd->htj", x, k) * scale
        ago = p[ctx:, None] - p[None]
        s = s.masked_fill((ago < 0) | (ago >= window), -torch.inf)
        o = torch.einsum("htj,jhd->thd", torch.softmax(s, -1), v)
        out.append(o * torch.sigmoid(gate[at:at + n].to(F64))[..., None])
        at += n
    ref = torch.cat(out).reshape(T, H * dv)
    d, rms = got.cpu().to(F64) - ref, ref.pow(2).mean().sqrt()
    assert float(d.pow(2).mean().sqrt() / rms) < 0.015
    assert float((d.abs() / torch.maximum(rms, ref.abs())).max()) < 0.1
