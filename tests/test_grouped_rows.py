"""Sorted rows times their experts' weights (the grouped GEMM for few rows per expert) against fp64.

Tolerance: products of bf16 inputs are exact in fp32, a sum of K of them errs by at most K 2^-24 of the sum of magnitudes;
the gated and squared results are rounded once to bf16 (2^-8 of their size), with the activation's slope in front of the sum's
error."""
import pytest
import torch

from xgserve.ops import seqmix as sq
from xgserve.ops._native import mixers, stream_ptr

pytestmark = pytest.mark.gpu


def run(x, w, rows, tile_e, tm, top, N, K, mode, kind=0, limit=0.0, scale=None):
    out = torch.full((rows.numel(), N), -7.0, device="cuda", dtype=torch.float32 if mode == 0 else torch.bfloat16)
    mixers().grouped_gemm(x.data_ptr(), False, x.stride(0), w.data_ptr(), rows.data_ptr(), tile_e.data_ptr(), rows.numel(), tm,
                          top, N, K, mode, out.data_ptr(), kind, limit, 1.702, 0 if scale is None else scale.data_ptr(), True,
                          stream_ptr())
    return out


@pytest.mark.parametrize("tm", [16, 32, 64])
@pytest.mark.parametrize("N,K", [(16, 64), (80, 192), (208, 1024), (2064, 320)])
@pytest.mark.parametrize("T,E,top", [(1, 3, 2), (16, 4, 1), (33, 5, 2), (150, 2, 1)])
def test_modes(tm, N, K, T, E, top):
    g = torch.Generator().manual_seed(T + N)
    h = torch.randn(T, K + 8, generator=g).bfloat16().cuda()[:, :K]           # rows of a wider tensor
    ids = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(T)]).to(torch.int32).cuda()
    if E > 2:
        ids[ids == E - 1] = 0                                                 # an expert without rows
    pairs = T * top
    cap = (pairs + E * (tm - 1) + tm - 1) // tm * tm
    i32 = dict(dtype=torch.int32, device="cuda")
    rows, tile_e, dest = torch.empty(cap, **i32), torch.empty(cap // tm, **i32), torch.empty(pairs, **i32)
    words = torch.full((9,), 5, **i32)
    mixers().moe_align(ids.data_ptr(), pairs, E, cap, tm, rows.data_ptr(), tile_e.data_ptr(), dest.data_ptr(), 0,
                       words.data_ptr(), 8, stream_ptr())
    assert words.tolist() == [0] * 8 + [5]
    e, d = ids.flatten().long(), dest.long()
    free = torch.ones(cap, dtype=torch.bool, device="cuda")
    free[d] = False
    w13 = (torch.randn(E, 2 * N, K, generator=g) / K ** 0.5).bfloat16().cuda()
    src = h.double()[torch.arange(pairs, device="cuda") // top]
    z = torch.stack([w13[a].double() @ v for a, v in zip(e, src)])
    err = K * 2.0 ** -24 * float(torch.stack([w13[a].double().abs() @ v.abs() for a, v in zip(e, src)]).max()) + 2.0 ** -20
    top_z = float(z.abs().max())

    def check(out, want, slope, bits):
        assert bool((out[free] == -7).all())                                  # rows without a pair stay as they were
        assert bool(((out[d].double() - want).abs() <= slope * err + want.abs() * bits).all())

    a, u = z[:, :N], z[:, N:]
    check(run(h, w13, rows, tile_e, tm, top, N, K, 1, sq.GLU_SILU), a * torch.sigmoid(a) * u, 3 * top_z + 3, 2.0 ** -8)
    ac, uc = a.clamp(max=1.0), u.clamp(-1.0, 1.0)
    check(run(h, w13, rows, tile_e, tm, top, N, K, 1, sq.GLU_CLAMPED, 1.0), ac * torch.sigmoid(1.702 * ac) * (uc + 1),
          3 * top_z + 3, 2.0 ** -8)
    w1 = w13[:, :N].contiguous()
    s = (torch.rand(pairs, generator=g) + 0.5).cuda()
    check(run(h, w1, rows, tile_e, tm, top, N, K, 2, sq.ACT_RELU2, scale=s), (a * s.double()[:, None]).clamp(min=0) ** 2,
          6 * top_z + 3, 2.0 ** -8)
    lay = torch.full((cap, K), float("nan"), device="cuda", dtype=torch.bfloat16)   # padding rows may hold anything
    lay[d] = h[torch.arange(pairs, device="cuda") // top]
    check(run(lay, w1, rows, tile_e, tm, top, N, K, 0), a, 1.0, 2.0 ** -22)


@pytest.mark.parametrize("T", [8, 200])
def test_weights_in_front_of_a_gate_are_refused(T):
    """Whatever the rows per expert: no gated form multiplies the product by the row's weight."""
    h, w13 = torch.zeros(T, 128, device="cuda").bfloat16(), torch.zeros(2, 256, 128, device="cuda").bfloat16()
    w2, ids = torch.zeros(2, 256, 128, device="cuda").bfloat16(), torch.zeros(T, 1, device="cuda", dtype=torch.int32)
    with pytest.raises((ValueError, RuntimeError)):
        sq.routed_experts(h, w13, w2, ids, torch.full((T, 1), 0.5, device="cuda"), sq.GLU_SILU, scale_input=True)


@pytest.mark.parametrize("kind", [sq.GLU_GELU_TANH, sq.GLU_CLAMPED, sq.GLU_SILU])
@pytest.mark.parametrize("E,top,K,F_,W,form", [(4, 2, 256, 128, 256, "gemm_pf_grouped"), (5, 1, 512, 384, 512, "gemm_pf_grouped"),
                                               (66, 4, 128, 128, 256, "gemm_pf_grouped"),     # more experts than the tiles take
                                               (4, 2, 256, 192, 128, "grouped_gemm"), (66, 4, 128, 64, 96, "grouped_gemm")])
def test_gated_experts_that_the_tiles_do_not_take(kind, E, top, K, F_, W, form, monkeypatch):
    """Many rows per expert on gemm_pf's grouped form and on the 128-row tiles, against fp64."""
    from _seq_util import record_native
    if E <= 64:
        monkeypatch.setattr(sq, "GROUPED_EXPERTS_MAX", 0)
    T = -(-140 * E // top)
    g = torch.Generator("cuda").manual_seed(E + F_)
    h = torch.randn(T, K, generator=g, device="cuda").bfloat16()
    w13 = (torch.randn(E, 2 * F_, K, generator=g, device="cuda") * 2 * K ** -0.5).bfloat16()
    w2 = (torch.randn(E, W, F_, generator=g, device="cuda") * F_ ** -0.5).bfloat16()
    ids = torch.rand(T, E, generator=g, device="cuda").topk(top, -1).indices.to(torch.int32)
    wts = torch.rand(T, top, generator=g, device="cuda")
    calls = record_native(monkeypatch, sq)
    got = sq.routed_experts(h, w13, w2, ids, wts, kind, 2.0, 1.702).double()
    assert calls.count(form) == 2 and "tile_grouped" not in calls
    ref, size = torch.zeros_like(got), torch.zeros_like(got)
    for e in range(E):
        t, j = torch.nonzero(ids == e, as_tuple=True)
        z = h[t].double() @ w13[e].double().t()
        a = sq._glu_ref(z[:, :F_], z[:, F_:], kind, 2.0, 1.702)
        ref.index_add_(0, t, wts[t, j, None].double() * (a @ w2[e].double().t()))
        size.index_add_(0, t, wts[t, j, None].double() * (a.abs() @ w2[e].double().abs().t()))
    # activations in bf16 (2^-9 of each term), sums in fp32
    assert ((got - ref).abs() <= (2.0 ** -9 + F_ * 2.0 ** -23) * size + 1e-5).all(), float(((got - ref).abs() / size).max())
