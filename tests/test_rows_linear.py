"""Products of a few rows (ops.seqmix.linear, linear_xielu, linear_relu2, linear_glu) against fp64.

Tolerance: the products of bf16 inputs are exact in fp32 and their sums err by at most K 2^-24 of the sum of magnitudes
(any order), the activation follows in fp32, and the result is rounded once to bf16: 2^-8 of its size at most. The
activations' slopes over the inputs used here stay below the bound SLOPE that the tests put on them."""
import types

import pytest
import torch

from xgserve.ops import seqmix as sq

from _seq_util import record_native

gpu = pytest.mark.gpu
# rows on both sides of the tiles of 16; columns and K on both sides of a workgroup's share and of the parts of K
ROWS = (1, 16, 17, 33, 64)
SHAPES = ((4, 128), (60, 256), (68, 1024), (1088, 2048), (2052, 4096), (16392, 128))


def test_plans_stay_within_the_words_and_the_chunks():
    for N in list(range(4, 600, 4)) + [2048, 8192, 16384, 16388, 32000, 128256]:
        for K in (128, 256, 768, 1024, 2048, 4096, 8192, 14336, 28672):
            for gated in (False, True):
                wide, S = sq._rows_plan(N, K, gated)
                tiles = -(-N // (128 if wide else 64))
                assert S in (1, 2, 4, 8) and S <= K // 128 and (wide or not gated)
                assert S == 1 or tiles <= sq._ROWS_TICKETS


def test_other_inputs_keep_the_general_product():
    x, w = torch.randn(3, 128), torch.randn(8, 128)
    sm = types.SimpleNamespace(tickets=None)
    assert sq._rows_plan_of(x, w, sm, None, False) is None and sq.step_tickets(w, 3) is None
    torch.testing.assert_close(sq.linear(x, w, sm), x @ w.t())
    torch.testing.assert_close(sq.linear_relu2(x, w), sq.relu2(x @ w.t()))


def data(T, N, K, seed=0):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(T, K, generator=g).bfloat16().cuda()
    w = (torch.randn(N, K, generator=g) / K ** 0.5).bfloat16().cuda()
    sm = types.SimpleNamespace(tickets=torch.zeros(sq._ROWS_TICKETS, dtype=torch.int32, device="cuda"))
    return g, x, w, sm


def check(got, want, scale, K, slope):
    """scale: the largest sum of magnitudes of a product (what its sum's error is a part of)."""
    assert got.dtype == torch.bfloat16 and got.shape == want.shape
    err = (got.double() - want).abs()
    assert bool((err <= want.abs() * 2.0 ** -8 + slope * scale * (K * 2.0 ** -24 + 2.0 ** -21)).all()), err.max()


@gpu
@pytest.mark.parametrize("N,K", SHAPES)
@pytest.mark.parametrize("T", ROWS)
def test_products(T, N, K, monkeypatch):
    calls = record_native(monkeypatch, sq)
    g, x, w, sm = data(T, N, K)
    z, mag = x.double() @ w.double().t(), float((x.double().abs() @ w.double().abs().t()).max())
    assert sq._rows_plan_of(x, w, sm, None, False) is not None
    check(sq.linear(x, w, sm), z, mag, K, 1.0)
    b16 = torch.randn(N, generator=g).bfloat16().cuda()
    check(sq.linear(x, w, sm, b16), z + b16.double(), mag + 8, K, 1.0)
    b = torch.randn(N, generator=g).cuda()
    v = z + b.double()
    slope = 2 * float(v.abs().max()) + 2                   # of relu2, and of xielu with sp, cn <= 1
    check(sq.linear_relu2(x, w, b, sm), v.clamp(min=0) ** 2, mag + 8, K, slope)
    neg = 0.9 * (torch.expm1(v.clamp(max=0)) - v) + 0.5 * v
    check(sq.linear_xielu(x, w, b, 0.6, 0.9, sm), torch.where(v > 0, 0.6 * v * v + 0.5 * v, neg), mag + 8, K, slope)
    assert not bool(sm.tickets.any())                      # every launch leaves the words zero
    assert calls == ["rows_linear"] * 4
    # rows of a wider activation tensor
    wide = torch.full((T, K + 16), float("nan"), device="cuda", dtype=torch.bfloat16)
    wide[:, 8:8 + K] = x
    assert torch.equal(sq.linear(wide[:, 8:8 + K], w, sm), sq.linear(x, w, sm))


@gpu
@pytest.mark.parametrize("N,K", [(8, 128), (136, 1024), (2048, 2048), (16400, 256)])
@pytest.mark.parametrize("T", ROWS)
def test_gated_products(T, N, K, monkeypatch):
    calls = record_native(monkeypatch, sq)
    _, x, w, sm = data(T, N, K, 1)
    z, mag = x.double() @ w.double().t(), float((x.double().abs() @ w.double().abs().t()).max())
    a, u = z[:, :N // 2], z[:, N // 2:]
    slope = 3 * float(z.abs().max()) + 3
    assert sq._rows_plan_of(x, w, sm, None, True) is not None
    check(sq.linear_glu(x, w, sq.GLU_SILU, sm=sm), a * torch.sigmoid(a) * u, mag, K, slope)
    tanh = torch.tanh((2 / torch.pi) ** 0.5 * (a + 0.044715 * a ** 3))
    check(sq.linear_glu(x, w, sq.GLU_GELU_TANH, sm=sm), 0.5 * a * (1 + tanh) * u, mag, K, slope)
    ac, uc = a.clamp(max=2.0), u.clamp(-2.0, 2.0)
    check(sq.linear_glu(x, w, sq.GLU_CLAMPED, 2.0, 1.702, sm), ac * torch.sigmoid(1.702 * ac) * (uc + 1), mag, K, slope)
    assert calls == ["rows_linear"] * 3


@gpu
def test_nan_rows_stay_rows_and_unfit_rows_take_the_library():
    _, x, w, sm = data(17, 2048, 2048, 2)
    ref = sq.linear(x, w, sm)
    x[5, 7], x[9, 3] = float("nan"), float("inf")
    got = sq.linear_relu2(x, w, None, sm)
    bad = torch.zeros(17, dtype=torch.bool, device="cuda")
    bad[5] = bad[9] = True
    assert bool(got[5].isnan().all()) and bool((got[9].isinf() | (got[9] == 0)).all()) and bool(got[~bad].isfinite().all())
    assert torch.equal(sq.linear(x, w, sm)[~bad], ref[~bad])
    odd = torch.randn(3, 2049, device="cuda").bfloat16()[:, 1:]             # rows that are not 16-byte aligned
    assert sq._rows_plan_of(odd, w, sm, None, False) is None
    torch.testing.assert_close(sq.linear(odd, w, sm), odd @ w.t())
    assert sq._rows_plan_of(x, w, None, None, False) is None                # parts of K without words
    assert sq.linear(x[:0], w, sm).shape == (0, 2048)


@gpu
def test_embed_clears_the_words_and_replays_agree():
    """A captured step: words cleared by the embedding launch, then products in parts on them, replayed."""
    _, x, w, _ = data(17, 2048, 4096, 3)
    ids, table = torch.arange(17, dtype=torch.int32, device="cuda"), x.clone()
    sm = types.SimpleNamespace(tickets=None)

    def step():
        sm.tickets = sq.step_tickets(table, 17)
        h = sq.embed_rows(ids, table, tickets=sm.tickets).bfloat16()
        y = sq.linear(h, w, sm)
        return sq.linear(h, w, sm), y

    want = sq.linear(x, w, types.SimpleNamespace(tickets=torch.zeros(sq._ROWS_TICKETS, dtype=torch.int32, device="cuda")))
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        step()
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        a, b = step()
    for _ in range(5):
        a.zero_(), b.zero_(), sm.tickets.fill_(77)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(a, want) and torch.equal(b, want)
        torch.full((64, 1024), 3.0, device="cuda").sum().item()


@gpu
@pytest.mark.parametrize("T", [17, 64, 65, 200])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
def test_nan_through_the_squared_relu_whatever_the_rows(T, dtype):
    """As torch.relu keeps it: in the product's epilogue (up to 64 rows), in a launch of its own, and between expert products."""
    g = torch.Generator().manual_seed(T)
    x, w = torch.randn(T, 256, generator=g).to(dtype).cuda(), (torch.randn(128, 256, generator=g) / 16).to(dtype).cuda()
    x[5, 7] = float("nan")
    rows = torch.arange(T, device="cuda") != 5
    y = sq.linear_relu2(x, w, None, types.SimpleNamespace(tickets=None))
    assert bool(y[5].isnan().all()) and bool(y[rows].isfinite().all())
    z = sq.relu2(torch.randn(T, 30, generator=g).to(dtype).cuda().index_fill(0, torch.tensor([5], device="cuda"), float("nan")))
    assert bool(z[5].isnan().all()) and bool(z[rows].isfinite().all())
    for E, K in ((1, 256), (1, 96), (4, 256)):
        h = torch.randn(T, K, generator=g).to(dtype).cuda()
        h[5, 7] = float("nan")
        up, down = (torch.randn(E, *s, generator=g).to(dtype).cuda() / 16 for s in ((64, K), (K, 64)))
        ids = (torch.arange(T, device="cuda") % E).to(torch.int32)[:, None].contiguous()
        o = sq.routed_experts(h, up, down, ids, torch.ones(T, 1, device="cuda"), sq.ACT_RELU2)
        assert bool(o[5].isnan().all()) and bool(o[rows].isfinite().all()), (E, K)


def test_whole_tiles_fit_one_round_and_parts_stay_where_they_cost_less():
    for T in (1, 16, 17, 33, 49, 64):
        for N in [*range(8, 20000, 56), 32000, 128256]:
            for K in (128, 768, 2048, 4096, 8192, 14336):
                for gated in (False, True):
                    wide, S = sq._rows_plan(N, K, gated)
                    cols = sq._rows_cols(T, N, K, gated, wide, S)
                    assert cols == (128 if wide else 64) or (cols in ((32, 64) if gated else (16, 32, 48)) and -(-N // cols) <= 256)
    assert [sq._rows_cols(T, 2048, K, False, *sq._rows_plan(2048, K, False)) for T, K in ((64, 2048), (64, 8192), (1, 2048))] == \
        [16, 64, 16]


@pytest.mark.parametrize("T,N,K,cols", [(64, 3072, 5120, 64), (64, 4096, 5120, 64), (48, 2560, 6144, 64), (64, 8192, 8192, 64),
                                        (64, 12288, 512, 64), (64, 10272, 256, 64), (1, 10272, 128, 64), (16, 4096, 8192, 16), (17, 2048, 4096, 16),
                                        (64, 1088, 2048, 16), (48, 3072, 768, 16), (1, 6176, 4096, 32), (17, 6176, 4096, 32)])
def test_the_form_that_measured_faster(T, N, K, cols):
    """Sizes at which the forms differ by 5 to 36 %."""
    assert sq._rows_cols(T, N, K, False, *sq._rows_plan(N, K, False)) == cols


@gpu
@pytest.mark.parametrize("N,K,cols", [(4, 128, 16), (2052, 1152, 16), (4092, 640, 16), (4100, 256, 32), (8188, 640, 32), (8196, 128, 48),
                                      (12284, 384, 48), (8, 256, -32), (2056, 1152, -32), (8184, 128, -32), (8200, 640, -64),
                                      (16376, 128, -64)])
@pytest.mark.parametrize("T", [1, 16, 17, 32, 33, 48, 49, 64])
def test_whole_tiles(T, N, K, cols, monkeypatch):
    """Tiles of 16 to 64 weight rows over the whole K (cols < 0: gated): partial tiles, fewer chunks than the ring, more than it."""
    calls = record_native(monkeypatch, sq)
    monkeypatch.setattr(sq, "_rows_cols", lambda *a: abs(cols))   # (at these small sizes mostly not the faster form)
    g, x, w, sm = data(T, N, K, N + T)
    z, mag = x.double() @ w.double().t(), float((x.double().abs() @ w.double().abs().t()).max())
    assert sq._rows_plan_of(x, w, sm, None, cols < 0) == (abs(cols), 1)
    if cols < 0:
        a, u = z[:, :N // 2], z[:, N // 2:]
        check(sq.linear_glu(x, w, sq.GLU_SILU, sm=sm), a * torch.sigmoid(a) * u, mag, K, 3 * float(z.abs().max()) + 3)
    else:
        check(sq.linear(x, w, sm), z, mag, K, 1.0)
        b = torch.randn(N, generator=g).cuda()
        v = z + b.double()
        check(sq.linear_relu2(x, w, b, sm), v.clamp(min=0) ** 2, mag + 8, K, 2 * float(v.abs().max()) + 2)
    assert calls == ["rows_linear"] * (1 if cols < 0 else 2)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,native", [(1, 128256, 4096, True), (16, 32000, 4096, True), (17, 32000, 4096, False), (3, 32004, 2048, True),
                                          (2, 32002, 2048, False), (1, 512, 4096, False), (4, 32000, 2112, False)])
def test_heads_of_few_rows(M, N, K, native, monkeypatch):
    """lm_head_linear: up to 16 rows on rows_linear where it takes the sizes in one part, the library's product else."""
    from xgserve.ops.linear import lm_head_linear
    calls = record_native(monkeypatch, sq)
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = (torch.randn(N, K, generator=g, device="cuda") / K ** 0.5).bfloat16()
    got = lm_head_linear(x, w).double()
    want = x.double() @ w.double().T
    # one rounding to bf16, and fp32 sums of K products of size 1 / sqrt(K)
    assert bool(((got - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -22 * 5).all())
    assert ("rows_linear" in calls) == native
    assert lm_head_linear(x.float(), w.float()).dtype == torch.float32 if M <= 16 else True
    if M <= 16:
        xr = x.clone().requires_grad_()
        assert lm_head_linear(xr, w).grad_fn is not None


@pytest.mark.gpu
@pytest.mark.parametrize("N,K,native", [(32768, 1024, True), (32772, 1024, False), (50304, 1024, False), (32772, 1536, True)])
def test_wide_heads_of_short_rows_stay_with_the_library(N, K, native, monkeypatch):
    test_heads_of_few_rows(2, N, K, native, monkeypatch)
