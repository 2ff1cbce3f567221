"""Products of many rows (csrc/mixers/tile_linear.h): every tile at its edges, parts of K, what follows the product."""
import pytest
import torch
import torch.nn.functional as F

from xgserve.ops import seqmix as sq
from xgserve.ops import tile_linear as tl

from _seq_util import record_native


def test_plans_fit_the_kernel():
    for M in (65, 66, 127, 200, 401, 1000, 2601, 8192):
        for N, K in ((8, 64), (40, 4096), (1088, 2048), (2048, 8192), (28672, 4096), (4096, 14336)):
            fm, fn, S = tl.tile_plan(M, N, K)
            assert (fm, fn) in tl._TILES and 1 <= S <= K // 64
            assert S == 1 or -(-M // (32 * fm)) * -(-N // (32 * fn)) * S <= tl._SPLIT_TILES


def test_refused_products_stay_with_torch():
    x, w = torch.zeros(128, 64, dtype=torch.bfloat16), torch.zeros(256, 64, dtype=torch.bfloat16)
    assert tl.tile_plan_of(x, w) is None                     # not on the GPU
    assert torch.equal(sq.linear(x, w), F.linear(x, w))
    assert tl.library_better(4096, 4096, 4096)
    assert not tl.library_better(300, 4096, 14336) and not tl.library_better(4001, 10304, 2048)


def _close(y, ref, K):
    # one rounding to bf16 (2^-9 of the value) and fp32 sums of K products: K 2^-24 of the sum of the products' sizes (about
    # sqrt(K) times a result of unit variance) at most
    assert torch.isfinite(y.float()).all()
    err = (y.double() - ref).abs()
    assert (err <= 2.0 ** -8 * ref.abs() + K * 2.0 ** -24 * K ** 0.5 + 1e-6).all(), float(err.max())


@pytest.mark.gpu
@pytest.mark.parametrize("tile", sorted(tl._TILES))
@pytest.mark.parametrize("M,N,K,S", [(1, 8, 64, 1), (33, 264, 128, 1), (257, 520, 192, 3), (300, 1096, 320, 2), (513, 384, 640, 4)])
def test_tiles_at_their_edges(tile, M, N, K, S):
    g = torch.Generator("cuda").manual_seed(M + N)
    x = torch.randn(M, K + 8, generator=g, device="cuda").to(torch.bfloat16)[:, :K]     # rows with a stride of their own
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16)
    b = torch.randn(N, generator=g, device="cuda")
    ref = x.double() @ w.double().t()
    for parts in (1, S):
        plan = (*tile, parts)
        _close(tl.tile_linear(plan, x, w), ref, K)
        _close(tl.tile_linear(plan, x, w, b.to(torch.bfloat16)), ref + b.to(torch.bfloat16).double(), K)
        z = ref + b.double()
        # the square doubles the sum's relative error and takes its size
        y = tl.tile_linear(plan, x, w, b, sq.ACT_RELU2).double()
        assert ((y - z.clamp(min=0) ** 2).abs() <= 2.0 ** -8 * z ** 2 + 2 * z.abs() * K ** 1.5 * 2.0 ** -24 + 1e-6).all()
        y = tl.tile_linear(plan, x, w, b, sq.ACT_XIELU, 0.7, 0.9).double()
        r = torch.where(z > 0, 0.7 * z * z, 0.9 * (torch.expm1(z.clamp(max=0)) - z)) + 0.5 * z
        # (its slope is at most 1.4 z + 0.5 above zero and 1.4 below)
        assert ((y - r).abs() <= 2.0 ** -8 * r.abs() + (1.4 * z.abs() + 1.4) * (K ** 1.5 * 2.0 ** -24 + 2.0 ** -22) + 1e-6).all()


@pytest.mark.gpu
@pytest.mark.parametrize("tile", sorted(tl._TILES))
@pytest.mark.parametrize("M,F_,K,S", [(1, 8, 64, 1), (70, 132, 128, 2), (270, 528, 192, 3)])
@pytest.mark.parametrize("kind", [sq.GLU_GELU_TANH, sq.GLU_CLAMPED, sq.GLU_SILU])
def test_gated_tiles(tile, M, F_, K, S, kind):
    g = torch.Generator("cuda").manual_seed(M + F_)
    x = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn(2 * F_, K, generator=g, device="cuda") * 3 * K ** -0.5).to(torch.bfloat16)
    z = x.double() @ w.double().t()
    ref = sq._glu_ref(z[:, :F_], z[:, F_:], kind, 2.0, 1.702)
    forms = [(w, tl.PAIR_HALVES)]
    if F_ % 16 == 0:
        forms.append((torch.stack([w[:F_].view(-1, 16, K), w[F_:].view(-1, 16, K)], 1).reshape(2 * F_, K), tl.PAIR_BLOCKS))
    for ww, pairs in forms:
        for parts in (1, S):
            y = tl.tile_linear((*tile, parts), x, ww, None, sq.ACT_GLU + kind, 2.0, 1.702, pairs).double()
            # slopes of the gate up to 1.2 and of the other factor 1, each times the other side
            room = (1.5 * z[:, F_:].abs() + 1.5 * z[:, :F_].abs() + 2) * (3 * K ** 1.5 * 2.0 ** -24 + 2.0 ** -22)
            assert ((y - ref).abs() <= 2.0 ** -8 * ref.abs() + room).all()


@pytest.mark.gpu
@pytest.mark.parametrize("tile", sorted(tl._TILES))
@pytest.mark.parametrize("K,S", [(192, 1), (256, 1), (320, 1), (384, 1), (448, 1), (704, 2), (1216, 3)])   # K of every ring's length and one more
def test_tiles_one_after_another(tile, K, S, monkeypatch):
    """Workgroups that go through many tiles of the result, rows and columns left over, give the bits that one per tile gives."""
    M, N = 64 * tile[0] + 41, 96 * tile[1] + 24
    g = torch.Generator("cuda").manual_seed(K)
    x = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16)
    b = torch.randn(N, generator=g, device="cuda")

    def results():
        out = [tl.tile_linear((*tile, S), x, w, b), tl.tile_linear((*tile, S), x, w, b.to(torch.bfloat16), sq.ACT_RELU2),
               tl.tile_linear((*tile, S), x, w, b, sq.ACT_XIELU, 0.7, 0.9), tl.tile_linear((*tile, S), x, w)]
        out += [tl.tile_linear((*tile, S), x, w, None, sq.ACT_GLU + k, 2.0, 1.702, tl.PAIR_HALVES)
                for k in (sq.GLU_GELU_TANH, sq.GLU_CLAMPED, sq.GLU_SILU)]
        return out + ([tl.tile_parts((*tile, S), x, w).part] if S > 1 else [])
    got = {}
    for cus in (1, 3, 1 << 20):
        monkeypatch.setattr(tl, "cu_count", lambda d, n=cus: n)
        got[cus] = results()
    for few, three, own in zip(got[1], got[3], got[1 << 20]):
        assert torch.equal(few, own) and torch.equal(three, own)
    _close(got[1][3], x.double() @ w.double().t(), K)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", sorted(tl._TILES))
@pytest.mark.parametrize("tiles,S", [(2, 1), (3, 1), (4, 2), (8, 1), (9, 1)])
def test_equal_rows_give_equal_bits(tile, tiles, S):
    """Wherever they are in the step: two to nine tiles of rows, weights beyond 24 MB, K tiles that begin at another place (up to 256 rows)."""
    M, N, K = 32 * tile[0] * tiles - 13, 1544, 8192 + 192
    g = torch.Generator("cuda").manual_seed(M)
    few = torch.randn(7, K, generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16)
    at = torch.arange(M, device="cuda") % 7
    y = tl.tile_linear((*tile, S), few[at], w)
    assert torch.equal(y, y[:7][at])
    _close(y[-7:], few[at[-7:]].double() @ w.double().t(), K)
    glu = tl.tile_linear((*tile, S), few[at], w, None, sq.ACT_GLU + sq.GLU_SILU, 0.0, 1.702, tl.PAIR_HALVES)
    assert torch.equal(glu, glu[:7][at])


@pytest.mark.gpu
@pytest.mark.parametrize("K", [64, 128, 192, 256, 320, 384, 448, 1024])
def test_sizes_of_tiles_sum_in_the_same_order(K):
    """More than 256 rows: every size of the tile gives the same bits, K of a few tiles (forms without a ring) and longer."""
    g = torch.Generator("cuda").manual_seed(K)
    x = torch.randn(300, K, generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn(1544, K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16)
    got = [tl.tile_linear((*tile, 1), x, w) for tile in sorted(tl._TILES)]
    assert all(torch.equal(y, got[0]) for y in got)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", sorted(tl._TILES))
@pytest.mark.parametrize("K", [64, 128, 192, 256, 320, 384, 448])
@pytest.mark.parametrize("S", [1, 2, 3])
def test_columns_begin_where_their_size_says(tile, K, S):
    """Up to 256 rows column tile n of the size that was asked for takes a part's K tiles from number 37 n on and around, whatever size
    runs in its place: the bits are those of more rows (which begin at the first) with x's and w's K tiles in that order."""
    nk, width, N = K // 64, 32 * tile[1], 1544
    if S > nk:
        pytest.skip("fewer K tiles than parts")
    g = torch.Generator("cuda").manual_seed(K + S)
    x = torch.randn(300, K, generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16)
    got = tl.tile_linear((*tile, S), x[:200], w)
    for n in range(-(-N // width)):
        order = []
        for s in range(S):
            lo, k = s * nk // S, (s + 1) * nk // S - s * nk // S
            order += [64 * (lo + (37 * n + i) % k) + e for i in range(k) for e in range(64)]
        cols = slice(width * n, min(width * (n + 1), N))
        want = tl.tile_linear((4, 4, S), x[:, order].contiguous(), w[cols, order].contiguous())
        assert torch.equal(got[:, cols], want[:200])


def test_results_of_2_31_bytes_a_wave_are_refused():
    from xgserve.ops._native import mixers
    with pytest.raises(ValueError):
        mixers().tile_linear(64, 64, 64, 0, False, 0, 64, 65, 1 << 22, 64, 1, 0, 0, 0.0, 0.0, 4, 4, 256, 0)


@pytest.mark.gpu
def test_prompt_products_take_the_tiles():
    x = torch.randn(300, 2048, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(10304, 2048, device="cuda", dtype=torch.bfloat16) * 2048 ** -0.5
    assert tl.tile_plan_of(x, w, plain=True) is not None and tl.tile_plan_of(x[:64], w) is None
    assert tl.tile_plan_of(x, torch.nn.Parameter(w)) is None            # a derivative is torch's
    with torch.no_grad():
        assert tl.tile_plan_of(x, torch.nn.Parameter(w)) is not None
    assert tl.tile_plan_of(x.t().contiguous().t(), w) is None and tl.tile_plan_of(x[:, 1:], w[:, 1:]) is None
    _close(sq.linear(x, w), x.double() @ w.double().t(), 2048)


def test_grouped_plans_are_the_kernels():
    for pairs, E, N, K in ((56, 1, 8, 64), (450, 8, 7168, 4096), (16384, 8, 4096, 3584), (100000, 64, 2048, 1024)):
        assert tl.grouped_plan(pairs, E, N, K) in tl._GROUPED


@pytest.mark.gpu
@pytest.mark.parametrize("tile", tl._GROUPED)
@pytest.mark.parametrize("kind", [sq.GLU_GELU_TANH, sq.GLU_CLAMPED, sq.GLU_SILU])
def test_grouped_tiles(tile, kind, monkeypatch):
    """Shares of every size: no row, one, a tile's worth and one more, several tiles; columns left over."""
    K, F_, W, top = 128, 192, 136, 2
    share = [0, 1, 32 * tile[0], 32 * tile[0] + 1, 7, 0, 2 * 32 * tile[0] - 5, 500]
    E, g = len(share), torch.Generator().manual_seed(tile[0])
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(share))
    if ids.numel() % 2:
        ids = torch.cat([ids, ids[-1:]])
    ids = ids[torch.randperm(ids.numel(), generator=g)].view(-1, top).to(torch.int32)
    T = ids.shape[0]
    h = torch.randn(T, K, generator=g).to(torch.bfloat16)
    w13 = (torch.randn(E, 2 * F_, K, generator=g) * 3 * K ** -0.5).to(torch.bfloat16)
    w2 = (torch.randn(E, W, F_, generator=g) * F_ ** -0.5).to(torch.bfloat16)
    wts = torch.rand(T, top, generator=g)
    monkeypatch.setattr(sq, "grouped_plan", lambda *a: tile)
    calls = record_native(monkeypatch, sq)
    got = sq.routed_experts(h.cuda(), w13.cuda(), w2.cuda(), ids.cuda(), wts.cuda(), kind, 2.0, 1.702).cpu().double()
    assert calls.count("tile_grouped") == 2
    ref = torch.zeros(T, W, dtype=torch.float64)
    size = torch.zeros(T, W, dtype=torch.float64)
    for e in range(E):
        t, j = torch.nonzero(ids == e, as_tuple=True)
        z = h[t].double() @ w13[e].double().t()
        a = sq._glu_ref(z[:, :F_], z[:, F_:], kind, 2.0, 1.702)
        ref.index_add_(0, t, wts[t, j, None].double() * (a @ w2[e].double().t()))
        size.index_add_(0, t, wts[t, j, None].double() * (a.abs() @ w2[e].double().abs().t()))
    # the activations are rounded to bf16 (2^-9 of each term of the second product), the sums are fp32
    assert ((got - ref).abs() <= (2.0 ** -9 + F_ * 2.0 ** -23) * size + 1e-5).all(), float(((got - ref).abs() / size).max())


@pytest.mark.gpu
@pytest.mark.parametrize("tile", tl._GROUPED)
def test_grouped_tiles_one_after_another(tile, monkeypatch):
    """Workgroups that go through the tiles of several experts give the bits that one per tile gives."""
    K, F_, W, top, E = 448, 576, 136, 2, 6
    g = torch.Generator("cuda").manual_seed(tile[1])
    T = 64 * tile[0] + 77
    ids = torch.stack([torch.randperm(E, generator=g, device="cuda")[:top] for _ in range(T)]).to(torch.int32)
    h = torch.randn(T, K, generator=g, device="cuda").to(torch.bfloat16)
    w13 = (torch.randn(E, 2 * F_, K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16)
    w2 = (torch.randn(E, W, F_, generator=g, device="cuda") * F_ ** -0.5).to(torch.bfloat16)
    wts = torch.rand(T, top, generator=g, device="cuda")
    monkeypatch.setattr(sq, "grouped_plan", lambda *a: tile)
    monkeypatch.setattr(sq, "_experts_on_tiles", lambda *a: True)
    got = []
    for cus in (1, 5, 1 << 20):
        monkeypatch.setattr(sq, "cu_count", lambda d, n=cus: n)
        got.append(sq.routed_experts(h, w13, w2, ids, wts, sq.GLU_SILU))
    assert torch.equal(got[0], got[2]) and torch.equal(got[1], got[2])


@pytest.mark.gpu
@pytest.mark.parametrize("F_,K,T,tiled", [(4096, 2048, 179, False), (4096, 2048, 180, True),      # 45 rows an expert: 16 M weights each
                                          (256, 128, 383, False), (256, 128, 384, True)])         # 96: smaller experts
def test_which_experts_take_the_tiles(F_, K, T, tiled, monkeypatch):
    E, W, top = 8, 256, 2
    g = torch.Generator("cuda").manual_seed(T)
    h = torch.randn(T, K, generator=g, device="cuda").to(torch.bfloat16)
    w13 = (torch.randn(E, 2 * F_, K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16)
    w2 = (torch.randn(E, W, F_, generator=g, device="cuda") * F_ ** -0.5).to(torch.bfloat16)
    ids = (torch.arange(T * top, device="cuda", dtype=torch.int32) % E).view(T, top)
    wts = torch.rand(T, top, generator=g, device="cuda")
    calls = record_native(monkeypatch, sq)
    got = sq.routed_experts(h, w13, w2, ids, wts, sq.GLU_SILU).double()
    assert calls.count("tile_grouped") == (2 if tiled else 0)
    ref, size = torch.zeros(T, W, dtype=torch.float64, device="cuda"), torch.zeros(T, W, dtype=torch.float64, device="cuda")
    for e in range(E):
        t, j = torch.nonzero(ids == e, as_tuple=True)
        z = h[t].double() @ w13[e].double().t()
        a = sq._glu_ref(z[:, :F_], z[:, F_:], sq.GLU_SILU, 0.0, 0.0)
        ref.index_add_(0, t, wts[t, j, None].double() * (a @ w2[e].double().t()))
        size.index_add_(0, t, wts[t, j, None].double() * (a.abs() @ w2[e].double().abs().t()))
    # activations in bf16 (2^-9 of each term), sums in fp32
    assert ((got - ref).abs() <= (2.0 ** -9 + F_ * 2.0 ** -23) * size + 1e-5).all(), float(((got - ref).abs() / size).max())


@pytest.mark.parametrize("rows", [8, 128])
@pytest.mark.parametrize("kind", [-1, 2, 4])
def test_unknown_gates_go_to_the_activation_that_refuses_them(rows, kind, monkeypatch):
    seen = []
    monkeypatch.setattr(sq, "_rows_plan_of", lambda *a, **k: (True, 1))
    monkeypatch.setattr(sq, "tile_plan_of", lambda *a, **k: (3, 2, 1))
    monkeypatch.setattr(sq, "_rows_linear", lambda *a: seen.append("rows"))
    monkeypatch.setattr(sq, "tile_linear", lambda *a: seen.append("tiles"))
    monkeypatch.setattr(sq, "glu_act", lambda z, k, *a: seen.append(k))
    sq.linear_glu(torch.zeros(rows, 128), torch.zeros(256, 128), kind)
    assert seen == [kind]


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [8, 128])
@pytest.mark.parametrize("kind", [-1, 2, 4])
def test_unknown_gates_are_refused(rows, kind):
    x, w = torch.zeros(rows, 128, device="cuda", dtype=torch.bfloat16), torch.zeros(256, 128, device="cuda", dtype=torch.bfloat16)
    with pytest.raises(ValueError):
        sq.linear_glu(x, w, kind)


@pytest.mark.parametrize("rows", [8, 128])
def test_products_on_another_device_stay_with_torch(rows, monkeypatch):
    """Launches go to the current device's stream; torch's products run where their tensors are."""
    x, w = torch.zeros(rows, 256, dtype=torch.bfloat16), torch.zeros(64, 256, dtype=torch.bfloat16)
    for m in (sq, tl):
        monkeypatch.setattr(m, "native_device", lambda t: True)
    monkeypatch.setattr(tl, "cu_count", lambda d: 256)
    plan = (lambda: sq._rows_plan_of(x, w, None, None, False)) if rows <= 64 else (lambda: tl.tile_plan_of(x, w))
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: 1, raising=False)
    monkeypatch.setattr(torch.Tensor, "get_device", lambda t: 1)
    assert plan() is not None
    monkeypatch.setattr(torch.Tensor, "get_device", lambda t: 0)
    assert plan() is None


class _Seen(torch.overrides.TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def test_modes_that_choose_or_see_a_product_keep_it_with_torch():
    x, w = torch.zeros(128, 64, dtype=torch.bfloat16), torch.zeros(256, 64, dtype=torch.bfloat16)
    assert tl.forward_only(x, w, None)
    with torch.autocast("cpu", dtype=torch.float16):
        assert not tl.forward_only(x, w, None)
        with torch.autocast("cpu", enabled=False):
            assert tl.forward_only(x, w, None)
    with _Seen():
        assert not tl.forward_only(x, w, None)
    with torch.device("cpu"):
        assert tl.forward_only(x, w, None)
        with _Seen():
            assert not tl.forward_only(x, w, None)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [8, 128])
def test_autocast_chooses_the_type(rows):
    x, w = torch.ones(rows, 128, device="cuda", dtype=torch.bfloat16), torch.ones(256, 128, device="cuda", dtype=torch.bfloat16)
    with torch.autocast("cuda", dtype=torch.float16):
        y = sq.linear(x, w)
    assert y.dtype == torch.float16 and bool((y == 128).all())
    assert sq.linear(x, w).dtype == torch.bfloat16


def test_grouped_sizes_end_where_the_kernel_refuses():
    """Activations of 2^31 elements in the sorted layout (one expert: up to 30 rows more than there are pairs) are past a lane's
    offset: pairs just below stay on the streamed products."""
    F_ = 2048
    for pairs in range((1 << 20) - 40, (1 << 20) + 2):
        cap = sq._sorted_rows(pairs, 1, 16)
        assert sq._experts_on_tiles(pairs, 1, 64, F_, 64, pairs) == (cap * F_ < 1 << 31)
    assert not sq._experts_on_tiles((1 << 20) - 17, 1, 64, F_, 64, (1 << 20) - 17)   # 2^20 rows


def test_llama_products_run_in_torch_where_the_kernels_are_missing(monkeypatch):
    """XGS_ALLOW_TORCH_FALLBACK=1 without a built library: no plan is asked for, torch's products run."""
    from xgserve.models import llama
    monkeypatch.setattr(llama, "use_native", lambda t: False, raising=False)
    monkeypatch.setattr(llama, "tile_plan_of", lambda *a, **k: pytest.fail("a plan without kernels"))
    x, w = torch.randn(128, 64).bfloat16(), torch.randn(256, 64).bfloat16()
    assert torch.equal(llama._product(x, w, parts=True), F.linear(x, w))
    assert llama._silu_gate(x, w).shape == (128, 128)


def _priced(M, N, K, cus):
    """The cheapest tile and parts of K by the prices, counted out plainly (the first of equals)."""
    out = []
    for (fm, fn), (kt, per) in tl._TILES.items():
        rows = -(-M // (32 * fm))
        tiles = rows * -(-N // (32 * fn))
        if 32 * fm >= 2 * M + 64:
            continue
        kt = max(kt, tl._X_READ * fm + tl._W_READ * fn / rows ** 0.25 + (tl._SMALL if (fm, fn) == (3, 2) else 0))
        for S in tl._SPLITS:
            if S > 1 and (K // S < tl._SPLIT_K or tiles * S > tl._SPLIT_TILES):
                continue
            last = tl._SUM + tl._PART * S + 4 * M * N * S / tl._PART_BYTES if S > 1 else 2 * M * N / tl._OUT_BYTES
            out.append((-(-tiles * S // cus) * (-(-(K // 64) // S) * kt + per) + last, fm, fn, S))
    return min(out, key=lambda c: c[0])[1:]


def test_the_native_search_finds_the_cheapest_plan():
    for M in (65, 96, 97, 400, 401, 1000, 2600, 2601, 8191):
        for N, K in ((8, 64), (1088, 2048), (4096, 14336), (18560, 4096)):
            for cus in (8, 256):
                assert tl.tile_plan(M, N, K, cus) == _priced(M, N, K, cus)
    with pytest.raises(ValueError):
        tl.tile_plan(128, 256, 0)


def test_small_tiles_pay_for_their_reads():
    """Products at which the smallest tiles over the whole of K are 15 to 35 % slower than others, and two at which they are the fastest."""
    for M, N, K in ((224, 4096, 4096), (768, 2048, 8192), (384, 4096, 8192), (128, 7168, 4096), (257, 5120, 5120)):
        assert tl.tile_plan(M, N, K) != (3, 2, 1), (M, N, K)
    for M, N, K in ((288, 18560, 4096), (288, 20512, 4096), (768, 4096, 11008)):
        assert tl.tile_plan(M, N, K) != (3, 4, 1), (M, N, K)
    assert tl.tile_plan(668, 768, 2048) == (3, 2, 1) and tl.tile_plan(1200, 2048, 4096) == (3, 4, 1)


def test_a_new_row_count_costs_no_search_in_python():
    """A server's prompt steps have another token count nearly every time: a plan that was not asked for before is some microseconds
    (in Python 20 to 140)."""
    def cost(plan, *args):
        import time
        best = 1.0
        for _ in range(5):
            t = time.perf_counter()
            for M in range(500, 700):
                plan.__wrapped__(M, *args)
            best = min(best, (time.perf_counter() - t) / 200)
        return best
    assert cost(tl.tile_plan, 4096, 4096) < 12e-6
    assert cost(tl.grouped_plan, 8, 4096, 4096) < 12e-6


@pytest.mark.parametrize("plan,split,want", [((3, 2, 4), True, "parts"), ((8, 8, 1), True, "tiles"), (None, True, "split"),
                                             (None, False, "torch")])
def test_llama_down_asks_for_one_plan(plan, split, want, monkeypatch):
    from xgserve.models import llama
    asked, layer = [], llama.LlamaLayer.__new__(llama.LlamaLayer)
    torch.nn.Module.__init__(layer)
    layer.down = torch.zeros(64, 128)
    monkeypatch.setattr(llama, "_tile_plan", lambda *a, **k: asked.append(k) or plan)
    monkeypatch.setattr(llama, "splitk_prefill_ok", lambda *a: split)
    for name, tag in (("tile_parts", "parts"), ("tile_linear", "tiles"), ("splitk_linear", "split")):
        monkeypatch.setattr(llama, name, lambda *a, tag=tag: tag)
    monkeypatch.setattr(llama.F, "linear", lambda *a: "torch")
    assert layer._down(torch.zeros(70, 128)) == want and asked == [dict(plain=True)]


# ---- workgroups that take tile after tile: the next tile's loads go out ahead of a whole tile's stores, which the waits then count.
# A launch told of 3 compute units has several rounds at small sizes. K tiles of 64: fewer than a ring has slots, as many, more.
_ROUNDS_K = (64, 192, 256, 384, 832)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", sorted(tl._TILES))
@pytest.mark.parametrize("rotated", [False, True])     # (up to 256 rows column tiles start at different places in K)
@pytest.mark.parametrize("K", _ROUNDS_K)
def test_a_workgroup_takes_several_tiles(tile, rotated, K, monkeypatch):
    monkeypatch.setattr(tl, "cu_count", lambda d: 3)
    fm, fn = tile
    M, N = 256 if rotated else max(32 * fm * 3, 288) + 5, 32 * fn * 7 + 8
    assert -(-M // (32 * fm)) * -(-N // (32 * fn)) >= 8 and (M <= 256) == rotated
    g = torch.Generator("cuda").manual_seed(K + fm)
    x = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16)
    b = torch.randn(N, generator=g, device="cuda")
    ref = x.double() @ w.double().t()
    for S in (1, 2) if K >= 128 else (1,):
        _close(tl.tile_linear((*tile, S), x, w), ref, K)
        _close(tl.tile_linear((*tile, S), x, w, b), ref + b.double(), K)
        if S > 1:
            part = tl.tile_parts((*tile, S), x, w).part
            # fp32 sums of K products (see _close)
            assert ((part.double().sum(0) - ref).abs() <= K * 2.0 ** -24 * K ** 0.5 + 1e-6).all()


@pytest.mark.gpu
@pytest.mark.parametrize("tile", sorted(tl._TILES))
@pytest.mark.parametrize("rotated", [False, True])
@pytest.mark.parametrize("K", _ROUNDS_K)
def test_a_workgroup_takes_several_gated_tiles(tile, rotated, K, monkeypatch):
    monkeypatch.setattr(tl, "cu_count", lambda d: 3)
    fm, fn = tile
    M, F_ = 256 if rotated else max(32 * fm * 3, 288) + 5, 16 * fn * 7 + 16
    g = torch.Generator("cuda").manual_seed(K + fn)
    x = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn(2 * F_, K, generator=g, device="cuda") * 3 * K ** -0.5).to(torch.bfloat16)
    blocks = torch.stack([w[:F_].view(-1, 16, K), w[F_:].view(-1, 16, K)], 1).reshape(2 * F_, K)
    z = x.double() @ w.double().t()
    ref = sq._glu_ref(z[:, :F_], z[:, F_:], sq.GLU_SILU, 0.0, 0.0)
    room = (1.5 * z[:, F_:].abs() + 1.5 * z[:, :F_].abs() + 2) * (3 * K ** 1.5 * 2.0 ** -24 + 2.0 ** -22)   # (as in test_gated_tiles)
    for S in (1, 2) if K >= 128 else (1,):
        for ww, pairs in ((w, tl.PAIR_HALVES), (blocks, tl.PAIR_BLOCKS)):
            y = tl.tile_linear((*tile, S), x, ww, None, sq.ACT_GLU + sq.GLU_SILU, pairs=pairs).double()
            assert ((y - ref).abs() <= 2.0 ** -8 * ref.abs() + room).all()


@pytest.mark.gpu
@pytest.mark.parametrize("tile", tl._GROUPED)
@pytest.mark.parametrize("idle", [0, 9])     # experts without rows: with them 256 rows an expert are not reached, and columns rotate
def test_grouped_workgroups_take_several_tiles(tile, idle, monkeypatch):
    K, F_, W, top = 512, 512, 264, 1
    share = [700, 32 * tile[0] * 2, 32 * tile[0], 300] + [0] * idle
    E, T, g = len(share), sum(share), torch.Generator().manual_seed(tile[1])
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(share))[torch.randperm(T, generator=g)].view(T, 1).to(torch.int32)
    assert (T > 256 * E) == (idle == 0)
    h = torch.randn(T, K, generator=g).to(torch.bfloat16)
    w13 = (torch.randn(E, 2 * F_, K, generator=g) * K ** -0.5).to(torch.bfloat16)
    w2 = (torch.randn(E, W, F_, generator=g) * F_ ** -0.5).to(torch.bfloat16)
    wts = torch.rand(T, top, generator=g)
    monkeypatch.setattr(sq, "grouped_plan", lambda *a: tile)
    monkeypatch.setattr(sq, "cu_count", lambda d: 3)
    calls = record_native(monkeypatch, sq)
    got = sq.routed_experts(h.cuda(), w13.cuda(), w2.cuda(), ids.cuda(), wts.cuda(), sq.GLU_SILU).cpu().double()
    assert calls.count("tile_grouped") == 2
    for e in range(4):
        t = torch.nonzero(ids[:, 0] == e).view(-1)
        z = h[t].double() @ w13[e].double().t()
        a = sq._glu_ref(z[:, :F_], z[:, F_:], sq.GLU_SILU, 0.0, 0.0)
        ref, size = wts[t].double() * (a @ w2[e].double().t()), wts[t].double() * (a.abs() @ w2[e].double().abs().t())
        assert ((got[t] - ref).abs() <= (2.0 ** -9 + F_ * 2.0 ** -23) * size + 1e-5).all()   # (as in test_grouped_tiles)


@pytest.mark.parametrize("M,N,K,library", [(2048, 16384, 2048, True), (6144, 2048, 2048, True),       # 512 and 192 of the library's tiles
                                           (2049, 16384, 2048, True), (5889, 2048, 2048, True),       # 576 of 768 and 192: three quarters
                                           (2560, 4096, 4096, False), (3100, 6144, 4096, False),      # 160 of 256, 312 of 512
                                           (1792, 16384, 2048, False), (8192, 10304, 2048, False)])
def test_the_library_keeps_full_rounds(M, N, K, library):
    assert tl.library_better(M, N, K) is library
