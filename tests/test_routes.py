"""Which kernel a call takes: the rules in Python against the kernels' own contracts, over all that they accept. No GPU is needed
(a rule looks at sizes, strides, types and alignment; CPU tensors stand for the device's)."""
import os
import subprocess
import sys
import types

import pytest
import torch

from xgserve.ops import seqmix as sq
from xgserve.ops._native import mixers

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_single_token_states_are_those_the_kernel_takes():
    """Every (dk, dv) that the rule sends to the one-token kernel fits it, and every one that fits is sent there."""
    rows, sm = mixers().gla_step_rows, types.SimpleNamespace(max_q=1, num_seqs=4)
    v = torch.zeros(4, 8)
    for dk in range(0, 260):
        for dv in range(0, 262):
            assert sq._gla_step_ok(v, sm, dk, dv) == (rows(dk, dv) > 0), (dk, dv)
    for dk, dv in ((88, 176), (168, 96), (152, 104), (136, 120), (72, 208)):   # 17 or 18 rows within 128 x 128 elements
        assert dk * dv <= 128 * 128 and not sq._gla_step_ok(v, sm, dk, dv)


@pytest.fixture
def as_if_native(monkeypatch):
    """CPU tensors pass for the device's (rules only: no kernel is called)."""
    monkeypatch.setattr(sq, "native_device", lambda t: t.device.type in ("cpu", "cuda"))


def test_products_that_torch_refuses_or_differentiates_stay_with_it(as_if_native):
    x, w, b = torch.randn(3, 256).bfloat16(), torch.randn(64, 256).bfloat16(), torch.randn(64).bfloat16()
    sm = types.SimpleNamespace(tickets=torch.zeros(128, dtype=torch.int32))

    def plan(x, w, b=None):
        return sq._rows_plan_of(x, w, sm, b, False)
    assert plan(x, w) is not None and plan(x, w, b) is not None and plan(x, w, b.float()) is not None
    # another device: F.linear raises, a kernel would read a pointer of the other device
    meta = dict(device="meta", dtype=torch.bfloat16)
    assert plan(x, torch.empty(64, 256, **meta)) is None and plan(x, w, torch.empty(64, **meta)) is None
    assert plan(x, w[None]) is None and plan(x, w[0]) is None and plan(x[None], w) is None
    with pytest.raises(RuntimeError):
        sq.linear(x, w, sm, b.float())                      # a bias of another type than the rows
    # something that follows the values
    xg, wg = x.clone().requires_grad_(), w.clone().requires_grad_()
    assert plan(xg, w) is None and plan(x, wg) is None and plan(x, w, b.clone().requires_grad_()) is None
    y = sq.linear(xg, w, sm)
    y.float().sum().backward()
    torch.testing.assert_close(xg.grad.float(), w.float().sum(0).expand(3, 256), rtol=2e-2, atol=0.1)
    with torch.no_grad():
        assert plan(xg, wg) is not None
    ref = torch.nn.functional.linear(x.expand(2, 3, 256), w)
    torch.testing.assert_close(torch.func.vmap(lambda h: sq.linear(h, w, sm))(x.expand(2, 3, 256)), ref)
    _, tangent = torch.func.jvp(lambda h: sq.linear(h, w, sm), (x,), (torch.ones_like(x),))
    torch.testing.assert_close(tangent, torch.nn.functional.linear(torch.ones_like(x), w))
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
        out = torch.autograd.forward_ad.unpack_dual(sq.linear(dual, w, sm)).tangent
        torch.testing.assert_close(out, torch.nn.functional.linear(torch.ones_like(x), w))
    assert plan(x, w) is not None


def test_products_that_are_recorded_stay_with_torch(as_if_native):
    """A tracer, a dispatch mode or a tensor type of its own sees torch's operator (a kernel's result would be a constant to it)."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.utils.flop_counter import FlopCounterMode
    x, w = torch.randn(3, 256).bfloat16(), torch.randn(64, 256).bfloat16()
    sm = types.SimpleNamespace(tickets=torch.zeros(128, dtype=torch.int32))
    want = torch.nn.functional.linear(2 * x, w)
    traced = torch.jit.trace(lambda h: sq.linear(h, w, sm), (x,), check_trace=False)
    torch.testing.assert_close(traced(2 * x), want)
    torch.testing.assert_close(make_fx(lambda h: sq.linear(h, w, sm))(x)(2 * x), want)
    with FlopCounterMode(display=False) as count:
        sq.linear(x, w, sm)
    assert count.get_total_flops() == 2 * 3 * 256 * 64
    with FakeTensorMode() as mode:
        assert sq.linear(mode.from_tensor(x), mode.from_tensor(w), sm).shape == (3, 64)
    fake = mode.from_tensor(x), mode.from_tensor(w)
    assert sq.linear(*fake, sm).shape == (3, 64)
    assert sq._rows_plan_of(x, torch.nn.Parameter(w, requires_grad=False), sm, None, False) is not None


def test_tensors_that_lie_off_16_bytes_keep_the_general_kernels(as_if_native):
    """The wide kernels refuse them, which would raise; the general ones take them."""
    sm = types.SimpleNamespace(max_q=1, num_seqs=2, block_tables=torch.zeros(2, 4, dtype=torch.int32))

    def off(*shape, dtype=torch.float32):
        n = torch.Size(shape).numel()
        return torch.zeros(n + 1, dtype=dtype)[1:].view(shape)
    v, state = torch.zeros(2, 64), torch.zeros(2, 1, 64, 64)
    assert sq._gla_step_ok(v, sm, 64, 64, state) and not sq._gla_step_ok(v, sm, 64, 64, off(2, 1, 64, 64))
    proj, w2 = torch.zeros(2, 5 * 64 + 8).bfloat16(), torch.zeros(64, 8).bfloat16()
    assert sq._delta_step_ok(proj, w2, state, 64, sm, torch.bfloat16)
    assert not sq._delta_step_ok(proj, w2, off(2, 1, 64, 64), 64, sm, torch.bfloat16)
    q, uv, cache = torch.zeros(2, 4, 96).bfloat16(), torch.zeros(256, 256).bfloat16(), torch.zeros(8, 288).bfloat16()
    assert sq._latent_shares(q, uv, 256, 32, 64, 64, 16, sm, cache) == 1
    assert sq._latent_shares(q, uv, 256, 32, 64, 64, 16, sm, off(8, 288, dtype=torch.bfloat16)) == 0
    x, y, w = torch.zeros(2, 64), torch.zeros(2, 64).bfloat16(), torch.zeros(64)
    assert sq._rows_aligned(y, None, x, w, None) and sq._rows_aligned(sq.Parts(torch.zeros(2, 2, 64)), y, x)
    assert not sq._rows_aligned(y, None, x, off(64)) and not sq._rows_aligned(y, off(2, 64, dtype=torch.bfloat16), x)
    assert not sq._rows_aligned(torch.zeros(2, 66).bfloat16()[:, :64], None, x)


@pytest.mark.parametrize("H,dn,rd,dv,R", [(32, 64, 32, 64, 256), (64, 128, 64, 128, 512), (128, 128, 64, 128, 512), (256, 128, 64, 128, 512)])
def test_expanded_latents_stay_within_their_bytes(as_if_native, H, dn, rd, dv, R):
    """Portions behind long contexts: the expansion is chosen only while keys, values and gathered rows stay within 1 GiB, which
    the cache's sizing leaves free. (Rows alone let 64 heads of 128 + 128 take 2.1 GB and 128 heads 4.3 GB.)"""
    chosen = []
    for T, ctx in ((64, 0), (2048, 30000), (2100, 65000), (4096, 65536), (8192, 57344), (8192, 200000)):
        q = torch.empty(1, H, dn + rd, dtype=torch.bfloat16).expand(T, -1, -1)
        cache = torch.empty(8, R + rd, dtype=torch.bfloat16)
        sm = types.SimpleNamespace(max_q=T, num_seqs=1, block_tables=torch.zeros(1, -(-(T + ctx) // 16), dtype=torch.int32))
        nk = sq._latent_expands(q, dn, R, dv, rd, 1 << 20, 16, sm, cache)
        keys = sq._latent_key_rows(sm, T, 1 << 20, 16)
        size = keys * (H * (dn + dv) + R + rd) * 2
        assert nk == (keys if keys <= 32 * T and size <= 1 << 30 else 0)
        chosen.append(nk > 0)
    assert chosen[0] and not chosen[-1]


def test_tuning_keys_choose_the_kernels_that_they_name(as_if_native, monkeypatch):
    """latent_mfma, delta_two_pass, scan_cols and scan_two_pass ask for the kernels they asked for before the chunked, expanded
    and one-token forms came in front of them."""
    step, prompt = types.SimpleNamespace(max_q=1, num_seqs=2, block_tables=torch.zeros(2, 4, dtype=torch.int32)), \
        types.SimpleNamespace(max_q=4001, num_seqs=1, block_tables=torch.zeros(1, 256, dtype=torch.int32))
    q, uv, cache = torch.zeros(2, 4, 96).bfloat16(), torch.zeros(256, 256).bfloat16(), torch.zeros(8, 288).bfloat16()
    qp = torch.zeros(1, 4, 96).bfloat16().expand(4001, -1, -1)
    proj, w2, state = torch.zeros(2, 5 * 64 + 8).bfloat16(), torch.zeros(64, 8).bfloat16(), torch.zeros(2, 1, 64, 64)
    v = torch.zeros(2, 64)

    def routes():
        return {"latent step": sq._latent_shares(q, uv, 256, 32, 64, 64, 16, step, cache) > 0,
                "latent prompt": sq._latent_expands(qp, 64, 256, 64, 32, 1024, 16, prompt, cache) > 0,
                "delta step": sq._delta_step_ok(proj, w2, state, 64, step, torch.bfloat16),
                "delta prompt": sq._delta_chunk_ok(proj, 0, 64, prompt),
                "scan step": sq._gla_step_ok(v, step, 64, 64, state), "scan prompt": sq._chunk_scan_ok(prompt, 64),
                "segments": sq._chunk_scan_segments(prompt, 4001, 16, 64, 128, 128, "cpu")[1] is not None}
    assert all(routes().values())
    for key, value, off in (("LATENT_MFMA", False, {"latent step", "latent prompt"}), ("DELTA_TWO_PASS", False, {"delta step", "delta prompt"}),
                            ("SCAN_COLS", 32, {"scan step", "scan prompt"}), ("SCAN_TWO_PASS", False, {"segments"})):
        with monkeypatch.context() as m:
            m.setattr(sq, key, value)
            assert {k for k, on in routes().items() if not on} == off, key


def test_the_32_row_tiles_follow_their_key():
    """moe_tile32_min reaches every kind of expert."""
    code = "from xgserve.ops import seqmix as sq; print(dict(sq.MOE_TILES)[32], dict(sq.MOE_TILES_GENERAL)[32])"
    for spec, want in (("", "8 12"), ("moe_tile32_min=20", "20 20")):
        out = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, XGS_TUNE=spec), cwd=ROOT, capture_output=True,
                             text=True, check=True)
        assert out.stdout.split() == want.split()
