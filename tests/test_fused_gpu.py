"""The fused layer-layout forward (spear_phalanx_mix_forward / phalanx_mix / Phalanx(method="fused"))
against the float64 composition of the pinned BTP oracle with sigmoid gates, and against the
unfused HIP path of the layer."""

import numpy as np
import pytest
import torch

from helpers import BF16_ATOL, BF16_RTOL, assert_close, f64
from oracle import btp_oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def make_mix_inputs(B, L, H, Hkv, seed, dtype=torch.bfloat16, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    a = (torch.randn(B, L, H, generator=g) * scale).to(dtype)
    b = (torch.randn(B, L, Hkv * 16, generator=g) * scale).to(dtype)
    c = torch.randn(B, L, Hkv * 16, generator=g).to(dtype)
    v = torch.randn(B, L, H * 16, generator=g).to(dtype)
    return a, b, c, v


def run_mix(a, b, c, v, H, Hkv):
    from spear_amd import _btp

    out = torch.full(v.shape, float("nan"), device=DEV, dtype=v.dtype)
    _btp.mix_forward(a.to(DEV), b.to(DEV), c.to(DEV), v.to(DEV), out, H, Hkv)
    torch.cuda.synchronize()
    return out.cpu()


# head counts and groupings as the reference's KVRepeat accepts them (spear/nn/phalanx/swr.py:37-38: any
# heads % kv_heads == 0): head counts that do not fill a wavefront's 8 heads or are odd (gate logits then do not pair
# up into aligned 32-bit words), groups of 1, 2, 4, 8 heads per kv head (summed inside a wavefront in backward) and
# every other group size (3, 5, 6, 7: whole groups per wavefront; 12, 16, 20, 24, 32: worked through 8 heads at a time)
ODD_GROUPINGS = [(2, 48, 6, 3), (1, 80, 12, 12), (2, 64, 3, 1), (1, 32, 1, 1), (2, 96, 5, 5), (1, 144, 10, 2),
                 (2, 64, 16, 1), (1, 80, 32, 2), (2, 48, 6, 2), (1, 112, 12, 2), (2, 64, 7, 1), (1, 272, 12, 1),
                 (1, 64, 24, 1), (2, 80, 40, 2), (1, 48, 9, 3), (3, 64, 36, 6), (1, 2064, 16, 1)]


@pytest.mark.parametrize("B,L,H,Hkv", [
    (1, 16, 4, 4), (2, 32, 4, 4), (2, 48, 8, 8), (1, 80, 4, 2), (3, 128, 8, 2), (2, 144, 16, 4),
    (1, 512, 32, 32), (2, 272, 12, 3), (1, 1040, 4, 1), (1, 4096, 8, 8), (2, 2064, 16, 2),
    (5, 64, 32, 8), (3, 272, 128, 16),
    # grids beyond one window of the dealing of workgroups to XCDs (1024 workgroups), with a tail
    # that keeps the launch order: 1096 and 1500 workgroups
    (137, 128, 32, 32), (100, 272, 24, 8),
] + ODD_GROUPINGS)
def test_fused_forward_matches_oracle(B, L, H, Hkv):
    a, b, c, v = make_mix_inputs(B, L, H, Hkv, seed=1000 + L + H)
    print(f"fused B={B} L={L} H={H} Hkv={Hkv}", flush=True)
    out = run_mix(a, b, c, v, H, Hkv)
    ref = orc.phalanx_mix_forward(f64(a), f64(b), f64(c), f64(v), H, Hkv)
    assert_close(f64(out), ref, BF16_ATOL, BF16_RTOL, "out")


def test_fused_forward_fp16_and_steep_gates():
    a, b, c, v = make_mix_inputs(2, 96, 8, 4, seed=5, dtype=torch.float16, scale=4.0)
    a[0, :10, :] = -30.0  # decay ~ 1e-13: counts as zero
    a[1, 20:40, 3] = 30.0  # decay -> 1
    out = run_mix(a, b, c, v, 8, 4)
    ref = orc.phalanx_mix_forward(f64(a), f64(b), f64(c), f64(v), 8, 4)
    assert_close(f64(out), ref, 4e-3, 4e-3, "out fp16")


def run_mix_backward(a, b, c, v, dout, H, Hkv=None):
    from spear_amd import _btp

    dev = [t.to(DEV) for t in (a, b, c, v, dout)]
    outs = [torch.full(t.shape, float("nan"), device=DEV, dtype=t.dtype) for t in (a, b, c, v)]
    _btp.mix_backward(*dev, *outs, H, H if Hkv is None else Hkv)
    torch.cuda.synchronize()
    return [t.cpu() for t in outs]


@pytest.mark.parametrize("B,L,H", [(1, 16, 4), (2, 32, 4), (2, 48, 8), (1, 80, 12), (3, 128, 8), (2, 144, 16), (1, 512, 32), (1, 1040, 4), (1, 4096, 8), (2, 2064, 16),
                                   (5, 64, 32), (2, 112, 24), (3, 272, 64),
                                   # grids beyond one window of the dealing of workgroups to XCDs (1024
                                   # workgroups), with a tail that keeps the launch order: 1096 and 1500 workgroups
                                   (137, 128, 32), (100, 272, 24)])
def test_fused_backward_matches_oracle(B, L, H):
    a, b, c, v = make_mix_inputs(B, L, H, H, seed=2000 + L + H)
    dout = torch.randn(B, L, H * 16, generator=torch.Generator().manual_seed(L)).bfloat16()
    print(f"fused bwd B={B} L={L} H={H}", flush=True)
    da, db, dc, dv = run_mix_backward(a, b, c, v, dout, H)
    rda, rdb, rdc, rdv = orc.phalanx_mix_backward(f64(a), f64(b), f64(c), f64(v), f64(dout), H, H)
    assert_close(f64(dv), rdv, BF16_ATOL, BF16_RTOL, "dv")
    assert_close(f64(dc), rdc, BF16_ATOL, BF16_RTOL, "dc")
    assert_close(f64(db), rdb, BF16_ATOL, BF16_RTOL, "db")
    assert_close(f64(da), rda, BF16_ATOL, BF16_RTOL, "da")


@pytest.mark.parametrize("B,L,H,Hkv", [(2, 48, 8, 4), (1, 80, 12, 3), (2, 144, 16, 2), (1, 272, 32, 8), (2, 64, 4, 2),
                                       (1, 2064, 8, 1)] + ODD_GROUPINGS)
def test_fused_backward_with_shared_kv_heads(B, L, H, Hkv):
    """Every head grouping at the bf16 bound: the sums over a group are taken in fp32 and rounded once."""
    a, b, c, v = make_mix_inputs(B, L, H, Hkv, seed=3000 + L + H)
    dout = torch.randn(B, L, H * 16, generator=torch.Generator().manual_seed(L + 1)).bfloat16()
    print(f"fused bwd kv B={B} L={L} H={H} Hkv={Hkv}", flush=True)
    da, db, dc, dv = run_mix_backward(a, b, c, v, dout, H, Hkv)
    rda, rdb, rdc, rdv = orc.phalanx_mix_backward(f64(a), f64(b), f64(c), f64(v), f64(dout), H, Hkv)
    assert_close(f64(dv), rdv, BF16_ATOL, BF16_RTOL, "dv")
    assert_close(f64(dc), rdc, BF16_ATOL, BF16_RTOL, "dc")
    assert_close(f64(db), rdb, BF16_ATOL, BF16_RTOL, "db")
    assert_close(f64(da), rda, BF16_ATOL, BF16_RTOL, "da")
    # a second run gives the same bits: every sum is taken in a fixed order
    again = run_mix_backward(a, b, c, v, dout, H, Hkv)
    for x, y in zip((da, db, dc, dv), again):
        assert torch.equal(x, y)


@pytest.mark.parametrize("B,L,H,Hkv", [(1, 16, 4, 4), (3, 128, 8, 8), (2, 144, 16, 2), (1, 80, 12, 3), (1, 272, 32, 4),
                                       (2, 2064, 8, 1), (40, 64, 32, 32), (1, 8192, 8, 8), (3, 112, 128, 16),
                                       (70, 272, 32, 32), (2, 80, 6, 2), (1, 144, 16, 1), (3, 48, 40, 2), (2, 64, 7, 7),
                                       (1, 96, 12, 1), (2, 64, 10, 2)])
def test_fused_backward_column_sums_match_oracle(B, L, H, Hkv):
    """The partial sums the backward kernel leaves (one row per batch row and tile of 64 time steps) add up to the
    oracle's gradients summed over batch and time (the bias gradients of proj_a, proj_b, proj_c); the gradients
    themselves are unchanged by asking."""
    from spear_amd import _btp

    a, b, c, v = make_mix_inputs(B, L, H, Hkv, seed=5000 + L + H)
    dout = torch.randn(B, L, H * 16, generator=torch.Generator().manual_seed(L + 2)).bfloat16()
    print(f"fused bwd sums B={B} L={L} H={H} Hkv={Hkv}", flush=True)
    plain = run_mix_backward(a, b, c, v, dout, H, Hkv)
    dev = [t.to(DEV) for t in (a, b, c, v, dout)]
    outs = [torch.full(t.shape, float("nan"), device=DEV, dtype=t.dtype) for t in (a, b, c, v)]
    rows = _btp.mix_backward_sum_rows(B, L, H)
    assert rows == B * -(-(L // 16) // 4)
    sums = tuple(torch.full((rows, w), float("nan"), device=DEV) for w in (H, Hkv * 16, Hkv * 16))
    _btp.mix_backward(*dev, *outs, H, Hkv, sums=sums)
    torch.cuda.synchronize()
    for got, want in zip(outs, plain):
        assert torch.equal(got.cpu(), want)
    rda, rdb, rdc, _ = orc.phalanx_mix_backward(f64(a), f64(b), f64(c), f64(v), f64(dout), H, Hkv)
    for name, s, ref in (("da", sums[0], rda), ("db", sums[1], rdb), ("dc", sums[2], rdc)):
        got = f64(s.cpu()).sum(0)
        want, mass = ref.sum((0, 1)), np.abs(ref).sum((0, 1))
        # fp32 arithmetic on bf16 inputs; the sums are taken before any rounding to bf16
        assert np.all(np.abs(got - want) <= 2e-4 * mass + 1e-5), (name, np.abs(got - want).max(), mass.max())
    with pytest.raises(RuntimeError, match="shape"):
        _btp.mix_backward(*dev, *outs, H, Hkv,
                          sums=tuple(torch.empty(rows + 1, w, device=DEV) for w in (H, Hkv * 16, Hkv * 16)))


@pytest.mark.parametrize("B,L,H,Hkv", [(1, 16, 4, 4), (3, 128, 8, 8), (2, 144, 16, 2), (1, 80, 12, 3), (2, 2064, 8, 1), (40, 64, 32, 32),
                                       (2, 48, 6, 2), (1, 80, 16, 1), (2, 64, 5, 5)])
def test_fused_backward_into_column_blocks_of_one_buffer(B, L, H, Hkv):
    """The four gradients written side by side into one [B, L, ld] buffer are bit-identical to the dense
    ones, and the columns between and after the blocks are left alone."""
    from spear_amd import _btp
    from spear_amd.nn.phalanx.projections import packed_columns

    a, b, c, v = make_mix_inputs(B, L, H, Hkv, seed=6000 + L + H)
    dout = torch.randn(B, L, H * 16, generator=torch.Generator().manual_seed(L + 3)).bfloat16()
    print(f"fused bwd packed B={B} L={L} H={H} Hkv={Hkv}", flush=True)
    plain = run_mix_backward(a, b, c, v, dout, H, Hkv)
    cols, ld = packed_columns(H, Hkv)
    assert ld % 64 == 0 and ld >= cols["a"][0] + cols["a"][1]
    ld += 64                                              # more slack than needed, so there is padding to check
    dev = [t.to(DEV) for t in (a, b, c, v, dout)]
    marker = 12345.0
    packed = torch.full((B, L, ld), marker, device=DEV, dtype=torch.bfloat16)
    views = [packed[..., cols[k][0]:cols[k][0] + cols[k][1]] for k in "abcv"]
    _btp.mix_backward(*dev, *views, H, Hkv)
    torch.cuda.synchronize()
    for got, want in zip(views, plain):
        assert torch.equal(got.cpu(), want)
    used = cols["a"][0] + cols["a"][1]
    assert bool((packed[..., used:] == marker).all())
    # a block that is not a column block of a dense buffer is refused
    with pytest.raises(RuntimeError, match="column block"):
        every_other = torch.empty(B, L, 2 * H * 16, device=DEV, dtype=torch.bfloat16)[..., ::2]
        _btp.mix_backward(*dev, views[0], views[1], views[2], every_other, H, Hkv)


def test_fused_backward_fp16_and_steep_gates():
    a, b, c, v = make_mix_inputs(2, 96, 8, 4, seed=6, dtype=torch.float16, scale=3.0)
    a[0, :10, :] = -30.0  # decay ~ 1e-13: counts as zero
    a[1, 20:40, 3] = 30.0  # decay -> 1
    dout = torch.randn(2, 96, 128, generator=torch.Generator().manual_seed(7)).half()
    da, db, dc, dv = run_mix_backward(a, b, c, v, dout, 8, 4)
    rda, rdb, rdc, rdv = orc.phalanx_mix_backward(f64(a), f64(b), f64(c), f64(v), f64(dout), 8, 4)
    # fp16 storage: 11 significant bits; sums over two heads and up to 32 steps of undamped states
    for name, got, want in (("dv", dv, rdv), ("dc", dc, rdc), ("db", db, rdb), ("da", da, rda)):
        assert_close(f64(got), want, 2e-2, 4e-3, name + " fp16")


@pytest.mark.parametrize("H,Hkv", [(8, 4), (16, 1), (32, 2), (6, 3), (12, 12), (6, 2)])
def test_fused_op_autograd_matches_unfused_composition(H, Hkv):
    """Gradients of phalanx_mix against autograd through the same composition built from torch ops
    and the float64 reference recurrence, at the bf16 bound for every head grouping."""
    from spear_amd import phalanx_mix
    from spear_amd.ops.btp.reference import block_two_pass_ref

    B, L = 2, 64
    a, b, c, v = make_mix_inputs(B, L, H, Hkv, seed=21)
    dout = torch.randn(B, L, H * 16, generator=torch.Generator().manual_seed(22)).bfloat16()

    leaves = [t.clone().to(DEV).requires_grad_(True) for t in (a, b, c, v)]
    out = phalanx_mix(*leaves, heads=H, kv_heads=Hkv)
    out.backward(dout.to(DEV))

    ref_leaves = [t.clone().double().requires_grad_(True) for t in (a, b, c, v)]
    ra, rb, rc, rv = ref_leaves
    g = H // Hkv
    heads = lambda t, h: t.view(B, L, h, 16).permute(0, 2, 3, 1)
    A = torch.sigmoid(ra).transpose(1, 2)
    G = torch.sigmoid(heads(rb, Hkv)).repeat_interleave(g, 1)
    C = heads(rc, Hkv).repeat_interleave(g, 1)
    V = heads(rv, H)
    hh = block_two_pass_ref(A.contiguous(), (G * V).contiguous())
    ref_out = (hh * C + V).permute(0, 3, 1, 2).reshape(B, L, H * 16)
    ref_out.backward(dout.double())

    assert_close(f64(out), ref_out.detach().numpy(), BF16_ATOL, BF16_RTOL, "out")
    for name, got, want in zip("abcv", leaves, ref_leaves):
        assert_close(f64(got.grad), want.grad.numpy(), BF16_ATOL, BF16_RTOL, f"d{name}")


def test_phalanx_fused_method_matches_default_and_pytorch():
    from spear_amd import Phalanx
    from spear_amd.testing.numerics import compute_error_metrics

    torch.manual_seed(0)
    ref = Phalanx(dim=512, length=128, method="pytorch", dtype=torch.bfloat16)
    fused = Phalanx(dim=512, length=128, method="fused", dtype=torch.bfloat16).to(DEV)
    dflt = Phalanx(dim=512, length=128, method="default", dtype=torch.bfloat16).to(DEV)
    fused.load_state_dict(ref.state_dict())
    dflt.load_state_dict(ref.state_dict())
    x = torch.randn(8, 128, 512, generator=torch.Generator().manual_seed(1)).bfloat16()
    y_ref, y_f, y_d = ref(x), fused(x.to(DEV)).cpu(), dflt(x.to(DEV)).cpu()
    for name, y in (("fused", y_f), ("default", y_d)):
        m = compute_error_metrics(y, y_ref)
        assert m["max_abs"] <= 1e-1 and m["rmse"] <= 5e-2, (name, m)  # layer forward limits of the reference tests
    assert_close(f64(y_f), f64(y_ref), 2e-2, 2e-2, "fused layer y")

    # and it trains: gradients reach every parameter
    fused.zero_grad()
    fused(x.to(DEV)).float().square().mean().backward()
    assert all(p.grad is not None and torch.isfinite(p.grad.float()).all() for p in fused.parameters())


def test_fused_method_needs_k_2_and_takes_every_head_count():
    from spear_amd import Phalanx

    with pytest.raises(ValueError, match="k == 2"):
        Phalanx(dim=128, method="fused", dtype=torch.bfloat16, k=1)
    for dim, kv_heads in ((96, None), (96, 2), (48, 1), (256, 1)):  # 6 heads, groups of 3, 3 heads shared, groups of 16
        torch.manual_seed(5)
        ref = Phalanx(dim=dim, length=64, method="pytorch", dtype=torch.bfloat16, kv_heads=kv_heads)
        fused = Phalanx(dim=dim, length=64, method="fused", dtype=torch.bfloat16, kv_heads=kv_heads).to(DEV)
        fused.load_state_dict(ref.state_dict())
        x = torch.randn(2, 64, dim, generator=torch.Generator().manual_seed(6)).bfloat16()
        assert_close(f64(fused(x.to(DEV))), f64(ref(x)), 2e-2, 2e-2, f"fused layer y, dim {dim} kv_heads {kv_heads}")
        fused.zero_grad()
        fused(x.to(DEV)).float().square().mean().backward()
        assert all(p.grad is not None and torch.isfinite(p.grad.float()).all() for p in fused.parameters())


def test_default_method_rerouted_by_environment_gives_the_fused_results(monkeypatch):
    from spear_amd import Phalanx

    torch.manual_seed(3)
    fused = Phalanx(dim=128, length=64, method="fused", dtype=torch.bfloat16).to(DEV)
    monkeypatch.setenv("SPEAR_PHALANX_DEFAULT", "fused")
    rerouted = Phalanx(dim=128, length=64, dtype=torch.bfloat16).to(DEV)
    rerouted.load_state_dict(fused.state_dict())
    x = torch.randn(2, 64, 128, generator=torch.Generator().manual_seed(4)).bfloat16().to(DEV)
    assert torch.equal(rerouted(x), fused(x))


@pytest.mark.parametrize("H,Hkv", [(16, 4), (12, 2), (16, 1)])
def test_qkv_form_backward_against_the_oracle(H, Hkv):
    """The q/k/v/gate form of the backward kernel, with groups summed inside a wavefront and through LDS."""
    from spear_amd import _btp

    B, L = 3, 176
    g = torch.Generator().manual_seed(8102)
    gate = -torch.nn.functional.softplus(torch.randn(B, L, H, generator=g))
    q, k, vv, dd = ((0.5 * torch.randn(B, L, w, generator=g)).bfloat16() for w in (Hkv * 16, Hkv * 16, H * 16, H * 16))
    outs = [torch.full(t.shape, float("nan"), device=DEV, dtype=t.dtype) for t in (gate, k, q, vv)]
    _btp.mix_backward(gate.to(DEV), k.to(DEV), q.to(DEV), vv.to(DEV), dd.to(DEV), *outs, H, Hkv, qkv_gate=True)
    torch.cuda.synchronize()
    rgate, rk, rq, rv = orc.qkv_gate_backward(f64(q), f64(k), f64(vv), f64(gate), f64(dd), H, Hkv)
    assert_close(f64(outs[0]), rgate, 1e-4, 1e-4, "dgate")
    assert_close(f64(outs[1]), rk, BF16_ATOL, BF16_RTOL, "dk")
    assert_close(f64(outs[2]), rq, BF16_ATOL, BF16_RTOL, "dq")
    assert_close(f64(outs[3]), rv, BF16_ATOL, BF16_RTOL, "dv")


@pytest.mark.parametrize("B,L,dim,kv_heads", [(1, 16, 16, None), (3, 48, 96, 2), (8, 128, 512, None), (64, 144, 80, 1)])
def test_default_layer_mixes_in_the_fused_kernels(B, L, dim, kv_heads):
    """A plain bf16 call of a default layer lies as close to the fused layer and to the stand-alone composition as their bf16
    roundings allow, with weight gradients in one split and in several."""
    from spear_amd import Phalanx, btp

    torch.manual_seed(11)
    layer = Phalanx(dim=dim, length=L, dtype=torch.bfloat16, kv_heads=kv_heads).to(DEV)
    fused = Phalanx(dim=dim, length=L, method="fused", dtype=torch.bfloat16, kv_heads=kv_heads).to(DEV)
    fused.load_state_dict(layer.state_dict())
    x = torch.randn(B, L, dim, generator=torch.Generator().manual_seed(12)).bfloat16().to(DEV)
    dy = torch.randn(B, L, dim, generator=torch.Generator().manual_seed(13)).bfloat16().to(DEV)

    def run(model):
        model.zero_grad()
        xx = x.clone().requires_grad_(True)
        y = model(xx)
        y.backward(dy)
        return [y.detach(), xx.grad] + [p.grad for p in model.parameters()]

    assert layer._as_one_node(x) is not None
    got = run(layer)
    for i, (a, b) in enumerate(zip(got, run(fused))):  # they differ in roundings to 16 bits on the way
        assert (a.float() - b.float()).norm() <= 2 ** -9 * 10 * b.float().norm(), i
    layer.btp_module = lambda *args: btp(*args)  # a replaced recurrence is called: the stand-alone composition
    assert layer._as_one_node(x) is None
    for i, (a, b) in enumerate(zip(got, run(layer))):
        # each of the about ten roundings between input and gradient is 2^-9 relative; they are independent
        assert (a.float() - b.float()).norm() <= 2 ** -9 * 10 * b.float().norm(), i


def test_calls_that_stay_with_the_stand_alone_kernels():
    from spear_amd import Phalanx

    x = torch.randn(2, 32, 64, device=DEV).bfloat16()
    for kwargs, xx in ((dict(k=1), x), (dict(output_dtype=torch.float32), x), (dict(wpb=3), x), (dict(), x[:, :17]), (dict(), x[:0]),
                       (dict(), x[0])):
        assert Phalanx(dim=64, dtype=torch.bfloat16, **kwargs).to(DEV)._as_one_node(xx) is None
    layer = Phalanx(dim=64, dtype=torch.bfloat16).to(DEV)
    assert layer._as_one_node(x) is not None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert layer._as_one_node(x) is None
    with torch.device(DEV):  # a function mode
        assert layer._as_one_node(x) is None
    with torch.autograd.forward_ad.dual_level():
        assert layer._as_one_node(x) is None
    with torch.no_grad():  # a trace records the ops and not one call's result
        traced, other = torch.jit.trace(layer, x, check_trace=False), x.flip(0, 1)
        assert (traced(other).float() - layer(other).float()).norm() <= 10 * 2 ** -9 * layer(other).float().norm()
    handle = layer.param.proj_c.register_forward_hook(lambda *a: None)
    assert layer._as_one_node(x) is None
    handle.remove()
    with pytest.raises(AssertionError, match="multiple"):
        layer(x[:, :17])


# The last ones: few tokens of many weights, whose gradients are the library's products; past 32768 tokens a narrow layer, whose weight gradients are the
# library's in slices, and one of dim 64, whose input gradients are too; products in 256 x 256 tiles; the front's projections by the library.
@pytest.mark.parametrize("B,L,dim,kv_heads", [(2, 16, 16, 1), (3, 48, 80, None), (8, 128, 96, 2), (64, 128, 256, 4), (1, 48, 4096, None), (264, 128, 128, 2),
                                              (264, 128, 64, None), (256, 128, 512, None), (93, 128, 1024, None)])
def test_layer_node_against_separate_modules(B, L, dim, kv_heads):
    """Every gradient of the one-node layer against the modules' own autograd (a hook keeps them separate), for every subset of
    frozen tensors that changes what backward computes; padding columns of the packed gradients at odd head counts included."""
    from spear_amd import Phalanx

    torch.manual_seed(21)
    layer = Phalanx(dim=dim, length=L, method="fused", dtype=torch.bfloat16, kv_heads=kv_heads).to(DEV)
    x = torch.randn(B, L, dim, generator=torch.Generator().manual_seed(22)).bfloat16().to(DEV)
    dy = torch.randn(B, dim, L, generator=torch.Generator().manual_seed(23)).bfloat16().to(DEV).transpose(1, 2)  # not dense

    def run():
        layer.zero_grad()
        xx = x.clone().requires_grad_(x_grad)
        y = layer(xx)
        y.backward(dy)
        return {"y": y.detach(), "x": xx.grad, **{n: p.grad for n, p in layer.named_parameters()}}

    names = [n for n, _ in layer.named_parameters()]
    for x_grad, trained in ((True, names), (False, names), (True, []), (False, ["proj_out.weight"]), (False, ["param.proj_b.bias"]),
                            (True, ["param.proj_a.weight"])):
        for n, p in layer.named_parameters():
            p.requires_grad_(n in trained)
        got = run()
        handle = layer.param.proj_a.register_forward_hook(lambda *a: None)
        want = run()
        handle.remove()
        for n in want:
            assert (got[n] is None) == (want[n] is None), n
            if want[n] is not None:
                # bf16 roundings of the modules' intermediate gradients, which the node does not make: fewer than ten of 2^-9
                assert (got[n].float() - want[n].float()).norm() <= 10 * 2 ** -9 * want[n].float().norm() + 1e-6, (n, x_grad, trained)


def test_layer_node_is_differentiable_once_and_says_so():
    from spear_amd import Phalanx

    layer = Phalanx(dim=64, dtype=torch.bfloat16).to(DEV)
    x = torch.randn(2, 32, 64, device=DEV).bfloat16().requires_grad_(True)
    plain, = torch.autograd.grad(layer(x).float().sum(), x)
    again, = torch.autograd.grad(layer(x).float().sum(), x, create_graph=True)
    assert torch.equal(plain, again.detach())
    with pytest.raises(RuntimeError, match="differentiated again"):
        again.float().square().sum().backward()


@pytest.mark.parametrize("method", ["default", "fused"])
@pytest.mark.parametrize("B,L,dim", [(2, 16, 16), (8, 128, 512), (4, 32, 1024), (64, 144, 80)])
def test_a_layers_results_can_be_worked_on_in_place(B, L, dim, method):
    """Residual connections, scales and masks written into a layer's output, under autograd and after no_grad, and trainable terms
    added to the input's gradient: with the output projection in a kernel of this library and in the library's product."""
    from spear_amd import Phalanx
    from spear_amd.nn.phalanx.inference import phalanx_prefill

    torch.manual_seed(31)
    layer = Phalanx(dim=dim, length=L, method=method, dtype=torch.bfloat16).to(DEV)
    x = torch.randn(B, L, dim, device=DEV).bfloat16().requires_grad_(True)
    dy = torch.randn(B, L, dim, device=DEV).bfloat16()

    def grads(y):
        return torch.autograd.grad(y, [x, *layer.parameters()], dy)

    y = layer(x)
    y += x
    y *= 2
    want = grads((layer(x) + x) * 2)
    assert all(torch.equal(a, b) for a, b in zip(grads(y), want))
    scale = torch.full((dim,), 2.0, device=DEV, dtype=torch.bfloat16, requires_grad=True)
    with torch.no_grad():
        plain = [layer(x), phalanx_prefill(layer, x)[0]]
    for t in plain + [torch.autograd.grad(layer(x), x, dy)[0]]:
        before = t.clone()
        t *= scale
        assert torch.equal(t, before * 2) and t.requires_grad


@pytest.mark.parametrize("method,owner,name", [
    ("default", "layer", "_mix_and_project"), ("default", "layer", "_project_out"), ("default", "param", "forward_axcv"),
    ("default", "param", "_compute_base_projections"), ("default", "param", "project"), ("fused", "layer", "_project_out"),
    ("fused", "param", "project")])
@pytest.mark.parametrize("where", ["instance", "class"])
def test_a_replaced_method_is_called(method, owner, name, where, monkeypatch):
    from spear_amd import Phalanx

    layer = Phalanx(dim=32, method=method, dtype=torch.bfloat16).to(DEV)
    x = torch.randn(2, 32, 32, device=DEV).bfloat16()
    obj, calls = (layer if owner == "layer" else layer.param), []
    own = getattr(type(obj), name)

    def replacement(*args):
        calls.append(name)
        return own(*(args if where == "class" else (obj, *args)))

    monkeypatch.setattr(type(obj) if where == "class" else obj, name, replacement)
    layer(x)
    assert calls == [name]


@pytest.mark.parametrize("B,L,dim,kv_heads", [(2, 32, 48, 1), (64, 128, 64, 2)])
def test_layer_node_with_saved_tensor_hooks(B, L, dim, kv_heads):
    """Tensors that come back in another layout or off the 16-byte grid give the same gradients; another type, shape or device raises."""
    from spear_amd import Phalanx

    layer = Phalanx(dim=dim, length=L, dtype=torch.bfloat16, kv_heads=kv_heads).to(DEV)
    x = torch.randn(B, L, dim, device=DEV).bfloat16().requires_grad_(True)
    dy = torch.randn(B, L, dim, device=DEV).bfloat16()

    def run(pack, unpack):
        with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
            y = layer(x)
        return torch.autograd.grad(y, [x, *layer.parameters()], dy)

    def shifted(t):
        return torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view(t.shape)

    want = run(lambda t: t, lambda t: t)
    with torch.autograd.graph.save_on_cpu():
        y = layer(x)
    other = [torch.autograd.grad(y, [x, *layer.parameters()], dy),
             run(lambda t: t.transpose(0, -1).contiguous(), lambda t: t.transpose(0, -1)), run(lambda t: t, shifted)]
    for got in other:
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    for unpack in (torch.Tensor.float, torch.Tensor.half, torch.Tensor.cpu, lambda t: t[..., :-1].contiguous(), lambda t: t.flatten()):
        with pytest.raises(RuntimeError, match="came back with another"):
            run(lambda t: t, unpack)


@pytest.mark.parametrize("method,names", [("default", ["proj_out.weight", "param.proj_c.weight", "param.proj_c.bias"]),
                                          ("fused", ["proj_out.weight"])])
@pytest.mark.parametrize("B,L,kv_heads", [(2, 32, 4), (3, 48, 2)])
def test_gradients_without_a_part_of_the_mixing_kernels_can_be_differentiated_again(method, names, B, L, kv_heads):
    """Hessian-vector products of what enters the layer after the recurrence, against the PyTorch statement of the layer in 64 bits."""
    from spear_amd import Phalanx
    from spear_amd.ops.btp import reference

    torch.manual_seed(41)
    layer = Phalanx(dim=64, method=method, dtype=torch.bfloat16, kv_heads=kv_heads).to(DEV)
    x = torch.randn(B, L, 64, device=DEV).bfloat16()
    params = dict(layer.named_parameters())
    vectors = {n: torch.randn_like(params[n]) for n in names}

    def products(forward, ps, cast):
        y = forward()
        gs = torch.autograd.grad((y * y).sum(), [ps[n] for n in names], create_graph=True)
        return torch.autograd.grad(sum((g * cast(vectors[n])).sum() for g, n in zip(gs, names)), list(ps.values()), allow_unused=True)

    ps = {n: p.detach().double().requires_grad_(True) for n, p in params.items()}

    def exact():
        lin = lambda n: torch.nn.functional.linear(x.double(), ps[f"param.proj_{n}.weight"], ps.get(f"param.proj_{n}.bias")).transpose(1, 2)
        heads = lambda t: t.view(B, -1, 16, L).repeat_interleave(4 * 16 // t.shape[1], 1)
        v = heads(lin("v"))
        h = reference.block_two_pass_linspace(torch.sigmoid(lin("a")), torch.sigmoid(heads(lin("b"))) * v, 16)
        return (h * heads(lin("c")) + v).permute(0, 3, 1, 2).reshape(B, L, 64) @ ps["proj_out.weight"].T

    want = products(exact, ps, torch.Tensor.double)
    got = products(lambda: layer(x).float(), params, torch.Tensor.float)
    with pytest.raises(RuntimeError, match="differentiated again"):
        g, = torch.autograd.grad(layer(x).float().square().sum(), params["param.proj_a.weight"], create_graph=True)
        g.float().sum().backward()
    for n, a, b in zip(params, got, want):
        # two layer passes and two backward ones, about ten bf16 roundings each
        assert (a.double() - b).norm() <= 40 * 2 ** -9 * b.norm(), (n, ((a.double() - b).norm() / b.norm()).item())


def _rounding_layer_in_64_bits(a, b, c, v, dout, H, Hkv):
    """The mixing stage with the decay, the input gate, the gated input and the recurrence's upstream gradient rounded to the operands'
    type, everything else in 64 bits: out and the gradients of a, b, c and v."""
    B, L, _ = v.shape
    to_type = lambda t: t.to(a.dtype).double()

    class Gate(torch.autograd.Function):
        @staticmethod
        def forward(ctx, z):
            y = to_type(torch.sigmoid(z))
            ctx.save_for_backward(y)
            return y

        @staticmethod
        def backward(ctx, g):
            y, = ctx.saved_tensors
            return g * y * (1 - y)

    leaves = [t.double().requires_grad_(True) for t in (a, b, c, v)]
    aa, bb, cc, vv = leaves
    expand = lambda t: t.view(B, L, Hkv, 16).repeat_interleave(H // Hkv, 2)
    A, V = Gate.apply(aa), vv.view(B, L, H, 16)
    product = expand(Gate.apply(bb)) * V
    X = product + (to_type(product) - product).detach()
    ys, h, last = [], torch.zeros_like(X[:, 0]), None
    for t in range(L):
        if t % 16 == 0:
            last, h, r = h, torch.zeros_like(h), torch.ones_like(A[:, 0])
        h, r = A[:, t, :, None] * h + X[:, t], r * A[:, t]
        ys.append(h + r[..., None] * last)
    Y = torch.stack(ys, 1)
    Y.register_hook(to_type)
    out = (Y * expand(cc) + V).reshape(B, L, H * 16)
    return [out.detach(), *torch.autograd.grad(out, leaves, dout.double())]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("H,Hkv", [(8, 8), (5, 5), (16, 8), (6, 3), (16, 4), (12, 3), (16, 2), (24, 3), (6, 2), (16, 1)])
def test_mixing_kernels_round_gates_and_products_on_request(H, Hkv, dtype):
    """SPEAR_MIX_ROUND in every instance of the backward kernel (one, two, four, eight and other numbers of heads per kv head) and both
    widths of the forward one, against the same roundings in 64 bits. The fp32 column sums tell the rounded kernel from the plain one."""
    from spear_amd import _btp

    ext = _btp.load_extension()
    for B, L in ((2, 80), (1, 528)):
        g = torch.Generator(device=DEV).manual_seed(H + Hkv + L)
        a, b, c, v, dout = (torch.randn(B, L, w, device=DEV, generator=g).to(dtype) for w in (H, Hkv * 16, Hkv * 16, H * 16, H * 16))
        want = _rounding_layer_in_64_bits(a, b, c, v, dout, H, Hkv)
        worst = {}
        print(f"rounding kernels B={B} L={L} H={H} Hkv={Hkv} {dtype}", flush=True)
        for rounds in (True, False):
            got = [torch.full_like(t, float("nan")) for t in (v, a, b, c, v)]
            sums = [torch.full((_btp.mix_backward_sum_rows(B, L, H), t.shape[2]), float("nan"), device=DEV) for t in (a, b, c)]
            ext.mix_forward(a, b, c, v, got[0], H, Hkv, False, rounds)
            ext.mix_backward(a, b, c, v, dout, *got[1:], H, Hkv, sums, False, rounds)
            far = lambda x, y: ((x.double() - y).norm() / y.norm()).item()
            totals = [t.double().sum(0) for t in sums]
            worst[rounds] = (max(map(far, got, want)), max(map(far, totals, (w.sum((0, 1)) for w in want[1:4]))))
        # results: one rounding, below eps / 2 each; sums: fp32 additions, and here and there a gate whose fp32 value rounds the other
        # way (plain kernels: every gate and product lies up to eps / 2 away)
        assert worst[True][0] <= torch.finfo(dtype).eps / 2, worst
        assert worst[True][1] <= torch.finfo(dtype).eps / 32 and worst[False][1] >= 2 * worst[True][1], worst


@pytest.mark.parametrize("dim,kv_heads", [(64, 2), (64, 1), (128, 1), (256, 2), (192, 4)])
def test_default_layer_gradients_with_shared_kv_heads(dim, kv_heads):
    """Groups of 2, 4, 8, 8 and 3 heads per kv head, the instances that a default layer's backward runs, against its composition."""
    from spear_amd import Phalanx, btp

    torch.manual_seed(13)
    layer = Phalanx(dim=dim, dtype=torch.bfloat16, kv_heads=kv_heads).to(DEV)
    x = torch.randn(4, 80, dim, device=DEV).bfloat16().requires_grad_(True)
    dy = torch.randn(4, 80, dim, device=DEV).bfloat16()
    run = lambda: [y := layer(x), *torch.autograd.grad(y, [x, *layer.parameters()], dy)]
    assert layer._as_one_node(x) is not None
    got = run()
    layer.btp_module = lambda *args: btp(*args)  # the stand-alone composition
    for i, (a, b) in enumerate(zip(got, run())):
        # each of the about ten roundings between input and gradient is 2^-9 relative; they are independent
        assert (a.float() - b.float()).norm() <= 2 ** -9 * 10 * b.float().norm(), i


@pytest.mark.parametrize("method", ["default", "fused"])
@pytest.mark.parametrize("B,L,dim", [(2, 48, 64), (1, 32, 1040), (64, 144, 80)])
def test_layer_node_off_the_16_byte_grid_and_on_another_stream(B, L, dim, method):
    from spear_amd import Phalanx

    torch.manual_seed(51)
    layer = Phalanx(dim=dim, length=L, method=method, dtype=torch.bfloat16).to(DEV)
    x = torch.randn(B, L, dim, device=DEV).bfloat16()
    dy = torch.randn(B, L, dim, device=DEV).bfloat16()

    def run(x, dy):
        xx = x.requires_grad_(True)
        assert layer._as_one_node(xx) is not None
        y = layer(xx)
        return [y.detach(), *torch.autograd.grad(y, [xx, *layer.parameters()], dy)]

    def shifted(t):
        return torch.cat([t.new_zeros(1), t.detach().view(-1)])[1:].view(t.shape)

    want = run(x, dy)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = run(x, dy)
    torch.cuda.current_stream().wait_stream(side)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    for i, (a, b) in enumerate(zip(run(shifted(x), shifted(dy)), want)):  # the library's products for the input projections
        assert (a.float() - b.float()).norm() <= 2 ** -9 * 10 * b.float().norm(), i


@pytest.mark.parametrize("method", ["default", "fused"])
def test_biases_may_change_between_forward_and_backward(method):
    """No gradient depends on a bias' value, so nothing keeps one from being updated before backward, create_graph included."""
    from spear_amd import Phalanx

    torch.manual_seed(61)
    layer = Phalanx(dim=64, method=method, dtype=torch.bfloat16).to(DEV)
    x = torch.randn(2, 32, 64, device=DEV).bfloat16().requires_grad_(True)

    def run(change, create_graph):
        biases = [p.detach().clone() for n, p in layer.named_parameters() if n.endswith("bias")]
        y = layer(x)
        with torch.no_grad():
            for p in (p for n, p in layer.named_parameters() if n.endswith("bias") and change):
                p.mul_(3)
        got = torch.autograd.grad(y, [x, *layer.parameters()], torch.ones_like(y), create_graph=create_graph)
        with torch.no_grad():
            for p, old in zip((p for n, p in layer.named_parameters() if n.endswith("bias")), biases):
                p.copy_(old)
        return got

    for create_graph in (False, True):
        assert all(torch.equal(a, b) for a, b in zip(run(True, create_graph), run(False, create_graph)))


@pytest.mark.parametrize("kv_heads", [4, 2, 1])
@pytest.mark.parametrize("bias", [float("nan"), float("inf"), float("-inf"), -30.0, -80.0, 30.0])
def test_default_layer_gradients_at_the_ends_of_the_decay(bias, kv_heads):
    """A NaN decay logit reaches the gradients that it reaches through the layer's own sigmoid; decays below the recurrences' floor keep
    the gradient of their logit."""
    from spear_amd import Phalanx, btp

    torch.manual_seed(71)
    layer = Phalanx(dim=64, dtype=torch.bfloat16, kv_heads=kv_heads).to(DEV)
    with torch.no_grad():
        layer.param.proj_a.bias[1] = bias
    x = torch.randn(2, 80, 64, device=DEV).bfloat16().requires_grad_(True)
    dy = torch.randn(2, 80, 64, device=DEV).bfloat16()
    run = lambda: [y := layer(x), *torch.autograd.grad(y, [x, *layer.parameters()], dy)]
    assert layer._as_one_node(x) is not None
    got = run()
    layer.btp_module = lambda *args: btp(*args)  # the stand-alone composition
    want = run()
    assert torch.isnan(want[1]).all() if bias != bias else not torch.isnan(want[1]).any()
    for i, (a, b) in enumerate(zip(got, want)):
        assert torch.equal(torch.isnan(a), torch.isnan(b)), i
        a, b = a.double().nan_to_num(), b.double().nan_to_num()
        assert (a - b).norm() <= 2 ** -9 * 10 * b.norm(), i
    a, b = got[3][1].double(), want[3][1].double()  # the bias of that head alone
    assert bias != bias or abs(a - b) <= 0.1 * abs(b), (a, b)
